// Rotate + quantise activations, one row (token) per workgroup, single pass.
//
// Maths (core/host/quant.cpp:109-169, device form core/kernels/int8_gemm.cpp:699-802):
//   per 256-group: y = H x with H = (J - 2R)^{(x)4} / 16, applied as four radix-4
//   passes over the base-4 digits of the in-group index (stride 1, 4, 16, 64);
//   each pass maps (x0,x1,x2,x3) to y[j] = (((x0+x1)+x2)+x3) - 2 x[3-j], then
//   every element is multiplied by 1/16;
//   amax = max |y| over the row; scale = amax > 1e-30 ? amax/qmax : 1;
//   q = clamp(round(y * (1/scale)), +-qmax), ties away from zero by default.
//
// Layout of the work.  A 16-lane team owns one 256-group.  In phase A lane l
// loads elements 16l..16l+15 (coalesced 64-B / 32-B runs), so digits 0 and 1
// of the index are in-lane and the first two passes run in registers.  The
// values go to LDS; in phase B lane l reads back the 16 elements whose low two
// digits equal l (a transpose through LDS), so digits 2 and 3 are in-lane and
// the last two passes also run in registers.  The rotated row stays in LDS
// (the reference reads the row from global memory twice instead), the row
// amax is reduced across the workgroup, and phase C quantises 16 contiguous
// elements per lane and writes them with one 16-byte store.
//
// An element-wise pre-op can run on every input element before the rotation,
// so the tensor between it and the linear never goes through memory: the
// adaLN modulation (QR_MOD), GELU-tanh (QR_GELU) or the SiLU gate over a
// [gate | value] row (QR_SILU_GATE).  They use the same per-element functions
// as the standalone kernels, so fused and unfused agree bit for bit where the
// unfused intermediate is fp32.
//
// LDS: a group's 256 floats sit as 16 slots of 20 floats (16 values + 4 pad,
// so the 16-B slot accesses of 8 lanes land on 8 distinct 4-bank windows), and
// groups are 336 floats apart (a 16-bank shift between the teams of a wave).
#include <cstdlib>

#include "device_common.hpp"
#include "i8_gemm.hpp"
#include "persist_common.hpp"
#include "qr_tiles.hpp"

namespace phi_dev {

constexpr int QR_PITCH = 20;
constexpr int QR_GSTRIDE = 16 * QR_PITCH + 16;

template <bool BF16_IN>
__global__ __launch_bounds__(1024) void quant_rotate_rows(const void* __restrict__ x, int64_t ldx,
                                                          int K, int8_t* __restrict__ q,
                                                          int64_t ldq, float* __restrict__ s,
                                                          float qmax, int half_even, int rotate,
                                                          QrPre pre) {
    extern __shared__ __align__(16) float lds[];
    const int row = blockIdx.x;
    const int tid = threadIdx.x;
    const int nthreads = blockDim.x;
    const int team = tid >> 4, tl = tid & 15, nteams = nthreads >> 4;
    const int G = K >> 8;
    float* red = lds + G * QR_GSTRIDE;

    // ---- phase A: load, passes over digits 0 and 1, stage into LDS ----
    for (int g = team; g < G; g += nteams) {
        float v[16];
        const int64_t e0 = (int64_t)g * 256 + tl * 16;
        load16<BF16_IN>(x, (int64_t)row * ldx + e0, v);
        if (pre.op == QR_MOD) {
            modulate16(v, pre.sc, pre.sh, e0);
        } else if (pre.op == QR_GELU) {
#pragma unroll
            for (int i = 0; i < 16; i++) v[i] = gelu_tanh(v[i]);
        } else if (pre.op == QR_SILU_GATE) {
            float u[16];
            load16<BF16_IN>(x, (int64_t)row * ldx + pre.off2 + e0, u);
#pragma unroll
            for (int i = 0; i < 16; i++) v[i] = silu_mul(v[i], u[i]);
        }
        if (rotate) {
            bfly16<1>(v);
            bfly16<4>(v);
        }
        float4* dst = (float4*)(lds + g * QR_GSTRIDE + tl * QR_PITCH);
#pragma unroll
        for (int i = 0; i < 4; i++) dst[i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
    }
    __syncthreads();

    // ---- phase B: transposed read, passes over digits 2 and 3, x 1/16, amax ----
    float amax = 0.0f;
    for (int g = team; g < G; g += nteams) {
        float* base = lds + g * QR_GSTRIDE + tl;
        float w[16];
#pragma unroll
        for (int j = 0; j < 16; j++) w[j] = base[j * QR_PITCH];
        if (rotate) {
            bfly16<1>(w);
            bfly16<4>(w);
#pragma unroll
            for (int j = 0; j < 16; j++) w[j] = w[j] * (1.0f / 16.0f);
#pragma unroll
            for (int j = 0; j < 16; j++) base[j * QR_PITCH] = w[j];
        }
#pragma unroll
        for (int j = 0; j < 16; j++) amax = fmaxf(amax, fabsf(w[j]));
    }
    amax = wave_max(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    float rmax = red[0];
    for (int w = 1; w < (nthreads >> 6); w++) rmax = fmaxf(rmax, red[w]);
    const float scale = rmax > 1e-30f ? rmax / qmax : 1.0f;
    const float inv = 1.0f / scale;

    // ---- phase C: quantise 16 contiguous elements per lane, 16-B store ----
    for (int g = team; g < G; g += nteams) {
        const float4* src = (const float4*)(lds + g * QR_GSTRIDE + tl * QR_PITCH);
        uint32_t packed[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float4 t = src[i];
            packed[i] = pack4(quant_code(t.x, inv, qmax, half_even), quant_code(t.y, inv, qmax, half_even),
                              quant_code(t.z, inv, qmax, half_even), quant_code(t.w, inv, qmax, half_even));
        }
        uint4* dst = (uint4*)(q + (int64_t)row * ldq + (int64_t)g * 256 + tl * 16);
        *dst = make_uint4(packed[0], packed[1], packed[2], packed[3]);
    }
    if (tid == 0) s[row] = scale;
}

// One block's share of a W4Expand job: item i (idx * threads + thread)
// turns 32 consecutive codes of one weight row into 32 int8, as
// w4_lut_expand_kernel's thread i does.
__device__ __forceinline__ void w4_expand_part(const W4Expand& ex, int idx) {
    const int nt = blockDim.x * blockDim.y;
    const int64_t per_row = ex.K / 32;
    const int64_t i = (int64_t)idx * nt + threadIdx.y * blockDim.x + threadIdx.x;
    if (i >= ex.N * per_row) return;
    const int64_t row = i / per_row, c32 = i - row * per_row;
    using persist::u32x4;
    const u32x4 c = *(const u32x4*)(ex.codes + row * ex.ldb + c32 * 16);
    const u32x4 t = ex.w4_signed ? persist::signed_nibble_table()
                                 : *(const u32x4*)(ex.lut + (row * ex.lut_groups + ((c32 * 32) >> ex.group_shift)) * 16);
    int8_t* o0 = ex.out + (ex.kt ? k_tiled_offset(row, c32 * 32, ex.K, ex.N) : row * ex.K + c32 * 32);
    int8_t* o1 = ex.out + (ex.kt ? k_tiled_offset(row, c32 * 32 + 16, ex.K, ex.N) : row * ex.K + c32 * 32 + 16);
    *(v4i*)o0 = persist::expand16b(c[0], c[1], t);
    *(v4i*)o1 = persist::expand16b(c[2], c[3], t);
}

template <bool BF16_IN, bool HALF_EVEN, int R, int OP>
__global__ __launch_bounds__(1024) void quant_rotate_tiles(const void* __restrict__ x, int64_t ldx, int rows,
                                                           int G, int8_t* __restrict__ q, int64_t ldq,
                                                           float* __restrict__ s, float qmax, float qrcp,
                                                           int rotate, QrPre pre_op, int qkt, int lg_run) {
    extern __shared__ __align__(16) float lds[];
    // The wave's index in its row and its row within the block are the same
    // for all its lanes; read as such, the row's address arithmetic runs on
    // the scalar unit instead of as 64-bit VALU work in every wave.
    const int lane = threadIdx.x & 63, wpr = blockDim.x >> 6;
    const int wr = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int wave = ty * wpr + wr;
    // Blocks are dealt to the 8 XCDs in turn.  Each XCD takes runs of
    // 2^lg_run consecutive blocks' rows, so the rows that share the 128-byte
    // lines of the K-tiled codes (two rows a line) are written through one
    // L2.  The last partial set of runs keeps its order.
    int blk = blockIdx.x;
    unsigned nblk = gridDim.x;
    if (OP == QR_PLAIN && pre_op.ex.blocks) {
        // Beside a W4Expand job: groups of 16 blocks, 8 of the prologue then 8
        // of the expansion (each kind on all 8 XCDs), while both last; then
        // the rest of the longer one.
        const int nq = pre_op.ex.nq, ne = pre_op.ex.blocks, full = min(nq, ne) / 8;
        int kind, idx;
        if (blk < 16 * full) {
            kind = (blk >> 3) & 1;
            idx = 8 * (blk >> 4) + (blk & 7);
        } else {
            const int rest = blk - 16 * full, qrem = nq - 8 * full;
            kind = rest >= qrem;
            idx = 8 * full + (kind ? rest - qrem : rest);
        }
        if (kind) {
            w4_expand_part(pre_op.ex, idx);
            return;
        }
        blk = idx;
        nblk = (unsigned)nq;
    }
    {
        const int span = 8 << lg_run;
        if (blk < (int)(nblk & ~(unsigned)(span - 1))) {
            const int c = blk & (span - 1);
            blk += ((c & 7) << lg_run) + (c >> 3) - c;
        }
    }
    const int team = lane >> 4, tl = lane & 15, sw = tl >> 2;
    const int g0 = wr * 4 * R + team;  // round r works on group g0 + 4 r
    float* T = lds + wave * QT_WAVE + team * QT_TILE;
    float* trow = T + tl * 16;
    uint32_t* red = (uint32_t*)(lds + blockDim.y * wpr * QT_WAVE);

    // Lanes past the row's last group, or in a row past the last, read valid
    // data of another group and discard it.
    const int row = blk * blockDim.y + ty;
    const int64_t roff = (int64_t)min(row, rows - 1) * ldx;
    const void* xr = BF16_IN ? (const void*)((const uint16_t*)x + roff) : (const void*)((const float*)x + roff);
    uint32_t raw[R][qt_ns<OP>][qt_nw<BF16_IN>];
#pragma unroll
    for (int r = 0; r < R; r++) qt_load<BF16_IN, OP>(xr, tl * 16 + min(g0 + 4 * r, G - 1) * 256, pre_op, raw[r]);
    qt_row<BF16_IN, HALF_EVEN, R, OP>(raw, xr, row, rows, G, q, ldq, s, qmax, qrcp, rotate, pre_op, qkt, red, T, trow,
                                      lane, wr, wpr, wave, g0, tl, sw);
}

// Rounds per wave for G groups.  For a large problem R minimises the
// instructions per element: ~14.3 per element plus ~90 per wave and
// round-set spread over the 16 R elements a lane holds, times the share of
// lanes doing live work, with 10 % more for R >= 4 (at most five waves per
// SIMD).  A small one (under 2^17 groups, about two waves of waves on the
// chip) is bound by latency, and the most waves (R = 1) wins.
static int tile_rounds(int64_t rows, int G) {
    const int forced = env_switch("PHI_QR_ROUNDS", 0, 1, QT_MAX_ROUNDS);  // A/B switch: force R where it fits
    if (forced && (G + 4 * forced - 1) / (4 * forced) <= 16) return forced;
    if (rows * G < (1 << 17) && G <= 64) return 1;
    int best = 1;
    double best_cost = 1e30;
    for (int R = 1; R <= QT_MAX_ROUNDS; R++) {
        const int wpr = (G + 4 * R - 1) / (4 * R);
        if (wpr > 16) continue;
        const double cost = (double)(4 * R * wpr) / G * (14.3 + 90.0 / (16 * R)) * (R >= 4 ? 1.1 : 1.0);
        if (cost < best_cost - 1e-9) best = R, best_cost = cost;
    }
    return best;
}

template <bool BF16_IN, bool HALF_EVEN, int R, int OP>
static hipError_t launch_tiles_r(hipStream_t stream, const void* x, int64_t rows, int G, int64_t ldx, int8_t* q,
                                 int64_t ldq, float* s, float qmax, int rotate, const QrPre& pre, int qkt) {
    // Blocks of about four waves: against eight, 9.4 against 10.1 us at
    // 4352 x 3072, 28 against 30.5 at 4352 x 12288 and 92.5 against 97.4 at
    // 32760 x 5120 (one to sixteen waves measured).
    const int wpr = (G + 4 * R - 1) / (4 * R);
    const int rpb = wpr >= 4 ? 1 : 4 / wpr;
    const size_t lds = ((size_t)rpb * wpr * QT_WAVE + 16) * sizeof(float);
    static bool lds_set = false;  // one attribute call per instantiation and process
    if (!lds_set) {
        const hipError_t e = hipFuncSetAttribute((const void*)quant_rotate_tiles<BF16_IN, HALF_EVEN, R, OP>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)((16 * QT_WAVE + 16) * sizeof(float)));
        if (e != hipSuccess) return e;
        lds_set = true;
    }
    dim3 grid((unsigned)((rows + rpb - 1) / rpb)), block((unsigned)(64 * wpr), (unsigned)rpb);
    QrPre p2 = pre;
    if (OP == QR_PLAIN && pre.ex.on) {
        const int64_t items = pre.ex.N * (pre.ex.K / 32), nt = 64 * wpr * rpb;
        p2.ex.nq = (int)grid.x;
        p2.ex.blocks = (int)((items + nt - 1) / nt);
        grid.x += (unsigned)p2.ex.blocks;
    } else {
        p2.ex.blocks = 0;
    }
    // Runs of 8 blocks a XCD: config 1's prologue 11.0 -> 10.4 us, config 1
    // down's 32.3 -> 29.0 us (K-tiled codes; runs of 2 and 4 measured too).
    // A/B switch: log2 of the run length, 0..4 (the kernel shifts by it)
    const int lg_run = env_switch("PHI_QR_RUN", 3, 0, 4);
    hipLaunchKernelGGL((quant_rotate_tiles<BF16_IN, HALF_EVEN, R, OP>), grid, block, lds, stream, x, ldx, (int)rows,
                       G, q, ldq, s, qmax, 1.0f / qmax, rotate, p2, qkt, lg_run);
    return hipGetLastError();
}

// A pre-op keeps R at 1 or 2: the modulation holds per-round scale/shift
// registers and the SiLU gate a second set of loads, and GELU's VALU work
// per element dwarfs the per-wave costs a larger R spreads.
template <bool BF16_IN, bool HALF_EVEN, int OP>
static hipError_t launch_tiles_op(hipStream_t stream, const void* x, int64_t rows, int G, int64_t ldx, int8_t* q,
                                  int64_t ldq, float* s, float qmax, int rotate, const QrPre& pre, int qkt) {
    if (tile_rounds(rows, G) == 1)
        return launch_tiles_r<BF16_IN, HALF_EVEN, 1, OP>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
    return launch_tiles_r<BF16_IN, HALF_EVEN, 2, OP>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
}

template <bool BF16_IN, bool HALF_EVEN>
static hipError_t launch_tiles(hipStream_t stream, const void* x, int64_t rows, int G, int64_t ldx, int8_t* q,
                               int64_t ldq, float* s, float qmax, int rotate, const QrPre& pre, int qkt) {
    switch (pre.op) {
        case QR_MOD: return launch_tiles_op<BF16_IN, HALF_EVEN, QR_MOD>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
        case QR_GELU: return launch_tiles_op<BF16_IN, HALF_EVEN, QR_GELU>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
        case QR_SILU_GATE:
            return launch_tiles_op<BF16_IN, HALF_EVEN, QR_SILU_GATE>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
        default: break;
    }
    switch (tile_rounds(rows, G)) {
        case 1: return launch_tiles_r<BF16_IN, HALF_EVEN, 1, QR_PLAIN>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
        case 2: return launch_tiles_r<BF16_IN, HALF_EVEN, 2, QR_PLAIN>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
        case 3: return launch_tiles_r<BF16_IN, HALF_EVEN, 3, QR_PLAIN>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
        case 4: return launch_tiles_r<BF16_IN, HALF_EVEN, 4, QR_PLAIN>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
        default: return launch_tiles_r<BF16_IN, HALF_EVEN, 5, QR_PLAIN>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
    }
}

// Host-side launcher.  Validation is done by the C ABI layer.
hipError_t launch_quant_rotate(hipStream_t stream, const void* x, bool bf16_in, int64_t rows,
                               int64_t K, int64_t ldx, int8_t* q, int64_t ldq, float* s,
                               float qmax, int half_even, int rotate, const QrPre& pre, int qkt) {
    const int G = (int)(K / 256);
    if (rows == 0) return hipSuccess;
    if (qkt && G > 64) return hipErrorInvalidValue;  // the row kernel writes row-major q only
    // A W4Expand job rides only on the plain tiles kernel.
    if (pre.ex.on && (G > 64 || pre.op != QR_PLAIN)) return hipErrorInvalidValue;
    if (G <= 64) {
        if (bf16_in)
            return half_even ? launch_tiles<true, true>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt)
                             : launch_tiles<true, false>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
        return half_even ? launch_tiles<false, true>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt)
                         : launch_tiles<false, false>(stream, x, rows, G, ldx, q, ldq, s, qmax, rotate, pre, qkt);
    }
    int threads = ((16 * G + 63) / 64) * 64;
    if (threads > 1024) threads = 1024;
    const size_t lds_bytes = ((size_t)G * QR_GSTRIDE + 16) * sizeof(float);
    if (lds_bytes > 65536) {
        hipError_t e = hipFuncSetAttribute(bf16_in ? (const void*)quant_rotate_rows<true> : (const void*)quant_rotate_rows<false>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        if (e != hipSuccess) return e;
    }
    if (bf16_in) {
        hipLaunchKernelGGL(quant_rotate_rows<true>, dim3((unsigned)rows), dim3(threads), lds_bytes,
                           stream, x, ldx, (int)K, q, ldq, s, qmax, half_even, rotate, pre);
    } else {
        hipLaunchKernelGGL(quant_rotate_rows<false>, dim3((unsigned)rows), dim3(threads), lds_bytes,
                           stream, x, ldx, (int)K, q, ldq, s, qmax, half_even, rotate, pre);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The rotation alone, fp32 in and out (phi_hip_convrot_rows): a wave takes
// four consecutive 256-groups of a row, one 16-lane team each, as the register
// form above does, with its tiles and the reference's butterflies (multiply
// and subtract).  y may be x: a team has read its group before it writes it.
// 302 MB of traffic at 12288 x 3072: 58 us; one element a thread with eight
// barriers took 108.
__global__ __launch_bounds__(256) void convrot_teams_kernel(const float* x, int64_t ldx, float* y, int64_t ldy,
                                                            int64_t groups, int gpr) {
    __shared__ __align__(16) float lds[4 * QT_WAVE];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, team = lane >> 4, tl = lane & 15, sw = tl >> 2;
    const int64_t at = ((int64_t)blockIdx.x * 4 + wave) * 4 + team, g = at < groups ? at : groups - 1;
    const int64_t row = g / gpr, col = (g - row * gpr) * 256 + tl * 16;
    float* T = lds + wave * QT_WAVE + team * QT_TILE;
    float* trow = T + tl * 16;
    float v[16], w[16];
    load16<false>(x, row * ldx + col, v);
    bfly16<1>(v);
    bfly16<4>(v);
#pragma unroll
    for (int c = 0; c < 4; c++)
        *(float4*)(trow + 4 * (c ^ sw)) = make_float4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
    wave_lds_fence();
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const float* cp = T + 64 * k + 4 * (sw ^ k) + (tl & 3);
#pragma unroll
        for (int i = 0; i < 4; i++) w[4 * k + i] = cp[16 * i];
    }
    wave_lds_fence();
    bfly16<1>(w);
    bfly16<4>(w);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        float* cp = T + 64 * k + 4 * (sw ^ k) + (tl & 3);
#pragma unroll
        for (int i = 0; i < 4; i++) cp[16 * i] = w[4 * k + i] * (1.0f / 16.0f);
    }
    wave_lds_fence();
    if (at >= groups) return;
    float4* dst = (float4*)(y + row * ldy + col);
#pragma unroll
    for (int k = 0; k < 4; k++) dst[k] = *(const float4*)(trow + 4 * (k ^ sw));
}

hipError_t launch_convrot_teams(hipStream_t stream, const float* x, int64_t ldx, float* y, int64_t ldy, int64_t rows,
                                int64_t K) {
    const int64_t groups = rows * (K / 256);
    hipLaunchKernelGGL(convrot_teams_kernel, dim3((unsigned)((groups + 15) / 16)), dim3(256), 0, stream, x, ldx, y, ldy,
                       groups, (int)(K / 256));
    return hipGetLastError();
}

size_t quant_rotate_lds_bytes(int64_t K) { return ((size_t)(K / 256) * QR_GSTRIDE + 16) * sizeof(float); }

}  // namespace phi_dev
