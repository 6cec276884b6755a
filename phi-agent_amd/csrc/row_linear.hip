// The W8A8 linear of a few rows in one launch: rotate + quantise, int8 GEMM,
// epilogue (linear_gemm's int8 branch, core/models/model_common.cpp:1384-1411;
// the two halves are quant_rotate.hip's register form and the small-problem
// GEMM of i8_gemm_skinny.hip, so every code, scale and output is theirs).
//
// For one row the two launches are most of the time: each costs the host
// about 4 us and the device a start and a drain, around a prologue that works
// on 6 KB.  Here every block rotates and quantises the rows itself, into LDS, a
// group a 16-lane team and under the first loads of its weight rows.  At one
// row, device time of a graph of calls, the weight in cache (new weights each
// call): 3072 -> 3072 5.9 -> 4.7 us (7.9 -> 7.2), 3072 -> 12288 10.8 -> 10.0
// (13.0 -> 12.6), 12288 -> 3072 11.5 -> 9.8 (14.0 -> 12.6); called back to back
// the first 11.1 -> 7.5.  Rows that need a second round of the block's waves run as two
// launches: 5 rows of 3072 took 9.7 us here against 7.9.
#include <atomic>

#include "device_common.hpp"
#include "i8_gemm.hpp"
#include "persist_common.hpp"
#include "qr_tiles.hpp"
#include "skinny_tile.hpp"

namespace phi_dev {

// LDS: the waves' weight stages (2 KB NT a wave; afterwards the partial
// sums), the rotation's tiles and words, the rows' scales, and their codes.
struct RowLds {
    int tiles, red, s, codes, total;
};
template <int NT>
__host__ __device__ constexpr RowLds row_lds(int waves, int M, int K) {
    RowLds l{};
    l.tiles = waves * NT * 2048;
    l.red = l.tiles + waves * QT_WAVE * 4;
    l.s = l.red + 64;
    l.codes = l.s + 64;
    l.total = l.codes + M * K;
    return l;
}

template <bool BF16_IN, bool HALF_EVEN, int NT>
__device__ __forceinline__ void row_linear(const GemmParams& p, const void* __restrict__ x, int64_t ldx,
                                           int8_t* __restrict__ q8, float* __restrict__ s8, int8_t* smem) {
    const int tid = threadIdx.y * blockDim.x + threadIdx.x, lane = tid & 63, g = lane >> 4, tl = lane & 15;
    const int wpr = blockDim.x >> 6, rpb = blockDim.y, NW = wpr * rpb;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ty = __builtin_amdgcn_readfirstlane(threadIdx.y), wr = wave - ty * wpr;
    const int G = p.K >> 8, n0 = persist::xcd_remap(blockIdx.x, gridDim.x) * 16 * NT;
    const RowLds L = row_lds<NT>(NW, p.M, p.K);
    int8_t* stage = persist::opaque_lds(smem + wave * (NT * 2048));
    int8_t* codes = smem + L.codes;
    float* sc = (float*)(smem + L.s);

    // The first rows' inputs, then the wave's first weight rows: the loads of
    // both are in flight together.
    const int g0 = wr * 4 + g, gc = min(g0, G - 1) * 256 + tl * 16;
    const int64_t xoff = (int64_t)min(ty, p.M - 1) * ldx;
    const void* xr = BF16_IN ? (const void*)((const uint16_t*)x + xoff) : (const void*)((const float*)x + xoff);
    const QrPre pre{};
    uint32_t raw[1][1][qt_nw<BF16_IN>];
    qt_load<BF16_IN, QR_PLAIN>(xr, gc, pre, raw[0]);
    Tile16 b[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) b[j] = tile16(p.B, p.ldb, p.kt, min(n0 + 16 * j, p.N - 1), p.N, p.K, lane);
    auto issue = [&](int pair) {
#pragma unroll
        for (int j = 0; j < NT; j++) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(b[j].rsrc, (persist::lptr_t)(stage + j * 2048), 16, b[j].vo0, pair * b[j].step, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(b[j].rsrc, (persist::lptr_t)(stage + j * 2048 + 1024), 16, b[j].vo1, pair * b[j].step, 0, 0);
        }
    };
    const int pairs = p.K >> 7, n = (pairs - wave + NW - 1) / NW;
    if (n > 0) issue(wave);

    float* T = (float*)(smem + L.tiles) + wave * QT_WAVE + g * QT_TILE;
    float* trow = T + tl * 16;
    qt_row<BF16_IN, HALF_EVEN, 1, QR_PLAIN>(raw, xr, ty, p.M, G, codes, p.K, sc, 127.0f, 1.0f / 127.0f, 1, pre, 0,
                                            (uint32_t*)(smem + L.red), T, trow, lane, wr, wpr, wave, g0, tl, tl >> 2);
    __syncthreads();

    // The caller's scratch, written once: row-major, or K-tiled beside a
    // K-tiled weight.
    if (blockIdx.x == 0) {
        for (int i = tid * 16; i < p.M * p.K; i += NW * 64 * 16) {
            const int r = i / p.K, c = i - r * p.K;
            *(uint4*)(q8 + (p.kt ? k_tiled_offset(r, c, p.K, p.M) : i)) = *(const uint4*)(codes + i);
        }
        if (tid < p.M) s8[tid] = sc[tid];
    }

    // Fragments: the weight's from the wave's stage, the rows' from the codes
    // (rows past the last repeat it), both columns 32 g + 16 f.. of the pair.
    const int8_t* arow = codes + min(tl, p.M - 1) * p.K + 32 * g;
    v4i acc[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) acc[j] = v4i{0, 0, 0, 0};
    for (int i = 0; i < n; i++) {
        __builtin_amdgcn_sched_barrier(0);
        persist::wait_vm_lgkm0<0>();
        __builtin_amdgcn_sched_barrier(0);
        v4i w[NT][2];
        const int pair = wave + i * NW;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            w[j][0] = *(const v4i*)(stage + j * 2048 + b[j].f0);
            w[j][1] = *(const v4i*)(stage + j * 2048 + b[j].f1);
        }
        const v4i a0 = *(const v4i*)(arow + pair * 128), a1 = *(const v4i*)(arow + pair * 128 + 16);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0): the fragments are read
        if (i + 1 < n) issue(pair + NW);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NT; j++) {
            acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[j][0], a0, acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[j][1], a1, acc[j], 0, 0, 0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NT; j++) ((v4i*)stage)[j * 64 + lane] = acc[j];
    __syncthreads();
    for (int e = tid; e < NT * 64; e += NW * 64) {
        const int8_t* part = persist::opaque_lds(smem) + e * 16;
        v4i s = *(const v4i*)part;
        for (int w = 1; w < NW; w++) s += *(const v4i*)(part + w * (NT * 2048));
        const int l = e & 63, m = l & 15, nn = n0 + 16 * (e >> 6) + 4 * (l >> 4);
        if (m < p.M && nn < p.N) skinny_store4(p, s, sc[m], m, nn);
    }
}

template <bool BF16_IN, bool HALF_EVEN, int NT>
__global__ __launch_bounds__(1024) void row_linear_kernel(GemmParams p, const void* x, int64_t ldx, int8_t* q8, float* s8) {
    extern __shared__ __align__(16) int8_t smem[];
    row_linear<BF16_IN, HALF_EVEN, NT>(p, x, ldx, q8, s8, smem);
}

// Waves over a row (a 256-group a team), and rows a block.
static int row_wpr(int K) { return (K / 256 + 3) / 4; }
static int row_rpb(int K) { return row_wpr(K) >= 8 ? 1 : 8 / row_wpr(K); }
static int row_waves(int K) { return row_wpr(K) * row_rpb(K); }

template <bool BF16_IN, bool HALF_EVEN, int NT>
static hipError_t launch_nt(hipStream_t stream, const GemmParams& p, const void* x, int64_t ldx, int8_t* q8, float* s8) {
    const size_t lds = (size_t)row_lds<NT>(row_waves(p.K), p.M, p.K).total;
    if (lds > 65536) {  // one attribute call per instantiation and device
        static std::atomic<uint64_t> set{0};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        const uint64_t bit = dev < 64 ? 1ull << dev : 0;
        if (!(set.load(std::memory_order_relaxed) & bit)) {
            e = hipFuncSetAttribute((const void*)row_linear_kernel<BF16_IN, HALF_EVEN, NT>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return e;
            set.fetch_or(bit, std::memory_order_relaxed);
        }
    }
    hipLaunchKernelGGL((row_linear_kernel<BF16_IN, HALF_EVEN, NT>), dim3((unsigned)((p.N + 16 * NT - 1) / (16 * NT))),
                       dim3(64 * row_wpr(p.K), row_rpb(p.K)), lds, stream, p, x, ldx, q8, s8);
    return hipGetLastError();
}

template <bool BF16_IN, bool HALF_EVEN>
static hipError_t launch_rows(hipStream_t stream, const GemmParams& p, const void* x, int64_t ldx, int8_t* q8, float* s8) {
    // One block a CU where columns allow it.
    if (p.N <= 4096) return launch_nt<BF16_IN, HALF_EVEN, 1>(stream, p, x, ldx, q8, s8);
    if (p.N <= 8192) return launch_nt<BF16_IN, HALF_EVEN, 2>(stream, p, x, ldx, q8, s8);
    return launch_nt<BF16_IN, HALF_EVEN, 4>(stream, p, x, ldx, q8, s8);
}

hipError_t launch_row_linear(hipStream_t stream, const GemmParams& p, const void* x, bool bf16_in, int64_t ldx,
                             int half_even, int8_t* q8, float* s8) {
    if (bf16_in) return half_even ? launch_rows<true, true>(stream, p, x, ldx, q8, s8)
                                  : launch_rows<true, false>(stream, p, x, ldx, q8, s8);
    return half_even ? launch_rows<false, true>(stream, p, x, ldx, q8, s8)
                     : launch_rows<false, false>(stream, p, x, ldx, q8, s8);
}

// One round of the block's waves, and one block a CU (up to 16384 columns:
// beyond, a CU would do the rows' work more than once).  All of a block fits
// one CU's LDS.
bool row_linear_ok(const GemmParams& p) {
    if (p.K % 256 != 0 || p.K > 16384 || p.M > row_rpb(p.K) || p.N > 16384 || p.gate || !skinny_ok(p, false)) return false;
    const int waves = row_waves(p.K);
    return (p.N <= 4096 ? row_lds<1>(waves, p.M, p.K) : p.N <= 8192 ? row_lds<2>(waves, p.M, p.K) : row_lds<4>(waves, p.M, p.K)).total <=
           160 * 1024;
}

}  // namespace phi_dev
