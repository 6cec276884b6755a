// The runtime LoRA correction of a linear, out += (x A^T) B^T, as the
// reference runs it (apply_lora_tail, core/models/model_common.cpp:1667-1700):
//
//   lora_down      h[m, r] = sum_k x[m, k] * A[r, k]          (dispatch_gemm_f16 with
//                  fp32 operands and no bias, core/kernels/gemm_f16.cpp:56-200)
//   lora_rank_add  out[m, n] += sum_r h[m, r] * B[n, r]       (dispatch_lora_rank_add,
//                  core/kernels/gemm_f16.cpp:237-308)
//
// Both are fp32 fma chains in a fixed order: the reference accumulates
// acc = fma(a, b, acc) (NVRTC's default --fmad=true) with k ascending from 0
// for h, and with r ascending from out's own value for the rank add.
//
// gfx950's fp32 MFMAs compute exactly such chains: D[i][j] is C[i][j] updated
// by one fma a k-slice, k ascending, each rounded once, denormals kept
// (16x16x4 and 32x32x2 compared with chains of fmaf over random, denormal,
// overflowing, signed-zero and non-finite operands: every bit the same).  So
// the matrix cores give the reference's bits at twice the rate of v_fmac_f32
// and with a fraction of its operand traffic.
//
// An operand fragment holds, in lane group g (16 lanes) of a 4-deep k-slice,
// column k0 + g of the lane's row.  Tiles are staged in LDS row by row at a
// pitch of 4 floats more than a multiple of 32, and read back one float a lane
// (two slices a ds_read2_b32): 16 rows x 4 columns hit 64 distinct banks.
// Reading 16 bytes a lane and exchanging registers between the groups instead
// (v_permlane16_swap / v_permlane32_swap) costs the wave more issue slots
// than it saves: with one or two waves a SIMD the kernels are bound by the
// instructions beside the MFMAs.
//
// Columns past K (or ranks past R) are padded with x = 0, A = -1: the product
// is -0, and fma adds it to any accumulator (-0 included) without a change.
// The reference's own padding of K to 32-deep tiles is with zero products,
// whose only effect is fma(0, 0, -0) = +0, reproduced by one extra fma when
// K % 32 != 0.
#include "device_common.hpp"
#include "lora.hpp"

namespace phi_dev {

// Four consecutive columns c.. of a row of `cols`, as loaded (bf16: in .x and
// .y); columns past the row's end are replaced by others of the row.  VEC: one
// access (cols % 4 == 0, the address aligned to it).  Branch-free: under a
// branch the compiler waits for each load before the next.
template <bool B16, bool VEC>
__device__ __forceinline__ uint4 load4(const char* __restrict__ row, int c, int cols) {
    constexpr int E = B16 ? 2 : 4;
    if (VEC) {
        const char* p = row + (uint64_t)((uint32_t)min(c, cols - 4) * (uint64_t)E);
        if (!B16) return *(const uint4*)p;
        const uint2 u = *(const uint2*)p;
        return make_uint4(u.x, u.y, 0u, 0u);
    }
    uint32_t e[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const char* p = row + (uint64_t)((uint32_t)min(c + i, cols - 1) * (uint64_t)E);
        e[i] = B16 ? *(const uint16_t*)p : *(const uint32_t*)p;
    }
    return B16 ? make_uint4(e[0] | e[1] << 16, e[2] | e[3] << 16, 0u, 0u) : make_uint4(e[0], e[1], e[2], e[3]);
}

// load4's value in fp32, and the same with columns from `cols` on replaced.
template <bool B16>
__device__ __forceinline__ float4 value4(const uint4& v) {
    if (B16)
        return make_float4(bf16_to_f32(v.x & 0xffffu), bf16_to_f32(v.x >> 16), bf16_to_f32(v.y & 0xffffu),
                           bf16_to_f32(v.y >> 16));
    return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
}
template <bool VEC>
__device__ __forceinline__ float4 pad4(const float4& v, int c, int cols, float pad) {
    const bool i0 = c < cols, i1 = VEC ? i0 : c + 1 < cols, i2 = VEC ? i0 : c + 2 < cols, i3 = VEC ? i0 : c + 3 < cols;
    return make_float4(i0 ? v.x : pad, i1 ? v.y : pad, i2 ? v.z : pad, i3 ? v.w : pad);
}

// ---- lora_down: h [M, R] = x [M, K] . A [R, K]^T -------------------------
// A wave owns 16 RT rows x 16 ranks as RT chains of 16x16x4 MFMAs, K / 4
// links each.  A chain is serial by contract, so the smallest output tile of
// a full-rate MFMA gives the shortest one (32 clocks a link of 4 columns,
// 10.2 us at K = 3072).  A block is 4 waves, WR of them over the ranks: 16 RT
// rows x 64 ranks reads x once where R > 32.
//
// With one wave a SIMD nothing hides a wave's own latencies, so they are laid
// under its MFMAs by hand.  Both operands' 64-column chunks go global ->
// registers (LD_AHEAD chunks ahead) -> LDS (three buffers) -> fragments.
// While the MFMAs of chunk c run, pair by pair, the fragments of c + 1 are
// read, c + 2 is written to LDS and c + 2 + LD_AHEAD fetched; one barrier a
// chunk.  The scheduling barriers keep that order: left alone the compiler
// gathers a chunk's MFMAs behind their own fragment reads.  4352 x 3072 x 64:
// 36.3 us, where one row a lane on v_fmac_f32 took 82.6.
constexpr int LD_KC = 64, LD_P = LD_KC + 4, LD_AHEAD = 6;

template <bool XB, bool VEC, int WR, int RT>
__global__ __launch_bounds__(256) void lora_down_kernel(const void* __restrict__ x, int64_t ldx,
                                                        const float* __restrict__ A, float* __restrict__ h, int M,
                                                        int K, int R) {
    constexpr int WM = 4 / WR, XS = RT * WM, BM = 16 * XS, BR = 16 * WR, NS = XS + WR, BUF = (BM + BR) * LD_P / 4;
    __shared__ float4 lds4[3 * BUF];
    const float* lds = (const float*)lds4;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.x * BM, r0 = blockIdx.y * BR;
    const int wm = wave / WR, wr = wave % WR;

    // Slot i of a thread: row tid / 16 + 16 i of the chunk's rows (x's, then
    // A's; rows past the last repeat it), columns 4 (tid % 16)..+3.
    constexpr int XE = XB ? 2 : 4;
    const int srow = tid >> 4, sc = (tid & 15) * 4;
    const char* src[NS];
#pragma unroll
    for (int i = 0; i < NS; i++)
        src[i] = i < XS ? (const char*)x + (int64_t)min(m0 + srow + 16 * i, M - 1) * ldx * XE
                        : (const char*)(A + (int64_t)min(r0 + srow + 16 * (i - XS), R - 1) * K);
    auto fetch = [&](int i, int k0) {
        return i < XS ? load4<XB, VEC>(src[i], k0 + sc, K) : load4<false, VEC>(src[i], k0 + sc, K);
    };
    auto stage = [&](int i, int buf, int k0, const uint4& v) {
        const float4 f = i < XS ? pad4<VEC>(value4<XB>(v), k0 + sc, K, 0.0f) : pad4<VEC>(value4<false>(v), k0 + sc, K, -1.0f);
        lds4[buf + (srow + 16 * i) * (LD_P / 4) + (tid & 15)] = f;
    };
    const int fx = (16 * RT * wm + (lane & 15)) * LD_P + (lane >> 4);
    const int fa = (BM + 16 * wr + (lane & 15)) * LD_P + (lane >> 4);
    auto frag_pair = [&](int buf, int q, float (&vx)[RT][16], float (&va)[16]) {  // links q and q + 1 of a chunk
#pragma unroll
        for (int e = 0; e < 2; e++) {
            va[q + e] = lds[4 * buf + fa + 4 * (q + e)];
#pragma unroll
            for (int t = 0; t < RT; t++) vx[t][q + e] = lds[4 * buf + fx + 16 * t * LD_P + 4 * (q + e)];
        }
    };
    v4f acc[RT];
#pragma unroll
    for (int t = 0; t < RT; t++) acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    const int nch = (K + LD_KC - 1) / LD_KC;
    uint4 ring[LD_AHEAD][NS];
    float vx[2][RT][16], va[2][16];
    uint4 first[2][NS];
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int i = 0; i < NS; i++) first[c][i] = fetch(i, c * LD_KC);
#pragma unroll
    for (int c = 2; c < 2 + LD_AHEAD; c++)
#pragma unroll
        for (int i = 0; i < NS; i++) ring[c % LD_AHEAD][i] = fetch(i, c * LD_KC);
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int i = 0; i < NS; i++) stage(i, c * BUF, c * LD_KC, first[c][i]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; q += 2) frag_pair(0, q, vx[0], va[0]);
    int rd = BUF, wr_at = 2 * BUF;  // LDS offsets (float4) of chunks c + 1 (read) and c + 2 (written)
    // Chunks in pairs: one past K holds only padding, which leaves the
    // accumulators as they are.
    for (int c = 0; c < nch; c += LD_AHEAD) {
#pragma unroll
        for (int u = 0; u < LD_AHEAD; u++) {
            if (u > 0 && u % 2 == 0 && c + u >= nch) break;
            const int cc = c + u;
#pragma unroll
            for (int q = 0; q < 16; q += 2) {
#pragma unroll
                for (int e = 0; e < 2; e++)
#pragma unroll
                    for (int t = 0; t < RT; t++)
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[u & 1][q + e], vx[u & 1][t][q + e], acc[t], 0, 0, 0);
                frag_pair(rd, q, vx[(u + 1) & 1], va[(u + 1) & 1]);
#pragma unroll
                for (int i = q / 2; i < NS; i += 8) {
                    stage(i, wr_at, (cc + 2) * LD_KC, ring[(u + 2) % LD_AHEAD][i]);
                    ring[(u + 2) % LD_AHEAD][i] = fetch(i, (cc + 2 + LD_AHEAD) * LD_KC);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            rd = wr_at;
            wr_at = wr_at == 2 * BUF ? 0 : wr_at + BUF;
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // Lane: row lane % 16 of each of its tiles, ranks 4 (lane / 16)..+3.
    const int r = r0 + 16 * wr + 4 * (lane >> 4);
    const bool pad = (K % 32) != 0;
#pragma unroll
    for (int t = 0; t < RT; t++) {
        const int m = m0 + 16 * (RT * wm + t) + (lane & 15);
        if (m >= M) continue;
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (r + e < R) h[(int64_t)m * R + r + e] = pad ? fmaf(0.0f, 0.0f, acc[t][e]) : acc[t][e];
    }
}

// ---- lora_rank_add: C [M, N] += h [M, R] . B [N, R]^T ---------------------
// C's read and write alone take 60 us at 4352 x 12288 (7.2 TB/s) and the
// MFMAs of 64 ranks 44; the kernel takes 93 (the chains on v_fmac_f32: 116).
// The MFMAs of some waves run under the memory phases of others: so small
// tiles and few registers (four waves a SIMD; with 32 x 128 outputs a wave and
// two waves a SIMD the two phases took turns, 120 us).
// Block: 64 x 128 outputs; wave: 32 rows x 64 columns as 2 x 4 16x16x4 MFMA
// tiles, tile t of a row holding columns 4 j + t (j = lane % 16), so that a
// lane's four tiles are four adjacent columns: every access of C is 16 bytes
// a lane (bf16: 8), a 256-byte piece of a row a lane group.  h and B are staged
// 32 ranks at a time, B's rows in tile order within each 64 (row n at (n % 4)
// 16 + n / 4).
constexpr int RA_BM = 64, RA_BN = 128, RA_RC = 32, RA_P = RA_RC + 4;

// CV: C's rows allow four-column accesses (N % 4 == 0, 16- or 8-byte aligned).
// RV: h's and B's rows allow four-rank accesses (R % 4 == 0, 16-byte aligned).
template <bool CB, bool CV, bool RV>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void lora_rank_add_kernel(
    const float* __restrict__ h, const float* __restrict__ B, void* __restrict__ C, int64_t ldc, int M, int N, int R) {
    __shared__ __align__(16) float sh[RA_BM * RA_P], sb[RA_BN * RA_P];
    constexpr int CE = CB ? 2 : 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Blocks are dealt to the 8 XCDs in turn: give each XCD a contiguous run of
    // blocks, rows first, so that its L2 serves B's panel and h again and again
    // beside C's stream (92.7 us against 102.9 with columns first).
    const int nblk = gridDim.x, xcd = blockIdx.x & 7, idx = blockIdx.x >> 3, tiles_m = (M + RA_BM - 1) / RA_BM;
    const int blk = xcd * (nblk >> 3) + min(xcd, nblk & 7) + idx;
    // Up to 16 ranks C's stream in fp32 is all the time there is: whole rows of C
    // at a time, over all XCDs (32760 x 12288 at rank 16 596 us against 668 rows
    // first, 4352 x 12288 68 either way).
    const bool by_row = !CB && R <= 16;
    const int tiles_n = (N + RA_BN - 1) / RA_BN;
    const int m0 = (by_row ? (int)blockIdx.x / tiles_n : blk % tiles_m) * RA_BM;
    const int n0 = (by_row ? (int)blockIdx.x % tiles_n : blk / tiles_m) * RA_BN;
    const int wm = 32 * (wave >> 1), wn = 64 * (wave & 1);
    const int col = n0 + wn + 4 * (lane & 15), row0 = m0 + wm + 4 * (lane >> 4);
    const int srow = tid >> 3, sc = (tid & 7) * 4;
    const char* src[6];
#pragma unroll
    for (int s = 0; s < 6; s++)
        src[s] = (const char*)(s < 2 ? h + (int64_t)min(m0 + srow + 32 * s, M - 1) * R
                                     : B + (int64_t)min(n0 + srow + 32 * (s - 2), N - 1) * R);
    uint4 v[6];
#pragma unroll
    for (int s = 0; s < 6; s++) v[s] = load4<false, RV>(src[s], sc, R);
    v4f acc[2][4];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int m = min(row0 + 16 * (i >> 2) + (i & 3), M - 1);
        const float4 f = value4<CB>(load4<CB, CV>((const char*)C + (int64_t)m * ldc * CE, col, N));
        acc[i >> 2][0][i & 3] = f.x, acc[i >> 2][1][i & 3] = f.y, acc[i >> 2][2][i & 3] = f.z, acc[i >> 2][3][i & 3] = f.w;
    }
    const int fh = (wm + (lane & 15)) * RA_P + (lane >> 4), fb = (wn + (lane & 15)) * RA_P + (lane >> 4);
    for (int r0 = 0; r0 < R; r0 += RA_RC) {
#pragma unroll
        for (int s = 0; s < 6; s++) {
            const int row = srow + 32 * (s < 2 ? s : s - 2);
            float* d = s < 2 ? &sh[row * RA_P + sc] : &sb[((row & 64) + (row & 3) * 16 + ((row & 63) >> 2)) * RA_P + sc];
            *(float4*)d = pad4<RV>(value4<false>(v[s]), r0 + sc, R, s < 2 ? 0.0f : -1.0f);
        }
        __syncthreads();
        if (r0 + RA_RC < R) {
#pragma unroll
            for (int s = 0; s < 6; s++) v[s] = load4<false, RV>(src[s], r0 + RA_RC + sc, R);
        }
        const int steps = (min(RA_RC, R - r0) + 7) / 8;  // 8 ranks a step
        for (int q = 0; q < steps; q++) {
            float th[2][2], tb[4][2];
#pragma unroll
            for (int e = 0; e < 2; e++) {
#pragma unroll
                for (int u = 0; u < 2; u++) th[u][e] = sh[fh + 16 * u * RA_P + 8 * q + 4 * e];
#pragma unroll
                for (int t = 0; t < 4; t++) tb[t][e] = sb[fb + 16 * t * RA_P + 8 * q + 4 * e];
            }
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int t = 0; t < 4; t++)
                        acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(th[u][e], tb[t][e], acc[u][t], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int m = row0 + 16 * (i >> 2) + (i & 3);
        if (m >= M) continue;
        const float f[4] = {acc[i >> 2][0][i & 3], acc[i >> 2][1][i & 3], acc[i >> 2][2][i & 3], acc[i >> 2][3][i & 3]};
        const int64_t off = (int64_t)m * ldc + col;
        if (CV) {
            if (col >= N) continue;
            if (CB) *(uint2*)((uint16_t*)C + off) = make_uint2(f32x2_to_bf16x2(f[0], f[1]), f32x2_to_bf16x2(f[2], f[3]));
            else *(float4*)((float*)C + off) = make_float4(f[0], f[1], f[2], f[3]);
            continue;
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (col + t >= N) continue;
            if (CB) ((uint16_t*)C)[off + t] = (uint16_t)f32_to_bf16(f[t]);
            else ((float*)C)[off + t] = f[t];
        }
    }
}

// The same chains on v_fmac_f32, one row a lane, for few columns or ranks: the
// kernel above always runs its 16-rank tiles over eight chunks' loads, with a
// block or two a CU; here a block (64 rows, a wave two ranks) needs 36 KB of
// LDS and few registers, and four fit a CU.  Each 64-k chunk of the rows' x and
// of the waves' A slices goes global -> registers -> LDS, double-buffered with
// one barrier a chunk, the next chunk's global loads in flight under the
// current chunk's fmas.  A lane reads its own row of x (68-float pitch: 16-byte
// aligned rows, conflict-free 16-byte reads and writes) and its wave's A
// values, which all the wave's lanes read at one address (a broadcast).
// 100000 x 64 x 4 fp32: 6.3 us, above 16.9; 4352 x 64 x 64 5.7 against 7.1.
constexpr int LR_TR = 2;

// 64 rows x 64 k of x into registers: lane t holds row t / 4, k 16 (t % 4)..+15
// (TAIL: zeros past K, a multiple of 16).
template <bool XB, bool TAIL>
__device__ __forceinline__ void fetch_x_tile(const void* __restrict__ x, int64_t ldx, int m0, int M, int K, int k0,
                                             float (&v)[16]) {
    const int row = threadIdx.x >> 2, kk = (threadIdx.x & 3) * 16;
    if (TAIL && k0 + kk >= K) {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = 0.0f;
        return;
    }
    const int64_t off = (int64_t)min(m0 + row, M - 1) * ldx + k0 + kk;
    if (XB) {
        const uint4 a = *(const uint4*)((const uint16_t*)x + off), b = *(const uint4*)((const uint16_t*)x + off + 8);
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[2 * i] = bf16_to_f32(w[i] & 0xffffu);
            v[2 * i + 1] = bf16_to_f32(w[i] >> 16);
        }
    } else {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float4 t = *(const float4*)((const float*)x + off + 4 * q);
            v[4 * q] = t.x, v[4 * q + 1] = t.y, v[4 * q + 2] = t.z, v[4 * q + 3] = t.w;
        }
    }
}

// x rows 16-byte aligned, K % 64 == 0, or (TAIL) K % 16 == 0: past K x = 0 and
// A = -1, as above.  Without it 100000 x 64 x 64 takes 39 us in bf16, with it 44.
template <bool XB, bool TAIL>
__global__ __launch_bounds__(256) void lora_down_rows_kernel(const void* __restrict__ x, int64_t ldx,
                                                             const float* __restrict__ A, float* __restrict__ h,
                                                             int M, int K, int R) {
    __shared__ __align__(16) float sx[2][64 * LD_P];
    __shared__ __align__(16) float sa[2][4][LR_TR * LD_KC];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m0 = blockIdx.x * 64;
    const int rb = (blockIdx.y * 4 + wave) * LR_TR;
    const bool live = rb < R;  // wave-uniform; a dead wave still stages x for the others
    // The wave's A slice of a chunk (LR_TR ranks x 64 k, rank-major): lane l
    // holds LR_TR consecutive k of rank l / LPR.  Ranks past R read rank R - 1.
    constexpr int LPR = LD_KC / LR_TR;
    const int at = lane / LPR, ak = (lane % LPR) * LR_TR;
    const float* arow = A + (int64_t)min(rb + at, R - 1) * K;
    auto fetch_a = [&](int k0) { return !TAIL || k0 + ak < K ? *(const float2*)(arow + k0 + ak) : make_float2(-1.0f, -1.0f); };
    float acc[LR_TR] = {0.0f, 0.0f};
    float xt[16];
    fetch_x_tile<XB, TAIL>(x, ldx, m0, M, K, 0, xt);
    float2 ta = fetch_a(0);
    const int srow = threadIdx.x >> 2, skk = (threadIdx.x & 3) * 16;
    for (int k0 = 0, buf = 0; k0 < K; k0 += LD_KC, buf ^= 1) {
        float* st = sx[buf] + srow * LD_P + skk;
#pragma unroll
        for (int q = 0; q < 4; q++) *(float4*)(st + 4 * q) = make_float4(xt[4 * q], xt[4 * q + 1], xt[4 * q + 2], xt[4 * q + 3]);
        *(float2*)&sa[buf][wave][at * LD_KC + ak] = ta;
        __syncthreads();
        if (k0 + LD_KC < K) {
            fetch_x_tile<XB, TAIL>(x, ldx, m0, M, K, k0 + LD_KC, xt);
            ta = fetch_a(k0 + LD_KC);
        }
        if (live) {
            const float* xr = sx[buf] + lane * LD_P;
            const float* as = sa[buf][wave];
#pragma unroll
            for (int kk = 0; kk < LD_KC; kk += 8) {
                const float4 x0 = *(const float4*)(xr + kk), x1 = *(const float4*)(xr + kk + 4);
                const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
                float av[LR_TR][8];
#pragma unroll
                for (int t = 0; t < LR_TR; t++) {
                    const float4 a0 = *(const float4*)(as + t * LD_KC + kk), a1 = *(const float4*)(as + t * LD_KC + kk + 4);
                    av[t][0] = a0.x, av[t][1] = a0.y, av[t][2] = a0.z, av[t][3] = a0.w;
                    av[t][4] = a1.x, av[t][5] = a1.y, av[t][6] = a1.z, av[t][7] = a1.w;
                }
#pragma unroll
                for (int i = 0; i < 8; i++)
#pragma unroll
                    for (int t = 0; t < LR_TR; t++) acc[t] = fmaf(xv[i], av[t][i], acc[t]);
            }
        }
        // The buffer written next iteration was last read two iterations ago,
        // before this iteration's barrier: one barrier per chunk suffices.
    }
    const int m = m0 + lane;
    if (!live || m >= M) return;
    const bool pad = TAIL && K % 32 != 0;
#pragma unroll
    for (int t = 0; t < LR_TR; t++)
        if (rb + t < R) h[(int64_t)m * R + rb + t] = pad ? fmaf(0.0f, 0.0f, acc[t]) : acc[t];
}

template <bool XB, bool VEC, int WR, int RT>
static hipError_t launch_down(hipStream_t stream, const void* x, int64_t ldx, const float* A, float* h, int M, int K,
                              int R) {
    constexpr int BM = 16 * RT * (4 / WR), BR = 16 * WR;
    const dim3 grid((unsigned)((M + BM - 1) / BM), (unsigned)((R + BR - 1) / BR));
    hipLaunchKernelGGL((lora_down_kernel<XB, VEC, WR, RT>), grid, dim3(256), 0, stream, x, ldx, A, h, M, K, R);
    return hipGetLastError();
}

// Waves over the ranks: as many 16-rank tiles as R has, up to four, so that no
// wave of a block idles and x is read as few times as possible.  One chain a
// wave while every chain finds a SIMD of its own (4 a CU), two beyond: the
// pair takes as long as two chains on one SIMD would, and A is read half as
// often.  Up to 16 ranks x is what the time goes to, and one chain a wave (two
// blocks a CU and not one) is the faster at any size: 65536 x 3072 x 16 163
// against 176 us, 100000 x 512 x 16 43 against 63.
template <bool XB, bool VEC>
static hipError_t launch_down_r(hipStream_t stream, const void* x, int64_t ldx, const float* A, float* h, int M, int K,
                                int R) {
    const bool one = ((int64_t)M + 15) / 16 * ((R + 15) / 16) <= 1024;
    if (R <= 16) return launch_down<XB, VEC, 1, 1>(stream, x, ldx, A, h, M, K, R);
    if (R <= 32) return one ? launch_down<XB, VEC, 2, 1>(stream, x, ldx, A, h, M, K, R)
                            : launch_down<XB, VEC, 2, 2>(stream, x, ldx, A, h, M, K, R);
    return one ? launch_down<XB, VEC, 4, 1>(stream, x, ldx, A, h, M, K, R)
               : launch_down<XB, VEC, 4, 2>(stream, x, ldx, A, h, M, K, R);
}

template <bool XB>
static hipError_t launch_down_rows(hipStream_t stream, const void* x, int64_t ldx, const float* A, float* h, int M, int K,
                                   int R) {
    const dim3 grid((unsigned)(((int64_t)M + 63) / 64), (unsigned)((R + 4 * LR_TR - 1) / (4 * LR_TR)));
    if (K % LD_KC == 0) hipLaunchKernelGGL((lora_down_rows_kernel<XB, false>), grid, dim3(256), 0, stream, x, ldx, A, h, M, K, R);
    else hipLaunchKernelGGL((lora_down_rows_kernel<XB, true>), grid, dim3(256), 0, stream, x, ldx, A, h, M, K, R);
    return hipGetLastError();
}

hipError_t launch_lora_down(hipStream_t stream, const void* x, bool x_bf16, int64_t ldx, const float* A, float* h,
                            int M, int K, int R) {
    const int esz = x_bf16 ? 2 : 4;
    // One row a lane: few columns, and few ranks of many rows (measured against
    // the tiles over 1350 sizes: 32760 x 1024 x 4 fp32 21.7 against 26.4 us, 4352
    // x 64 x 16 4.0 against 5.1; 4352 x 256 x 64 10.7 against 8.5, 32760 x 2048 x
    // 16 80 against 47).
    if ((K <= 64 || (K <= 192 && (R <= 16 || M <= 1024)) || (R <= 8 && M > 16384 && K <= 1024)) && K % 16 == 0 &&
        (uintptr_t)x % 16 == 0 && (ldx * esz) % 16 == 0 && (uintptr_t)A % 16 == 0)
        return x_bf16 ? launch_down_rows<true>(stream, x, ldx, A, h, M, K, R)
                      : launch_down_rows<false>(stream, x, ldx, A, h, M, K, R);
    const bool vec = K % 4 == 0 && ldx % 4 == 0 && (uintptr_t)x % (4 * esz) == 0 && (uintptr_t)A % 16 == 0;
    if (x_bf16) return vec ? launch_down_r<true, true>(stream, x, ldx, A, h, M, K, R)
                           : launch_down_r<true, false>(stream, x, ldx, A, h, M, K, R);
    return vec ? launch_down_r<false, true>(stream, x, ldx, A, h, M, K, R)
               : launch_down_r<false, false>(stream, x, ldx, A, h, M, K, R);
}

template <bool CB, bool CV>
static hipError_t launch_add(hipStream_t stream, const float* h, const float* B, void* C, int64_t ldc, int M, int N,
                             int R) {
    const int64_t blocks = (int64_t)((N + RA_BN - 1) / RA_BN) * ((M + RA_BM - 1) / RA_BM);
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    const dim3 grid((unsigned)blocks);
    if (R % 4 == 0 && (uintptr_t)h % 16 == 0 && (uintptr_t)B % 16 == 0)
        hipLaunchKernelGGL((lora_rank_add_kernel<CB, CV, true>), grid, dim3(256), 0, stream, h, B, C, ldc, M, N, R);
    else
        hipLaunchKernelGGL((lora_rank_add_kernel<CB, CV, false>), grid, dim3(256), 0, stream, h, B, C, ldc, M, N, R);
    return hipGetLastError();
}

hipError_t launch_lora_rank_add(hipStream_t stream, const float* h, const float* B, void* C, bool c_bf16, int64_t ldc,
                                int M, int N, int R) {
    const bool vec = N % 4 == 0 && ldc % 4 == 0 && (uintptr_t)C % (c_bf16 ? 8 : 16) == 0;
    if (c_bf16) return vec ? launch_add<true, true>(stream, h, B, C, ldc, M, N, R)
                           : launch_add<true, false>(stream, h, B, C, ldc, M, N, R);
    return vec ? launch_add<false, true>(stream, h, B, C, ldc, M, N, R)
               : launch_add<false, false>(stream, h, B, C, ldc, M, N, R);
}

}  // namespace phi_dev
