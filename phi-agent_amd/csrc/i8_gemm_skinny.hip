// int8 x int8 -> int32 GEMM for problems too small to fill the chip with
// 128 x 128 tiles: few rows, few columns, or both (a prompt's or a small
// image's tokens, a single row, the projection onto a few channels).  Same
// product and epilogue as the persistent kernels (core/kernels/int8_gemm.cpp:
// 466-621, epilogue :588-620; host gemm_int8 core/host/quant.cpp:223-236):
//   C[m,n] = fma((float)acc[m,n] * sA[m], sB[n], bias[n]), or with a gate
//   C[m,n] = fma(that, gate[n], C[m,n]) on fp32 C.
//
// What bounds such a problem is one pass over the weight, and latency: at one
// row the weight's bytes are all the traffic there is.  A 128 x 128 tile walks
// K alone on one CU (3072 -> 3072 has 24 of them, 11.9 us at one row on 24 of
// 256 CUs).  Here a block owns a small tile, (16 MT) x (16 NT) outputs, and
// its NW waves split K: wave w takes the 128-column pairs w, w + NW, ... The
// int32 partial sums are exact in any order and meet in LDS.  That needs no
// workspace and no second launch, and the tile can be as small as the shape
// wants: 192 blocks of 8 waves for the example.
//
// A wave streams its operands through LDS of its own (no barriers): the
// 16-byte chunks of a 128-column pair by direct-to-LDS loads, whole 128-byte
// lines of 8 rows (row-major) or 1 KB of a K-tiled block an instruction, then
// 16-byte fragment reads.  Loading the fragments straight into registers puts
// 16 different rows into each 16-lane quarter of a load, 64 line accesses an
// instruction, and ran at 16 bytes a clock and CU (31 K-tiled).  In a pair
// lane group g (16 lanes) multiplies columns 32 g .. +31 as two fragments
// (the sum over k may take them in any order, if A and B agree): packed 4-bit
// weights are the same 32 columns in one 16-byte read, expanded in registers.
#include <atomic>
#include <cmath>

#include "device_common.hpp"
#include "i8_gemm.hpp"
#include "persist_common.hpp"
#include "skinny_tile.hpp"

namespace phi_dev {

using persist::u32x4;

enum SkinnyB { SB_I8 = 0, SB_LUT = 1, SB_S4 = 2 };

// 32 signed nibbles (16 bytes, column order) as two fragments of int8 values
// times 16: a nibble in the high half of a byte is its signed value times 16.
// The sums come out times 16 exactly and are shifted back (K <= 65536 keeps
// them in 32 bits).
__device__ __forceinline__ void expand_s4(const u32x4& c, v4i& f0, v4i& f1) {
    uint32_t o[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t even = (c[i] << 4) & 0xf0f0f0f0u, odd = c[i] & 0xf0f0f0f0u;
        o[2 * i] = __builtin_amdgcn_perm(odd, even, 0x05010400u);
        o[2 * i + 1] = __builtin_amdgcn_perm(odd, even, 0x07030602u);
    }
    f0 = v4i{(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
    f1 = v4i{(int)o[4], (int)o[5], (int)o[6], (int)o[7]};
}

// Bytes of a wave's stage (one pair of its tile's rows), and its loads.
template <int MT, int NT, int SB>
constexpr int skinny_stage = MT * 2048 + NT * (SB == SB_I8 ? 2048 : SB == SB_S4 ? 1024 : 1536);
template <int MT, int NT, int SB>
constexpr int skinny_loads = 2 * MT + (SB == SB_S4 ? 1 : 2) * NT;

// A wave's LDS: its stages, and after the last pair its partial sums.
template <int MT, int NT, int S, int SB>
constexpr int skinny_region = S * skinny_stage<MT, NT, SB> > MT * NT * 1024 ? S * skinny_stage<MT, NT, SB> : MT * NT * 1024;

template <int MT, int NT, int NW, int S, int SB>
__device__ __forceinline__ void skinny_tile(const GemmParams& p, int8_t* smem) {
    constexpr int BM = 16 * MT, BN = 16 * NT, T = MT * NT, STG = skinny_stage<MT, NT, SB>, D = skinny_loads<MT, NT, SB>;
    constexpr int REG = skinny_region<MT, NT, S, SB>;
    static_assert((S - 1) * D < 64, "vmcnt is six bits");
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Each XCD takes a contiguous run of blocks, rows first: the blocks that
    // read one panel of the weight run together on one L2.
    const int tiles_m = (p.M + BM - 1) / BM;
    const int blk = persist::xcd_remap(blockIdx.x, gridDim.x);
    const int m0 = blk % tiles_m * BM, n0 = blk / tiles_m * BN;
    int8_t* ring = persist::opaque_lds(smem + wave * REG);

    Tile16 a[MT], b[NT];
    int tv[NT];  // SB_LUT: the lane's byte offset into the tables, group 0
    const __amdgpu_buffer_rsrc_t rl = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(SB == SB_LUT ? p.lut + (int64_t)n0 * p.lut_groups * 16 : p.A), (short)0, 0x7fffffff, persist::kRsrcWord3);
#pragma unroll
    for (int i = 0; i < MT; i++) a[i] = tile16(p.A, p.lda, p.kt, min(m0 + 16 * i, p.M - 1), p.M, p.K, lane);
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int r0 = min(n0 + 16 * j, p.N - 1), last = p.N - 1 - r0;
        if (SB == SB_I8) {
            b[j] = tile16(p.B, p.ldb, p.kt && !p.b_rm, r0, p.N, p.K, lane);
        } else {
            // 16 rows x 64 bytes of codes a load; chunk c of row r in slot c ^ ((r >> 2) & 3).
            b[j].rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(p.B + (int64_t)r0 * p.ldb), (short)0, 0x7fffffff,
                                                          persist::kRsrcWord3);
            const int row = lane >> 2, r = lane & 15;
            b[j].vo0 = min(row, last) * (int)p.ldb + (((lane & 3) ^ ((row >> 2) & 3)) << 4);
            b[j].f0 = r * 64 + ((g ^ ((r >> 2) & 3)) << 4);
            tv[j] = (r0 - n0 + min(r, last)) * (int)p.lut_groups * 16;
        }
    }
    // The tables of a pair: lane l < 32 loads the one of row l % 16 for columns
    // 64 (l / 16).. of the pair (with groups of 128 and up, the same twice).
    auto issue = [&](int st, int pair) {
        int8_t* d = ring + st * STG;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            if (SB == SB_I8) {
                __builtin_amdgcn_raw_ptr_buffer_load_lds(b[j].rsrc, (persist::lptr_t)(d + j * 2048), 16, b[j].vo0, pair * b[j].step, 0, 0);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(b[j].rsrc, (persist::lptr_t)(d + j * 2048 + 1024), 16, b[j].vo1, pair * b[j].step, 0, 0);
            } else {
                __builtin_amdgcn_raw_ptr_buffer_load_lds(b[j].rsrc, (persist::lptr_t)(d + j * 1024), 16, b[j].vo0, pair * 64, 0, 0);
            }
        }
        int8_t* da = d + STG - MT * 2048;
#pragma unroll
        for (int i = 0; i < MT; i++) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(a[i].rsrc, (persist::lptr_t)(da + i * 2048), 16, a[i].vo0, pair * a[i].step, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(a[i].rsrc, (persist::lptr_t)(da + i * 2048 + 1024), 16, a[i].vo1, pair * a[i].step, 0, 0);
        }
        if (SB == SB_LUT && lane < 32) {
            const int gi = (pair * 128 + (lane >> 4) * 64) >> p.group_shift;
#pragma unroll
            for (int j = 0; j < NT; j++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rl, (persist::lptr_t)(d + NT * 1024 + j * 512), 16, tv[j] + gi * 16, 0, 0, 0);
        }
    };

    v4i acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = v4i{0, 0, 0, 0};
    v4i fa[MT][2], fb[NT][2];
    auto read = [&](int st) {
        const int8_t* d = ring + st * STG;
        const int8_t* da = d + STG - MT * 2048;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            if (SB == SB_I8) {
                fb[j][0] = *(const v4i*)(d + j * 2048 + b[j].f0);
                fb[j][1] = *(const v4i*)(d + j * 2048 + b[j].f1);
            } else {
                fb[j][0] = *(const v4i*)(d + j * 1024 + b[j].f0);
                if (SB == SB_LUT) fb[j][1] = *(const v4i*)(d + NT * 1024 + j * 512 + ((g >> 1) * 16 + (lane & 15)) * 16);
            }
        }
#pragma unroll
        for (int i = 0; i < MT; i++) {
            fa[i][0] = *(const v4i*)(da + i * 2048 + a[i].f0);
            fa[i][1] = *(const v4i*)(da + i * 2048 + a[i].f1);
        }
    };
    auto multiply = [&] {
#pragma unroll
        for (int j = 0; j < NT; j++) {
            v4i w0 = fb[j][0], w1 = fb[j][1];
            if (SB != SB_I8) {
                const u32x4 c = __builtin_bit_cast(u32x4, fb[j][0]), t = __builtin_bit_cast(u32x4, fb[j][1]);
                if (SB == SB_S4) {
                    expand_s4(c, w0, w1);
                } else {
                    w0 = persist::expand16b(c[0], c[1], t);
                    w1 = persist::expand16b(c[2], c[3], t);
                }
            }
#pragma unroll
            for (int i = 0; i < MT; i++) {
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, fa[i][0], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, fa[i][1], acc[i][j], 0, 0, 0);
            }
        }
    };

    // Pairs wave, wave + NW, ...: S of them in flight.  A pair's stage is
    // refilled as soon as its fragments are in registers.
    const int pairs = p.K >> 7, n = (pairs - wave + NW - 1) / NW;
    for (int i = 0; i < S && i < n; i++) issue(i, wave + i * NW);
    for (int i = 0, st = 0; i < n; i++) {
        // Loads complete in order: stage i has landed when only the younger
        // stages' loads are left.
        const int young = min(S - 1, n - 1 - i);
        __builtin_amdgcn_sched_barrier(0);
        if (S > 3 && young >= 3) persist::wait_vm_lgkm0<(S > 3 ? 3 * D : 0)>();
        else if (S > 2 && young == 2) persist::wait_vm_lgkm0<(S > 2 ? 2 * D : 0)>();
        else if (S > 1 && young == 1) persist::wait_vm_lgkm0<(S > 1 ? D : 0)>();
        else persist::wait_vm_lgkm0<0>();
        __builtin_amdgcn_sched_barrier(0);
        read(st);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0): the fragments are read
        if (i + S < n) issue(st, wave + (i + S) * NW);
        __builtin_amdgcn_sched_barrier(0);
        multiply();
        st = st + 1 == S ? 0 : st + 1;
    }

    // The wave's partial sums into its own stages (its loads and reads are
    // over), then the block's sum.
    __builtin_amdgcn_sched_barrier(0);
    v4i* mine = (v4i*)ring;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) mine[(i * NT + j) * 64 + lane] = acc[i][j];
    __syncthreads();

    // Lane l of tile (i, j): row 16 i + l % 16, columns 16 j + 4 (l / 16)..+3.
    for (int e = tid; e < T * 64; e += NW * 64) {
        const int8_t* part = persist::opaque_lds(smem) + e * 16;
        v4i s = *(const v4i*)part;
#pragma unroll
        for (int w = 1; w < NW; w++) s += *(const v4i*)(part + w * REG);
        if (SB == SB_S4) s >>= 4;
        const int tile = e >> 6, l = e & 63;
        const int m = m0 + 16 * (tile / NT) + (l & 15), nn = n0 + 16 * (tile % NT) + 4 * (l >> 4);
        if (m >= p.M || nn >= p.N) continue;
        skinny_store4(p, s, p.sA ? p.sA[m] : 0.0f, m, nn);
    }
}

// The tiles the kernel is built for: wave tile, waves a block, stages a wave.
// More waves beat more stages a wave (4 x 4 tiles over K = 12288 at 256 rows:
// 26.3 us with 8 waves of one stage, 27.0 with 4 of two).  Then, as fitted (see
// skinny_us), in us by what B is (SkinnyB): the tile's part of the fixed time,
// and what a round of blocks takes for a 128-column pair and apart from its
// pairs.
struct SkinnyCfg {
    int mt, nt, nw, s;
    double fixed[3], pair[3], block[3];
};
constexpr SkinnyCfg kSkinny[] = {
    {1, 1, 8, 2, {0.59, 0.13, 0.73}, {0.0345, 0.0476, 0.0254}, {0.45, 0.45, 0.29}},
    {1, 2, 8, 1, {0.99, 0.52, 1.00}, {0.0533, 0.0895, 0.0411}, {0.10, 0.07, 0.13}},
    {1, 4, 8, 1, {1.16, 0.61, 1.20}, {0.0917, 0.1810, 0.0681}, {0.16, 0.09, 0.11}},
    {2, 1, 8, 1, {0.97, 0.57, 0.99}, {0.0492, 0.0521, 0.0386}, {0.15, 0.21, 0.18}},
    {2, 2, 8, 1, {0.98, 0.61, 1.08}, {0.0699, 0.0914, 0.0506}, {0.25, 0.26, 0.21}},
    {2, 4, 8, 1, {0.13, 1.11, 1.25}, {0.1170, 0.1797, 0.0874}, {1.47, 0.00, 0.28}},
    {4, 1, 8, 1, {1.05, 0.75, 0.91}, {0.0821, 0.0851, 0.0727}, {0.32, 0.30, 0.50}},
    {4, 2, 8, 1, {0.15, 0.09, 1.21}, {0.1073, 0.1370, 0.0870}, {1.48, 1.17, 0.44}},
    {4, 4, 8, 1, {0.00, 0.42, 0.15}, {0.1666, 0.2422, 0.1438}, {2.11, 1.31, 2.00}},
    {5, 2, 8, 1, {0.14, 0.16, 0.00}, {0.1277, 0.1617, 0.1151}, {1.77, 1.43, 1.97}},
    {5, 4, 8, 1, {0.19, 0.71, 0.28}, {0.1880, 0.2646, 0.1744}, {2.23, 1.37, 2.28}},
    {6, 4, 4, 2, {0.24, 0.44, 0.53}, {0.2088, 0.3776, 0.2304}, {3.23, 2.23, 3.21}},
    {3, 8, 4, 1, {0.42, 0.31, 0.52}, {0.2332, 0.4556, 0.2131}, {3.49, 2.48, 3.22}},
    {5, 8, 4, 1, {0.52, 1.86, 0.80}, {0.2641, 0.5525, 0.3079}, {5.67, 2.98, 5.17}},
};
constexpr int kSkinnyCfgs = (int)(sizeof kSkinny / sizeof kSkinny[0]);

int skinny_configs() { return kSkinnyCfgs; }

// Time of p on tile cfg in us: a fixed part, the rounds of blocks and the
// operands' pass from memory (the weight once; A once a column panel, rows
// first, unless the L2s hold it) as the two sides of a right triangle, for they
// overlap and disturb each other, the weight's share of a first pass, and the
// stores.  Fitted over 2400 random shapes x 14 tiles (1 to 16384 rows, 8 to
// 40000 columns, K 512 to 16384, both layouts, every output), the weight in
// cache and not, to their geometric mean, rms error 7 % (signed nibbles 6 %);
// codes through tables over 970 shapes with the weight in cache, 10 %.  On 630
// other int8 and nibble shapes the error is 7 %, and the tile it picks within
// 0.8 % of the best on average, within 5 % on 95 of 100.
static double skinny_us(const GemmParams& p, bool w4, int num_cus, int cfg) {
    const SkinnyCfg c = kSkinny[cfg];
    const int b = !w4 ? SB_I8 : p.w4_signed ? SB_S4 : SB_LUT;
    const double tiles_m = (p.M + 16 * c.mt - 1) / (16 * c.mt), tiles_n = (p.N + 16 * c.nt - 1) / (16 * c.nt);
    const double rounds = ceil(tiles_m * tiles_n / num_cus), pairs = p.K / 128.0, out = 1e-6 * p.M * p.N;
    const double weight = 1e-6 * p.N * p.K * (w4 ? 0.5 : 1.0), a = 1e-6 * p.M * p.K;
    // By what B is: fixed, a MB from memory, a MB of the weight, a million
    // outputs, and a 16 x 16 tile of a block's.
    constexpr double kUs[3][5] = {{1.53, 0.083, 0.046, 1.8, 0.013}, {2.08, 0.159, 0.0, 2.3, 0.0}, {1.49, 0.083, 0.056, 1.4, 0.010}};
    double fixed = kUs[b][0], store = kUs[b][3], tile = kUs[b][4];
    const bool wide = p.c_kind != C_BF16;
    if (p.gate) fixed += 0.65, store = 5.7, tile = 0.016;
    else if (!w4 && wide) store = 2.5, tile = 0.021;
    if (!wide && !(p.c_vec && p.N % 4 == 0)) store = 4.5;
    const double blocks = rounds * (pairs * c.pair[b] + c.block[b] + tile * c.mt * c.nt);
    const double memory = kUs[b][1] * (weight + a * (a > 4.0 ? tiles_n : fmin(tiles_n, 8.0)));
    return c.fixed[b] + fixed + hypot(blocks, memory) + kUs[b][2] * weight + store * out;
}

int skinny_best(const GemmParams& p, bool w4, int num_cus, double* us) {
    int best = 0;
    double t = 1e300;
    for (int i = 0; i < kSkinnyCfgs; i++) {
        const double ti = skinny_us(p, w4, num_cus, i);
        if (ti < t) t = ti, best = i;
    }
    *us = t;
    return best;
}

template <int MT, int NT, int NW, int S, int SB>
__global__ __launch_bounds__(NW * 64) void i8_gemm_skinny_kernel(GemmParams p) {
    extern __shared__ __align__(16) int8_t smem[];
    skinny_tile<MT, NT, NW, S, SB>(p, smem);
}

template <int MT, int NT, int NW, int S, int SB>
static hipError_t launch_one(hipStream_t stream, const GemmParams& p) {
    const int64_t blocks = (int64_t)((p.M + 16 * MT - 1) / (16 * MT)) * ((p.N + 16 * NT - 1) / (16 * NT));
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    constexpr int lds = NW * skinny_region<MT, NT, S, SB>;
    if (lds > 65536) {  // one attribute call per instantiation and device
        static std::atomic<uint64_t> set{0};
        int dev = 0;
        const hipError_t d = hipGetDevice(&dev);
        if (d != hipSuccess) return d;
        const uint64_t bit = dev < 64 ? 1ull << dev : 0;
        if (!(set.load(std::memory_order_relaxed) & bit)) {
            const hipError_t e = hipFuncSetAttribute((const void*)i8_gemm_skinny_kernel<MT, NT, NW, S, SB>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e != hipSuccess) return e;
            set.fetch_or(bit, std::memory_order_relaxed);
        }
    }
    hipLaunchKernelGGL((i8_gemm_skinny_kernel<MT, NT, NW, S, SB>), dim3((unsigned)blocks), dim3(NW * 64), lds, stream, p);
    return hipGetLastError();
}

template <int MT, int NT, int NW, int S>
static hipError_t launch_cfg(hipStream_t stream, const GemmParams& p, int sb) {
    // A second stage where the partial sums' region holds one anyway.
    constexpr int SL = S == 1 && 2 * skinny_stage<MT, NT, SB_LUT> <= MT * NT * 1024 ? 2 : S;
    constexpr int S4 = S == 1 && 2 * skinny_stage<MT, NT, SB_S4> <= MT * NT * 1024 ? 2 : S;
    switch (sb) {
        case SB_I8: return launch_one<MT, NT, NW, S, SB_I8>(stream, p);
        case SB_LUT: return launch_one<MT, NT, NW, SL, SB_LUT>(stream, p);
        default: return launch_one<MT, NT, NW, S4, SB_S4>(stream, p);
    }
}

template <int I>
static hipError_t launch_at(hipStream_t stream, const GemmParams& p, int sb) {
    return launch_cfg<kSkinny[I].mt, kSkinny[I].nt, kSkinny[I].nw, kSkinny[I].s>(stream, p, sb);
}

hipError_t launch_i8_gemm_skinny(hipStream_t stream, const GemmParams& p, bool w4, int cfg) {
    const int sb = !w4 ? SB_I8 : p.w4_signed ? SB_S4 : SB_LUT;
    switch (cfg) {
        case 0: return launch_at<0>(stream, p, sb);
        case 1: return launch_at<1>(stream, p, sb);
        case 2: return launch_at<2>(stream, p, sb);
        case 3: return launch_at<3>(stream, p, sb);
        case 4: return launch_at<4>(stream, p, sb);
        case 5: return launch_at<5>(stream, p, sb);
        case 6: return launch_at<6>(stream, p, sb);
        case 7: return launch_at<7>(stream, p, sb);
        case 8: return launch_at<8>(stream, p, sb);
        case 9: return launch_at<9>(stream, p, sb);
        case 10: return launch_at<10>(stream, p, sb);
        case 11: return launch_at<11>(stream, p, sb);
        case 12: return launch_at<12>(stream, p, sb);
        default: return launch_at<13>(stream, p, sb);
    }
}

// Whether the kernel takes p: whole 128-column pairs and 16-byte operand
// chunks; signed nibbles times 16 within 32 bits.
bool skinny_ok(const GemmParams& p, bool w4) {
    auto al = [](const void* q, int64_t ld) { return (uintptr_t)q % 16 == 0 && ld % 16 == 0; };
    if (p.K % 128 != 0 || !al(p.A, p.kt ? 16 : p.lda) || !al(p.B, p.kt && !p.b_rm ? 16 : p.ldb)) return false;
    if (w4 && p.w4_signed && p.K > 65536) return false;
    // 32-bit byte offsets within a tile's rows (at most 128) and along K.
    const int64_t lim = (int64_t)1 << 23;
    if (p.lda >= lim || p.ldb >= lim || p.K >= lim || p.lut_groups * 16 >= lim) return false;
    return true;
}

}  // namespace phi_dev
