// The register-resident rotate + quantise of one row (quant_rotate.hip), shared
// with the one-launch linear of a few rows (row_linear.hip).
#pragma once

#include "device_common.hpp"
#include "i8_gemm.hpp"
#include "qt_scale.hpp"

namespace phi_dev {

// One radix-4 pass over 16 in-register values: the digit with stride `st`
// (1 or 4) varies, the other digit selects the quadruple.
template <int ST>
__device__ __forceinline__ void bfly16(float (&v)[16]) {
#pragma unroll
    for (int o = 0; o < 4; o++) {
        const int b = ST == 1 ? 4 * o : o;
        const float x0 = v[b], x1 = v[b + ST], x2 = v[b + 2 * ST], x3 = v[b + 3 * ST];
        const float sum = ((x0 + x1) + x2) + x3;
        v[b] = sum - 2.0f * x3;
        v[b + ST] = sum - 2.0f * x2;
        v[b + 2 * ST] = sum - 2.0f * x1;
        v[b + 3 * ST] = sum - 2.0f * x0;
    }
}

// Modulation before the rotation (the DiT's adaLN ModAdd, fused):
// v = fma(v, 1 + scale[col], shift[col]), the reference's `a * (1 + b) + c`
// (core/kernels/ops.cpp:82, ModAdd core/kernels/gpu_ops.hpp:29-35) as NVRTC's
// default --fmad=true contracts it.  scale or shift may be NULL (0).
__device__ __forceinline__ void modulate16(float (&v)[16], const float* __restrict__ sc, const float* __restrict__ sh,
                                           int64_t col) {
    float b[16], c[16];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float4 tb = sc ? *(const float4*)(sc + col + 4 * i) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float4 tc = sh ? *(const float4*)(sh + col + 4 * i) : make_float4(0.f, 0.f, 0.f, 0.f);
        b[4 * i] = tb.x, b[4 * i + 1] = tb.y, b[4 * i + 2] = tb.z, b[4 * i + 3] = tb.w;
        c[4 * i] = tc.x, c[4 * i + 1] = tc.y, c[4 * i + 2] = tc.z, c[4 * i + 3] = tc.w;
    }
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = fmaf(v[i], 1.0f + b[i], c[i]);
}

// 16 consecutive input elements at element offset off, as fp32.
template <bool BF16_IN>
__device__ __forceinline__ void load16(const void* __restrict__ x, int64_t off, float (&v)[16]) {
    if (BF16_IN) {
        const uint4* src = (const uint4*)((const uint16_t*)x + off);
        const uint4 a = src[0], b = src[1];
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[2 * i] = bf16_to_f32(w[i] & 0xffffu);
            v[2 * i + 1] = bf16_to_f32(w[i] >> 16);
        }
    } else {
        const float4* src = (const float4*)((const float*)x + off);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float4 t = src[i];
            v[4 * i] = t.x;
            v[4 * i + 1] = t.y;
            v[4 * i + 2] = t.z;
            v[4 * i + 3] = t.w;
        }
    }
}

// ---------------------------------------------------------------------------
// Register-resident form, K <= 16384 (at most 64 groups).
//
// A wave works on 4R consecutive 256-groups of one row in R rounds of four,
// one 16-lane team per group, and keeps its rotated values in registers (16
// per lane per round) until the row amax is known.  WPR = ceil(G / 4R) waves
// cover a row (threadIdx.x) and a block holds RPB rows (threadIdx.y); only the
// amax crosses waves (one barrier, none when WPR is 1).  The two transposes
// of a round go through a 16x16 tile private to the team: a wave's LDS
// operations complete in issue order, so they need no barrier.
//
// Tile layout: row a holds group elements 16a..16a+15, and its 16-byte chunk c
// sits in chunk slot c ^ (a >> 2).  Row accesses (16 lanes x 16 B) and column
// accesses (one float per lane) are then free of bank conflicts; the four
// tiles of a wave are 272 floats apart, so the teams' column accesses use
// different banks.
//
// About fifteen VALU instructions an element against four bytes of HBM
// traffic (bf16 in, int8 out).  At one round a wave the prologue is bound by
// VALU issue (at 4352 x 3072 the VALU instructions fill 0.9 of the busy
// clocks, and the same loads and stores alone take 5.7 us against its
// 9.2 us); with more rounds a wave there are fewer waves, and it waits on
// memory instead.  Hence few instructions: one fma per butterfly output
// (exact as sum - 2x while 2x does not overflow), the final 1/16 folded into
// the scale, the amax as v_max3 over |.|, half-away rounding as add +
// truncate (pre_half_away) without the clamp on rows that cannot need it,
// the bytes packed by the conversions themselves (cvt_pack4), the row's
// address arithmetic on the scalar unit, and the scale's two divisions in
// nine instructions (qt_scale_fast).  R > 1 spreads the per-wave costs
// (addresses, scale divisions, reductions) over more elements.
constexpr int QT_TILE = 272;
constexpr int QT_WAVE = 4 * QT_TILE;
constexpr int QT_MAX_ROUNDS = 5;

// Orders one wave's LDS accesses across lanes for the compiler: the hardware
// already completes a wave's LDS operations in issue order, and a wavefront-
// scope fence emits no instruction, but it keeps the compiler from moving a
// load of another lane's slot above the store that fills it.
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// bfly16 with y = fma(-2, x[3-j], sum): bit-identical, one instruction fewer
// per output.
template <int ST>
__device__ __forceinline__ void bfly16f(float (&v)[16]) {
#pragma unroll
    for (int o = 0; o < 4; o++) {
        const int b = ST == 1 ? 4 * o : o;
        const float x0 = v[b], x1 = v[b + ST], x2 = v[b + 2 * ST], x3 = v[b + 3 * ST];
        const float sum = ((x0 + x1) + x2) + x3;
        v[b] = fmaf(-2.0f, x3, sum);
        v[b + ST] = fmaf(-2.0f, x2, sum);
        v[b + 2 * ST] = fmaf(-2.0f, x1, sum);
        v[b + 3 * ST] = fmaf(-2.0f, x0, sum);
    }
}

// bfly16f<4> that also returns (s0 + s1) + (s2 + s3) over its four quadruple
// sums.  That value is finite only if all 16 inputs are: an inf or NaN input
// makes its quadruple's sum inf or NaN (never finite).  With finite inputs the
// outputs fma(-2, x, sum) are finite or +-inf, never NaN.
__device__ __forceinline__ float bfly16f_last(float (&v)[16]) {
    float s[4];
#pragma unroll
    for (int o = 0; o < 4; o++) {
        const float x0 = v[o], x1 = v[o + 4], x2 = v[o + 8], x3 = v[o + 12];
        s[o] = ((x0 + x1) + x2) + x3;
        v[o] = fmaf(-2.0f, x3, s[o]);
        v[o + 4] = fmaf(-2.0f, x2, s[o]);
        v[o + 8] = fmaf(-2.0f, x1, s[o]);
        v[o + 12] = fmaf(-2.0f, x0, s[o]);
    }
    return (s[0] + s[1]) + (s[2] + s[3]);
}

// max(m, |a|, |b|) in one instruction (fmaxf would first canonicalise each
// operand separately).
__device__ __forceinline__ float max3_abs(float m, float a, float b) {
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}

// Wave-wide max of non-negative floats, as their bit patterns (same order):
// four DPP steps leave each 16-lane row's max in all its lanes, then the four
// row maxima are read out.  The result is wave-uniform.
__device__ __forceinline__ uint32_t wave_max_bits(uint32_t u) {
    u = max(u, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u, 0xB1, 0xF, 0xF, false));   // quad_perm 1,0,3,2
    u = max(u, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u, 0x4E, 0xF, 0xF, false));   // quad_perm 2,3,0,1
    u = max(u, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u, 0x141, 0xF, 0xF, false));  // row_half_mirror
    u = max(u, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u, 0x140, 0xF, 0xF, false));  // row_mirror
    const uint32_t a = __builtin_amdgcn_readlane(u, 0), b = __builtin_amdgcn_readlane(u, 16);
    const uint32_t c = __builtin_amdgcn_readlane(u, 32), d = __builtin_amdgcn_readlane(u, 48);
    return max(max(a, b), max(c, d));
}

// For ties away from zero: min(|v| inv + (0.5 - 2^-25), qmax) with v's sign,
// whose truncation toward zero is the code.  For every non-negative fp32 d,
// floor(fl(d + (0.5 - 2^-25))) is d rounded half away from zero (checked over
// all fp32 d < 2^25; above that d is an integer and the addition returns d),
// and |v| * inv is |v * inv| exactly.  The clamp commutes with the truncation
// because qmax is an integer.  A NaN product (a NaN value, or inf * 0 in a
// row whose amax is inf) gives -qmax, as the reference's clamp
// fminf(fmaxf(d, -qmax), qmax) does (core/kernels/int8_gemm.cpp:779).
__device__ __forceinline__ float pre_half_away(float v, float inv, float qmax) {
    const float p = fabsf(v) * inv;
    return p != p ? -qmax : copysignf(fminf(p + 0.49999997f, qmax), v);
}

// fmaxf returns -qmax for a NaN product here.
__device__ __forceinline__ float pre_half_even(float v, float inv, float qmax) {
    return fminf(fmaxf(rintf(v * inv), -qmax), qmax);
}

// The fast path's codes: pre_half_away and pre_half_even without the clamp.
// They give the clamped codes whenever |v| inv < qmax + 1/2 and v inv is not
// NaN, which holds on every element of a row whose rotated values are all
// finite: there |v| <= amax, so |v| inv <= qmax (1 + 3 2^-24), and qmax is an
// integer in [1, 127] (checked by the C ABI).
__device__ __forceinline__ float pre_half_away_nc(float v, float inv) {
    return copysignf(fabsf(v) * inv + 0.49999997f, v);
}
__device__ __forceinline__ float pre_half_even_nc(float v, float inv) { return rintf(v * inv); }

// Four fp32 values truncated to int and packed little-endian into one dword:
// each conversion writes the low byte of its int32 result into its byte of
// the dword (SDWA dst_sel), the first clearing the others.  Callers pass
// values whose truncations fit int8.
__device__ __forceinline__ uint32_t cvt_pack4(float a, float b, float c, float d) {
    uint32_t r;
    asm("v_cvt_i32_f32_sdwa %0, %1 dst_sel:BYTE_0 dst_unused:UNUSED_PAD src0_sel:DWORD" : "=v"(r) : "v"(a));
    asm("v_cvt_i32_f32_sdwa %0, %1 dst_sel:BYTE_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD" : "+v"(r) : "v"(b));
    asm("v_cvt_i32_f32_sdwa %0, %1 dst_sel:BYTE_2 dst_unused:UNUSED_PRESERVE src0_sel:DWORD" : "+v"(r) : "v"(c));
    asm("v_cvt_i32_f32_sdwa %0, %1 dst_sel:BYTE_3 dst_unused:UNUSED_PRESERVE src0_sel:DWORD" : "+v"(r) : "v"(d));
    return r;
}

template <int OP> constexpr int qt_ns = OP == QR_SILU_GATE ? 2 : 1;  // input sets (the SiLU gate has two)
template <bool BF16_IN> constexpr int qt_nw = BF16_IN ? 8 : 16;        // input dwords per lane and set

// One round's inputs: the lane's 16 elements of a group at element offset
// off of the row at xr, and for the SiLU gate the value operand's 16 at
// off + off2.
template <bool BF16_IN, int OP>
__device__ __forceinline__ void qt_load(const void* __restrict__ xr, int off, const QrPre& pre_op,
                                        uint32_t (&raw)[qt_ns<OP>][qt_nw<BF16_IN>]) {
#pragma unroll
    for (int h = 0; h < qt_ns<OP>; h++) {
        const int o = off + (h ? (int)pre_op.off2 : 0);
        const uint4* src = BF16_IN ? (const uint4*)((const uint16_t*)xr + o) : (const uint4*)((const float*)xr + o);
#pragma unroll
        for (int i = 0; i < qt_nw<BF16_IN> / 4; i++) {
            const uint4 t = src[i];
            raw[h][4 * i] = t.x;
            raw[h][4 * i + 1] = t.y;
            raw[h][4 * i + 2] = t.z;
            raw[h][4 * i + 3] = t.w;
        }
    }
}

// One round's rotation: the pre-op on the raw inputs, passes 1 and 4 in
// registers, the transpose through the team's tile, passes 16 and 64.  w[j]
// receives element 16 j + tl of the group (before the final 1/16).  SUB =
// false forms each butterfly output as fma(-2, x, sum), one rounding; SUB =
// true as sum - 2 x, the reference's mul and subtract.  The product 2x is
// exact unless it overflows (|x| >= 2^127), so the two agree on every group
// whose rotated values stay below 2^126: one radix-4 pass applied twice is
// 4 I, so each value inside the rotation is bounded by about the largest
// output of the pass after it.  For SUB = false the result is the last pass's
// check sum (bfly16f_last): finite only if every value entering that pass is.
template <bool BF16_IN, int OP, bool SUB>
__device__ __forceinline__ float qt_round(const uint32_t (&raw)[qt_ns<OP>][qt_nw<BF16_IN>], int64_t col0, int rotate,
                                          const QrPre& pre_op, float* T, float* trow, int tl, int sw,
                                          float (&w)[16]) {
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        if (BF16_IN) v[i] = __uint_as_float(i & 1 ? raw[0][i >> 1] & 0xffff0000u : raw[0][i >> 1] << 16);
        else v[i] = __uint_as_float(raw[0][i]);
    }
    if (OP == QR_MOD) modulate16(v, pre_op.sc, pre_op.sh, col0);
    if (OP == QR_GELU) {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = gelu_tanh(v[i]);
    }
    if (OP == QR_SILU_GATE) {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t u = raw[qt_ns<OP> - 1][BF16_IN ? i >> 1 : i];
            v[i] = silu_mul(v[i], __uint_as_float(BF16_IN ? (i & 1 ? u & 0xffff0000u : u << 16) : u));
        }
    }
    if (rotate) {
        if (SUB) {
            bfly16<1>(v);
            bfly16<4>(v);
        } else {
            bfly16f<1>(v);
            bfly16f<4>(v);
        }
    }
    // Row tl of the tile, then column tl: w[j] = element 16 j + tl.
#pragma unroll
    for (int c = 0; c < 4; c++)
        *(float4*)(trow + 4 * (c ^ sw)) = make_float4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
    wave_lds_fence();
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const float* col = T + 64 * k + 4 * (sw ^ k) + (tl & 3);
#pragma unroll
        for (int i = 0; i < 4; i++) w[4 * k + i] = col[16 * i];
    }
    wave_lds_fence();
    float f = 0.0f;
    if (rotate) {
        if (SUB) {
            bfly16<1>(w);
            bfly16<4>(w);
        } else {
            bfly16f<1>(w);
            f = bfly16f_last(w);
        }
    }
    return f;
}

// max |w[j]| over a round, as bits (NaN values are passed over, as the
// reference's `if (a > amax)` and fmaxf pass them over).
__device__ __forceinline__ uint32_t qt_amax16(const float (&w)[16]) {
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; j += 2) m = max3_abs(m, w[j], w[j + 1]);
    return __float_as_uint(m);
}

// One round's codes: column tl back into the tile, row tl out (16 contiguous
// elements), quantised and stored as one 16-byte write when live.  FAST
// leaves out the clamp (pre_half_away_nc).
template <bool HALF_EVEN, bool FAST>
__device__ __forceinline__ void qt_store(const float (&w)[16], float* T, float* trow, int tl, int sw,
                                         const QtScale& c, float qmax, int8_t* dst, bool live) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
        float* col = T + 64 * k + 4 * (sw ^ k) + (tl & 3);
#pragma unroll
        for (int i = 0; i < 4; i++) col[16 * i] = w[4 * k + i];
    }
    wave_lds_fence();
    uint32_t packed[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        float4 u = *(const float4*)(trow + 4 * (k ^ sw));
        // Wave-uniform and rare; never on a fast row (amax < 2^126 makes
        // inv >= 2^-122, so the 1/16 is folded).
        if (!FAST && !c.fold) u = make_float4(u.x * c.pre, u.y * c.pre, u.z * c.pre, u.w * c.pre);
        if (FAST) {
            if (HALF_EVEN)
                packed[k] = cvt_pack4(pre_half_even_nc(u.x, c.post), pre_half_even_nc(u.y, c.post),
                                      pre_half_even_nc(u.z, c.post), pre_half_even_nc(u.w, c.post));
            else
                packed[k] = cvt_pack4(pre_half_away_nc(u.x, c.post), pre_half_away_nc(u.y, c.post),
                                      pre_half_away_nc(u.z, c.post), pre_half_away_nc(u.w, c.post));
        } else {
            if (HALF_EVEN)
                packed[k] = cvt_pack4(pre_half_even(u.x, c.post, qmax), pre_half_even(u.y, c.post, qmax),
                                      pre_half_even(u.z, c.post, qmax), pre_half_even(u.w, c.post, qmax));
            else
                packed[k] = cvt_pack4(pre_half_away(u.x, c.post, qmax), pre_half_away(u.y, c.post, qmax),
                                      pre_half_away(u.z, c.post, qmax), pre_half_away(u.w, c.post, qmax));
        }
    }
    wave_lds_fence();
    if (live) *(uint4*)dst = make_uint4(packed[0], packed[1], packed[2], packed[3]);
}

// One row's work after its loads: the rotation of the wave's R rounds, the
// row amax across the row's waves (red: one word a wave of the block), the
// reference-form second pass for rows that need it, and the codes and scale.
template <bool BF16_IN, bool HALF_EVEN, int R, int OP>
__device__ __forceinline__ void qt_row(const uint32_t (&raw)[R][qt_ns<OP>][qt_nw<BF16_IN>],
                                       const void* __restrict__ xr, int row, int rows, int G,
                                       int8_t* __restrict__ q, int64_t ldq, float* __restrict__ s, float qmax,
                                       float qrcp, int rotate, const QrPre& pre_op, int qkt, uint32_t* red, float* T,
                                       float* trow,
                                       int lane, int wr, int wpr, int wave, int g0, int tl, int sw) {
    auto gcol = [&](int r) { return min(g0 + 4 * r, G - 1) * 256; };

    // First pass, on the inputs the caller loaded.
    float rot[R][16];
    uint32_t amax = 0;
    bool nonfinite = false;  // an inf or NaN among a live round's values
    {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const float f = qt_round<BF16_IN, OP, false>(raw[r], gcol(r) + tl * 16, rotate, pre_op, T, trow, tl, sw, rot[r]);
            if (g0 + 4 * r < G) {
                amax = max(amax, qt_amax16(rot[r]));
                nonfinite |= !__builtin_isfinite(f);
            }
        }
    }

    // The lane's 16 bytes of group g land at qrow + g * gstep: row-major, or
    // K-tiled (256-row strips of h rows; the group's four 64-byte K-steps are
    // blocks h x 64 bytes apart; chunk tl & 3 of K-step tl >> 2 in slot
    // (tl & 3) ^ ((row >> 2) & 3)).
    int8_t* qrow;
    int64_t gstep;
    if (qkt) {
        const int64_t st = row >> 8, rr = row & 255, h = min(256, rows - (int)(st << 8));
        qrow = q + st * 256 * (int64_t)G * 256 + (tl >> 2) * h * 64 + rr * 64 + (((tl & 3) ^ ((rr >> 2) & 3)) * 16);
        gstep = 4 * h * 64;
    } else {
        qrow = q + (int64_t)row * ldq + tl * 16;
        gstep = 256;
    }

    // The row's amax (non-negative, so bit 31 is free) travels with a flag
    // for a non-finite value in bit 31.  A row is fast when its rotated
    // values are finite and below 2^126: the fma butterflies then give the
    // reference's values, and the codes need no clamp (pre_half_away_nc).
    // Other rows are rotated again in the reference's form, one round at a
    // time, and quantised with the clamp.  Where waves share barriers
    // (several waves a row), the whole block does so when any of its rows
    // needs it; a fast row gets the same values and codes that way.
    amax = wave_max_bits(amax);
    uint32_t flag = __builtin_amdgcn_ballot_w64(nonfinite) ? 0x80000000u : 0u;
    bool redo;
    if (wpr > 1) {
        // Lane l reads wave l's word (at most 16 waves a block; the lanes
        // past them repeat the last), then one reduction gives the row's
        // amax and flag, and one ballot whether any row of the block is slow.
        if (lane == 0) red[wave] = amax | flag;
        __syncthreads();
        const int nw = blockDim.y * wpr, first = __builtin_amdgcn_readfirstlane(threadIdx.y) * wpr;
        const uint32_t e = red[min(lane, nw - 1)];
        const bool mine = lane >= first && lane < first + wpr;
        amax = wave_max_bits(mine ? e & 0x7fffffffu : 0u);
        flag = __builtin_amdgcn_ballot_w64(mine && (e >> 31) != 0) ? 0x80000000u : 0u;
        redo = __builtin_amdgcn_ballot_w64((e >> 31) != 0 || (e & 0x7fffffffu) >= 0x7e800000u) != 0;
    } else {
        redo = (flag >> 31) != 0 || amax >= 0x7e800000u;
    }

    if (__builtin_amdgcn_readfirstlane(rotate && redo)) {
        // The inputs are loaded again each time: the opaque base keeps the
        // compiler from holding earlier loads live across the passes.
        uint32_t a2 = 0;
#pragma unroll 1
        for (int r = 0; r < R; r++) {
            const void* xo = xr;
            asm volatile("" : "+s"(xo));
            uint32_t raw[qt_ns<OP>][qt_nw<BF16_IN>];
            qt_load<BF16_IN, OP>(xo, tl * 16 + gcol(r), pre_op, raw);
            float w[16];
            qt_round<BF16_IN, OP, true>(raw, gcol(r) + tl * 16, rotate, pre_op, T, trow, tl, sw, w);
            if (g0 + 4 * r < G) a2 = max(a2, qt_amax16(w));
        }
        amax = wave_max_bits(a2);
        if (wpr > 1) {
            __syncthreads();  // every wave has read the first pass's entries
            if (lane == 0) red[wave] = amax;
            __syncthreads();
            for (int i = 0; i < wpr; i++) amax = max(amax, red[__builtin_amdgcn_readfirstlane(threadIdx.y) * wpr + i]);
        }
        const QtScale c = qt_scale(amax, qmax, rotate);
#pragma unroll 1
        for (int r = 0; r < R; r++) {
            const void* xo = xr;
            asm volatile("" : "+s"(xo));
            uint32_t raw[qt_ns<OP>][qt_nw<BF16_IN>];
            qt_load<BF16_IN, OP>(xo, tl * 16 + gcol(r), pre_op, raw);
            float w[16];
            qt_round<BF16_IN, OP, true>(raw, gcol(r) + tl * 16, rotate, pre_op, T, trow, tl, sw, w);
            qt_store<HALF_EVEN, false>(w, T, trow, tl, sw, c, qmax, qrow + (int64_t)(g0 + 4 * r) * gstep,
                                       row < rows && g0 + 4 * r < G);
        }
        if (wr == 0 && lane == 0 && row < rows) s[row] = c.scale;
    } else {
        // Here every row of the block is fast, or there is no rotation (then
        // nothing was checked, and the codes are clamped).
        if (__builtin_amdgcn_readfirstlane(rotate)) {
            const QtScale c = qt_scale_fast(amax, qmax, qrcp);
#pragma unroll
            for (int r = 0; r < R; r++)
                qt_store<HALF_EVEN, true>(rot[r], T, trow, tl, sw, c, qmax, qrow + (int64_t)(g0 + 4 * r) * gstep,
                                          row < rows && g0 + 4 * r < G);
            if (wr == 0 && lane == 0 && row < rows) s[row] = c.scale;
        } else {
            const QtScale c = qt_scale(amax, qmax, rotate);
#pragma unroll
            for (int r = 0; r < R; r++)
                qt_store<HALF_EVEN, false>(rot[r], T, trow, tl, sw, c, qmax, qrow + (int64_t)(g0 + 4 * r) * gstep,
                                           row < rows && g0 + 4 * r < G);
            if (wr == 0 && lane == 0 && row < rows) s[row] = c.scale;
        }
    }
}

}  // namespace phi_dev
