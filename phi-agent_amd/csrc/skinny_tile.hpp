// Pieces shared by the small-problem GEMM (i8_gemm_skinny.hip) and the
// one-launch linear of a few rows (row_linear.hip): a wave's 16-row operand
// tile as direct-to-LDS loads and fragment reads, and the epilogue of four
// adjacent outputs.
#pragma once

#include "device_common.hpp"
#include "i8_gemm.hpp"
#include "persist_common.hpp"

namespace phi_dev {

// One operand's 16-row tile as the wave loads and reads it: a buffer resource
// at the tile, the lane's byte offsets for a pair's two 1 KB loads, the bytes
// from a pair to the next, and the offsets of the lane's two fragments in the
// 2 KB the loads fill.
struct Tile16 {
    __amdgpu_buffer_rsrc_t rsrc;
    int vo0, vo1, step, f0, f1;
};

// Rows r0.. of a row-major operand (pitch ld), or of a K-tiled one.  Rows past
// the last read it again; their products are not stored.  Row-major: load j
// fetches rows 8 j + l / 8, slot l % 8 of a row's 128 bytes holding chunk
// slot ^ ((row >> 1) & 7), so that the fragment reads of 16 rows hit 16
// distinct bank windows; K-tiled: load j is K-step j of the pair, swizzled in
// memory already (k_tiled_offset).
__device__ __forceinline__ Tile16 tile16(const int8_t* base, int64_t ld, bool kt, int r0, int rows, int K, int lane) {
    Tile16 t;
    const int r = lane & 15, g = lane >> 4, last = rows - 1 - r0;
    if (!kt) {
        t.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(base + (int64_t)r0 * ld), (short)0, 0x7fffffff, persist::kRsrcWord3);
        const int ra = lane >> 3, rb = 8 + ra;
        t.vo0 = min(ra, last) * (int)ld + (((lane & 7) ^ ((ra >> 1) & 7)) << 4);
        t.vo1 = min(rb, last) * (int)ld + (((lane & 7) ^ ((rb >> 1) & 7)) << 4);
        t.step = 128;
        t.f0 = r * 128 + (((2 * g) ^ ((r >> 1) & 7)) << 4);
        t.f1 = r * 128 + (((2 * g + 1) ^ ((r >> 1) & 7)) << 4);
    } else {
        const int s = r0 >> 8, rr = r0 & 255, h = min(256, rows - (s << 8));
        t.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(base + (int64_t)s * 256 * K + rr * 64), (short)0, 0x7fffffff,
                                                   persist::kRsrcWord3);
        t.vo0 = min(lane >> 2, last) * 64 + (lane & 3) * 16;
        t.vo1 = t.vo0 + h * 64;
        t.step = h * 128;
        const int x = (r >> 2) & 3, c = (2 * g) & 3, at = (g >> 1) * 1024 + r * 64;
        t.f0 = at + ((c ^ x) << 4);
        t.f1 = at + (((c + 1) ^ x) << 4);
    }
    return t;
}

// The epilogue (core/kernels/int8_gemm.cpp:588-620) of row m's outputs nn..+3,
// s their int32 sums, sa the row's scale; columns past N are not stored.
__device__ __forceinline__ void skinny_store4(const GemmParams& p, const v4i& s, float sa, int m, int nn) {
    const int64_t off = (int64_t)m * p.ldc + nn;
    const bool whole = p.c_vec && nn + 4 <= p.N;
    if (p.c_kind == C_I32) {
        int32_t* C = (int32_t*)p.C + off;
        if (whole) {
            *(v4i*)C = s;
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (nn + k < p.N) C[k] = s[k];
        }
        return;
    }
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int nk = min(nn + k, p.N - 1);
        const float sb = p.sB[p.sb_scalar ? 0 : nk];
        float bz = 0.0f;
        if (p.bias_kind == BIAS_F32) bz = ((const float*)p.bias)[nk];
        else if (p.bias_kind == BIAS_BF16) bz = bf16_to_f32(((const uint16_t*)p.bias)[nk]);
        v[k] = fmaf((float)s[k] * sa, sb, bz);
    }
    if (p.c_kind == C_BF16) {
        uint16_t* C = (uint16_t*)p.C + off;
        if (whole) {
            *(uint2*)C = make_uint2(f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]));
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (nn + k < p.N) C[k] = (uint16_t)f32_to_bf16(v[k]);
        }
        return;
    }
    float* C = (float*)p.C + off;
    if (p.gate) {
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (nn + k < p.N) C[k] = fmaf(v[k], p.gate[nn + k], C[k]);
    } else if (whole) {
        *(float4*)C = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (nn + k < p.N) C[k] = v[k];
    }
}

}  // namespace phi_dev
