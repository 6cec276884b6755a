// Grouped low-bit weights (asym_w4a8_int8 nibble4, w6a8_int8 packed6) onto the
// int8 GEMM operand.
//
// Decode (core/host/quant.cpp:315-389, device core/kernels/w4a8_expand.cpp:99-257):
//   level = codebook ? codebook[code] : code - 8      (nibble4; low nibble = even col)
//         = code - 32                                 (packed6: k/2 low-nibble bytes,
//                                                      then k/4 bytes of top-2 bits)
//   v     = rint_clamp127(level * s_rel[row, col/group]) * s_channel[row] (+ corr[g][row])
// Requantise per row (core/host/quant.cpp:134-169, no rotation):
//   scale = amax > 1e-30 ? amax/127 : 1;  q = clamp(round_half_away(v * (1/scale)), +-127)
//
// expand: writes q [rows, k] and s [rows] -- the reference's expand pass.
// prepare: writes s [rows] and, per (row, group), the 16 codes the expand would
//   produce for nibbles 0..15 (lut [rows, groups, 16]), so a GEMM can turn packed
//   nibbles into the same int8 operand in registers (nibble4 only).
//
// Nibble codes in whole 16-byte chunks of one group each take
// w4a8_table_kernel where that pays (w4a8_table_pays), one wave a row: a group
// has 16 possible values, so the row needs 16 decodes a group and not one an
// element.  The general kernel (packed6, other groups and alignments) runs one
// workgroup per row, each thread decoding 16 consecutive columns at a time:
// pass 1 reduces the row amax, pass 2 decodes again and quantises.
#include "device_common.hpp"
#include "persist_common.hpp"
#include "w4a8.hpp"

namespace phi_dev {

__device__ __forceinline__ float rel_at(const uint8_t* row, int dtype, int64_t g) {
    switch (dtype) {
        case W_F32: return ((const float*)row)[g];
        case W_F16: return f16_to_f32(((const uint16_t*)row)[g]);
        case W_BF16: return bf16_to_f32(((const uint16_t*)row)[g]);
        case W_E5M2: return e5m2_to_f32(row[g]);
        default: return e4m3_to_f32(row[g]);  // W_E4M3 and the byte-container spelling
    }
}

// The packer's int8 grid: nearest integer with ties to even, clamped to +-127.
__device__ __forceinline__ float grid8(float v) { return fminf(fmaxf(rintf(v), -127.0f), 127.0f); }

// Decode 16 consecutive columns starting at c0 (c0 % 16 == 0) of one row.
__device__ __forceinline__ void decode16(const W4a8Params& p, int64_t row, int64_t c0,
                                         const float* cb, float (&v)[16]) {
    const uint8_t* codes = p.codes + row * p.codes_row_bytes;
    const uint8_t* rel_row = (const uint8_t*)p.s_rel + row * p.srel_row_bytes;
    const float sch = p.s_channel ? (p.sch_scalar ? p.s_channel[0] : p.s_channel[row]) : 1.0f;
    int code[16];
    if (p.layout == 0) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t b = codes[c0 / 2 + j];
            code[2 * j] = (int)(b & 15u);
            code[2 * j + 1] = (int)(b >> 4);
        }
    } else {
        // Column i's top two bits sit in hi-plane byte i/4 at bit 2*(i & 3).
        const uint8_t* hi = codes + p.k / 2 + c0 / 4;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t b = codes[c0 / 2 + j];
            const uint32_t h = hi[j / 2];
            const int i0 = 2 * j, i1 = 2 * j + 1;
            code[i0] = (int)((b & 15u) | (((h >> (2 * (i0 & 3))) & 3u) << 4));
            code[i1] = (int)((b >> 4) | (((h >> (2 * (i1 & 3))) & 3u) << 4));
        }
    }
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int64_t col = c0 + i;
        const int64_t g = col / p.group;
        float level;
        if (p.layout == 0) level = cb ? cb[code[i]] : (float)(code[i] - 8);
        else level = (float)(code[i] - 32);
        const float rel = p.s_rel ? rel_at(rel_row, p.s_rel_dtype, g) : 1.0f;
        float val = grid8(level * rel) * sch;
        if (p.correction) val = val + p.correction[g * p.rows + row];
        v[i] = val;
    }
}

__device__ float block_max(float v, float* red) {
    v = wave_max(v);
    const int tid = threadIdx.x;
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    float m = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); w++) m = fmaxf(m, red[w]);
    return m;
}

template <bool LUT>
__global__ __launch_bounds__(256) void w4a8_rows_kernel(W4a8Params p, int8_t* __restrict__ out,
                                                        float* __restrict__ s) {
    __shared__ float cb[16];
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const int tid = threadIdx.x;
    if (tid < 16) cb[tid] = p.codebook ? p.codebook[tid] : 0.0f;
    __syncthreads();
    const float* cbp = p.codebook ? cb : nullptr;
    const int64_t chunks = p.k / 16;

    float amax = 0.0f;
    for (int64_t c = tid; c < chunks; c += blockDim.x) {
        float v[16];
        decode16(p, row, c * 16, cbp, v);
#pragma unroll
        for (int i = 0; i < 16; i++) amax = fmaxf(amax, fabsf(v[i]));
    }
    const float rmax = block_max(amax, red);
    const float scale = rmax > 1e-30f ? rmax / 127.0f : 1.0f;
    const float inv = 1.0f / scale;
    if (tid == 0) s[row] = scale;

    if (!LUT) {
        for (int64_t c = tid; c < chunks; c += blockDim.x) {
            float v[16];
            decode16(p, row, c * 16, cbp, v);
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
                w[i] = pack4(quant_code(v[4 * i], inv, 127.0f, 0), quant_code(v[4 * i + 1], inv, 127.0f, 0),
                             quant_code(v[4 * i + 2], inv, 127.0f, 0), quant_code(v[4 * i + 3], inv, 127.0f, 0));
            *(uint4*)(out + row * p.k + c * 16) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    } else {
        // One table per (row, group): the code each nibble value would expand to.
        const int64_t groups = p.k / p.group;
        const uint8_t* rel_row = (const uint8_t*)p.s_rel + row * p.srel_row_bytes;
        const float sch = p.s_channel ? (p.sch_scalar ? p.s_channel[0] : p.s_channel[row]) : 1.0f;
        for (int64_t g = tid; g < groups; g += blockDim.x) {
            const float rel = p.s_rel ? rel_at(rel_row, p.s_rel_dtype, g) : 1.0f;
            const float corr = p.correction ? p.correction[g * p.rows + row] : 0.0f;
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                int qv[4];
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const int code = 4 * i + t;
                    const float level = cbp ? cbp[code] : (float)(code - 8);
                    float val = grid8(level * rel) * sch;
                    if (p.correction) val = val + corr;
                    qv[t] = quant_code(val, inv, 127.0f, 0);
                }
                w[i] = pack4(qv[0], qv[1], qv[2], qv[3]);
            }
            *(uint4*)(out + (row * groups + g) * 16) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

// One wave a row.  Pass 1 collects, per group, which of the 16 codes occur
// (two instructions a code); then lane e of 16 G decodes table entry e (group
// e / 16, code e % 16) once, the row amax is the largest of those that occur,
// and pass 2 turns codes into bytes through the quantised table, as the GEMM
// does.  The same functions on the same values as the general kernel, which
// decodes every element twice and was bound by that (its per-element 64-bit
// division by the group above all): 12288 x 3072, group 128 with a correction
// plane, 154 us; this kernel 23, against 57 MB of traffic (11 us at the card's
// copy rate).  LDS a wave: the table as fp32 and as bytes, and the masks.
__host__ __device__ constexpr size_t w4a8_table_bytes(int64_t groups) { return ((size_t)groups * 84 + 15) & ~(size_t)15; }

template <bool LUT>
__global__ __launch_bounds__(256) void w4a8_table_kernel(W4a8Params p, int8_t* __restrict__ out, float* __restrict__ s) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row = (int64_t)blockIdx.x * 4 + wave;
    if (row >= p.rows) return;  // waves share nothing
    const int G = (int)(p.k / p.group), chunks = (int)(p.k / 32), cpg = (int)(p.group / 32);
    uint8_t* mine = smem + (size_t)wave * w4a8_table_bytes(G);
    float* val = (float*)mine;
    uint8_t* q8 = mine + 64 * G;
    uint32_t* used = (uint32_t*)(mine + 80 * G);
    const persist::u32x4* codes = (const persist::u32x4*)(p.codes + row * p.codes_row_bytes);

    for (int g = lane; g < G; g += 64) used[g] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int c = lane; c < chunks; c += 64) {
        const persist::u32x4 w = codes[c];
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < 32; i++) m |= 1u << ((w[i >> 3] >> (4 * (i & 7))) & 15u);
        atomicOr(&used[c / cpg], m);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");

    const uint8_t* rel_row = (const uint8_t*)p.s_rel + row * p.srel_row_bytes;
    const float sch = p.s_channel ? (p.sch_scalar ? p.s_channel[0] : p.s_channel[row]) : 1.0f;
    const float level = p.codebook ? p.codebook[lane & 15] : (float)((lane & 15) - 8);
    float amax = 0.0f;
    for (int e = lane; e < 16 * G; e += 64) {
        const int g = e >> 4;
        const float rel = p.s_rel ? rel_at(rel_row, p.s_rel_dtype, g) : 1.0f;
        float v = grid8(level * rel) * sch;
        if (p.correction) v = v + p.correction[g * p.rows + row];
        val[e] = v;
        if ((used[g] >> (lane & 15)) & 1u) amax = fmaxf(amax, fabsf(v));
    }
    const float rmax = wave_max(amax);
    const float scale = rmax > 1e-30f ? rmax / 127.0f : 1.0f;
    const float inv = 1.0f / scale;
    if (lane == 0) s[row] = scale;
    for (int e = lane; e < 16 * G; e += 64) q8[e] = (uint8_t)quant_code(val[e], inv, 127.0f, 0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");

    if (LUT) {
        for (int g = lane; g < G; g += 64) *(uint4*)(out + (row * G + g) * 16) = *(const uint4*)(q8 + 16 * g);
        return;
    }
    for (int c = lane; c < chunks; c += 64) {
        const persist::u32x4 w = codes[c], t = *(const persist::u32x4*)(q8 + 16 * (c / cpg));
        v4i* o = (v4i*)(out + row * p.k + (int64_t)c * 32);
        o[0] = persist::expand16b(w[0], w[1], t);
        o[1] = persist::expand16b(w[2], w[3], t);
    }
}

// Where the table kernel beats the general one (189 sizes a function).  Its
// LDS holds 84 bytes a group and wave: above 240 groups one block fits a CU.
// With groups of 32 the general kernel, which spreads a row over four waves,
// is then as fast where there are rows enough to fill the chip otherwise
// (expand, 3072 rows x 8192: 138 us against 121).  Prepare decodes each table
// entry, half the work of an element's in expand, so the line lies lower: with
// few rows a wave's own chain bounds it, 16 entries a group, where the general
// kernel takes a step of 4096 columns (256 x 3072 in groups of 32, 96 of them:
// 14 us against 10); with many, two blocks a CU (3072 x 6144, 192 groups: 74
// against 58; 160 groups 30 against 54).  Groups of 128 and up have few
// entries a column: never.
static bool w4a8_table_pays(const W4a8Params& p, bool lut) {
    const int64_t G = p.k / p.group;
    if (!lut) return G <= 240 || p.group >= 64 || p.rows <= 2048;
    if (p.group >= 128) return true;
    if (p.rows < 1024) return G <= 60 * ((p.k + 4095) / 4096);
    return G <= 160 || (p.group >= 64 && p.rows <= 2048);
}

// The table kernel's limits: 16-byte code chunks that lie in one group, and
// four rows' tables in LDS.
static bool w4a8_table_ok(const W4a8Params& p) {
    return p.layout == 0 && p.group % 32 == 0 && p.k % 32 == 0 && (uintptr_t)p.codes % 16 == 0 &&
           p.codes_row_bytes % 16 == 0 && p.k / p.group <= 480;
}

template <bool LUT>
static hipError_t launch_table(hipStream_t stream, const W4a8Params& p, int8_t* out, float* s) {
    const size_t lds = 4 * w4a8_table_bytes(p.k / p.group);
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute((const void*)w4a8_table_kernel<LUT>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)(4 * w4a8_table_bytes(480)));
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(w4a8_table_kernel<LUT>, dim3((unsigned)((p.rows + 3) / 4)), dim3(256), lds, stream, p, out, s);
    return hipGetLastError();
}

hipError_t launch_w4a8_rows(hipStream_t stream, const W4a8Params& p, int8_t* out, float* s, bool lut) {
    if (w4a8_table_ok(p) && w4a8_table_pays(p, lut)) return lut ? launch_table<true>(stream, p, out, s) : launch_table<false>(stream, p, out, s);
    if (lut)
        hipLaunchKernelGGL(w4a8_rows_kernel<true>, dim3((unsigned)p.rows), dim3(256), 0, stream, p, out, s);
    else
        hipLaunchKernelGGL(w4a8_rows_kernel<false>, dim3((unsigned)p.rows), dim3(256), 0, stream, p, out, s);
    return hipGetLastError();
}

}  // namespace phi_dev
