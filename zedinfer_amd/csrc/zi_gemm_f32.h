// What the float32 products (gemm_f32.hip, gemm_f32_split.hip) share: the list of their kernels, loads, stores and the activation.
#pragma once
#include "zi_common.h"

typedef __attribute__((ext_vector_type(4))) float gf_f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned gf_u32x4_t;
typedef __attribute__((ext_vector_type(8))) __bf16 gf_bf16x8_t;

#define GF_PARTS 8           // runs of k; the wavefronts of the stream kernels
#define GF_OUT 0x7fffffff    // an offset past the end of every buffer: the load gives zeros and fetches nothing

// Products of more columns than this go as products of bfloat16 parts (gemm_f32_split.hip), the others through the float32 instruction
// (gemm_f32.hip): a rule on k alone, so that a row's bits do not depend on the rows beside it.  Time by parts over that of the instruction,
// ranges over 1,024 to 65,536 weight rows, by columns:
//                        1,028           1,152           1,408           1,536           2,048
//   1 and 4 rows         0.96 to 1.15    0.93 to 1.03    0.94 to 1.05    0.96 to 1.05    0.94 to 1.15
//   8 to 24 rows         0.92 to 1.17    0.80 to 0.99    0.83 to 1.02    0.81 to 1.02    0.78 to 1.06
//   64 and 200 rows      0.74 to 1.17    0.72 to 1.14    0.74 to 1.02    0.75 to 1.04    0.74 to 1.01
//   450 and 1,000 rows   0.76 to 1.15    0.74 to 1.15    0.74 to 0.99    0.74 to 0.99    0.74 to 1.01
// (1 and 4 rows before gf_few, which takes 2 to 10 % off them.)  Three chunks a run are 24; 1,028 columns fill 17 of them, 1,408 22, and a round of
// tiles is up to 1.15 of the other's time until they are full.
#define GF_SPLIT_ABOVE 1408

// The kernels a product can take; all of one k give the same bits.
enum gf_kernel { GF_PAIRS, GF_ROWS16, GF_ROWS32, GF_HELD_PAIRS, GF_HELD_ROWS16, GF_TILE_64, GF_TILE_32, GF_TILE_32_HALVES, GF_TILE_96_HALVES, GF_TILE_64_QUARTERS };

gf_kernel zi_gemm_f32_split_kernel(int M, int64_t N, int K);
bool zi_gemm_f32_takes(const void* x, const void* w, int N, int K, int64_t ldx, int64_t ldw);
extern "C" int zi_gemm_f32_swiglu_takes(const void* x, const void* w, int M, int inter, int K, int64_t ldx, int64_t ldw);
int zi_gemm_f32_split_launch(bool gated, float* out, const float* x, const float* w, const float* bias, int M, int N, int K, int64_t ldx,
                             int64_t ldw, int64_t ldo, hipStream_t stream);

union gf_pack {
    gf_u32x4_t u;
    gf_f32x4_t f;
    gf_bf16x8_t b;
};

// Rows base .. base + rows - 1 of a row-major matrix as a buffer whose range ends with the last row's K values.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gf_rows(const float* base, int64_t ld, int rows, int K) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, (int)(((int64_t)(rows - 1) * ld + K) * 4), 0x00020000);
}

template <int AUX>
__device__ __forceinline__ gf_f32x4_t gf_load(__amdgpu_buffer_rsrc_t rows, int offset, int all = 0) {
    gf_pack p;
    p.u = __builtin_amdgcn_raw_buffer_load_b128(rows, offset, all, AUX);
    return p.f;
}

// Four outputs of one row of x, columns n .. n + 3.
__device__ __forceinline__ void gf_store4(float* __restrict__ out, const float* __restrict__ bias, gf_f32x4_t s, int n, int N, int vec_out) {
    if (bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += n + e < N ? bias[n + e] : 0.f;
    }
    if (vec_out && n + 3 < N) {
        *reinterpret_cast<gf_f32x4_t*>(out + n) = s;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < N) out[n + e] = s[e];
    }
}

// up * silu(gate), the arithmetic of the activation's own kernel (elementwise.hip).
__device__ __forceinline__ float gf_gate(float gate, float up) { return up * (gate / (1.f + expf(-gate))); }
