// What the kernels of the gated delta rule share (delta.hip, delta_chunks.hip).
#pragma once
#include "zi_common.h"

// Tokens of a chunk.  The chunks of entries of at least `shortest` tokens are numbered entry by entry, and marks [chunk][head]
// are kept by that number.
#define DELTA_CHUNK 64

__device__ __forceinline__ int delta_chunks_of(int len, int shortest) { return len >= shortest ? (len + DELTA_CHUNK - 1) / DELTA_CHUNK : 0; }

// All lanes of a wavefront: the number of entry e's first chunk.
__device__ __forceinline__ int delta_first_chunk(int e, const int32_t* __restrict__ entry_len, int shortest) {
    int sum = 0;
    for (int i = threadIdx.x & (ZI_WAVE - 1); i < e; i += ZI_WAVE) sum += delta_chunks_of(entry_len[i], shortest);
#pragma unroll
    for (int o = ZI_WAVE / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, ZI_WAVE);
    return __builtin_amdgcn_readfirstlane(sum);
}

// All lanes of a wavefront: the first of the `chunks` chunks from number `first` on that is marked for head h, counted from
// `first`; `chunks` if none is.
__device__ __forceinline__ int delta_first_mark(int first, int chunks, const int32_t* __restrict__ marks, int heads, int h) {
    const int lane = threadIdx.x & (ZI_WAVE - 1);
    for (int i0 = 0; i0 < chunks; i0 += ZI_WAVE) {
        const uint64_t marked = __ballot(i0 + lane < chunks && marks[(int64_t)(first + i0 + lane) * heads + h] != 0);
        if (marked) return i0 + __builtin_ctzll(marked);
    }
    return chunks;
}

// The recurrence token by token.  `marks` (or null): of entries of at least `shortest` tokens only a head's tokens from its first
// marked chunk on are done, from the state that the chunks before it left.
int zi_delta_rule_launch(float* out, const float* qk, const float* v, const float* beta_g, float* state, int64_t state_stride,
                         const int32_t* entry_start, const int32_t* entry_len, const int32_t* entry_slot, int entries, int heads,
                         int kvh, int dim, int vdim, int shortest, const int32_t* marks, hipStream_t stream);
