// The gated delta rule over portions of a prompt, in chunks of 64 tokens on the matrix cores' float32 instruction
// (v_mfma_f32_16x16x4_f32: float32 products and sums).  delta.hip has the rule, token by token; with it, for the tokens i
// of a chunk, S the state before it, r_ij the product of the decays of the tokens j + 1 .. i and r_i that of the first i + 1,
//
//   u_i = beta_i (v_i - r_i S^T k_i - sum_{j < i} r_ij (k_j . k_i) u_j),     o_i = r_i S^T q_i + sum_{j <= i} r_ij (k_j . q_i) u_j,
//   S <- r_last S + sum_j r_last,j k_j u_j^T.
//
// With M_ij = beta_i r_ij (k_i . k_j) below the diagonal and T = (1 + M)^-1 that is u = T (beta v) - T (beta r k) S.  Products of
// decays are multiplied up and never divided, so a decay of any size, zero included, is as exact as token by token.  The
// entries of T are bounded by one (they are beta_i k_i^T (product of 1 - beta k k^T) k_j, contractions), so it is made by
// forward substitution: 16 x 16 blocks on the diagonal lane by lane, the others as products of blocks.
//
// delta_chunk_kernel makes, for all chunks and heads at once, what does not depend on the state: W = T (beta r k), U = T (beta v),
// A_ij = r_ij (k_j . q_i), r q, the keys turned and scaled for the state's update.  It is a chain of short steps through LDS
// (18 us for one chunk as for 200).  delta_chunk_walk_kernel walks an entry's chunks in order, a workgroup for 16 columns of one
// head's state: u = U - W S on four wavefronts beside r S^T q on the other four, u through LDS, then the state's update beside
// A u.  Bound by that chain: 2.3 us a chunk, of which the instructions are 1.5 (3,584 cycles on every SIMD), on heads x vdim / 16
// workgroups.
//
// Measured, a prompt of 2,000 tokens, 12 heads of 128 x 128: 28 + 77 us a layer and 5 for the launch that finds nothing left to
// do, against 992 us token by token.  Against 64 bits, on the tensors of a model's six such layers, the read-out is 1.7e-7 off
// (token by token 1.8e-7) and the state 1.5e-7 (2.1e-7): the long sums are made of a sum for every 16 values.
//
// The two take DC_ROUND bytes' worth of chunks in turn, so that the workspace has a bound whatever the step: 148 KB a (chunk, head)
// at those sizes, where a round is 151 chunks.  A round more costs its launches and the end of a chain (with rounds of 128 MB 28
// heads took 531 us for 8,192 tokens, against 527 in one of 534 MB; 32 heads 189 for 2,000 against 165).
//
// A NaN or an infinity would pass, as zero times it, from a token to earlier ones of its chunk.  Chunks with a value that
// is not finite, or so large that sums of them may not be (DC_LARGEST; a decay above one, which grows), are marked, and an entry's head is left to delta_rule_kernel from its first marked chunk on.
#include "zi_common.h"
#include "zi_delta.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(4))) float dc_f32x4_t;

#define DC_TOKS DELTA_CHUNK
#define DC_LD (DC_TOKS + 4)
#define DC_LARGEST 0x1p60f        // (keys are unit vectors, T's entries at most one: sums of a chunk's values stay far from infinity)

__device__ __forceinline__ dc_f32x4_t dc_mfma(dc_f32x4_t a, dc_f32x4_t b, dc_f32x4_t c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
    return c;
}

// The sum of N parts, halves first.
template <int N>
__device__ __forceinline__ dc_f32x4_t dc_total(const dc_f32x4_t* part) {
    if constexpr (N == 1) return part[0];
    else return dc_total<N / 2>(part) + dc_total<N - N / 2>(part + N / 2);
}

// 16 x 16 sums over N x 16 values: the rows' pieces in registers, the columns' 16 values apart in LDS (or, turned, the other way
// round).  A sum for every 16, added at the end: less rounding than in one chain.
template <int N, bool TURNED>
__device__ __forceinline__ dc_f32x4_t dc_dot(const dc_f32x4_t (&held)[N], const float* lds) {
    const dc_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    dc_f32x4_t s[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const dc_f32x4_t x = *reinterpret_cast<const dc_f32x4_t*>(lds + i * 16);
        s[i] = TURNED ? dc_mfma(x, held[i], zero) : dc_mfma(held[i], x, zero);
    }
    return dc_total<N>(s);
}

// Chunks are numbered entry by entry.  All lanes of a wavefront: the entry and the chunk within it that number `id` stands for
// (entry -1: none).
__device__ __forceinline__ void dc_find(int id, const int32_t* __restrict__ entry_len, int entries, int shortest, int* entry, int* chunk) {
    const int lane = threadIdx.x & (ZI_WAVE - 1);
    int before = 0;
    *entry = -1;
    for (int e0 = 0; e0 < entries; e0 += ZI_WAVE) {
        const int own = e0 + lane < entries ? delta_chunks_of(entry_len[e0 + lane], shortest) : 0;
        int upto = own;
#pragma unroll
        for (int o = 1; o < ZI_WAVE; o <<= 1) {
            const int x = __shfl_up(upto, o, ZI_WAVE);
            if (lane >= o) upto += x;
        }
        const uint64_t past = __ballot(before + upto > id);
        if (past) {
            const int l = __builtin_ctzll(past);
            *entry = __builtin_amdgcn_readfirstlane(e0 + l);
            *chunk = id - before - __builtin_amdgcn_readlane(upto - own, l);
            return;
        }
        before += __builtin_amdgcn_readlane(upto, ZI_WAVE - 1);
    }
}

// What a (chunk, head) is given in the workspace, in floats: W [64][dim], r q [64][dim], the keys [dim][64], U [64][vdim], A [64][64],
// r of the last token; each in 16 x 16 blocks as the walk's lanes hold them, so that a load takes 1 KB in a run (rows in their
// natural order, sixteen half lines an instruction, took the walk 4.0 instead of 2.3 us a chunk).
__host__ __device__ __forceinline__ int64_t dc_cell(int dim, int vdim) { return (int64_t)DC_TOKS * (3 * dim + vdim + DC_TOKS + 1); }

template <int DT>        // dim / 16
__global__ void __launch_bounds__(512)
delta_chunk_kernel(float* __restrict__ ws, int32_t* __restrict__ marks, const float* __restrict__ qk, const float* __restrict__ v,
                   const float* __restrict__ beta_g, const int32_t* __restrict__ entry_start, const int32_t* __restrict__ entry_len,
                   int entries, int shortest, int heads, int kvh, int vdim, int id0) {
    constexpr int D = DT * 16, LDK = D + 4, VP = (DC_TOKS * D / 4 + 511) / 512;
    __shared__ __attribute__((aligned(16))) float ks[DC_TOKS * LDK];      // keys; then dim columns of v at a time
    __shared__ __attribute__((aligned(16))) float rt[DC_TOKS * DC_LD], ms[DC_TOKS * DC_LD];        // r_ij, then T; M
    __shared__ __attribute__((aligned(16))) float gs[DC_TOKS], bs[DC_TOKS], br[DC_TOKS];
    __shared__ int odd;
    const int tid = threadIdx.x, lane = tid & (ZI_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / ZI_WAVE);
    const int c = lane & 15, g = lane >> 4;
    int e, chunk;
    dc_find(id0 + blockIdx.x, entry_len, entries, shortest, &e, &chunk);
    if (e < 0) return;
    const int h = blockIdx.y, kh = h / (heads / kvh), qkc = 2 * kvh * D;
    const int len = entry_len[e], cnt = len - chunk * DC_TOKS < DC_TOKS ? len - chunk * DC_TOKS : DC_TOKS;
    const int t0 = entry_start[e] + chunk * DC_TOKS;
    float* const cell = ws + ((int64_t)blockIdx.x * heads + h) * dc_cell(D, vdim);
    dc_f32x4_t* const W = reinterpret_cast<dc_f32x4_t*>(cell) + lane, *const Q = W + DC_TOKS * D / 4, *const KT = Q + DC_TOKS * D / 4,
                     *const U = KT + DC_TOKS * D / 4, *const A = U + DC_TOKS * vdim / 4;
    const dc_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    if (tid == 0) odd = 0;
    bool bad = false;
    auto check = [&](const dc_f32x4_t& x) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) bad |= !(fabsf(x[j]) < DC_LARGEST);
    };
    // The blocks of K K^T (wavefronts 0 .. 3) and Q K^T (4 .. 7) on and below the diagonal, a row of blocks a wavefront, the long
    // rows of one beside the short ones of the other on a SIMD.  Queries go straight into registers (rows past the end repeat
    // the last token's; their results are not used).
    const bool of_q = wave >= 4;
    const int ib = of_q ? 7 - wave : wave;
    dc_f32x4_t a[DT];
    if (of_q) {
        const int t = ib * 16 + c < cnt ? ib * 16 + c : cnt - 1;
#pragma unroll
        for (int i = 0; i < DT; ++i) a[i] = *reinterpret_cast<const dc_f32x4_t*>(qk + (int64_t)(t0 + t) * qkc + kh * D + i * 16 + g * 4);
    }
    for (int i = tid; i < DC_TOKS * D / 4; i += 512) {
        const int t = i / (D / 4), d = i % (D / 4) * 4;
        dc_f32x4_t x = zero;
        if (t < cnt) x = *reinterpret_cast<const dc_f32x4_t*>(qk + (int64_t)(t0 + t) * qkc + (kvh + kh) * D + d);
        check(x);
        *reinterpret_cast<dc_f32x4_t*>(ks + t * LDK + d) = x;
    }
    if (tid < DC_TOKS) {       // (tokens past the end: nothing is written, nothing decays)
        const float* row = beta_g + (int64_t)(t0 + (tid < cnt ? tid : 0)) * 2 * heads + h;
        bs[tid] = tid < cnt ? row[0] : 0.f;
        gs[tid] = tid < cnt ? row[heads] : 1.f;
        bad |= !(fabsf(bs[tid]) < DC_LARGEST) || !(fabsf(gs[tid]) <= 1.f);
    }
    __syncthreads();
    // r_ij for i >= j: a thread has column j and 8 rows i0 ..; what comes before them is the rest of j's own 8, then whole 8s
    {
        const int j = tid & 63, i0 = wave * 8, end = (j | 7) + 1;
        float own[8], p = 1.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) own[i] = gs[i0 + i];
        if (end <= i0) {
#pragma unroll
            for (int i = 1; i < 8; ++i) {
                const float x = gs[(j & 56) + i];
                p *= i > (j & 7) ? x : 1.f;
            }
            for (int b = end; b < i0; b += 8) {
                float q = 1.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) q *= gs[b + i];
                p *= q;
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            p *= i0 + i > j ? own[i] : 1.f;
            rt[(i0 + i) * DC_LD + j] = i0 + i >= j ? p : 0.f;
        }
    }
    if (of_q) {
#pragma unroll
        for (int i = 0; i < DT; ++i) check(a[i]);
    } else {
#pragma unroll
        for (int i = 0; i < DT; ++i) a[i] = *reinterpret_cast<const dc_f32x4_t*>(ks + (ib * 16 + c) * LDK + i * 16 + g * 4);
    }
    __syncthreads();
    if (tid < DC_TOKS) br[tid] = bs[tid] * gs[0] * rt[tid * DC_LD];
    if (tid == 0) cell[dc_cell(D, vdim) - DC_TOKS] = gs[0] * rt[(cnt - 1) * DC_LD];
    for (int jb = 0; jb < 4; ++jb) {
        if (of_q) {       // lane (c, g): token i = c of the block, tokens j = 4 g ..
            const int i = ib * 16 + c, j = jb * 16 + g * 4;
            dc_f32x4_t x = zero;
            if (jb <= ib) x = dc_dot<DT, true>(a, ks + (jb * 16 + c) * LDK + g * 4) * *reinterpret_cast<const dc_f32x4_t*>(rt + i * DC_LD + j);
#pragma unroll
            for (int n = 0; n < 4; ++n) x[n] = j + n <= i ? x[n] : 0.f;
            A[(ib * 4 + jb) * ZI_WAVE] = x;
        } else {
            dc_f32x4_t x = zero;
            if (jb <= ib) x = dc_dot<DT, false>(a, ks + (jb * 16 + c) * LDK + g * 4);
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                const int i = ib * 16 + g * 4 + n, j = jb * 16 + c;
                ms[i * DC_LD + j] = j < i ? bs[i] * rt[i * DC_LD + j] * x[n] : 0.f;
            }
        }
    }
    if (of_q) {
        const float r = gs[0] * rt[(ib * 16 + c) * DC_LD];
#pragma unroll
        for (int i = 0; i < DT; ++i) Q[(ib * DT + i) * ZI_WAVE] = a[i] * r;
    }
    // the keys turned, times the decays to the chunk's end (rows past cnt are zero)
    for (int b = wave; b < DT * 4; b += 8) {
        const int d = b / 4 * 16 + c, t = b % 4 * 16 + g * 4;
        dc_f32x4_t x;
#pragma unroll
        for (int n = 0; n < 4; ++n) x[n] = ks[(t + n) * LDK + d];
        KT[b * ZI_WAVE] = x * *reinterpret_cast<const dc_f32x4_t*>(rt + (cnt - 1) * DC_LD + t);
    }
    // v's first columns travel while T is made
    dc_f32x4_t ahead[VP];
    auto request_v = [&](int e0, int wide) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int at = tid + i * 512, t = at / (wide / 4), d = at % (wide / 4) * 4;
            ahead[i] = zero;
            if (t < cnt) ahead[i] = *reinterpret_cast<const dc_f32x4_t*>(v + ((int64_t)(t0 + t) * heads + h) * vdim + e0 + d);
        }
    };
    request_v(0, vdim < D ? vdim : D);
    __syncthreads();
    // T, in the place of r: the diagonal blocks, a column a lane
    if (wave < 4 && g == 0) {
        float x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float s = 0.f;
#pragma unroll
            for (int j = 0; j < i; ++j) s += ms[(wave * 16 + i) * DC_LD + wave * 16 + j] * x[j];
            x[i] = i < c ? 0.f : i == c ? 1.f : -s;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) rt[(wave * 16 + i) * DC_LD + wave * 16 + c] = x[i];
    }
    __syncthreads();
    // the blocks below: a wavefront makes block column `wave` from the diagonal down, T_ij = - T_ii sum_k M_ik T_kj
    if (wave < 3) {
        dc_f32x4_t t[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            t[i] = zero;
            if (i == wave) {
#pragma unroll
                for (int n = 0; n < 4; ++n) t[i][n] = rt[(i * 16 + g * 4 + n) * DC_LD + i * 16 + c];
            } else if (i > wave) {
                dc_f32x4_t s = zero;
#pragma unroll
                for (int k = 0; k < i; ++k)
                    if (k >= wave) s += dc_mfma(*reinterpret_cast<const dc_f32x4_t*>(ms + (i * 16 + c) * DC_LD + k * 16 + g * 4), t[k], zero);
                s = dc_mfma(*reinterpret_cast<const dc_f32x4_t*>(rt + (i * 16 + c) * DC_LD + i * 16 + g * 4), s, zero);
                t[i] = -s;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i > wave) {
#pragma unroll
                for (int n = 0; n < 4; ++n) rt[(i * 16 + g * 4 + n) * DC_LD + wave * 16 + c] = t[i][n];
            }
    }
    __syncthreads();
    // W = T (beta r k) and U = T (beta v): a wavefront takes 16 columns, all four blocks of rows
    auto product = [&](dc_f32x4_t (&sum)[4], int at, const float* scale, auto turned) __attribute__((always_inline)) {   // columns at .. at + 15 of ks
        dc_f32x4_t b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] = zero;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int n = 0; n < 4; ++n) b[j][n] = ks[(j * 16 + g * 4 + n) * LDK + at + c];
            b[j] *= *reinterpret_cast<const dc_f32x4_t*>(scale + j * 16 + g * 4);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (i >= j) {
                    const dc_f32x4_t t = *reinterpret_cast<const dc_f32x4_t*>(rt + (i * 16 + c) * DC_LD + j * 16 + g * 4);
                    sum[i] += decltype(turned)::value ? dc_mfma(b[j], t, zero) : dc_mfma(t, b[j], zero);
                }
    };
    dc_f32x4_t sum[4];
    for (int d = wave; d < DT; d += 8) {
        product(sum, d * 16, br, std::true_type{});       // a token's four dims a lane
#pragma unroll
        for (int i = 0; i < 4; ++i) W[(i * DT + d) * ZI_WAVE] = sum[i];
    }
    for (int e0 = 0; e0 < vdim; e0 += D) {          // v comes through the keys' place, D columns at a time
        const int wide = vdim - e0 < D ? vdim - e0 : D;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int at = tid + i * 512, t = at / (wide / 4), d = at % (wide / 4) * 4;
            check(ahead[i]);
            if (t < DC_TOKS) *reinterpret_cast<dc_f32x4_t*>(ks + t * LDK + d) = ahead[i];
        }
        __syncthreads();
        if (e0 + D < vdim) request_v(e0 + D, vdim - e0 - D < D ? vdim - e0 - D : D);
        for (int d = wave; d < wide / 16; d += 8) {
            product(sum, d * 16, bs, std::false_type{});      // four tokens of a column a lane
#pragma unroll
            for (int i = 0; i < 4; ++i) U[((e0 / 16 + d) * 4 + i) * ZI_WAVE] = sum[i];
        }
    }
    if (bad) odd = 1;
    __syncthreads();
    if (tid == 0) marks[(int64_t)(id0 + blockIdx.x) * heads + h] = odd;
}

// The chunks id_lo .. id_hi - 1 (of all entries; those of the round), as far as no mark of an entry's head comes before them.
template <int DT>        // dim / 16, at most 8: a wavefront holds 16 rows of the state
__global__ void __launch_bounds__(512)
delta_chunk_walk_kernel(float* __restrict__ out, const float* __restrict__ ws, const int32_t* __restrict__ marks,
                        float* __restrict__ state, int64_t state_stride, const int32_t* __restrict__ entry_start,
                        const int32_t* __restrict__ entry_len, const int32_t* __restrict__ entry_slot, int shortest, int heads,
                        int vdim, int id_lo, int id_hi) {
    constexpr int D = DT * 16;
    __shared__ __attribute__((aligned(16))) float st[16 * (D + 4)], xt[16 * DC_LD];      // [column][row of S], [column][token]
    const int lane = threadIdx.x & (ZI_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE);
    const int c = lane & 15, g = lane >> 4;
    // a head's workgroups read the same operands: they are put on one XCD (workgroup i runs on XCD i mod 8)
    const int blocks = vdim / 16, in_xcd = blockIdx.x / 8;
    const int e = blockIdx.z, h = blockIdx.x % 8 + in_xcd / blocks * 8, col = in_xcd % blocks * 16 + c;
    if (h >= heads) return;
    const int len_all = entry_len[e], chunks_all = delta_chunks_of(len_all, shortest);
    if (chunks_all == 0) return;
    const int id0 = delta_first_chunk(e, entry_len, shortest);
    const int first = id_lo > id0 ? id_lo - id0 : 0, before = id_hi - id0 < chunks_all ? id_hi - id0 : chunks_all;
    if (first >= before) return;
    const int chunks = delta_first_mark(id0, before, marks, heads, h) - first;       // (the marks of earlier rounds are there)
    if (chunks <= 0) return;
    // from here on the entry is this round's part of it
    const int start = entry_start[e] + first * DC_TOKS;
    const int len = len_all - first * DC_TOKS < chunks * DC_TOKS ? len_all - first * DC_TOKS : chunks * DC_TOKS;
    const int64_t cell = dc_cell(D, vdim);
    const float* const base = ws + ((int64_t)(id0 + first - id_lo) * heads + h) * cell;
    float* const S = state + (int64_t)entry_slot[e] * state_stride + (int64_t)h * D * vdim;
    const dc_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    const int rb = wave & 3;                                  // the block of tokens
    float* const s_col = st + c * (D + 4) + g * 4;             // this lane's column of the state, of u
    float* const u_col = xt + c * DC_LD + g * 4;
    // the float4s of chunk i that this lane holds
    auto cell_of = [&](int i) __attribute__((always_inline)) {
        return reinterpret_cast<const dc_f32x4_t*>(base + (int64_t)(i < chunks ? i : chunks - 1) * heads * cell) + lane;
    };
    constexpr int QS = DC_TOKS * D / 4;                       // float4s of W, of r q, of the keys
    // A chunk's operands are requested two chunks ahead, each as soon as the products have taken the one in its place, so that
    // the loads' turns at the memory pipeline pass under the products.  Loads and stores stand under no branch: the compiler then
    // knows how many are on their way (a wait behind a branch is a wait for all).
    if (wave < 4) {
        // u = U - W S for 16 tokens, then the state's rows 16 wave .. and 16 (wave + 4) .. (as far as there are)
        const bool own = wave < DT, two = wave + 4 < DT;
        dc_f32x4_t s[2] = {zero, zero};
        auto put = [&]() __attribute__((always_inline)) {
            if (own) *reinterpret_cast<dc_f32x4_t*>(s_col + wave * 16) = s[0];
            if (two) *reinterpret_cast<dc_f32x4_t*>(s_col + wave * 16 + 64) = s[1];
        };
#pragma unroll
        for (int t = 0; t < 2; ++t)
            if (t == 0 ? own : two) {
#pragma unroll
                for (int n = 0; n < 4; ++n) s[t][n] = S[(int64_t)(wave * 16 + t * 64 + g * 4 + n) * vdim + col];
            }
        put();
        dc_f32x4_t w[2][DT], u0[2], kt[2][2][4];
        float last[2];
        const int k0 = 2 * QS + (own ? wave : 0) * 4 * ZI_WAVE, k1 = 2 * QS + (two ? wave + 4 : 0) * 4 * ZI_WAVE;
        const int u_at = 3 * QS + (col / 16 * 4 + rb) * ZI_WAVE;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const dc_f32x4_t* p = cell_of(i);
#pragma unroll
            for (int d = 0; d < DT; ++d) w[i][d] = p[(rb * DT + d) * ZI_WAVE];
            u0[i] = p[u_at];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                kt[i][0][j] = p[k0 + j * ZI_WAVE];
                kt[i][1][j] = p[k1 + j * ZI_WAVE];
            }
            last[i] = reinterpret_cast<const float*>(p - lane)[cell - DC_TOKS];
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        auto step = [&](const int slot, int i) __attribute__((always_inline)) {
            const dc_f32x4_t* p = cell_of(i + 2);
            dc_f32x4_t x[DT];
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                x[d] = dc_mfma(w[slot][d], *reinterpret_cast<const dc_f32x4_t*>(s_col + d * 16), zero);
                __builtin_amdgcn_sched_barrier(0);
                w[slot][d] = p[(rb * DT + d) * ZI_WAVE];
            }
            *reinterpret_cast<dc_f32x4_t*>(u_col + rb * 16) = u0[slot] - dc_total<DT>(x);
            u0[slot] = p[u_at];
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            // (the chunk's sum is made apart and added once: less rounding than into the larger state)
            dc_f32x4_t add[2][4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const dc_f32x4_t u = *reinterpret_cast<const dc_f32x4_t*>(u_col + j * 16);
                add[0][j] = dc_mfma(kt[slot][0][j], u, zero);
                if (DT > 4) add[1][j] = dc_mfma(kt[slot][1][j], u, zero);
                __builtin_amdgcn_sched_barrier(0);
                kt[slot][0][j] = p[k0 + j * ZI_WAVE];
                kt[slot][1][j] = p[k1 + j * ZI_WAVE];
            }
#pragma unroll
            for (int t = 0; t < (DT > 4 ? 2 : 1); ++t) {
                const dc_f32x4_t grown = s[t] * last[slot] + dc_total<4>(add[t]);
                s[t] = i < chunks ? grown : s[t];         // (an odd number of chunks is rounded up by a step that changes nothing)
            }
            put();
            last[slot] = reinterpret_cast<const float*>(p - lane)[cell - DC_TOKS];
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
        };
        for (int i = 0; i < chunks; i += 2) {
            step(0, i);
            step(1, i + 1);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
            if (t == 0 ? own : two) {
#pragma unroll
                for (int n = 0; n < 4; ++n) S[(int64_t)(wave * 16 + t * 64 + g * 4 + n) * vdim + col] = s[t][n];
            }
    } else {
        // o = r S^T q + A u for 16 tokens
        dc_f32x4_t q[2][DT], att[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const dc_f32x4_t* p = cell_of(i);
#pragma unroll
            for (int d = 0; d < DT; ++d) q[i][d] = p[QS + (rb * DT + d) * ZI_WAVE];
#pragma unroll
            for (int j = 0; j < 4; ++j) att[i][j] = p[3 * QS + DC_TOKS * vdim / 4 + (rb * 4 + j) * ZI_WAVE];
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        auto step = [&](const int slot, int i) __attribute__((always_inline)) {
            const dc_f32x4_t* p = cell_of(i + 2);
            dc_f32x4_t x[DT];
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                x[d] = dc_mfma(q[slot][d], *reinterpret_cast<const dc_f32x4_t*>(s_col + d * 16), zero);
                __builtin_amdgcn_sched_barrier(0);
                q[slot][d] = p[QS + (rb * DT + d) * ZI_WAVE];
            }
            __syncthreads();
            dc_f32x4_t add[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                add[j] = dc_mfma(att[slot][j], *reinterpret_cast<const dc_f32x4_t*>(u_col + j * 16), zero);
                __builtin_amdgcn_sched_barrier(0);
                att[slot][j] = p[3 * QS + DC_TOKS * vdim / 4 + (rb * 4 + j) * ZI_WAVE];
            }
            x[0] = dc_total<DT>(x) + dc_total<4>(add);
            // (rows past the entry's end are past the buffer's and go nowhere)
            const int rows = len - i * DC_TOKS < DC_TOKS ? len - i * DC_TOKS : DC_TOKS;
            const __amdgpu_buffer_rsrc_t dst = __builtin_amdgcn_make_buffer_rsrc(out + (int64_t)(start + i * DC_TOKS) * heads * vdim, 0,
                                                                                 rows > 0 ? rows * heads * vdim * 4 : 0, 0x00020000);
#pragma unroll
            for (int n = 0; n < 4; ++n)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[0][n]), dst, (((rb * 16 + g * 4 + n) * heads + h) * vdim + col) * 4, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
        };
        for (int i = 0; i < chunks; i += 2) {
            step(0, i);
            step(1, i + 1);
        }
    }
}

// Tokens of an entry from which it is done in chunks: one chunk's launches take 32 us, as delta_rule_kernel does for 64 tokens.
#define DC_SHORTEST 64

// Bytes of workspace that a round of chunks may take (marks apart).
#define DC_ROUND (256 << 20)

static int64_t dc_most_chunks(int n, int entries) { return n / DC_TOKS + (entries < n / DC_SHORTEST ? entries : n / DC_SHORTEST); }

// Chunks of a round; 0: not even one chunk's heads fit.
static int64_t dc_round(int n, int entries, int heads, int dim, int vdim) {
    const int64_t fit = DC_ROUND / 4 / (heads * dc_cell(dim, vdim)), most = dc_most_chunks(n, entries);
    return fit < most ? fit : most;
}

extern "C" int64_t zi_delta_rule_workspace(int n, int entries, int heads, int dim, int vdim);

// Whether a step whose entries of at least DC_SHORTEST tokens are `long_entries` with `long_tokens` tokens, the longest `longest`, is the
// faster with them in chunks than token by token.  Token by token the longest entry's chain, or, where there are more wavefronts
// than one (two from dim 64 down) a SIMD, all tokens' share of the chip; in chunks the chain of the longest entry's chunks and the
// walk's workgroups, 40 a microsecond past the first 256.  (Constants from one MI355X; the chip is scaled by its units.)  Measured,
// us, token by token against chunks: 12 heads of 128 x 128 one entry of 64 tokens 40 against 31, 32 of them 237 against 168, 20 of 100
// 241 against 124; 2 heads one of 64 39 against 30, 32 of them 46 against 90, 20 of 100 65 against 67; 16 heads of 32 x 64 one of 64
// 20.9 against 22.5, one of 100 30 against 23, 32 of 64 45 against 63; 6 heads of 64 x 64 32 of 64 35 against 49, 8 of 300 108 against 43.
extern "C" int zi_delta_rule_chunks_pay(int long_tokens, int longest, int long_entries, int heads, int dim, int vdim) {
    if (long_entries < 1 || longest < DC_SHORTEST || zi_delta_rule_workspace(long_tokens, long_entries, heads, dim, vdim) == 0) return 0;
    const double chip = zi_compute_units() / 256.;
    const double share = (double)long_tokens * heads * ((vdim + 7) / 8) / ((dim > 64 ? 1024. : 2048.) * chip);
    const double tokens = (0.2 + 0.003 * dim) * (share > longest ? share : longest);
    const double groups = (double)long_entries * ((heads + 7) / 8 * 8) * (vdim / 16) - 256. * chip;
    const double chunks = 17. + 0.09 * dim + 0.018 * dim * ((longest - 1) / DC_TOKS) + (groups > 0 ? 0.025 * groups / chip : 0.);
    return chunks < tokens;
}

// Floats of workspace with which zi_delta_rule_chunked takes n tokens of so many entries in chunks; 0: it would not, the
// entries are too short, the head sizes no multiples of 16 or the heads too many for a round.
extern "C" int64_t zi_delta_rule_workspace(int n, int entries, int heads, int dim, int vdim) {
    if (entries < 1 || n - (entries - 1) < DC_SHORTEST || (int64_t)heads * vdim > (1 << 20) || dim % 16 || dim < 16 || dim > 128 || vdim % 16 || vdim < 16) return 0;
    const int64_t round = dc_round(n, entries, heads, dim, vdim);
    return round > 0 ? heads * (round * dc_cell(dim, vdim) + dc_most_chunks(n, entries)) : 0;
}

extern "C" int zi_delta_rule_chunked(float* out, const float* qk, const float* v, const float* beta_g, float* state, int64_t state_stride,
                                     const int32_t* entry_start, const int32_t* entry_len, const int32_t* entry_slot, int n,
                                     int entries, int heads, int kvh, int dim, int vdim, float* workspace, int64_t workspace_floats,
                                     hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && entries >= 0 && entries <= 65535 && heads > 0 && heads <= 65535 && kvh > 0 && heads % kvh == 0 && dim > 0 &&
               vdim > 0, "delta_rule: bad sizes");
    ZI_REQUIRE(state_stride >= (int64_t)heads * dim * vdim, "delta_rule: the state row is too short");
    const int64_t need = zi_delta_rule_workspace(n, entries, heads, dim, vdim);
    ZI_REQUIRE(need > 0 && workspace && workspace_floats >= need, "delta_rule: workspace of %lld floats is too small (%lld needed)",
               (long long)workspace_floats, (long long)need);
    ZI_REQUIRE(((uintptr_t)qk | (uintptr_t)v | (uintptr_t)workspace) % 16 == 0, "delta_rule: rows must be 16-byte aligned");
    const int64_t chunks = dc_most_chunks(n, entries), round = dc_round(n, entries, heads, dim, vdim);
    int32_t* marks = (int32_t*)(workspace + round * heads * dc_cell(dim, vdim));
#define ZI_DC(DT)                                                                                                                       \
    case DT:                                                                                                                            \
        for (int64_t lo = 0; lo < chunks; lo += round) {                                                                                \
            const int hi = (int)(lo + round < chunks ? lo + round : chunks);                                                             \
            delta_chunk_kernel<DT><<<dim3(hi - lo, heads), 512, 0, stream>>>(workspace, marks, qk, v, beta_g, entry_start, entry_len,    \
                                                                             entries, DC_SHORTEST, heads, kvh, vdim, (int)lo);          \
            delta_chunk_walk_kernel<DT><<<dim3((heads + 7) / 8 * 8 * (vdim / 16), 1, entries), 512, 0, stream>>>(                        \
                out, workspace, marks, state, state_stride, entry_start, entry_len, entry_slot, DC_SHORTEST, heads, vdim, (int)lo, hi);  \
        }                                                                                                                               \
        break
    switch (dim / 16) {
        ZI_DC(1); ZI_DC(2); ZI_DC(3); ZI_DC(4); ZI_DC(5); ZI_DC(6); ZI_DC(7); ZI_DC(8);
    }
#undef ZI_DC
    const int rc = zi_check_launch("delta_rule_chunked");
    if (rc) return rc;
    // the short entries, and the heads of long ones from a mark on
    return zi_delta_rule_launch(out, qk, v, beta_g, state, state_stride, entry_start, entry_len, entry_slot, entries, heads, kvh, dim,
                                vdim, DC_SHORTEST, marks, stream);
}
