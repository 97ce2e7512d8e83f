// Mixture of experts, all on the device: nothing of a step's routing is seen by the host, so a step's launches
// are the same whatever the tokens choose (a step can be recorded and replayed).
//
//   zi_moe_route    z [n][E] float32 router logits -> s = softmax(z); choice = s + correction; the `top` experts
//                   of largest choice (the lowest index among equals), weights s * scale
//   zi_moe_route_table  the experts of a token are read from a table by its id, equal weights
//   zi_moe_group    the (token, choice) pairs sorted by expert: offsets, the order and its inverse, and the list
//                   of row tiles (expert, first row, rows) that the products walk
//   zi_moe_linear   out[row] = act(W[expert of row] . x[source of row]) for every row of the sorted order
//   zi_moe_combine  out[t] = sum_k weight[t][k] * y[place of (t, k)], float32, k in rising order
//
// A row's sums depend on its own values and its expert's weights only, never on where in the order it stands.
#include "zi_common.h"
#include "zi_api.h"

#define MOE_MAX_EXPERTS 1024
#define MOE_PER_LANE (MOE_MAX_EXPERTS / ZI_WAVE)

template <int PER>
__global__ void __launch_bounds__(256)
moe_route_kernel(int32_t* __restrict__ idx, float* __restrict__ wt, const float* __restrict__ z,
                 const float* __restrict__ correction, int n, int E, int top, float scale) {
    const int lane = threadIdx.x % ZI_WAVE;
    const int t = blockIdx.x * (blockDim.x / ZI_WAVE) + threadIdx.x / ZI_WAVE;
    if (t >= n) return;
    float s[PER], choice[PER];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + i * ZI_WAVE;
        s[i] = e < E ? z[(int64_t)t * E + e] : -INFINITY;
        m = fmaxf(m, s[i]);
    }
    m = zi_wave_max(m);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + i * ZI_WAVE;
        s[i] = e < E ? expf(s[i] - m) : 0.f;
        sum += s[i];
    }
    sum = zi_wave_sum(sum);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + i * ZI_WAVE;
        s[i] = s[i] / sum;
        choice[i] = e < E ? s[i] + correction[e] : -INFINITY;
    }
    for (int k = 0; k < top; ++k) {
        float best = -INFINITY, best_s = 0.f;
        int best_e = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = lane + i * ZI_WAVE;
            if (e < E && (choice[i] > best || (choice[i] == best && e < best_e))) {
                best = choice[i];
                best_e = e;
                best_s = s[i];
            }
        }
#pragma unroll
        for (int o = ZI_WAVE / 2; o > 0; o >>= 1) {
            const float ob = __shfl_xor(best, o, ZI_WAVE), os = __shfl_xor(best_s, o, ZI_WAVE);
            const int oe = __shfl_xor(best_e, o, ZI_WAVE);
            if (ob > best || (ob == best && oe < best_e)) {
                best = ob;
                best_e = oe;
                best_s = os;
            }
        }
        if (lane == 0) {
            idx[(int64_t)t * top + k] = best_e;
            wt[(int64_t)t * top + k] = best_s * scale;
        }
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + i * ZI_WAVE == best_e) choice[i] = -INFINITY;
    }
}

extern "C" int zi_moe_route(int32_t* idx, float* wt, const float* z, const float* correction, int n, int experts,
                            int top, float scale, hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && experts > 0 && experts <= MOE_MAX_EXPERTS && top > 0 && top <= experts,
               "moe_route: bad sizes (experts %d, top %d; at most %d experts)", experts, top, MOE_MAX_EXPERTS);
    if (n == 0) return 0;
    const int blocks = (n + 3) / 4;
#define ZI_MOE_ROUTE(PER) moe_route_kernel<PER><<<blocks, 256, 0, stream>>>(idx, wt, z, correction, n, experts, top, scale)
    if (experts <= ZI_WAVE) ZI_MOE_ROUTE(1);
    else if (experts <= 2 * ZI_WAVE) ZI_MOE_ROUTE(2);
    else if (experts <= 4 * ZI_WAVE) ZI_MOE_ROUTE(4);
    else ZI_MOE_ROUTE(MOE_PER_LANE);
#undef ZI_MOE_ROUTE
    return zi_check_launch("moe_route");
}

// The other router: the `top` largest logits themselves are chosen (the lowest index among equals) and the weights
// are the softmax over the chosen logits only.  z [n][E] float32; `bias` [E] (or null) is added to it first.
template <int PER>
__global__ void __launch_bounds__(256)
moe_route_top_kernel(int32_t* __restrict__ idx, float* __restrict__ wt, const float* __restrict__ z,
                     const float* __restrict__ bias, int n, int E, int top) {
    const int lane = threadIdx.x % ZI_WAVE;
    const int t = blockIdx.x * (blockDim.x / ZI_WAVE) + threadIdx.x / ZI_WAVE;
    if (t >= n) return;
    float choice[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + i * ZI_WAVE;
        choice[i] = e < E ? z[(int64_t)t * E + e] + (bias ? bias[e] : 0.f) : -INFINITY;
    }
    float first = 0.f, sum = 0.f;
    for (int k = 0; k < top; ++k) {
        float best = -INFINITY;
        int best_e = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = lane + i * ZI_WAVE;
            if (e < E && (choice[i] > best || (choice[i] == best && e < best_e))) {
                best = choice[i];
                best_e = e;
            }
        }
#pragma unroll
        for (int o = ZI_WAVE / 2; o > 0; o >>= 1) {
            const float ob = __shfl_xor(best, o, ZI_WAVE);
            const int oe = __shfl_xor(best_e, o, ZI_WAVE);
            if (ob > best || (ob == best && oe < best_e)) {
                best = ob;
                best_e = oe;
            }
        }
        if (k == 0) first = best;      // the largest of all: the softmax's maximum
        const float p = expf(best - first);
        sum += p;
        if (lane == 0) {
            idx[(int64_t)t * top + k] = best_e;
            wt[(int64_t)t * top + k] = p;
        }
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + i * ZI_WAVE == best_e) choice[i] = -INFINITY;
    }
    if (lane == 0)
        for (int k = 0; k < top; ++k) wt[(int64_t)t * top + k] /= sum;
}

extern "C" int zi_moe_route_top(int32_t* idx, float* wt, const float* z, const float* bias, int n, int experts, int top,
                                hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && experts > 0 && experts <= MOE_MAX_EXPERTS && top > 0 && top <= experts,
               "moe_route_top: bad sizes (experts %d, top %d; at most %d experts)", experts, top, MOE_MAX_EXPERTS);
    if (n == 0) return 0;
    const int blocks = (n + 3) / 4;
#define ZI_MOE_ROUTE(PER) moe_route_top_kernel<PER><<<blocks, 256, 0, stream>>>(idx, wt, z, bias, n, experts, top)
    if (experts <= ZI_WAVE) ZI_MOE_ROUTE(1);
    else if (experts <= 2 * ZI_WAVE) ZI_MOE_ROUTE(2);
    else if (experts <= 4 * ZI_WAVE) ZI_MOE_ROUTE(4);
    else ZI_MOE_ROUTE(MOE_PER_LANE);
#undef ZI_MOE_ROUTE
    return zi_check_launch("moe_route_top");
}

// Experts named by a table instead of a router: token id v uses the experts table[v][0 .. top), each with the
// weight 1 / top.  An id outside the table, or an entry that names no expert, gives expert 0 with weight NaN so
// that the fault shows.
__global__ void __launch_bounds__(256)
moe_route_table_kernel(int32_t* __restrict__ idx, float* __restrict__ wt, const int32_t* __restrict__ ids,
                       const int32_t* __restrict__ table, int pairs, int vocab, int E, int top) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= pairs) return;
    const int id = ids[i / top];
    const int e = (id >= 0 && id < vocab) ? table[(int64_t)id * top + i % top] : -1;
    const bool ok = e >= 0 && e < E;
    idx[i] = ok ? e : 0;
    wt[i] = ok ? 1.f / (float)top : NAN;
}

extern "C" int zi_moe_route_table(int32_t* idx, float* wt, const int32_t* ids, const int32_t* table, int n, int vocab,
                                  int experts, int top, hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && vocab > 0 && experts > 0 && experts <= MOE_MAX_EXPERTS && top > 0 && top <= experts,
               "moe_route_table: bad sizes (experts %d, top %d; at most %d experts)", experts, top, MOE_MAX_EXPERTS);
    if (n == 0) return 0;
    const int pairs = n * top;
    moe_route_table_kernel<<<(pairs + 255) / 256, 256, 0, stream>>>(idx, wt, ids, table, pairs, vocab, experts, top);
    return zi_check_launch("moe_route_table");
}

// One workgroup sorts the M = n * top pairs by expert (a counting sort; within an expert the order is the order
// of arrival, which no result depends on).  plan: [0] = number of row tiles, then [1 + 3 i ...] = (expert, first
// row, rows) of tile i; order[place] = pair, place_of[pair] = place.
__global__ void __launch_bounds__(1024)
moe_group_kernel(int32_t* __restrict__ plan, int32_t* __restrict__ order, int32_t* __restrict__ place_of,
                 const int32_t* __restrict__ idx, int M, int E, int tile_rows) {
    __shared__ int count[MOE_MAX_EXPERTS], first[MOE_MAX_EXPERTS], tile0[MOE_MAX_EXPERTS], cursor[MOE_MAX_EXPERTS];
    for (int e = threadIdx.x; e < E; e += blockDim.x) count[e] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < M; i += blockDim.x) {
        const int e = idx[i];
        if ((unsigned)e < (unsigned)E) atomicAdd(&count[e], 1);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int at = 0, tiles = 0;
        for (int e = 0; e < E; ++e) {
            first[e] = at;
            tile0[e] = tiles;
            at += count[e];
            tiles += (count[e] + tile_rows - 1) / tile_rows;
        }
        plan[0] = tiles;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        cursor[e] = first[e];
        for (int r = 0, i = tile0[e]; r < count[e]; r += tile_rows, ++i) {
            plan[1 + 3 * i] = e;
            plan[2 + 3 * i] = first[e] + r;
            plan[3 + 3 * i] = count[e] - r < tile_rows ? count[e] - r : tile_rows;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < M; i += blockDim.x) {
        const int e = idx[i];
        if ((unsigned)e >= (unsigned)E) continue;
        const int at = atomicAdd(&cursor[e], 1);
        order[at] = i;
        place_of[i] = at;
    }
}

extern "C" int zi_moe_group(int32_t* plan, int32_t* order, int32_t* place_of, const int32_t* idx, int pairs,
                            int experts, int tile_rows, hipStream_t stream) {
    ZI_REQUIRE(pairs >= 0 && experts > 0 && experts <= MOE_MAX_EXPERTS && tile_rows > 0, "moe_group: bad sizes");
    moe_group_kernel<<<1, 1024, 0, stream>>>(plan, order, place_of, idx, pairs, experts, tile_rows);
    return zi_check_launch("moe_group");
}

#define MOE_ACT_NONE 0
#define MOE_ACT_GELU_ERF 1

__device__ __forceinline__ void moe_store4(float* p, float a, float b, float c, float d) {
    *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d);
}
__device__ __forceinline__ void moe_store4(zi_bf16* p, float a, float b, float c, float d) {
    uint2 v;
    v.x = zi_pack_bf16x2(a, b);
    v.y = zi_pack_bf16x2(c, d);
    *reinterpret_cast<uint2*>(p) = v;
}

__device__ __forceinline__ float moe_act(float z, int act) {
    return act == MOE_ACT_GELU_ERF ? 0.5f * z * (1.f + erff(z * 0.70710678118654752440f)) : z;
}

// The plain product: a workgroup of 256 threads makes 16 rows (of a larger tile: the blockIdx.z-th) x 64 columns, k in blocks
// of 32 through LDS.
#define MOE_TM 16
#define MOE_TN 64
#define MOE_KC 32

template <typename TX, typename TW, typename TO>
__global__ void __launch_bounds__(256)
moe_linear_kernel(TO* __restrict__ out, int64_t ldo, const TX* __restrict__ x, int64_t ldx, const TW* __restrict__ w,
                  const int32_t* __restrict__ plan, const int32_t* __restrict__ source, int source_div, int N, int K,
                  int act) {
    __shared__ float xs[MOE_TM][MOE_KC + 1], ws[MOE_TN][MOE_KC + 1];
    __shared__ int src[MOE_TM];
    const int tile = blockIdx.y;
    if (tile >= plan[0]) return;
    const int e = plan[1 + 3 * tile], r0 = plan[2 + 3 * tile] + blockIdx.z * MOE_TM, rows = plan[3 + 3 * tile] - (int)blockIdx.z * MOE_TM;
    if (rows <= 0) return;
    const int n0 = blockIdx.x * MOE_TN;
    if (threadIdx.x < MOE_TM) {
        const int r = r0 + (threadIdx.x < rows ? threadIdx.x : 0);
        src[threadIdx.x] = source ? source[r] / source_div : r;
    }
    const TW* we = w + (int64_t)e * N * K;
    const int c = threadIdx.x % MOE_TN, rg = threadIdx.x / MOE_TN;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += MOE_KC) {
        __syncthreads();
        for (int i = threadIdx.x; i < MOE_TM * MOE_KC; i += 256) {
            const int r = i / MOE_KC, kk = i % MOE_KC;
            xs[r][kk] = k0 + kk < K ? zi_load(x + (int64_t)src[r] * ldx + k0 + kk) : 0.f;
        }
        for (int i = threadIdx.x; i < MOE_TN * MOE_KC; i += 256) {
            const int cc = i / MOE_KC, kk = i % MOE_KC;
            ws[cc][kk] = (n0 + cc < N && k0 + kk < K) ? zi_load(we + (int64_t)(n0 + cc) * K + k0 + kk) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < MOE_KC; ++kk) {
            const float wv = ws[c][kk];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] += xs[rg * 4 + i][kk] * wv;
        }
    }
    if (n0 + c >= N) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = rg * 4 + i;
        if (r < rows) zi_store(out + (int64_t)(r0 + r) * ldo + n0 + c, moe_act(acc[i], act));
    }
}

// The same on the matrix cores (bfloat16 operands, float32 sums): a workgroup of four wavefronts makes a tile of RT x 16 rows
// and 64 CT columns, a wavefront all of the rows and 16 CT of the columns; the expert's weight rows are the first operand (lane:
// row l % 16, eight k from 8 (l / 16)), the tokens' rows the second, so a lane ends with four neighbouring columns of one row.
// Both operands go straight into LDS in whole lines of 128 bytes (1 KB an instruction; piece c of row q at place c xor (q / 2
// mod 8), so that a wavefront's reads meet no bank twice), k in steps of 64 through a ring of ST buffers; every wavefront
// issues as many loads a step as every other, so that each can wait for its own by count before the step's one barrier.
// Workgroups are dealt out so that an XCD takes neighbouring tiles: an expert's weights are then fetched into one L2.
// What it replaced read the operands' fragments from memory, 16 rows x 64 bytes an instruction, a quarter of the rate of whole
// lines.  Measured with 32 experts of 1536 x 1536 (151 MB of weights), the first product and the second: 8,000 pairs 203 and
// 195 to 98 and 87 us (two buffers, so that a unit holds two workgroups: with four buffers and one workgroup 141 and 115), 128
// pairs 41 and 40 to 24.8 and 24.6 us (6.1 TB/s; with four buffers 26.5 and 25.3).
// Tiles of 128 rows x 256 columns are eight wavefronts', 64 x 64 each, with three buffers in 144 KB: three fifths of the bytes an
// operation, two steps on their way, and one workgroup a unit, so that a last round of tiles costs more (which
// steps take them: moe_tile_rows).  8 experts of 4,096 x 14,336 with 256 rows each 0.84 of the time in tiles of 64, of 6,144 x 16,384 0.76; at
// 1,536 x 1,536 8,000 pairs 88 and 77 us for 92 and 83, but 9,200 pairs a fifth more than in tiles of 64.
typedef __attribute__((ext_vector_type(8))) __bf16 moe_bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float moe_f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned moe_u32x4_t;
union moe_pack {
    moe_u32x4_t u;
    moe_bf16x8_t b;
};

#define MOE_KB 64
#define MOE_XCDS 8
// Turns through the buffers in a row.  The compiler waits for all loads at the first read in a loop's body, also for those that were asked
// for a moment ago: once in TURNS turns.  More turns are more instructions, which every compute unit fetches once a launch, and with more
// than one a tile asks for ST - 1 steps past its last.  Time over that of one turn, of two and four turns, geometric means over 2 to 3
// numbers of pairs of five sets of experts (8 to 64, 512 to 4,096 columns), by columns of K:
//   tiles of 16 rows   64: 1.04, 1.05    256: 1.01, 1.00    384: 0.98, 0.98    640: 0.98, 0.96    1,536: 0.96, 0.94    3,584: 0.95, 0.94
//   of 32              64: 1.08, 1.16    384: 0.99, 1.07    512: 1.00, 1.06    640: 0.99, 1.04    1,536: 0.95, 1.01    3,584: 0.95, 1.00
//   of 128             64: 1.04, 1.08    384: 0.99, 1.02    512: 1.00, 1.01    640: 0.98, 0.99    1,536: 0.94, 0.94    3,584: 0.94, 0.94
// Tiles of 64 rows have two buffers and wait for every load in every step: four turns 1.02 to 1.06.  So 16 rows take four from 384
// columns on, 32 and 128 two beyond 512.  (Slower there: 8 experts of 4,096 columns at 12 rows, four turns 1.03 to 1.05.)
static int moe_turns(int tile_rows, int K) { return tile_rows == 16 ? (K >= 384 ? 4 : 1) : tile_rows == 64 ? 1 : K > 512 ? 2 : 1; }
// the longest row of weights whose tile of rows a buffer's 31-bit offsets reach
#define MOE_MAX_K (1 << 21)

// 16 bytes a lane into LDS, lane after lane from `to` on: from an address, or from a buffer (zeros past its end).
__device__ __forceinline__ void moe_to_lds(const zi_bf16* from, moe_u32x4_t* to) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host's pass knows loads of this size for no target)
    __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
#endif
}
template <int AUX>
__device__ __forceinline__ void moe_to_lds(__amdgpu_buffer_rsrc_t from, moe_u32x4_t* to, int lane_at) {
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_raw_ptr_buffer_load_lds(from, to, 16, lane_at, 0, 0, AUX);
#endif
}

// A wavefront's tile: a lane holds four consecutive columns of a row, one store of 16 (float32) or 8 bytes (bfloat16) where the rows allow it.
template <int RW, int CT, typename TO>
__device__ __forceinline__ void moe_store_tile(TO* out, int64_t ldo, moe_f32x4_t (&acc)[RW][CT], int act, int rows, int r0, int row0, int n1, int N, int r, int j) {
    const bool whole = ldo % 4 == 0 && ((uintptr_t)out % 16) == 0;
#pragma unroll
    for (int t = 0; t < RW; ++t) {
        const int row = row0 + t * 16 + r;
        if (row >= rows) continue;
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const int n = n1 + c * 16 + 4 * j;
            TO* dst = out + (int64_t)(r0 + row) * ldo + n;
            if (whole && n + 3 < N) {
                moe_store4(dst, moe_act(acc[t][c][0], act), moe_act(acc[t][c][1], act), moe_act(acc[t][c][2], act),
                           moe_act(acc[t][c][3], act));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < N) zi_store(dst + i, moe_act(acc[t][c][i], act));
            }
        }
    }
}

// WR: wavefronts along the rows of a tile, each with RT / WR of its sixteens; four times as many in all.  TURNS: see moe_turns.
template <typename TO, int RT, int CT, int ST, int WR, int TURNS>
__global__ void __launch_bounds__(4 * WR * ZI_WAVE)
moe_linear_mfma_kernel(TO* __restrict__ out, int64_t ldo, const zi_bf16* __restrict__ x, int64_t ldx,
                       const zi_bf16* __restrict__ w, const int32_t* __restrict__ plan,
                       const int32_t* __restrict__ source, int source_div, int N, int K, int act) {
    constexpr int WAVES = 4 * WR, RW = RT / WR;
    static_assert(RT % WR == 0 && 8 * CT % WAVES == 0, "whole shares");
    constexpr int XI = 2 * RT, WI = 8 * CT, XW = (XI + WAVES - 1) / WAVES, WW = WI / WAVES, PW = XW + WW;      // loads of a step; a wavefront's share
    constexpr int PIECES = (WAVES * XW + WI) * ZI_WAVE;
    // (arrays of their own, so that the compiler can tell a buffer that is read from those that loads are on their way to)
    __shared__ __attribute__((aligned(16))) moe_u32x4_t s0[PIECES], s1[PIECES], s2[ST > 2 ? PIECES : 1];
    static_assert(ST == 2 || ST == 3, "two or three buffers");
    const int blocks = (N + 64 * CT - 1) / (64 * CT), total = plan[0] * blocks, share = (total + MOE_XCDS - 1) / MOE_XCDS;
    const int at_share = blockIdx.x / MOE_XCDS, job = (int)(blockIdx.x % MOE_XCDS) * share + at_share;
    if (at_share >= share || job >= total) return;
    const int tile = job / blocks, n0 = job % blocks * 64 * CT;
    const int e = plan[1 + 3 * tile], r0 = plan[2 + 3 * tile], rows = plan[3 + 3 * tile];
    const int lane = threadIdx.x % ZI_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE);
    const int r = lane & 15, j = lane >> 4, wave_c = wave % 4, row0 = wave / 4 * RW * 16;      // this wavefront's columns and rows
    // Load i takes 8 rows: lane l row l / 8 of them, the piece that belongs at place l % 8.  (Rows of the tokens past the
    // tile's are its first row again, not stored; weight rows past N are past the buffer's end.)
    const int rows_w = N - n0 < 64 * CT ? N - n0 : 64 * CT;
    const __amdgpu_buffer_rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc(const_cast<zi_bf16*>(w + ((int64_t)e * N + n0) * K), 0,
                                                                        rows_w * K * 2, 0x00020000);
    const zi_bf16* xrow[XW];
    int xpiece[XW], w_at[WW], wpiece[WW];
#pragma unroll
    for (int i = 0; i < XW; ++i) {
        const int q = (i * WAVES + wave) * 8 + lane / 8, rr = q < rows ? q : 0;
        xrow[i] = x + (int64_t)(source ? source[r0 + rr] / source_div : r0 + rr) * ldx;
        xpiece[i] = ((lane & 7) ^ ((q >> 1) & 7)) * 8;
    }
#pragma unroll
    for (int i = 0; i < WW; ++i) {
        const int q = (i * WAVES + wave) * 8 + lane / 8;
        wpiece[i] = ((lane & 7) ^ ((q >> 1) & 7)) * 8;
        w_at[i] = (q < rows_w ? q * K + wpiece[i] : rows_w * K) * 2;
    }
    const int steps = (K + MOE_KB - 1) / MOE_KB;
    // (columns past K, a multiple of 8: the tokens' are the row's first again, the weights' the next row's or zeros; both masked, or, in
    // the steps past the last that are asked for too, not read)
    auto issue = [&](moe_u32x4_t* buf, int t) {
        const int k0 = t * MOE_KB;
        const bool whole = k0 + MOE_KB <= K;
#pragma unroll
        for (int i = 0; i < XW; ++i)
            moe_to_lds(xrow[i] + (whole || k0 + xpiece[i] < K ? k0 + xpiece[i] : 0), buf + (i * WAVES + wave) * ZI_WAVE);
#pragma unroll
        for (int i = 0; i < WW; ++i)
            moe_to_lds<RT == 1 ? 2 : 0>(wb, buf + (WAVES * XW + i * WAVES + wave) * ZI_WAVE,
                                        whole || k0 + wpiece[i] < K ? w_at[i] + k0 * 2 : rows_w * K * 2);
    };
    moe_f32x4_t acc[RW][CT];
#pragma unroll
    for (int t = 0; t < RW; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[t][c] = (moe_f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int sw = (r >> 1) & 7;
    auto step = [&](const moe_u32x4_t* buf, moe_u32x4_t* free, int t) __attribute__((always_inline)) {
        if (TURNS == 1 && t >= steps) return;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (TURNS > 1 || steps - 1 - t >= ST - 2) zi_wait_loads<(ST - 2) * PW>();      // the newest steps' loads may still be on their way
        else zi_wait_loads<0>();
        __builtin_amdgcn_s_barrier();          // all wavefronts' loads of the step are there, and all are done with `free`
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (TURNS > 1 || t + ST - 1 < steps) issue(free, t + ST - 1);
        __builtin_amdgcn_sched_barrier(0);
        const int left = K - t * MOE_KB;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int at = (kk * 4 + j) ^ sw;
            moe_pack a[CT], b[RW];
#pragma unroll
            for (int c = 0; c < CT; ++c) a[c].u = buf[(WAVES * XW * 8 + (wave_c * CT + c) * 16 + r) * 8 + at];
#pragma unroll
            for (int m = 0; m < RW; ++m) b[m].u = buf[(row0 + m * 16 + r) * 8 + at];
            if (left < MOE_KB) {
                const unsigned mask = 0u - (unsigned)(kk * 32 + j * 8 < left);
#pragma unroll
                for (int c = 0; c < CT; ++c) a[c].u &= mask;
#pragma unroll
                for (int m = 0; m < RW; ++m) b[m].u &= mask;
            }
#pragma unroll
            for (int m = 0; m < RW; ++m)
#pragma unroll
                for (int c = 0; c < CT; ++c)
                    acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c].b, b[m].b, acc[m][c], 0, 0, 0);
        }
    };
    issue(s0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (ST > 2 && (TURNS > 1 || steps > 1)) issue(s1, 1);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (TURNS == 1) {
        for (int t = 0; t < steps; t += ST) {
            step(s0, ST == 2 ? s1 : s2, t);
            step(s1, s0, t + 1);
            if constexpr (ST > 2) step(s2, s1, t + 2);
        }
    } else {
        for (int t = 0, left = 1; left;) {
#pragma unroll
            for (int turn = 0; turn < TURNS; ++turn) {
                step(s0, ST == 2 ? s1 : s2, t);
                if (!(left = ++t < steps)) break;
                step(s1, s0, t);
                if (!(left = ++t < steps)) break;
                if constexpr (ST > 2) {
                    step(s2, s1, t);
                    if (!(left = ++t < steps)) break;
                }
            }
        }
        zi_wait_loads<0>();
    }
    moe_store_tile<RW, CT>(out, ldo, acc, act, rows, r0, row0, n0 + wave_c * CT * 16, N, r, j);
}

// The tiles of 128 rows x 256 columns where k is whole steps: the same loads, places in LDS and sums as the kernel above, but a step is two
// halves, and while the products of one run, the operands of the next are read from LDS and a share of a later step's loads is issued; the step's
// one barrier stands between the halves.  Above, a step's loads, reads and products follow each other and only the second wavefront of a SIMD
// stands beside them.  (Past the last step that one is loaded again, so that every step waits alike.)  Bound by the weights' way from memory
// where an expert has few tiles, by LDS otherwise (its reads and loads are 1,792 cycles of a step, the products 1,024).
// us, the kernel above and this one, the first product and the second, everything from memory and the launch's 15 us included: 32 experts of
// 1,536 x 1,536, 8,000 pairs 101 and 101 to 97 and 97, 9,200 118 and 110 to 109 and 103, 16,384 159 and 163 to 145 and 151; of 2,560 x 3,584,
// 8,192 pairs 342 and 324 to 315 and 303; 8 of 4,096 x 14,336, 2,000 pairs 538 and 539 to 515 and 491.  Taken for every k of whole steps from three on.
template <typename TO>
__global__ void __launch_bounds__(8 * ZI_WAVE, 1)
moe_linear_halves_kernel(TO* __restrict__ out, int64_t ldo, const zi_bf16* __restrict__ x, int64_t ldx, const zi_bf16* __restrict__ w,
                         const int32_t* __restrict__ plan, const int32_t* __restrict__ source, int source_div, int N, int K, int act) {
    constexpr int RT = 8, CT = 4, ST = 3, WAVES = 8, RW = 4, XW = 2, WW = 4, PW = XW + WW, EARLY = PW / 2, PIECES = (2 * RT + 8 * CT) * ZI_WAVE;
    __shared__ __attribute__((aligned(16))) moe_u32x4_t all[ST * PIECES];
    const int blocks = (N + 64 * CT - 1) / (64 * CT), total = plan[0] * blocks, share = (total + MOE_XCDS - 1) / MOE_XCDS;
    const int at_share = blockIdx.x / MOE_XCDS, job = (int)(blockIdx.x % MOE_XCDS) * share + at_share;
    if (at_share >= share || job >= total) return;
    const int tile = job / blocks, n0 = job % blocks * 64 * CT;
    const int e = plan[1 + 3 * tile], r0 = plan[2 + 3 * tile], rows = plan[3 + 3 * tile];
    const int lane = threadIdx.x % ZI_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE);
    const int r = lane & 15, j = lane >> 4, wave_c = wave % 4, row0 = wave / 4 * RW * 16;
    const int rows_w = N - n0 < 64 * CT ? N - n0 : 64 * CT;
    const __amdgpu_buffer_rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc(const_cast<zi_bf16*>(w + ((int64_t)e * N + n0) * K), 0,
                                                                        rows_w * K * 2, 0x00020000);
    const zi_bf16* xrow[XW];
    int w_at[WW];
#pragma unroll
    for (int i = 0; i < XW; ++i) {
        const int q = (i * WAVES + wave) * 8 + lane / 8, rr = q < rows ? q : 0;
        xrow[i] = x + (int64_t)(source ? source[r0 + rr] / source_div : r0 + rr) * ldx + ((lane & 7) ^ ((q >> 1) & 7)) * 8;
    }
#pragma unroll
    for (int i = 0; i < WW; ++i) {
        const int q = (i * WAVES + wave) * 8 + lane / 8;
        w_at[i] = q < rows_w ? (q * K + ((lane & 7) ^ ((q >> 1) & 7)) * 8) * 2 : rows_w * K * 2;
    }
    const int steps = K / MOE_KB;
    auto issue = [&](int buf, int t, const int lo, const int hi) __attribute__((always_inline)) {
        const int k0 = (t < steps ? t : steps - 1) * MOE_KB;
#pragma unroll
        for (int i = lo; i < hi; ++i) {
            if (i < XW) moe_to_lds(xrow[i] + k0, all + buf + (i * WAVES + wave) * ZI_WAVE);
            else moe_to_lds<0>(wb, all + buf + (XW * WAVES + (i - XW) * WAVES + wave) * ZI_WAVE, w_at[i - XW] + k0 * 2);
        }
    };
    moe_f32x4_t acc[RW][CT];
#pragma unroll
    for (int t = 0; t < RW; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[t][c] = (moe_f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int sw = (r >> 1) & 7;
    moe_pack a0[CT], b0[RW], a1[CT], b1[RW];
    auto read = [&](int buf, const int half, moe_pack (&a)[CT], moe_pack (&b)[RW]) __attribute__((always_inline)) {
        const int at = buf + ((half * 4 + j) ^ sw);
#pragma unroll
        for (int m = 0; m < RW; ++m) b[m].u = all[at + (row0 + m * 16 + r) * 8];
#pragma unroll
        for (int c = 0; c < CT; ++c) a[c].u = all[at + (2 * RT * 8 + (wave_c * CT + c) * 16 + r) * 8];
    };
    auto multiply = [&](moe_pack (&a)[CT], moe_pack (&b)[RW]) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < RW; ++m)
#pragma unroll
            for (int c = 0; c < CT; ++c) acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c].b, b[m].b, acc[m][c], 0, 0, 0);
    };
    auto spread = [&](const int loads) __attribute__((always_inline)) {      // a read, a load, products between them
#pragma unroll
        for (int i = 0; i < RW + CT; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (i < loads) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < ST; ++i) {
        issue(i * PIECES, i, 0, i < ST - 1 ? PW : EARLY);
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("" ::: "memory");
    zi_wait_loads<(ST - 2) * PW + EARLY>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    int cur = 0, free = (ST - 1) * PIECES;
    read(0, 0, a0, b0);
    for (int t = 0; t < steps; ++t) {
        issue(free, t + ST - 1, EARLY, PW);
        read(cur, 1, a1, b1);
        multiply(a0, b0);
        spread(PW - EARLY);
        asm volatile("" ::: "memory");
        // the next step's loads have arrived, all wavefronts have read this step's
        zi_wait_loads<(ST - 2) * PW, true>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        free = cur;
        cur = cur == (ST - 1) * PIECES ? 0 : cur + PIECES;
        issue(free, t + ST, 0, EARLY);
        read(cur, 0, a0, b0);
        multiply(a1, b1);
        spread(EARLY);
    }
    zi_wait_loads<0>();       // (no load may arrive after the workgroup's LDS is another's)
    moe_store_tile<RW, CT>(out, ldo, acc, act, rows, r0, row0, n0 + wave_c * CT * 16, N, r, j);
}

extern "C" int zi_moe_linear(void* out, int out_dt, int64_t ldo, const void* x, int x_dt, int64_t ldx, const void* w,
                             int w_dt, const int32_t* plan, const int32_t* source, int source_div, int max_tiles,
                             int tile_rows, int N, int K, int act, hipStream_t stream) {
    ZI_REQUIRE(max_tiles >= 0 && max_tiles <= 65535 && N > 0 && K > 0 && ldx >= K && ldo >= N && source_div > 0,
               "moe_linear: bad sizes");
    ZI_REQUIRE(act == MOE_ACT_NONE || act == MOE_ACT_GELU_ERF, "moe_linear: unknown activation %d", act);
    if (max_tiles == 0) return 0;
    const dim3 grid((N + MOE_TN - 1) / MOE_TN, max_tiles, (tile_rows + MOE_TM - 1) / MOE_TM);
    const bool cores = x_dt == ZI_BF16 && w_dt == ZI_BF16 && K % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 16) == 0 &&
                       ((uintptr_t)w % 16) == 0 && (tile_rows == 16 || tile_rows == 32 || tile_rows == 64 || tile_rows == 128);
    // tiles of 64 rows (many rows an expert: prompts) are 256 columns wide, for a workgroup's reads of LDS: 8 operands for 16
    // products; smaller ones (decoded tokens) are bound by the weights' stream: narrow, so that every unit has several workgroups
    // (and what neither a buffer's offsets nor a grid of one dimension, 2^32 threads, reaches is left to the plain kernel)
    const int wide = cores ? (tile_rows < 64 ? 64 * (tile_rows / 16) : 256) : 64;       // columns of a workgroup
    const int64_t most = ((int64_t)N + wide - 1) / wide * max_tiles + MOE_XCDS;
    if (cores && K <= MOE_MAX_K && most * (tile_rows == 128 ? 512 : 256) < (1LL << 32)) {
#define ZI_MOE_CORES(RT, CT, ST, WR, TURNS)                                                                                                   \
    moe_linear_mfma_kernel<TO, RT, CT, ST, WR, TURNS><<<dim3((((N + 64 * CT - 1) / (64 * CT)) * (int64_t)max_tiles + MOE_XCDS - 1) / MOE_XCDS * \
                                                        MOE_XCDS), 256 * WR, 0, stream>>>((TO*)out, ldo, (const zi_bf16*)x, ldx,                      \
                                                                                       (const zi_bf16*)w, plan, source, source_div, N, K, act)
        ZI_DISPATCH_DTYPE(out_dt, TO, {
            const int turns = moe_turns(tile_rows, K);
            if (tile_rows == 16 && turns > 1) ZI_MOE_CORES(1, 1, 3, 1, 4);
            else if (tile_rows == 16) ZI_MOE_CORES(1, 1, 3, 1, 1);
            else if (tile_rows == 32 && turns > 1) ZI_MOE_CORES(2, 2, 3, 1, 2);
            else if (tile_rows == 32) ZI_MOE_CORES(2, 2, 3, 1, 1);
            else if (tile_rows == 64) ZI_MOE_CORES(4, 4, 2, 1, 1);
            else if (K % MOE_KB == 0 && K >= 3 * MOE_KB)
                moe_linear_halves_kernel<TO><<<dim3((((N + 255) / 256) * (int64_t)max_tiles + MOE_XCDS - 1) / MOE_XCDS * MOE_XCDS), 512, 0, stream>>>(
                    (TO*)out, ldo, (const zi_bf16*)x, ldx, (const zi_bf16*)w, plan, source, source_div, N, K, act);
            else if (turns > 1) ZI_MOE_CORES(8, 4, 3, 2, 2);
            else ZI_MOE_CORES(8, 4, 3, 2, 1);
        });
        return zi_check_launch("moe_linear");
    }
#undef ZI_MOE_CORES
    ZI_REQUIRE(cores || tile_rows == MOE_TM, "moe_linear: the plain product walks tiles of %d rows, not %d", MOE_TM, tile_rows);
    ZI_DISPATCH_DTYPE(x_dt, TX, ZI_DISPATCH_DTYPE(w_dt, TW, ZI_DISPATCH_DTYPE(out_dt, TO, {
        moe_linear_kernel<TX, TW, TO><<<grid, 256, 0, stream>>>((TO*)out, ldo, (const TX*)x, ldx, (const TW*)w, plan,
                                                                 source, source_div, N, K, act);
    })));
    return zi_check_launch("moe_linear");
}

__global__ void __launch_bounds__(256)
moe_combine_kernel(float* __restrict__ out, const float* __restrict__ y, const float* __restrict__ wt,
                   const int32_t* __restrict__ place_of, int top, int H) {
    const int64_t t = blockIdx.x;
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
        float acc = 0.f;
        for (int k = 0; k < top; ++k) acc += wt[t * top + k] * y[(int64_t)place_of[t * top + k] * H + c];
        out[t * H + c] = acc;
    }
}

// The same for widths that are whole 16-byte pieces: four columns a thread, a workgroup of one wavefront for 256 of a token's, the places
// and weights of four pairs and then their values asked for together.  A workgroup a token with a trip for every pair and 256 columns
// was a chain of 2 top x H / 256 trips: us, 32 tokens of 4 pairs x 1,536 5.3 to 2.9, of 8 x 3,584 32 to 5.0, 2,000 of 4 x 1,536 19.6 to 13.0.
__global__ void __launch_bounds__(ZI_WAVE)
moe_combine4_kernel(float* __restrict__ out, const float* __restrict__ y, const float* __restrict__ wt, const int32_t* __restrict__ place_of,
                    int top, int H) {
    const int64_t t = blockIdx.x;
    const int c = (blockIdx.y * ZI_WAVE + threadIdx.x) * 4;
    if (c >= H) return;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int k0 = 0; k0 < top; k0 += 4) {
        float g[4];
        float4 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int64_t at = t * top + (k0 + k < top ? k0 + k : top - 1);
            g[k] = wt[at];
            v[k] = *reinterpret_cast<const float4*>(y + (int64_t)place_of[at] * H + c);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (k0 + k >= top) break;
            acc.x += g[k] * v[k].x;
            acc.y += g[k] * v[k].y;
            acc.z += g[k] * v[k].z;
            acc.w += g[k] * v[k].w;
        }
    }
    *reinterpret_cast<float4*>(out + t * H + c) = acc;
}

extern "C" int zi_moe_combine(float* out, const float* y, const float* wt, const int32_t* place_of, int n, int top,
                              int hidden, hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && top > 0 && hidden > 0, "moe_combine: bad sizes");
    if (n == 0) return 0;
    if (hidden % 4 == 0 && ((uintptr_t)out | (uintptr_t)y) % 16 == 0 && hidden <= 65535 * 256)
        moe_combine4_kernel<<<dim3(n, (hidden + 4 * ZI_WAVE - 1) / (4 * ZI_WAVE)), ZI_WAVE, 0, stream>>>(out, y, wt, place_of, top, hidden);
    else
        moe_combine_kernel<<<n, 256, 0, stream>>>(out, y, wt, place_of, top, hidden);
    return zi_check_launch("moe_combine");
}

// ---- a router of independent scores --------------------------------------------------------------------------
// s = sigmoid(z); the `top` experts with the largest s are chosen (the lowest index among equals); their weights are
// the scores themselves, not renormalised.  z [n][ld] float32 of which the first E columns are the experts'.
template <int PER>
__global__ void __launch_bounds__(256)
moe_route_sigmoid_kernel(int32_t* __restrict__ idx, float* __restrict__ wt, const float* __restrict__ z, int64_t ld,
                         int n, int E, int top) {
    const int lane = threadIdx.x % ZI_WAVE;
    const int t = blockIdx.x * (blockDim.x / ZI_WAVE) + threadIdx.x / ZI_WAVE;
    if (t >= n) return;
    float choice[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + i * ZI_WAVE;
        choice[i] = e < E ? 1.f / (1.f + expf(-z[(int64_t)t * ld + e])) : -INFINITY;
    }
    for (int k = 0; k < top; ++k) {
        float best = -INFINITY;
        int best_e = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = lane + i * ZI_WAVE;
            if (e < E && (choice[i] > best || (choice[i] == best && e < best_e))) {
                best = choice[i];
                best_e = e;
            }
        }
#pragma unroll
        for (int o = ZI_WAVE / 2; o > 0; o >>= 1) {
            const float ob = __shfl_xor(best, o, ZI_WAVE);
            const int oe = __shfl_xor(best_e, o, ZI_WAVE);
            if (ob > best || (ob == best && oe < best_e)) {
                best = ob;
                best_e = oe;
            }
        }
        if (lane == 0) {
            idx[(int64_t)t * top + k] = best_e;
            wt[(int64_t)t * top + k] = best;
        }
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + i * ZI_WAVE == best_e) choice[i] = -INFINITY;
    }
}

extern "C" int zi_moe_route_sigmoid(int32_t* idx, float* wt, const float* z, int64_t ld, int n, int experts, int top,
                                    hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && experts > 0 && experts <= MOE_MAX_EXPERTS && top > 0 && top <= experts && ld >= experts,
               "moe_route_sigmoid: bad sizes (experts %d, top %d; at most %d experts)", experts, top, MOE_MAX_EXPERTS);
    if (n == 0) return 0;
    const int blocks = (n + 3) / 4;
#define ZI_MOE_ROUTE(PER) moe_route_sigmoid_kernel<PER><<<blocks, 256, 0, stream>>>(idx, wt, z, ld, n, experts, top)
    if (experts <= ZI_WAVE) ZI_MOE_ROUTE(1);
    else if (experts <= 2 * ZI_WAVE) ZI_MOE_ROUTE(2);
    else if (experts <= 4 * ZI_WAVE) ZI_MOE_ROUTE(4);
    else ZI_MOE_ROUTE(MOE_PER_LANE);
#undef ZI_MOE_ROUTE
    return zi_check_launch("moe_route_sigmoid");
}

// The gated middle of experts whose INPUT carries the routing weight: an expert is linear up to its activation, so
// gate (w x) = w gate(x) and up (w x) = w up(x): out = silu(w g) * (w u) for row r of the grouped pairs, w the weight
// of the pair that stands at place r (wt[order[r]]).  gu [pairs][2 ff] float32 (gate, then up).
template <typename TO>
__global__ void __launch_bounds__(256)
moe_weighted_glu_kernel(TO* __restrict__ out, int64_t ldo, const float* __restrict__ gu, int64_t ld,
                        const float* __restrict__ wt, const int32_t* __restrict__ order, int pairs, int ff) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)pairs * ff) return;
    const int64_t r = i / ff, c = i % ff;
    const float w = wt[order[r]];
    const float g = w * gu[r * ld + c], u = w * gu[r * ld + ff + c];
    zi_store(out + r * ldo + c, g / (1.f + expf(-g)) * u);
}

extern "C" int zi_moe_weighted_glu(void* out, int out_dt, int64_t ldo, const float* gu, int64_t ld, const float* wt,
                                   const int32_t* order, int pairs, int ff, hipStream_t stream) {
    ZI_REQUIRE(pairs >= 0 && ff > 0 && ld >= 2 * (int64_t)ff && ldo >= ff, "moe_weighted_glu: bad sizes");
    if (pairs == 0) return 0;
    const int64_t total = (int64_t)pairs * ff;
    ZI_DISPATCH_DTYPE(out_dt, TO, {
        moe_weighted_glu_kernel<TO><<<(unsigned)((total + 255) / 256), 256, 0, stream>>>((TO*)out, ldo, gu, ld, wt, order,
                                                                                         pairs, ff);
    });
    return zi_check_launch("moe_weighted_glu");
}

// out [n][H] = sum over a token's `top` pairs of y[place_of[pair]] (each counts once: the weight went into the
// expert's input) + sigmoid(gate[t * ld_gate]) * shared[t], where shared is the sum of `splits` float32 terms
// (`split_stride` apart) or null.
__global__ void __launch_bounds__(256)
moe_sum_shared_kernel(float* __restrict__ out, const float* __restrict__ y, const int32_t* __restrict__ place_of,
                      const float* __restrict__ shared, int splits, int64_t split_stride, const float* __restrict__ gate,
                      int64_t ld_gate, int top, int H) {
    const int64_t t = blockIdx.x;
    const float gs = (shared && gate) ? 1.f / (1.f + expf(-gate[t * ld_gate])) : 1.f;
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
        float acc = 0.f;
        for (int k = 0; k < top; ++k) acc += y[(int64_t)place_of[t * top + k] * H + c];
        if (shared) {
            float sv = shared[t * H + c];
            for (int s = 1; s < splits; ++s) sv += shared[s * split_stride + t * H + c];
            acc += gs * sv;
        }
        out[t * H + c] = acc;
    }
}

extern "C" int zi_moe_sum_shared(float* out, const float* y, const int32_t* place_of, const float* shared, int splits,
                                 int64_t split_stride, const float* gate, int64_t ld_gate, int n, int top, int hidden,
                                 hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && top > 0 && hidden > 0 && splits >= 1, "moe_sum_shared: bad sizes");
    if (n == 0) return 0;
    moe_sum_shared_kernel<<<n, 256, 0, stream>>>(out, y, place_of, shared, splits, split_stride, gate, ld_gate, top, hidden);
    return zi_check_launch("moe_sum_shared");
}
