// out[M,N] = x[M,K] . w[N,K]^T (+ bias) for 1..256 rows of x: the decode-time products, bound by the one
// pass over the weights (the entry points are in gemm_skinny.hip).  Up to 64 rows (and for rows of x or w too far apart for
// offsets of 31 bits) gemm_mid_kernel, from 65 on gemm_wide_kernel below it.
//
// A workgroup of gemm_mid_kernel, four to eight wavefronts, owns 16 weight rows a wavefront and a range of k.  It walks its
// k-blocks of 128: the block's slice of x (up to 64 rows x 128 values) is staged in LDS once for the four
// wavefronts, each wavefront reads its own 16 weight rows from memory as whole cache lines, turns them
// into matrix-core operands through a piece of LDS of its own (v_mfma_f32_16x16x32_bf16, float32
// accumulation) and keeps the sums of its 16 x M outputs in registers, so nothing is added across
// wavefronts.  The next two blocks' weights and x travel while the current one is worked on (a ring of
// three register buffers; loads are issued without branches so that they stay in flight).  The k dimension is cut over gridDim.y workgroups when N alone gives too few of them; those
// leave float32 partial sums [split][M][N] that the consumer adds in rising order.  The cut depends on N
// and K only.  Epilogues as in the few-rows kernel: plain (bias), partial sums, SwiGLU over gate/up rows
// interleaved in blocks of 8, an activation of every output.
#include "zi_common.h"
#include "zi_activation.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 gm_bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float gm_f32x4_t;
// 16 bytes as a native vector: copies of the struct uint4 are memcpys to the compiler, and an array of
// them that is only copied stays in memory instead of registers
typedef __attribute__((ext_vector_type(4))) unsigned gm_u32x4_t;

#define GM_MIN_WAVES 4      // wavefronts of a workgroup: 4 .. 8, 16 weight rows each
#define GM_MAX_WAVES 8
#define GM_KB 128
#define GM_XS GM_KB         // LDS row stride, in elements: rows of 16 pieces of 16 bytes, piece c of row r at place c xor (r mod 16)

#define GM_MODE_PLAIN 0
#define GM_MODE_PARTIAL 1
#define GM_MODE_SWIGLU 2
#define GM_MODE_CLAMPED 3      // like SWIGLU, with biases: g = min(gate, limit), u = clamp(up, -limit, limit), g sigmoid(1.702 g) (u + 1)
#define GM_MODE_ACT 4          // + the code of an activation (zi_activate_value), of the sum and the bias

union gm_pack {
    gm_u32x4_t u;
    gm_bf16x8_t b;
};

// v where `keep` holds, else zeros, by arithmetic: after a select the compiler may move the load that
// made v under a branch, and wait for it there.
__device__ __forceinline__ gm_u32x4_t gm_keep(gm_u32x4_t v, bool keep) {
    const unsigned mask = 0u - (unsigned)keep;
    return v & mask;
}

// What a wavefront does with its sums: C[n = n0 + j*4 + e][m = m0 + t*16 + r] in acc[t][e].
template <int MT>
__device__ __forceinline__ void gm_epilogue(const gm_f32x4_t (&acc)[MT], void* __restrict__ out, int mode, int out_f32,
                                            const zi_bf16* __restrict__ bias_in, int M, int N, int64_t ldo, int split,
                                            int n0, int r, int j, int vec_out, float limit, int m0 = 0) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        gm_f32x4_t s = acc[t];
        const zi_bf16* bias = bias_in;
        const int m = m0 + t * 16 + r;
        if (mode == GM_MODE_SWIGLU || mode == GM_MODE_CLAMPED) {
            if (mode == GM_MODE_CLAMPED && bias && n0 < N) {
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] += zi_load(bias + n0 + j * 4 + e);
            }
            // lanes j = 0,1 hold gate rows j*4 + e, lanes j = 2,3 the up rows of the same columns: they trade halves, so that each
            // lane makes two columns (nothing overlaps the exponentials at a product's end: 19.7 us for gate/up of 80 rows at the
            // 1.5B sizes, 21.5 when lanes 0, 1 made four)
            const bool low = j < 2;
            const float t0 = __shfl_xor(low ? s[2] : s[0], 32, ZI_WAVE), t1 = __shfl_xor(low ? s[3] : s[1], 32, ZI_WAVE);
            if (m >= M || n0 >= N) continue;
            const int col = (n0 / 16) * 8 + (j & 1) * 4 + (low ? 0 : 2);     // N / 2 columns of output; N % 16 == 0
            float act[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float gate = low ? s[e] : e ? t1 : t0, other = low ? (e ? t1 : t0) : s[2 + e];
                if (mode == GM_MODE_SWIGLU) {
                    act[e] = other * (gate / (1.f + expf(-gate)));
                } else {
                    const float g = fminf(gate, limit), u = fminf(fmaxf(other, -limit), limit);
                    act[e] = g / (1.f + expf(-1.702f * g)) * (u + 1.f);
                }
            }
            zi_bf16* dst = (zi_bf16*)out + (int64_t)m * ldo + col;
            if (vec_out) {
                *reinterpret_cast<uint32_t*>(dst) = zi_pack_bf16x2(act[0], act[1]);
            } else {
#pragma unroll
                for (int e = 0; e < 2; ++e) zi_store(dst + e, act[e]);
            }
            continue;
        }
        if (m >= M) continue;
        const int nb = n0 + j * 4;
        if (mode >= GM_MODE_ACT) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                s[e] = zi_activate_value<true, false>(s[e] + (bias && nb + e < N ? zi_load(bias + nb + e) : 0.f), mode - GM_MODE_ACT);
            bias = nullptr;
        }
        if (nb + 3 < N && vec_out) {
            if (mode == GM_MODE_PARTIAL) {
                if (bias && split == 0) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[e] += zi_load(bias + nb + e);
                }
                *reinterpret_cast<gm_f32x4_t*>((float*)out + ((int64_t)split * M + m) * N + nb) = s;
            } else {
                if (bias) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[e] += zi_load(bias + nb + e);
                }
                if (out_f32) {
                    *reinterpret_cast<gm_f32x4_t*>((float*)out + (int64_t)m * ldo + nb) = s;
                } else {
                    uint2 pk;
                    pk.x = zi_pack_bf16x2(s[0], s[1]);
                    pk.y = zi_pack_bf16x2(s[2], s[3]);
                    *reinterpret_cast<uint2*>((zi_bf16*)out + (int64_t)m * ldo + nb) = pk;
                }
            }
            continue;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = nb + e;
            if (n >= N) continue;
            if (mode == GM_MODE_PARTIAL) {
                ((float*)out)[((int64_t)split * M + m) * N + n] = s[e] + ((bias && split == 0) ? zi_load(bias + n) : 0.f);
            } else {
                const float v = s[e] + (bias ? zi_load(bias + n) : 0.f);
                if (out_f32) ((float*)out)[(int64_t)m * ldo + n] = v;
                else zi_store((zi_bf16*)out + (int64_t)m * ldo + n, v);
            }
        }
    }
}

// APART: rows blockIdx.z * 16 MT .. of x.
template <int MT, int GM_RING, int GM_WAVES, bool APART = false>
__global__ void __launch_bounds__(GM_WAVES* ZI_WAVE)
gemm_mid_kernel(void* __restrict__ out, int mode, int out_f32, const zi_bf16* __restrict__ x,
                const zi_bf16* __restrict__ w, const zi_bf16* __restrict__ bias, int M, int N, int K, int64_t ldx,
                int64_t ldw, int64_t ldo, int kb_per_split, int vec_out, float limit) {
    __shared__ __attribute__((aligned(16))) uint16_t xs[2][MT * 16 * GM_XS];
    __shared__ __attribute__((aligned(16))) uint16_t wt[GM_WAVES][16 * GM_XS];   // a wavefront's weight tile
    const int tid = threadIdx.x, lane = tid & (ZI_WAVE - 1), wave = tid / ZI_WAVE;
    const int r = lane & 15, j = lane >> 4;
    const int split = blockIdx.y;
    const int kb_total = (K + GM_KB - 1) / GM_KB;
    const int kb_lo = split * kb_per_split;
    const int kb_hi = (kb_lo + kb_per_split < kb_total) ? kb_lo + kb_per_split : kb_total;
    const int n0 = (blockIdx.x * GM_WAVES + wave) * 16, m0 = APART ? blockIdx.z * MT * 16 : 0;
    // Weights are read as whole cache lines: a load instruction takes 4 rows x 256 bytes (lane l: row
    // l / 16 of the four, 16-byte piece l % 16), four instructions a tile of 16 rows x 128 values.
    // Loads in the matrix-core operand layout (16 rows x 64 bytes an instruction) were measured a fifth
    // slower.  The tile is turned into that layout through a piece of LDS that the wavefront owns.
    const int wq = lane & 15;
    const zi_bf16* wrow[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int n = n0 + c * 4 + j;
        wrow[c] = w + (int64_t)(n < N ? n : N - 1) * ldw;
    }
    // LDS rows are not padded but swizzled (16-byte reads in operand order then run at the full LDS rate)
    uint16_t* const wt_w = &wt[wave][0];

    // what this thread stages of a block's x slice: XP pieces of 16 bytes (rows srow[p], piece spc).  The slice's
    // MT * 256 pieces are dealt out over all the workgroup's threads, a row of 16 pieces to 16 neighbours; the
    // last round may pass the slice's end (its loads repeat the last row and go nowhere).
    constexpr int THREADS = GM_WAVES * ZI_WAVE, XP = (MT * 256 + THREADS - 1) / THREADS;
    const int spc = tid % 16;
    int srow[XP];
#pragma unroll
    for (int p = 0; p < XP; ++p) srow[p] = p * (THREADS / 16) + tid / 16;
    // the weights of GM_RING k-blocks are in flight at once (a ring of register buffers); the x slice of
    // the next block is fetched while this one is worked on
    gm_u32x4_t ring[GM_RING][4], xring[GM_RING][XP];
    // Loads are issued without branches and their results are not touched before the products need
    // them: only then does the compiler let several blocks' loads stay in flight.  Addresses are
    // clamped into the matrices.  Rows of x past M repeat the last row and give outputs that nobody
    // stores; columns past K would count the last eight twice, so the weights are zeroed there, when
    // they are used.  A block's x is requested before its weights: loads return in order, and x, which
    // comes from the cache and is wanted a step earlier, must not queue behind weights from memory.
    const zi_bf16* xrow[XP];
#pragma unroll
    for (int p = 0; p < XP; ++p) xrow[p] = x + (int64_t)(m0 + srow[p] < M ? m0 + srow[p] : M - 1) * ldx;
    auto fetch = [&](const int slot, int kb) __attribute__((always_inline)) {
        const int k0 = kb * GM_KB;
        const int kx = k0 + spc * 8 < K ? k0 + spc * 8 : K - 8;
#pragma unroll
        for (int p = 0; p < XP; ++p) xring[slot][p] = *reinterpret_cast<const gm_u32x4_t*>(xrow[p] + kx);
        const int k = k0 + wq * 8;
        // a weight is read once a step and the weights of a step are many times the caches: non-temporal loads keep
        // them out of L2 (decode at batch 8, 1.5B sizes: 5,403 to 5,518 tok/s)
#pragma unroll
        for (int c = 0; c < 4; ++c) ring[slot][c] = __builtin_nontemporal_load(reinterpret_cast<const gm_u32x4_t*>(wrow[c] + (k < K ? k : K - 8)));
    };
    auto stash = [&](const int slot, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < XP; ++p)
            if ((p + 1) * (THREADS / 16) <= MT * 16 || srow[p] < MT * 16)
                *reinterpret_cast<gm_u32x4_t*>(&xs[b][srow[p] * GM_XS + (spc ^ (srow[p] & 15)) * 8]) = xring[slot][p];
    };
    gm_f32x4_t acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = gm_f32x4_t{0.f, 0.f, 0.f, 0.f};

    // Blocks kb_lo .. kb_lo + GM_RING - 2 are requested up front; block kb's x goes to LDS one step
    // before it is used, GM_RING - 2 steps after it was requested.  Block kb lives in ring slot
    // (kb - kb_lo) % GM_RING.  The compiler counts how many loads may stay in flight at each use only
    // in straight-line code; behind a branch that may or may not have issued loads it waits for all of
    // them.  So the walk is cut into pieces without such branches: a steady loop of GM_RING steps that
    // all request a block, and one of GM_RING straight-line endings, chosen by how many blocks are
    // left to request.
    int cur = 0;
    auto step = [&](const int slot, int kb, const bool request) __attribute__((always_inline)) {
        if (request) fetch((slot + GM_RING - 1) % GM_RING, kb + GM_RING - 1);
        // all of the block's x operands are read from LDS before the first product: the reads' latency
        // is paid once, not once per product
        // the weight tile goes through the wavefront's LDS piece (zeros past K: the last block only);
        // LDS serves a wavefront's instructions in order, so no barrier stands between put and get
#pragma unroll
        for (int c = 0; c < 4; ++c)
            *reinterpret_cast<gm_u32x4_t*>(wt_w + (c * 4 + j) * GM_XS + (wq ^ (c * 4 + j)) * 8) =
                gm_keep(ring[slot][c], kb * GM_KB + wq * 8 < K);
        gm_pack bb[4][MT], a[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int t = 0; t < MT; ++t)
                bb[c][t].u = *reinterpret_cast<const gm_u32x4_t*>(&xs[cur][(t * 16 + r) * GM_XS + ((c * 4 + j) ^ r) * 8]);
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c].u = *reinterpret_cast<const gm_u32x4_t*>(wt_w + r * GM_XS + ((c * 4 + j) ^ r) * 8);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int t = 0; t < MT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c].b, bb[c][t].b, acc[t], 0, 0, 0);
        stash((slot + 1) % GM_RING, cur ^ 1);    // after the last block: something nobody reads
        __syncthreads();
        cur ^= 1;
    };
    // the ending for `left` blocks still to request: left + GM_RING - 1 blocks to work on
    auto ending = [&](auto left_c, int kb0) __attribute__((always_inline)) {
        constexpr int LEFT = decltype(left_c)::value;
#pragma unroll
        for (int i = 0; i < LEFT + GM_RING - 1; ++i) step(i % GM_RING, kb0 + i, i < LEFT);
    };
#pragma unroll
    for (int b = 0; b < GM_RING - 1; ++b) fetch(b, kb_lo + b < kb_hi ? kb_lo + b : kb_hi - 1);
    stash(0, 0);
    __syncthreads();
    int kb0 = kb_lo;
    for (; kb0 + 2 * GM_RING - 1 <= kb_hi; kb0 += GM_RING) {
#pragma unroll
        for (int b = 0; b < GM_RING; ++b) step(b, kb0 + b, true);
    }
    const int left = kb_hi - kb0 - (GM_RING - 1);    // < 0: fewer blocks than the ring requests up front
    if (left < 0) {
#pragma unroll
        for (int b = 0; b < GM_RING - 1; ++b)
            if (kb0 + b < kb_hi) step(b, kb0 + b, false);
    } else {
        static_assert(GM_RING >= 2 && GM_RING <= 4, "one ending per residue");
        switch (left) {
            case 0: ending(std::integral_constant<int, 0>{}, kb0); break;
            case 1: ending(std::integral_constant<int, 1>{}, kb0); break;
            case 2: if (GM_RING > 2) ending(std::integral_constant<int, 2>{}, kb0); break;
            default: if (GM_RING > 3) ending(std::integral_constant<int, 3>{}, kb0); break;
        }
    }
    gm_epilogue<MT>(acc, out, mode, out_f32, bias, M, N, ldo, split, n0, r, j, vec_out, limit, m0);
}

// The same product for 65 .. 256 rows of x (MT = 5 .. 16 tiles of 16 rows): one pass over the weights where two launches of the
// kernel above would make two.  With that many rows the reads of x from LDS bind a workgroup whose wavefronts each take all of
// them for 16 weight rows (16.3 us for a down product of 27 MB), so here wavefronts share the rows of x: four with 32 rows and all
// of the workgroup's NT x 16 weight rows, 2 + NT operands read for 2 NT products, or eight with half of the weight rows each.  Both operands go straight into LDS
// (global_load_lds_dwordx4, 1 KB an instruction, rows of 128 bytes with piece c of row q at place c xor (q / 2 mod 8)), k in
// steps of 64 through four buffers, three steps on their way while one is worked on (six buffers were no faster); every wavefront issues as many loads a step
// as every other, so that each can wait for its own by count before the step's one barrier.  The cut, the order of the
// sums and the epilogues are the kernel's above: a row's result does not depend on which of the two kernels makes it.
// Measured at 128 rows, weights from memory, against wavefronts of 16 weight rows: 1.5B sizes down 16.3 to 11.9 us, q/k/v 7.3 to
// 6.5, output 7.4 to 6.4; 7B sizes down 53 to 36, q/k/v 20 to 13.5, output 16 to 12.8.  With the SwiGLU epilogue 20.5 us at 128 rows
// and 18.0 at 80 (1.5B gate/up), where the library's product and the activation's launch take 27.2 and 22.8 together (for which
// products it pays: zi_gemm_skinny_swiglu_pays).  A step's instructions were what bound it first: loads whose addresses cost the
// lanes nothing took 80 rows of the 1.5B gate/up from 20.6 to 18.0 us.
//
// Two wavefronts a SIMD cover each other's waits, but read more of LDS for a product than four wavefronts of 32 rows of x and all weight
// rows, so up to 128 rows eight are for a short k and a long one keeps the four (gw_eight_most).  us at 65 and 128 rows, four to eight:
// 2,048 x 1,536 5.9 to 5.2 and 6.7 to 6.2, 4,608 x 3,584 12.9 to 11.2 and 14.6 to 13.3, gate/up of 8,960 columns x 1,536 at 128 rows 21.6 to
// 19.8, of 3,072 x 1,024 10.9 to 9.3 and 12.1 to 11.0; the other way round 8,192 x 8,192 31.6 to 36.8 and 40.8 to 42.0, 12,264 x 14,712 99 to
// 104 and 110 to 141, 16,384 x 4,096 30.9 to 34.8 at 65.
//
// Beyond 128 rows eight wavefronts, each with a quarter of the rows of x (gate/up at the 7B sizes, 10
// weight tiles, 160 rows 63 us; four wavefronts two by two 66, five of 32 rows each 71).  The cut is one of its own
// (zi_gemm_many_plan); with LDS for four buffers of a step gone, three.  Weights from memory, us at 160 and 256 rows, against the
// library's first proposal: 7B sizes q/k/v 15 and 18 against 25 and 35, output 14 and 17 against 25 and 20, down 37 and 43 against
// 106 and 125 (a kernel of 32 weight rows a wavefront, 32 x 32 instructions, took 59 at 160 rows and is gone), gate/up with
// the activation 63 and 79 against 83 and 88 with its launch; 1.5B gate/up 24 and 27 against 30 and 34; 32B q/k/v 24 and 30 against
// 38 and 52, output 20 and 25 against 37 and 50, down 60 and 73 against 194 and 267.  Bound by a step's barrier and LDS
// reads: 3.4 to 5.4 TB/s of weights where ten tiles share a slice of x (18,944 columns x 3,584 63 and 79 us, 20,480 x 7,168 108 and 145).
#define GW_KB 64

#define GW_STAGES 4
#define GW_MID_ROWS 128      // up to here the cut of the kernel above, beyond it zi_gemm_many_plan's
#define GW_MAX_TILES 10      // 16 weight rows each, of a workgroup

// Rows further apart than this (in elements; 128 of them then span 2^30 bytes) are past what the kernel's 31-bit offsets reach:
// they go to the kernel above, whose addresses have 64 bits, 64 rows a workgroup.
#define GW_MAX_LD (1 << 22)

// 16 bytes a lane from a buffer into LDS, lane after lane from `to` on; what lies past the buffer's end gives zeros.
template <int AUX>
__device__ __forceinline__ void gw_to_lds(__amdgpu_buffer_rsrc_t from, gm_u32x4_t* to, int lane_at) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host's pass knows loads of this size for no target)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(from, to, 16, lane_at, 0, 0, AUX);
#endif
}

// Column k (a multiple of 8) and all that follows of `rows` rows as a buffer: it ends with the last row's K values, and past
// the last column it holds nothing.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gw_rows(const zi_bf16* base, int64_t ld, int rows, int K, int k) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<zi_bf16*>(base + k), 0, k < K ? (int)(((rows - 1) * ld + K - k) * 2) : 0, 0x00020000);
}

// WN: the wavefronts along the weight rows, four times as many in all.
template <int MT, int NT, int WN>
struct gw_shape {
    static constexpr int WM = 4, WAVES = WM * WN;                                 // wavefronts along the rows of x, of a workgroup
    static constexpr int MW = MT <= 8 ? 2 : (MT + 3) / 4, NW = (NT + WN - 1) / WN;       // a wavefront's tiles
    static constexpr int STAGES = (MT + NT) * 8 + 1 <= 160 ? GW_STAGES : 3;       // 2 KB a tile and buffer in 160 KB of LDS
};

template <int MT, int NT, int WN>
__global__ void __launch_bounds__((gw_shape<MT, NT, WN>::WAVES) * ZI_WAVE)
gemm_wide_kernel(void* __restrict__ out, int mode, int out_f32, const zi_bf16* __restrict__ x,
                 const zi_bf16* __restrict__ w, const zi_bf16* __restrict__ bias, int M, int N, int K, int64_t ldx,
                 int64_t ldw, int64_t ldo, int kb_per_split, int vec_out, float limit) {
    typedef gw_shape<MT, NT, WN> S;
    constexpr int WAVES = S::WAVES, STAGES = S::STAGES, MW = S::MW, NW = S::NW;
    constexpr int XI = 2 * MT, LOADS = XI + 2 * NT, PW = (LOADS + WAVES - 1) / WAVES;       // 1 KB loads of x, of a step; a wavefront's share
    constexpr int PIECES = LOADS * ZI_WAVE;
    static_assert(STAGES * LOADS + 1 <= 160, "the buffers fit into LDS");
    // (arrays of their own, so that the compiler can tell a buffer that is read from those that loads are on their way to)
    __shared__ __attribute__((aligned(16))) gm_u32x4_t s0[PIECES], s1[PIECES], s2[PIECES], s3[STAGES > 3 ? PIECES : 1], spare[ZI_WAVE];       // (spare: where loads go that nobody needs)
    const int tid = threadIdx.x, lane = tid & (ZI_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / ZI_WAVE);
    const int r = lane & 15, j = lane >> 4;
    const int split = blockIdx.y;
    const int k_lo = split * kb_per_split * GM_KB, k_hi = k_lo + kb_per_split * GM_KB < K ? k_lo + kb_per_split * GM_KB : K;
    const int steps = (k_hi - k_lo + GW_KB - 1) / GW_KB;
    const int n0 = blockIdx.x * NT * 16;
    // Load i of a step takes 8 rows: lane l row l / 8 of them, the piece that belongs at place l % 8.  A step's place along k is in
    // the buffers it loads from (scalar registers), so that a load costs no arithmetic of the lanes (with one wavefront a SIMD every
    // instruction counts) and every address is checked by the lane's offset alone, the one part of an address that the buffer's
    // range is sure to be held against.
    // Rows past M or N are past the buffers' ends and zero; columns past K are the next row's, and masked when they are used.
    const int rows_w = N - n0 < NT * 16 ? N - n0 : NT * 16;
    const zi_bf16* const w0 = w + (int64_t)n0 * ldw;
    int lane_at[PW];
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int L = i * WAVES + wave;
        const int q = (L < XI ? L : L - XI) * 8 + lane / 8;
        lane_at[i] = (int)(q * (L < XI ? ldx : ldw) * 2) + ((lane & 7) ^ ((q >> 1) & 7)) * 16;
    }
    auto issue = [&](gm_u32x4_t* buf, int t) {
        const int k = t < steps ? k_lo + t * GW_KB : K;       // (steps past the end: nothing is fetched)
        const __amdgpu_buffer_rsrc_t xb = gw_rows(x, ldx, M, K, k), wb = gw_rows(w0, ldw, rows_w, K, k);
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            const int L = i * WAVES + wave;
            gm_u32x4_t* to = L < LOADS ? buf + L * ZI_WAVE : spare;
            if (i * WAVES + WAVES - 1 < XI) gw_to_lds<0>(xb, to, lane_at[i]);
            else if (i * WAVES >= XI) gw_to_lds<2>(wb, to, lane_at[i]);       // weights are read once: past L2
            else gw_to_lds<0>(L < XI ? xb : wb, to, lane_at[i]);
        }
    };
    gm_f32x4_t acc[NW][MW];
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
        for (int t = 0; t < MW; ++t) acc[n][t] = gm_f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int sw = (r >> 1) & 7;
    const int m_tile = wave % S::WM * MW, n_tile = wave / S::WM * NW;
    int tile_at[MW], wtile_at[NW];         // (past the rows: the last tile again, not stored)
#pragma unroll
    for (int m = 0; m < MW; ++m) tile_at[m] = ((m_tile + m < MT ? m_tile + m : MT - 1) * 16 + r) * 8;
#pragma unroll
    for (int n = 0; n < NW; ++n) wtile_at[n] = XI * ZI_WAVE + ((n_tile + n < NT ? n_tile + n : NT - 1) * 16 + r) * 8;
    auto step = [&](const gm_u32x4_t* buf, gm_u32x4_t* free, int t) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        zi_wait_loads<(STAGES - 2) * PW>();
        __builtin_amdgcn_s_barrier();          // all wavefronts' loads of the step are there, and all are done with `free`
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        issue(free, t + STAGES - 1);
        __builtin_amdgcn_sched_barrier(0);
        if (t >= steps) return;
        // all of the step's operands are asked for before the first product: their way is paid once
        gm_pack a[2][NW], b[2][MW];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int at = (kk * 4 + j) ^ sw;
#pragma unroll
            for (int m = 0; m < MW; ++m) b[kk][m].u = buf[tile_at[m] + at];
#pragma unroll
            for (int n = 0; n < NW; ++n) a[kk][n].u = buf[wtile_at[n] + at];
        }
        const int left = K - (k_lo + t * GW_KB);
        if (left < GW_KB) {
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
                for (int n = 0; n < NW; ++n) a[kk][n].u = gm_keep(a[kk][n].u, kk * 32 + j * 8 < left);
#pragma unroll
                for (int m = 0; m < MW; ++m) b[kk][m].u = gm_keep(b[kk][m].u, kk * 32 + j * 8 < left);
            }
        }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int n = 0; n < NW; ++n)
#pragma unroll
                for (int m = 0; m < MW; ++m)
                    acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kk][n].b, b[kk][m].b, acc[n][m], 0, 0, 0);
    };
    issue(s0, 0);
    __builtin_amdgcn_sched_barrier(0);
    issue(s1, 1);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (STAGES == 4) {
        issue(s2, 2);
        __builtin_amdgcn_sched_barrier(0);
        for (int t = 0; t < steps; t += 4) {
            step(s0, s3, t);
            step(s1, s0, t + 1);
            step(s2, s1, t + 2);
            step(s3, s2, t + 3);
        }
    } else {
        for (int t = 0; t < steps; t += 3) {
            step(s0, s2, t);
            step(s1, s0, t + 1);
            step(s2, s1, t + 2);
        }
    }
    zi_wait_loads<0>();       // (no load may arrive after the workgroup's LDS is another's)
#pragma unroll
    for (int n = 0; n < NW; ++n)
        if (n_tile + n < NT)
            gm_epilogue<MW>(acc[n], out, mode, out_f32, bias, M, N, ldo, split, n0 + (n_tile + n) * 16, r, j, vec_out, limit, m_tile * 16);
}

// How the product with a weight matrix [N, K] is cut: wavefronts a workgroup (16 weight rows each), splits
// of k over workgroups (at most 16: what the consumers add at once) and k-blocks per split.  A function of
// N and K alone.
//
// A compute unit works through the wavefronts it is given at a fixed rate (measured: 280 workgroups of
// four wavefronts on 256 compute units take almost twice as long as 140, because 24 units hold two), so
// what counts is the most work any unit gets when workgroups are dealt out in turn: rounds = ceil(workgroups
// / units), each of `waves * k-blocks` wavefront-blocks plus a start-up worth about ten of them.  Among
// the cuts the cheapest by that measure is taken, then the one with the fewest splits, then the fewest
// wavefronts.  A matrix with many times more rows than that keeps the units busy whatever the cut (its
// workgroups follow each other, two to a unit): four wavefronts, no split (measured on the 151,936 rows of
// the output head: 108 against 119 us with eight).  `whole`: the cheapest without a split.  Returns the cost.
int64_t zi_gemm_mid_plan(int N, int K, int whole, int* splits, int* kb_per_split, int* waves) {
    const int tiles = (N + 15) / 16;
    const int kb_total = (K + GM_KB - 1) / GM_KB;
    int64_t best_cost = -1;
    int best_s = 1, best_w = GM_MIN_WAVES, best_per = kb_total;
    const int cus = zi_compute_units();          // the cut is balanced over the device's compute units
    const bool many = (tiles + GM_MIN_WAVES - 1) / GM_MIN_WAVES > 4 * cus;
    for (int w = GM_MIN_WAVES; w <= (many ? GM_MIN_WAVES : GM_MAX_WAVES); ++w) {
        const int groups = (tiles + w - 1) / w;
        for (int s0 = 1; s0 <= (many || whole ? 1 : 16) && s0 <= (kb_total > 1 ? kb_total / 2 : 1); ++s0) {
            const int per = (kb_total + s0 - 1) / s0;
            const int s = (kb_total + per - 1) / per;
            if (s != s0) continue;      // the same cut under another name
            const int64_t wgs = (int64_t)groups * s;
            const int64_t rounds = (wgs + cus - 1) / cus;
            const int64_t cost = rounds * ((int64_t)w * per + 10);
            if (best_cost < 0 || cost < best_cost || (cost == best_cost && s < best_s)) {
                best_cost = cost; best_s = s; best_w = w; best_per = per;
            }
        }
    }
    *splits = best_s;
    *kb_per_split = best_per;
    *waves = best_w;
    return best_cost;
}

// How the product of 129 .. 256 rows is cut: weight tiles of 16 rows a workgroup, splits of k over workgroups (at most 16) and blocks of
// 128 per split; a function of N and K alone.  A cut's time in ns, as measured at the 7B and 32B sizes: a round of workgroups is 3 us
// and, a block, 500 and 150 for each tile (5 tiles 1.2 us a block, 10 tiles 1.8 to 2.1); a split's sums are written and read once
// more, at 5 TB/s.  us at 160 rows, the model's choice and the best of all cuts: 4,608 x 3,584 15.2 and 14.2, 3,584 x 3,584 14.1 and
// 13.1, 3,584 x 18,944 36.9 and 35.1 (10 splits), 7,168 x 5,120 24 and 23.3, 5,120 x 27,648 60.2 and 60.2.  `whole`: without a split.
// Returns the cost.
#define GW_PLAN_ROWS 192
int64_t zi_gemm_many_plan(int N, int K, int whole, int* splits, int* kb_per_split, int* tiles_wg) {
    const int tiles = (N + 15) / 16, kb_total = (K + GM_KB - 1) / GM_KB, cus = zi_compute_units();
    int64_t best = -1;
    for (int w = GM_MIN_WAVES; w <= GW_MAX_TILES; ++w) {
        if (w == 9) continue;       // (no kernel is made for nine)
        const int groups = (tiles + w - 1) / w;
        for (int s0 = 1; s0 <= (whole ? 1 : 16) && s0 <= (kb_total > 1 ? kb_total / 2 : 1); ++s0) {
            const int per = (kb_total + s0 - 1) / s0, s = (kb_total + per - 1) / per;
            if (s != s0) continue;      // the same cut under another name
            const int64_t rounds = ((int64_t)groups * s + cus - 1) / cus;
            const int64_t cost = rounds * ((int64_t)per * (150 * w + 500) + 3000) + (whole ? 0 : (int64_t)s * N * GW_PLAN_ROWS / 625);
            if (best < 0 || cost < best) {
                best = cost;
                *splits = s;
                *kb_per_split = per;
                *tiles_wg = w;
            }
        }
    }
    return best;
}

// The most blocks of 128 of k that eight wavefronts work faster than four: for sums that are parts and for whole products with the
// activation, 5 .. 8 tiles of 16 rows of x (down) and 4 .. 8 of weight rows, where the means of both ways cross, launches in turn at three
// random products for each of 1 .. 56 blocks (up to 96 rows below that: single products lost up to a tenth before the means crossed).
// Eight's time of four's at 3 / 9 / 28 blocks: 72 and 80 rows, 4 weight tiles 0.96 / 1.07 / 1.12, 8 weight tiles 0.86 / 0.94 / 0.98; 96 rows (a quarter of the wavefronts has none) 0.98 / 1.14 / 1.21 and 0.88 / 0.95 / 0.99; 128 rows 0.95 /
// 0.97 / 1.02 and 0.87 / 0.90 / 0.97; whole, 128 rows, 5 weight tiles 0.85 / 0.92 / 1.00.  Where rows do not begin at lines of 128 bytes
// eight lose sooner (128 rows, 6 weight tiles 0.96 / 1.03 / 1.12, whole 0.89 / 1.04 / 1.16): one bound for all of these.
static const int gw_eight_most[2][4][5] = {
    {{4, 3, 5, 5, 7}, {4, 4, 8, 8, 12}, {20, 20, 36, 36, 1000}, {18, 12, 28, 36, 1000}},
    {{8, 6, 12, 12, 12}, {8, 7, 12, 12, 12}, {36, 20, 36, 40, 1000}, {48, 20, 36, 40, 1000}}};
static const int gw_eight_most_apart[2] = {5, 7};

static bool gw_eight(int mt, int tiles, int per, bool whole, bool lines) {
    return mt > 8 || per <= (lines ? gw_eight_most[whole][mt < 5 ? 0 : mt - 5][tiles - GM_MIN_WAVES] : gw_eight_most_apart[whole]);
}

// (for tests: the wavefronts of a workgroup for M = 65 .. 256 rows of x and the weights [N, K], rows `ld` elements apart)
extern "C" int zi_gemm_wide_wavefronts(int M, int N, int K, int ld, int whole) {
    int splits, per, tiles;
    if (M > GW_MID_ROWS) zi_gemm_many_plan(N, K, whole, &splits, &per, &tiles);
    else zi_gemm_mid_plan(N, K, whole, &splits, &per, &tiles);
    return gw_eight((M + 15) / 16, tiles, per, whole, ld % 64 == 0) ? 8 : 4;
}

// The launch; the checks are the caller's (zi_gemm_skinny).
int zi_gemm_mid_launch(void* out, int out_f32, int mode, const zi_bf16* x, const zi_bf16* w, const zi_bf16* bias, int M,
                       int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, int vec_out, float limit, hipStream_t stream) {
    int splits, per, waves;
    if (M > GW_MID_ROWS) zi_gemm_many_plan(N, K, mode == GM_MODE_SWIGLU, &splits, &per, &waves);
    else zi_gemm_mid_plan(N, K, mode >= GM_MODE_ACT || (mode == GM_MODE_SWIGLU && M > 64), &splits, &per, &waves);
    const int64_t most_ld = M > GW_MID_ROWS ? GW_MAX_LD / 2 : GW_MAX_LD;
    const bool apart = M > 64 && (ldx > most_ld || ldw > most_ld);
    if (apart && waves > GM_MAX_WAVES) waves = GM_MAX_WAVES;       // (which weight rows share a workgroup changes no sum)
    const int tiles = (N + 15) / 16;
    const dim3 grid((tiles + waves - 1) / waves, splits);
    const int mt = apart ? 0 : (M + 15) / 16;
    const bool lines = ldx % 64 == 0 && ldw % 64 == 0 && ((uintptr_t)x | (uintptr_t)w) % 128 == 0;
    const bool eight = gw_eight(mt, waves, per, mode == GM_MODE_SWIGLU, lines);
#define ZI_GM3(MT, WV, APART, GRID)                                                                                            \
    gemm_mid_kernel<MT, 3, WV, APART><<<GRID, WV * ZI_WAVE, 0, stream>>>(out, mode, out_f32, x, w, bias, M, N, K, ldx, ldw, \
                                                                         ldo, per, vec_out, limit)
#define ZI_GM2(MT, WV) ZI_GM3(MT, WV, false, grid)
#define ZI_GA2(MT, WV) ZI_GM3(MT, WV, true, dim3(grid.x, grid.y, (M + 16 * MT - 1) / (16 * MT)))
#define ZI_GA(MT)                               \
    switch (waves) {                            \
        case 4: ZI_GA2(MT, 4); break;           \
        case 5: ZI_GA2(MT, 5); break;           \
        case 6: ZI_GA2(MT, 6); break;           \
        case 7: ZI_GA2(MT, 7); break;           \
        default: ZI_GA2(MT, 8); break;          \
    }
#define ZI_GM(MT)                               \
    switch (waves) {                            \
        case 4: ZI_GM2(MT, 4); break;           \
        case 5: ZI_GM2(MT, 5); break;           \
        case 6: ZI_GM2(MT, 6); break;           \
        case 7: ZI_GM2(MT, 7); break;           \
        default: ZI_GM2(MT, 8); break;          \
    }
#define ZI_GW3(MT, WV, WN)                                                                                     \
    gemm_wide_kernel<MT, WV, WN><<<grid, (gw_shape<MT, WV, WN>::WAVES) * ZI_WAVE, 0, stream>>>(out, mode, out_f32, x, w, bias, M, N, \
                                                                                               K, ldx, ldw, ldo, per, vec_out, limit)
#define ZI_GW2(MT, WV)                                                         \
    do {                                                                        \
        if (eight) ZI_GW3(MT, WV, 2);                                           \
        else ZI_GW3(MT, WV, (MT <= 8 && WV <= GM_MAX_WAVES ? 1 : 2));            \
    } while (0)
#define ZI_GW(MT)                               \
    switch (waves) {                            \
        case 4: ZI_GW2(MT, 4); break;           \
        case 5: ZI_GW2(MT, 5); break;           \
        case 6: ZI_GW2(MT, 6); break;           \
        case 7: ZI_GW2(MT, 7); break;           \
        default: ZI_GW2(MT, 8); break;          \
    }
// (rows beyond 128 in tiles of 32: the engine's steps have multiples of 32)
#define ZI_GW_MANY(MT)                          \
    switch (waves) {                            \
        case 10: ZI_GW2(MT, 10); break;         \
        default: ZI_GW(MT)                      \
    }
    switch (mt) {
        case 0: ZI_GA(4); break;
        case 1: ZI_GM(1); break;
        case 2: ZI_GM(2); break;
        case 3: ZI_GM(3); break;
        case 4: ZI_GM(4); break;
        case 5: ZI_GW(5); break;
        case 6: ZI_GW(6); break;
        case 7: ZI_GW(7); break;
        case 8: ZI_GW(8); break;
        case 9:
        case 10: ZI_GW_MANY(10); break;
        case 11:
        case 12: ZI_GW_MANY(12); break;
        case 13:
        case 14: ZI_GW_MANY(14); break;
        default: ZI_GW_MANY(16); break;
    }
#undef ZI_GM
#undef ZI_GM2
#undef ZI_GM3
#undef ZI_GA
#undef ZI_GA2
#undef ZI_GW_MANY
#undef ZI_GW
#undef ZI_GW2
#undef ZI_GW3
    return zi_check_launch("gemm_mid");
}
