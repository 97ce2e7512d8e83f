// out[M,N] = x[M,K] . w[N,K]^T (+ bias[N]), everything float32 and K above GF_SPLIT_ABOVE, on the matrix cores' bfloat16 instruction
// (v_mfma_f32_16x16x32_bf16, sixteen times the multiply-adds a cycle of the float32 one).
//
// A float32 value is the sum of three bfloat16 ones, exactly: itself rounded, what is left rounded, and what is left of that (8 + 8 + 8 bits).
// That needs the last part's last bit, 2^-23 of the value, to be a bfloat16 one: bfloat16 ends at 2^-133, so values below 2^-110 would lose
// theirs (below 2^-126 0.4 % and more).  Operands are therefore split times 2^24, an exact step that lifts the smallest float32 to 2^-125,
// where parts are not even subnormal, and finished sums take 2^-48.
// Of the nine products of two values' parts the six largest are added; two of the others reach 2^-25 of the product each, the third 2^-34.  Weights and x stay
// float32 in memory and are split on their way into the matrix cores; sums are float32.  A value that 2^24 takes past the range (2^104 and
// above), infinities and NaNs leave parts that are no numbers, and sums from 2^80 on leave the range: a sum that is not finite is made again from the
// float32 operands (gf_finite).
//
// The instruction cuts off what lies more than some three bits below its largest term's last bit, downwards whatever the sign, so sums come
// out low, by a quarter of their rounding errors at 8,960 columns, every output alike; over a model's layers that adds up.  So one of the two
// chains below is summed with x negated and subtracted, and the two change places from run to run: the errors cancel in the mean, also where
// x lies in one half of every chunk alone (mean over rms then, changing places or not: 1,536 columns 0.00 and 0.15,
// 8,960 0.01 and 0.22).
//
// Error against 64 bits, 2-norm over 2-norm, of the float32 instruction's kernels and of these: normal values 1.85e-7 and 1.38e-7 at 1,536 columns,
// 4.3e-7 and 3.6e-7 at 8,960, their absolute values 4.9e-8 and 4.2e-8, 1.0e-7 and 8.0e-8; the logits of a 28-layer model 3.7e-7 and 3.3e-7 (with one
// sign for all chains 4.5e-7).  These are further off where few products make a sum, a single one 2.5e-8 and 3.4e-8, eight 5.4e-8 and 6.1e-8, and
// at many columns where half of every chunk is empty, so that one chain adds up what are two there: 1,536 columns 1.37e-7 and 1.35e-7, absolute
// values 4.4e-8 and 5.0e-8; 8,960 3.06e-7 and 3.56e-7, 7.7e-8 and 1.04e-7.  That is the instruction's cutting, not the products left out: with the two
// of 2^-25 added the figures are the same (a single one 3.4e-8), at 8 to 15 % more time.
//
// One order of the sums, the same in every kernel here, so that a row's result does not depend on M, on the tile it falls in or on the rest
// of the batch: k is cut into GF_PARTS runs of whole chunks of 64 (a function of K alone); within a run the first and the second 32 of every
// chunk (in runs of odd number the second and the first) are two chains, each 32 an instruction for every product of parts, whose lane group
// g holds k = 4 g .. 4 g + 3 and 16 more; a run's sum is first - second chain; the sums of each half of the runs are added in rising order,
// then the two halves, then the bias.
//
// What bounds it: few rows the one pass over the weights; many rows, by counters at 2,048 rows of 4,096 x 4,096, the vector instructions
// (57 % of the cycles, eleven for every two values split, thirteen since they are split times 2^24) and the matrix cores (51 %), which mostly take turns, beside LDS (43 %).
//
// Measured, weights from memory, against the float32 instruction's kernels, us, launch included (N x K; act: with the activation):
//   1 row      2,048 x 1,536 5.1 and 5.1, 1,536 x 8,960 13.2 and 11.8, 17,920 x 1,536 act 19.8 and 20.1, 151,936 x 1,536 135.5 and 140.5
//   8 rows     5.9 and 5.6, 18.6 and 15.9, 21.2 and 20.4, 156.8 and 155.1
//   24 rows    9.4 and 8.8, 34.5 and 24.8, 151,936 x 1,536 317 and 248; 64 rows 11.9 and 10.0, 51.8 and 37.3, 297 and 240
//   450 rows   32.3 and 28.1, 122 and 112 (111 TFLOP/s), 230 and 187 (132)
//   2,048 rows 116 and 84.7, 473 and 428, 903 and 711 (159), 4,608 x 3,584 534 and 429 (158; the float32 instruction in a large library product: 152)
// Slower: up to 4 rows of 151,936 x 1,536 2 to 4 %, up to 8 of 37,888 x 3,584 act 1 to 3 %, and, where tiles are one or two rounds of workgroups, 96 to
// 256 rows of 2,048 x 1,536 1 to 4 %, 48 to 128 of 3,584 x 3,584 0 to 3 %, 200 of 4,608 x 3,584 9 % (69 and 75).
#include "zi_gemm_f32.h"

#define GF_KB 64             // k of a chunk
static_assert((GF_SPLIT_ABOVE / GF_KB + GF_PARTS) / GF_PARTS > 2, "a run has three chunks and more");
#define GF_HELD_CHUNKS 8     // chunks of a run that a wavefront can hold of 8 rows of x beside as many of weights (256 registers)

// The three bfloat16 parts of eight values, largest first.
struct gf_parts {
    gf_pack p[3];
};

typedef unsigned __attribute__((may_alias)) gf_u32_alias_t;

#define GF_UP 0x1p24f        // what operands are multiplied by before they are split (x of the negated chain by its negative), ...
#define GF_DOWN 0x1p-48f     // ... and sums when they are finished

// The parts of two values, packed, through set(part, both).
template <typename Set>
__device__ __forceinline__ void gf_split_two(float lo, float hi, float up, Set set) {
    lo *= up;
    hi *= up;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        const uint32_t u = zi_pack_bf16x2(lo, hi);
        set(p, u);
        if (p < 2) {
            lo -= __uint_as_float(u << 16);             // exactly: what is left fits a float32
            hi -= __uint_as_float(u & 0xffff0000u);
        }
    }
}

__device__ __forceinline__ gf_parts gf_split(gf_f32x4_t a, gf_f32x4_t b, float up) {
    gf_parts s;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        gf_split_two(i < 2 ? a[2 * i] : b[2 * i - 4], i < 2 ? a[2 * i + 1] : b[2 * i - 3], up, [&](int p, uint32_t u) { s.p[p].u[i] = u; });
    return s;
}

enum gf_sign { GF_PLUS, GF_MINUS, GF_MINUS_SECOND };

// A block of 16 lines of 128 bytes, loaded as whole lines (lane l, load i: piece l % 8 of line 8 i + l / 8), as the matrix cores' operand:
// lane (r, g) gets pieces g and 4 + g of line r, split.  Loads in the operand's own layout would take a line's pieces by lanes 16 apart,
// which the vector cache serves one lane at a time: 52 instead of 16 of its cycles for an instruction's 1 KB, 16 bytes a clock and unit.
// SIGN: the values, their negatives, or (of blocks that hold both chains) the negatives of the second chain's lines.
// `block` is 2 KB of LDS of this wavefront alone (piece c of line q at place c xor (q / 2 mod 8), free of bank conflicts both ways); a
// wavefront's LDS accesses are in order, so there is nothing to wait for between one block and the next.
template <gf_sign SIGN>
__device__ __forceinline__ gf_parts gf_turn(gf_f32x4_t* block, gf_f32x4_t line0, gf_f32x4_t line8, int lane) {
    const int r = lane & 15, g = lane >> 4, q = lane >> 3, c = lane & 7;
    block[q * 8 + (c ^ (q >> 1))] = line0;
    block[(8 + q) * 8 + (c ^ (4 + (q >> 1)))] = line8;
    gf_f32x4_t a = block[r * 8 + (g ^ (r >> 1))], b = block[r * 8 + ((4 + g) ^ (r >> 1))];
    return gf_split(a, b, SIGN == GF_MINUS || (SIGN == GF_MINUS_SECOND && (lane & 8)) ? -GF_UP : GF_UP);
}

// A block of x of chain h, or (PAIR) of both chains; the second chain's negated (see the top).
template <bool PAIR>
__device__ __forceinline__ gf_parts gf_turn_of_chain(int h, gf_f32x4_t* block, gf_f32x4_t line0, gf_f32x4_t line8, int lane) {
    if (PAIR) return gf_turn<GF_MINUS_SECOND>(block, line0, line8, lane);
    return h ? gf_turn<GF_MINUS>(block, line0, line8, lane) : gf_turn<GF_PLUS>(block, line0, line8, lane);
}

// x of up to V rows (V 2 or 4) where a block holds 8: a lane loads and splits V values of a chunk instead of 8, of which most would be
// rows that are not there (a row of x, us: 1,536 x 8,960 13.1 to 11.7, 2,048 x 1,536 5.5 to 5.15, 3,584 x 18,944 50.2 to 46.2; rows that
// are held were split for 2 us before the first weights were looked at: 4,608 x 3,584 17.1 to 15.8).  Lane l holds values V c .. V c + V - 1 of the chunk's 64 of row l / (64 / V), c = l mod (64 / V); the parts go
// through 2 KB of LDS, 64 bytes for a row and chain, into the same operand as gf_turn's; rows past V are one line of zeros.
template <int V>
struct gf_few {
    static constexpr int LANES = ZI_WAVE / V, PART = (2 * V + 1) * 64;      // lanes a row; bytes of one part, the zeros last
    static_assert(V == 2 || V == 4, "whole pairs, within 2 KB");
    float up;
    int put, get;
    __device__ __forceinline__ gf_few(char* block, int lane, int exchanged) {
        const int m = lane / LANES, k = lane % LANES * V, chain = (k / 32) ^ exchanged, piece = k % 32 / 4, r = lane & 15, g = lane >> 4;
        up = chain ? -GF_UP : GF_UP;
        put = (chain * V + m) * 64 + (piece & 3) * 16 + (piece >> 2) * 8 + (k & 3) * 2;
        get = (r % 8 < V ? r / 8 * V + r % 8 : 2 * V) * 64 + g * 16;
        if (lane < 12) *reinterpret_cast<gf_f32x4_t*>(block + lane / 4 * PART + 2 * V * 64 + lane % 4 * 16) = gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    __device__ __forceinline__ gf_parts turn(char* block, const gf_pack& x) const {
#pragma unroll
        for (int i = 0; i < V; i += 2)
            gf_split_two(x.f[i], x.f[i + 1], up, [&](int p, uint32_t u) { *reinterpret_cast<gf_u32_alias_t*>(block + p * PART + put + i * 2) = u; });
        gf_parts s;
#pragma unroll
        for (int p = 0; p < 3; ++p) s.p[p].f = *reinterpret_cast<const gf_f32x4_t*>(block + p * PART + get);
        return s;
    }
    __device__ __forceinline__ static gf_pack load(__amdgpu_buffer_rsrc_t rows, int offset) {
        gf_pack x;
        if constexpr (V == 4) {
            x.f = gf_load<0>(rows, offset);
        } else {
            const auto two = __builtin_amdgcn_raw_buffer_load_b64(rows, offset, 0, 0);
            x.u[0] = two[0];
            x.u[1] = two[1];
        }
        return x;
    }
};
// Where lane l's values lie: `row` bytes into x (GF_OUT: a row that is not there, see fetch), `k` bytes into the chunk.
struct gf_few_place {
    int row, k;
};
template <int V>
__device__ __forceinline__ gf_few_place gf_few_at(int lane, int rows_x, int64_t ldx) {
    const int m = lane / (ZI_WAVE / V), k = lane % (ZI_WAVE / V) * V * 4;
    return {m < rows_x ? (int)(m * ldx * 4) + k : GF_OUT, k};
}
template <>
struct gf_few<8> {      // (none: blocks of 8 rows)
    __device__ __forceinline__ gf_few(char*, int, int) {}
};

// acc += w . x over the 32 k of an instruction: the six products of parts that reach float32's last bits, the smallest first.
__device__ __forceinline__ gf_f32x4_t gf_multiply(const gf_parts& w, const gf_parts& x, gf_f32x4_t acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.p[2].b, x.p[0].b, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.p[0].b, x.p[2].b, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.p[1].b, x.p[1].b, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.p[1].b, x.p[0].b, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.p[0].b, x.p[1].b, acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.p[0].b, x.p[0].b, acc, 0, 0, 0);
}

// Finishes four sums of a lane, of row `row` of x and of rows w_row(e) of w.  One that is not finite (an operand was no number or too large
// to split, or the sum left the range: see the top) is made again from the float32 operands, by the whole wavefront (all its lanes come here
// together; mine(e): sum e is an output), so that a lane has K / 64 multiply-adds one after the other and the sum is at least as exact.  A
// row of x with a NaN, what a request whose values ran away brings to every product, has NaNs only: it is looked for first, four loads
// on their way, and remembered in nan_rows; a weight row with one gives them to all rows in hand.
// (Rows with a NaN, us, every lane for itself, summed by the wavefront before it is looked for, now, and without such rows.  One among 8:
// 17,920 x 1,536 with the activation 1,178, 32, 24.6 and 20.2; 1,536 x 8,960 1,053, 23, 18.2 and 15.9; 151,936 x 1,536 9,085, 185, 156 and 156.  Four among 72
// of 1,536 x 8,960 97.7 and 85.9, 20 among 450 158 and 117.  A weight row with one, 450 rows of 1,536 x 8,960: 376, 114 and, without, 107.)
template <typename Mine, typename Row>
__device__ __forceinline__ void gf_finite(gf_f32x4_t& s, int row, Mine mine, Row w_row, const float* x, int64_t ldx, const float* w, int64_t ldw, int K,
                                          uint64_t& nan_rows) {
    const float no_number = __uint_as_float(0x7fc00000u);
    const bool all = s[0] * 0.f + s[1] * 0.f + s[2] * 0.f + s[3] * 0.f == 0.f;      // (0 times what is not finite is a NaN)
    s *= GF_DOWN;
    if (__ballot(!all) == 0) return;
    const int lane = threadIdx.x & (ZI_WAVE - 1);
#pragma unroll 1
    for (int e = 0; e < 4; ++e) {
        float sum = e == 0 ? s[0] : e == 1 ? s[1] : e == 2 ? s[2] : s[3];
        const int row_w = w_row(e);
        const bool known = nan_rows >> row & 1;
        if (known) sum = no_number;
        uint64_t todo = __ballot(mine(e) && !known && (__float_as_uint(sum) & 0x7f800000u) == 0x7f800000u);
        while (todo) {
            const int of = __builtin_ctzll(todo), of_x = __builtin_amdgcn_readlane(row, of), of_w = __builtin_amdgcn_readlane(row_w, of);
            todo &= todo - 1;
            float again = 0.f;
            const float *a = x + of_x * ldx, *b = w + of_w * ldw;
            bool nan_x = false, nan_w = false;
            for (int k0 = lane * 4; k0 < K; k0 += ZI_WAVE * 16) {      // (four loads on their way)
                gf_f32x4_t u[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) u[i] = *reinterpret_cast<const gf_f32x4_t*>(a + (k0 + i * ZI_WAVE * 4 < K ? k0 + i * ZI_WAVE * 4 : k0));
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) nan_x |= u[i][j] != u[i][j];
            }
            if (__ballot(nan_x)) {
                nan_rows |= 1ull << of_x;
                todo &= ~__ballot(row == of_x);
                if (row == of_x) sum = no_number;
                continue;
            }
#pragma unroll 1
            for (int k = lane * 4; k < K; k += ZI_WAVE * 4) {
                const gf_f32x4_t u = *reinterpret_cast<const gf_f32x4_t*>(a + k), v = *reinterpret_cast<const gf_f32x4_t*>(b + k);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    again = fmaf(u[i], v[i], again);
                    nan_w |= v[i] != v[i];
                }
            }
            again = zi_wave_sum(again);
            if (__ballot(nan_w)) {
                todo &= ~__ballot(row_w == of_w);
                if (row_w == of_w) sum = no_number;
            }
            if (lane == of) sum = again;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = i == e ? sum : s[i];
    }
}

// PAIR: 8 weight rows and up to 8 rows of x (XV < 8: up to XV of them, see gf_few); else 16 weight rows and up to 16 * MT rows of x a
// workgroup.  RING chunks are on their way while one is worked on.
template <int MT, bool PAIR, int RING, int XV>
__global__ void __launch_bounds__(GF_PARTS* ZI_WAVE, 4)
gemm_f32_split_stream_kernel(float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w,
                       const float* __restrict__ bias, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, int per, int vec_out) {
    constexpr int NR = PAIR ? 8 : 16, MR = PAIR ? 8 : 16 * MT, H = PAIR ? 1 : 2;
    __shared__ __attribute__((aligned(16))) gf_f32x4_t part[GF_PARTS][MT][ZI_WAVE];
    const int lane = threadIdx.x & (ZI_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE);
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * NR, m0 = blockIdx.y * MR;
    const int rows_w = N - n0 < NR ? N - n0 : NR, rows_x = M - m0 < MR ? M - m0 : MR;
    const __amdgpu_buffer_rsrc_t wb = gf_rows(w + (int64_t)n0 * ldw, ldw, rows_w, K), xb = gf_rows(x + (int64_t)m0 * ldx, ldx, rows_x, K);
    __shared__ __attribute__((aligned(16))) gf_f32x4_t turn[GF_PARTS][1 + MT][128];
    // a block of 16 lines is the rows' lines of one chain, or (PAIR) both chains' lines of 8 rows
    constexpr int RB = PAIR ? 1 : 2;               // loads of different rows a block
    const int k_lane = (lane & 7) * 16;
    int w_row[RB], x_row[MT][RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        const int row = i * 8 + (lane >> 3);
        w_row[i] = row < rows_w ? (int)(row * ldw * 4) : GF_OUT;
#pragma unroll
        for (int t = 0; t < MT; ++t) x_row[t][i] = t * 16 + row < rows_x ? (int)((t * 16 + row) * ldx * 4) : GF_OUT;
    }
    const int chunks = (K + GF_KB - 1) / GF_KB;
    const int c0 = wave * per, c1 = c0 + per < chunks ? c0 + per : chunks;
    constexpr bool FEW = PAIR && XV < 8;
    char* const few_block = reinterpret_cast<char*>(turn[wave][1]);
    const gf_few<PAIR ? XV : 8> few(few_block, lane, wave & 1);
    const gf_few_place at_few = gf_few_at<XV>(lane, rows_x, ldx);

    gf_f32x4_t wr[RING][H][2], xr[RING][H][MT][2];
    gf_pack xf[RING];
    auto fetch = [&](const int slot, int c) __attribute__((always_inline)) {
        if constexpr (FEW) xf[slot] = few.load(xb, c < c1 && c * (GF_KB * 4) + at_few.k < K * 4 && at_few.row != GF_OUT ? at_few.row + c * (GF_KB * 4) : GF_OUT);
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int k = c * (GF_KB * 4) + ((PAIR ? i : h) ^ (wave & 1)) * 128 + k_lane;      // (see the top: the chains change places)
                const bool in = c < c1 && k < K * 4;
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    if constexpr (!FEW) xr[slot][h][t][i] = gf_load<0>(xb, in && x_row[t][i % RB] != GF_OUT ? x_row[t][i % RB] + k : GF_OUT);
                // a weight of up to 8 rows of x is read once by one workgroup: past L2
                wr[slot][h][i] = gf_load<PAIR ? 2 : 0>(wb, in && w_row[i % RB] != GF_OUT ? w_row[i % RB] + k : GF_OUT);
            }
    };
    gf_f32x4_t acc[H][MT];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[h][t] = gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < RING; ++s) {
        fetch(s, c0 + s);
        __builtin_amdgcn_sched_barrier(0);         // in this order: the loop waits for the oldest only
    }
    for (int c = c0; c < c1; c += RING) {
#pragma unroll
        for (int s = 0; s < RING; ++s) {
#pragma unroll
            for (int h = 0; h < H; ++h) {
                const gf_parts ws = gf_turn<GF_PLUS>(turn[wave][0], wr[s][h][0], wr[s][h][1], lane);
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    if constexpr (FEW) acc[h][t] = gf_multiply(ws, few.turn(few_block, xf[s]), acc[h][t]);
                    else acc[h][t] = gf_multiply(ws, gf_turn_of_chain<PAIR>(h, turn[wave][1 + t], xr[s][h][t][0], xr[s][h][t][1], lane), acc[h][t]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);     // the loads stay this far ahead of their use
            fetch(s, c + s + RING);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // lane (r, g) holds rows 4 g .. 4 g + 3 of column r; PAIR: the first chain in the quadrant of rows and columns 0 .. 7, the
    // second in the one of 8 .. 15 (the others mix the halves and are dropped)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        gf_f32x4_t s = acc[0][t];
        if (PAIR) {
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] -= __shfl(acc[0][t][e], (lane + 40) & 63, ZI_WAVE);
        } else {
            s -= acc[H - 1][t];
        }
        part[wave][t][lane] = s;
    }
    __syncthreads();
    uint64_t nan_rows = 0;
    for (int t = wave; t < MT; t += GF_PARTS) {
        const int m = t * 16 + r, n = g * 4;
        gf_f32x4_t s = part[0][t][lane], s2 = part[GF_PARTS / 2][t][lane];
#pragma unroll
        for (int p = 1; p < GF_PARTS / 2; ++p) {
            s += part[p][t][lane];
            s2 += part[GF_PARTS / 2 + p][t][lane];
        }
        s += s2;
        gf_finite(s, m, [&](int e) { return m < rows_x && n + e < rows_w; }, [&](int e) { return n0 + n + e; }, x + m0 * ldx, ldx, w, ldw, K, nan_rows);
        if (m < rows_x && n < rows_w) gf_store4(out + (int64_t)(m0 + m) * ldo, bias, s, n0 + n, N, vec_out);
    }
}

// The same for up to 16 rows of x and more groups of weight rows than there are compute units: a workgroup keeps its wavefronts' runs
// of x in registers, split into their parts once (PER chunks a wavefront, at most), and walks over groups of 8 (PAIR) or 16 weight rows,
// gridDim.x apart.  As soon as a chunk of weights has been used, its registers are filled with the same chunk of the next group: PER
// chunks are always on their way, x passes the loads once a workgroup instead of once a group, as many bytes again as the weights' for 8
// rows, and a workgroup's start and end come once.  The eight runs' sums meet in one of two LDS buffers, so a group costs one barrier,
// which does not wait for loads; the wavefronts take the adding and storing in turn.  GATED: a group is as many gate rows as up rows (row
// n and row N + n of w) and the outputs are up * silu(gate).
//
// Bound by the stream of the weights: 151,936 x 1,536 at 8 rows 161 us (5.8 TB/s).  Two workgroups a unit while a lane has registers for that
// (128): with 4 chunks of x they spill, and one is faster (5,000 x 2,048 with the activation, one row: 17.4 against 20.8 us).
template <bool PAIR, int PER, bool GATED, int XV>
__global__ void __launch_bounds__(GF_PARTS* ZI_WAVE, (PAIR ? 1 : 2) * PER <= 3 ? 4 : 2)
gemm_f32_split_held_kernel(float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                     int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, int per, int vec_out, int groups) {
    constexpr int NR = PAIR ? 8 : 16, NC = GATED ? NR / 2 : NR, H = PAIR ? 1 : 2;
    __shared__ __attribute__((aligned(16))) gf_f32x4_t part[2][GF_PARTS][ZI_WAVE];
    const int lane = threadIdx.x & (ZI_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE);
    __shared__ __attribute__((aligned(16))) gf_f32x4_t turn[GF_PARTS][2][128];
    constexpr int RB = PAIR ? 1 : 2;               // as above
    const int r = lane & 15, g = lane >> 4;
    const int chunks = (K + GF_KB - 1) / GF_KB, c0 = wave * per;
    const int mine = chunks - c0 < per ? chunks - c0 : per;       // chunks of this wavefront's run (none or fewer at the end of k)
    const int k0 = c0 * (GF_KB * 4) + (lane & 7) * 16;            // the first byte of a row that this lane loads
    const __amdgpu_buffer_rsrc_t xb = gf_rows(x, ldx, M, K);
    int x_row[RB], w_row[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        const int row = i * 8 + (lane >> 3);
        x_row[i] = row < M ? (int)(row * ldx * 4) : GF_OUT;
        w_row[i] = (int)((GATED && row >= NC ? N + row - NC : row) * ldw * 4);
    }
    // the weight rows of a group: what lies past the last one gives zeros (or, of a gate row past the last, an output that is not stored)
    auto weights = [&](int group) {
        const int64_t n0 = (int64_t)group * NC;
        const int rows = group >= groups ? 0 : (GATED ? N : 0) + (int)(N - n0 < NC ? N - n0 : NC);
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(w + (rows ? n0 * ldw : 0)), 0,
                                                 rows ? (int)(((int64_t)(rows - 1) * ldw + K) * 4) : 0, 0x00020000);
    };
    auto place = [&](int s, int h, int i) { return s * (GF_KB * 4) + ((PAIR ? i : h) ^ (wave & 1)) * 128; };      // (the chains change places)
    auto in = [&](int s, int h, int i) { return s < mine && k0 + place(s, h, i) < K * 4; };
    gf_f32x4_t wr[PER][H][2];
    gf_parts xs[PER][H];
    __amdgpu_buffer_rsrc_t wb = weights(blockIdx.x);
    auto fetch = [&](const int s) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int i = 0; i < 2; ++i) wr[s][h][i] = gf_load<2>(wb, in(s, h, i) ? w_row[i % RB] + k0 + place(s, h, i) : GF_OUT);
    };
    constexpr bool FEW = PAIR && XV < 8;
    {
        char* const few_block = reinterpret_cast<char*>(turn[wave][0]);
        const gf_few<PAIR ? XV : 8> few(few_block, lane, wave & 1);
        const gf_few_place at_few = gf_few_at<XV>(lane, M, ldx);
        gf_pack xf[PER];
        gf_f32x4_t xr[PER][H][2];
#pragma unroll
        for (int s = 0; s < PER; ++s)
            if constexpr (FEW)
                xf[s] = few.load(xb, s < mine && (c0 + s) * (GF_KB * 4) + at_few.k < K * 4 && at_few.row != GF_OUT ? at_few.row + (c0 + s) * (GF_KB * 4) : GF_OUT);
#pragma unroll
        for (int s = 0; s < PER && !FEW; ++s)
#pragma unroll
            for (int h = 0; h < H; ++h)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    xr[s][h][i] = gf_load<0>(xb, in(s, h, i) && x_row[i % RB] != GF_OUT ? x_row[i % RB] + k0 + place(s, h, i) : GF_OUT);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < PER; ++s) {
            fetch(s);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int s = 0; s < PER; ++s)
#pragma unroll
            for (int h = 0; h < H; ++h) {
                if constexpr (FEW) xs[s][h] = few.turn(few_block, xf[s]);
                else xs[s][h] = gf_turn_of_chain<PAIR>(h, turn[wave][(s * H + h) & 1], xr[s][h][0], xr[s][h][1], lane);
            }
    }
    int b = 0, whose = 0;
    uint64_t nan_rows = 0;
    for (int group = blockIdx.x; group < groups; group += gridDim.x, b ^= 1, whose = (whose + 1) % GF_PARTS) {
        wb = weights(group + (int)gridDim.x);
        gf_f32x4_t acc[H];
#pragma unroll
        for (int h = 0; h < H; ++h) acc[h] = gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < PER; ++s) {
#pragma unroll
            for (int h = 0; h < H; ++h) acc[h] = gf_multiply(gf_turn<GF_PLUS>(turn[wave][(s * H + h) & 1], wr[s][h][0], wr[s][h][1], lane), xs[s][h], acc[h]);
            __builtin_amdgcn_sched_barrier(0);
            fetch(s);
            __builtin_amdgcn_sched_barrier(0);
        }
        gf_f32x4_t sum = acc[0];
        if (PAIR) {
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] -= __shfl(acc[0][e], (lane + 40) & 63, ZI_WAVE);
        } else {
            sum -= acc[H - 1];
        }
        part[b][wave][lane] = sum;
        // all sums are in LDS (and the buffer's reader of two groups ago is past the barrier of the last one); loads travel on
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        if (wave != whose) continue;
        gf_f32x4_t s = part[b][0][lane], s2 = part[b][GF_PARTS / 2][lane];
#pragma unroll
        for (int p = 1; p < GF_PARTS / 2; ++p) {
            s += part[b][p][lane];
            s2 += part[b][GF_PARTS / 2 + p][lane];
        }
        s += s2;
        const int64_t n = (int64_t)group * NC + g * 4;
        // sum e of this lane is weight row g * 4 + e of the group, a gate row or, from NC on, an up row
        auto output = [&](int e) { return group * NC + (GATED && g * 4 + e >= NC ? g * 4 + e - NC : g * 4 + e); };
        gf_finite(s, r, [&](int e) { return r < M && g * 4 + e < NR && output(e) < N; }, [&](int e) { return output(e) + (GATED && g * 4 + e >= NC ? N : 0); },
                  x, ldx, w, ldw, K, nan_rows);
        if (GATED) {
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = gf_gate(s[e], __shfl(s[e], lane + (PAIR ? 16 : 32), ZI_WAVE));
        }
        if (r < M && g * 4 < NC && n < N) gf_store4(out + (int64_t)r * ldo, bias, s, (int)n, N, vec_out);
    }
}

// 16 MT rows of x by 16 NT WAVES weight rows a workgroup, 16 NT weight rows a wavefront; GROUPS (1 or 4) groups of WAVES wavefronts,
// each over as many eighths of k.  A step is half a chunk, 32 k, one of the two chains.  A wavefront's weight rows are its own: they go
// from memory into its registers, DEPTH steps ahead, and are split there.  x, which all wavefronts of a group share, is split by the
// threads that loaded it and goes through LDS as its parts, two buffers, one barrier a step that does not wait for loads.
// GATED (NT even): of a wavefront's blocks of 16 weight rows the even ones are gate rows and the odd ones the up rows of the same outputs
// (rows n and N + n of w), and half as many outputs, up * silu(gate), are what the tile leaves.
// With both operands loaded in the matrix cores' layout (see gf_turn) 512 rows of 1,536 x 8,960 took 126 us and now 109, 256 of 17,920 x 1,536
// 136 and 120; with two groups of wavefronts instead of four, and one wavefront a SIMD, 160.  Tiles of 128 x 128 with one wavefront a SIMD
// are no faster (2,048 rows of 4,096 x 4,096 406 against 403 us), nor is one more vector instruction less a pair by v_dot2 (the matrix
// cores do not run beside it).
template <int MT, int NT, int WAVES, int GROUPS, bool GATED>
__global__ void __launch_bounds__(ZI_WAVE* WAVES* GROUPS, GROUPS > 1 ? WAVES * GROUPS / 4 : MT * NT <= 4 ? 3 : 2)
gemm_f32_split_tile_kernel(float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w,
                     const float* __restrict__ bias, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, int per, int vec_out,
                     int m_tiles, int tiles) {
    static_assert(!GATED || NT % 2 == 0, "as many gate as up blocks a wavefront");
    constexpr int TM = 16 * MT, TN = 16 * NT * WAVES, NC = GATED ? TN / 2 : TN, NW = NC / WAVES;     // NW outputs a row and wavefront
    constexpr int THREADS = ZI_WAVE * WAVES, PIECES = TM * 4, XP = (PIECES + THREADS - 1) / THREADS;
    constexpr int DEPTH = GROUPS == 1 ? 2 : 1, RUNS = GF_PARTS / GROUPS, SUMS = GROUPS == 1 ? 1 : RUNS;
    constexpr bool TOGETHER = GROUPS == 1 && MT * NT > 4;     // two wavefronts a SIMD
    constexpr int BLOCKS = WAVES * MT * NT;                  // 16 x 16 blocks of the tile
    constexpr int X_BYTES = GROUPS * 2 * 3 * PIECES * 16, SUM_BYTES = GROUPS == 1 ? 0 : GF_PARTS * BLOCKS * ZI_WAVE * 16, FIRST_BYTES = GROUPS == 1 ? BLOCKS * ZI_WAVE * 16 : 0, TURN_BYTES = GROUPS * WAVES * NT * 2048;
    __shared__ __attribute__((aligned(16))) gf_u32x4_t lds_all[(GROUPS == 1 || X_BYTES + TURN_BYTES > SUM_BYTES ? X_BYTES + TURN_BYTES + FIRST_BYTES : SUM_BYTES) / 16];
    gf_u32x4_t(*lds)[2][3][PIECES] = reinterpret_cast<gf_u32x4_t(*)[2][3][PIECES]>(lds_all);
    gf_f32x4_t* first = reinterpret_cast<gf_f32x4_t*>(lds_all) + (X_BYTES + TURN_BYTES) / 16 + (int)threadIdx.x;      // one group: sums of the first half of the runs
    // the tiles that share weight rows follow each other on one XCD (workgroup i runs on XCD i mod 8)
    const int per_xcd = (tiles + 7) / 8, tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (tile >= tiles) return;
    const int m0 = (tile % m_tiles) * TM, n0 = (tile / m_tiles) * NC;
    const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE), group = wave_all / WAVES, wave = wave_all % WAVES;
    const int lane = threadIdx.x & (ZI_WAVE - 1), tid = wave * ZI_WAVE + lane;
    const int r = lane & 15, g = lane >> 4;
    const int rows_w = N - n0 < NC ? N - n0 : NC, rows_x = M - m0 < TM ? M - m0 : TM;
    const __amdgpu_buffer_rsrc_t wb = gf_rows(w + (int64_t)n0 * ldw, ldw, (GATED ? N : 0) + rows_w, K), xb = gf_rows(x + (int64_t)m0 * ldx, ldx, rows_x, K);
    // a thread's pieces of x: the eight values of lane group i % 4 of row i / 4, i = tid, tid + THREADS, ...; piece c of row q lies at
    // place c xor (-(q / 4) mod 4), which keeps the operand reads free of bank conflicts (a read of 16 bytes a lane serves lanes 0 to 3, 12 to
    // 15 and 20 to 27 in one turn)
    int x_row[XP], x_place[XP], w_row[NT][2];
    const int x_lane = (tid & 3) * 16, w_lane = (lane & 7) * 16;
    gf_f32x4_t* turn = reinterpret_cast<gf_f32x4_t*>(lds_all) + X_BYTES / 16 + wave_all * NT * 128;
#pragma unroll
    for (int p = 0; p < XP; ++p) {
        const int i = tid + p * THREADS, q = i >> 2;
        x_row[p] = q < rows_x && i < PIECES ? (int)(q * ldx * 4) + x_lane : GF_OUT;
        x_place[p] = q * 4 + ((i ^ -(q >> 2)) & 3);
    }
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int q = wave * NW + (GATED ? u / 2 : u) * 16 + i * 8 + (lane >> 3);
            w_row[u][i] = q < rows_w ? (int)((q + (GATED && (u & 1) ? N : 0)) * ldw * 4) + w_lane : GF_OUT;
        }
    const int chunks = (K + GF_KB - 1) / GF_KB, mine = per * RUNS;
    const int c0 = group * mine, c1 = GROUPS > 1 && c0 + mine < chunks ? c0 + mine : chunks;
    const int steps = GROUPS > 1 ? mine : chunks;      // chunks, the same number for all groups: they share the barriers
    gf_f32x4_t xr[DEPTH][XP][2], wr[DEPTH][NT][2];
    // (the step's place along k is the loads' scalar offset; bytes of a row from there on, none past the group's last chunk)
    auto left = [&](int at, int c) { return c < c1 ? K * 4 - at : 0; };
    int in_part = 0, parts = 0;      // the chunk's place in its run, runs done (a group's first run is of even number)
    // the chain of half h of the chunk `ahead` (at most 2, a run has 3 and more) after this one: the halves change places from run to run
    auto place = [&](const int h, int c, int ahead) { return c * (GF_KB * 4) + (h ^ ((parts + (in_part + ahead >= per)) & 1)) * 128; };
    auto fetch_x = [&](const int h, int c, int ahead) __attribute__((always_inline)) {
        const int at = place(h, c, ahead), rest = left(at, c);
#pragma unroll
        for (int p = 0; p < XP; ++p)
#pragma unroll
            for (int q = 0; q < 2; ++q) xr[h % DEPTH][p][q] = gf_load<0>(xb, x_lane + q * 64 < rest ? x_row[p] : GF_OUT, at + q * 64);
    };
    auto fetch_w = [&](const int h, int c, int ahead) __attribute__((always_inline)) {
        const int at = place(h, c, ahead), rest = left(at, c);
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) wr[h % DEPTH][u][i] = gf_load<0>(wb, w_lane < rest ? w_row[u][i] : GF_OUT, at);
    };
    auto stash = [&](const int h) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < XP; ++p) {
            const gf_parts s = gf_split(xr[h % DEPTH][p][0], xr[h % DEPTH][p][1], h ? -GF_UP : GF_UP);
            if (PIECES % THREADS == 0 || tid + p * THREADS < PIECES) {
#pragma unroll
                for (int i = 0; i < 3; ++i) lds[group][h][i][x_place[p]] = s.p[i].u;
            }
        }
    };
    const gf_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    gf_f32x4_t acc[2][MT][NT], sum[SUMS][MT][NT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            acc[0][t][u] = acc[1][t][u] = zero;
#pragma unroll
            for (int i = 0; i < SUMS; ++i) sum[i][t][u] = zero;
        }
    const int read_at = r * 4 + ((g ^ -(r >> 2)) & 3);
    // Half h of chunk c: its weights' parts lie in ws[h] and its x in buffer h.  While it is multiplied the next half's operands are split, one
    // vector instruction after the other in the time that the matrix cores take, and those of DEPTH halves later are asked for.
    gf_parts ws[2][NT];
    auto step = [&](const int h, int c) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NT; ++u) ws[h ^ 1][u] = gf_turn<GF_PLUS>(turn + u * 128, wr[(h ^ 1) % DEPTH][u][0], wr[(h ^ 1) % DEPTH][u][1], lane);
        if (DEPTH == 2) fetch_w(h ^ 1, h ? c + 2 : c + 1, h ? 2 : 1);
        else fetch_w(h, c + 1, 1);
        stash(h ^ 1);
        if (DEPTH == 2) fetch_x(h ^ 1, h ? c + 2 : c + 1, h ? 2 : 1);
        else fetch_x(h, c + 1, 1);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            gf_parts xs;
#pragma unroll
            for (int i = 0; i < 3; ++i) xs.p[i].u = lds[group][h][i][t * 64 + read_at];
#pragma unroll
            for (int u = 0; u < NT; ++u) acc[h][t][u] = gf_multiply(ws[h][u], xs, acc[h][t][u]);
        }
        // a product, a few vector instructions, and so on
        __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
        for (int i = 0; i < 6 * MT * NT; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, TOGETHER ? 4 : 3, 0);
            if (i % (6 * NT) == 0 && i / (6 * NT) + 2 < MT) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
        }
        if (TOGETHER) {
            // (the splitting done here: left to itself the compiler moves it past the barrier, where no product is under way)
#pragma unroll
            for (int u = 0; u < NT; ++u)
#pragma unroll
                for (int i = 0; i < 3; ++i) asm volatile("" : "+v"(ws[h ^ 1][u].p[i].u));
        }
        // x of the next half is in LDS, this half's has been read; loads travel on
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        __builtin_amdgcn_sched_barrier(0);
    };
    fetch_x(0, c0, 0);
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(0, c0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (DEPTH == 2) {
        fetch_x(1, c0, 0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_w(1, c0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
    stash(0);
    if (DEPTH == 2) fetch_x(0, c0 + 1, 1);
    else fetch_x(1, c0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < NT; ++u) ws[0][u] = gf_turn<GF_PLUS>(turn + u * 128, wr[0][u][0], wr[0][u][1], lane);
    if (DEPTH == 2) fetch_w(0, c0 + 1, 1);
    else fetch_w(1, c0, 0);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    for (int c = 0; c < steps; ++c) {
        step(0, c0 + c);
        step(1, c0 + c);
        if (++in_part == per) {           // a run of k ends
            in_part = 0;
            ++parts;
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    // one group: the sum of the runs of a half; else a sum for each of the group's runs
                    const gf_f32x4_t run = acc[0][t][u] - acc[1][t][u];
                    acc[0][t][u] = acc[1][t][u] = zero;
                    if (GROUPS == 1) {
                        sum[0][t][u] += run;
                        if (parts == GF_PARTS / 2) {
                            first[(t * NT + u) * THREADS] = sum[0][t][u];
                            sum[0][t][u] = zero;
                        }
                    } else if (parts == 1) {
                        sum[0][t][u] = run;
                    } else {
                        sum[SUMS - 1][t][u] = run;
                    }
                }
        }
    }
    constexpr int STEP = GATED ? 2 : 1;
    uint64_t nan_rows = 0;
    auto finish = [&](gf_f32x4_t* s, int t, int u0, int of) __attribute__((always_inline)) {
        // the sums of a wavefront's block (t, u0), or of its gate and up blocks: checked, activated, stored
        int l = lane;
        asm volatile("" : "+v"(l));        // (what is worked out of it is worked out here: kept, it takes the loop's registers)
        const int m = m0 + t * 16 + (l & 15), n = n0 + of * NW + (GATED ? u0 / 2 : u0) * 16 + (l >> 4) * 4;
#pragma unroll
        for (int i = 0; i < STEP; ++i)
            gf_finite(s[i], t * 16 + (l & 15), [&](int e) { return m < M && n + e < N; }, [&](int e) { return n + e + (i ? N : 0); }, x + m0 * ldx, ldx, w, ldw, K,
                      nan_rows);
        if (m >= M || n >= N) return;
        if (GATED) {
#pragma unroll
            for (int e = 0; e < 4; ++e) s[0][e] = gf_gate(s[0][e], s[GATED][e]);
        }
        gf_store4(out + (int64_t)m * ldo, GATED ? nullptr : bias, s[0], n, N, vec_out);
    };
    if (GROUPS == 1) {
        // (through this thread's own places in LDS, so that what checks and stores them is there once and takes no registers from the loop above)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int u = 0; u < NT; ++u) {          // (acc: zeros where the last run ended)
                gf_f32x4_t& at = first[(t * NT + u) * THREADS];
                const gf_f32x4_t s = sum[0][t][u] + (acc[0][t][u] - acc[1][t][u]);
                at = parts >= GF_PARTS / 2 ? at + s : s;
            }
#pragma unroll 1
        for (int b = 0; b < MT * NT; b += STEP) {
            gf_f32x4_t s[STEP];
#pragma unroll
            for (int i = 0; i < STEP; ++i) s[i] = first[(b + i) * THREADS];
            finish(s, b / NT, b % NT, wave);
        }
        return;
    }
    // the runs' sums meet in LDS (past the last barrier nobody reads x there)
    gf_f32x4_t* part = reinterpret_cast<gf_f32x4_t*>(lds_all);
#pragma unroll
    for (int i = 0; i < RUNS; ++i)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int u = 0; u < NT; ++u)
                part[(((group * RUNS + i) * WAVES + wave) * MT * NT + t * NT + u) * ZI_WAVE + lane] =
                    sum[i % SUMS][t][u];
    __syncthreads();
    for (int b = wave_all; b < BLOCKS / STEP; b += WAVES * GROUPS) {
        gf_f32x4_t s[STEP];
#pragma unroll
        for (int i = 0; i < STEP; ++i) {
            const gf_f32x4_t* at = part + (b * STEP + i) * ZI_WAVE + lane;
            s[i] = at[0];
            gf_f32x4_t s2 = at[GF_PARTS / 2 * BLOCKS * ZI_WAVE];
#pragma unroll
            for (int p = 1; p < GF_PARTS / 2; ++p) {
                s[i] += at[p * BLOCKS * ZI_WAVE];
                s2 += at[(GF_PARTS / 2 + p) * BLOCKS * ZI_WAVE];
            }
            s[i] += s2;
        }
        const int of = b * STEP / (MT * NT), tu = b * STEP % (MT * NT);
        finish(s, tu / NT, tu % NT, of);
    }
}

// Which kernel M rows of x and N weight rows take is a matter of filling the compute units only.
// Up to 8 rows a stream of the weights in groups of 8, up to 16 in groups of 16 unless two passes over groups of 8 are one round (1,024 weight
// rows); x is held in registers once there are more groups than units.  Beyond, groups of 16 weight rows with 16 or 32 rows of x while those are
// one round of workgroups, 32 up to 32 rows.  Then the tiles that take the least: rounds of workgroups times (a start + a time a chunk), us, or,
// with one group of wavefronts, where several workgroups share a unit, a start and a time a chunk for one, two and three of them, both fitted to 255
// products alone of 33 to 3,200 rows, 400 to 24,000 weight rows and 23 to 296 chunks.  The choice takes 0.8 % more than the best of the five in the
// mean, over 5 % in 12 of the 255 and at most 20 % (few rows and more weights than stream in that time: 115 rows of 9,988 x 2,148 82 us
// in tiles of 32 x 96, 68 in 64 x 128).  Chosen and next, us: 450 rows of 4,608 x 3,584 32 x 96 135, 64 x 64 159; 1,024 of 1,536 x 8,960 32 x 96 222, 64 x 128 237,
// 32 x 64 269; 2,048 of 4,608 x 3,584 64 x 128 430, 32 x 128 496; 256 of 17,920 x 1,536 with the activation 64 x 128 121, 32 x 128 130, 80 rows of it 32 x 128 62, 32 x 64 73;
// 512 of 2,048 x 1,536 64 x 64 28, 32 x 64 36; 256 of 1,536 x 8,960 32 x 64 92, 32 x 96 107.
static gf_kernel gf_choose(int M, int64_t N, int K, float* tiles_us) {      // (tiles_us: set where it is a tile)
    const int64_t cus = zi_compute_units(), n16 = (N + 15) / 16, m16 = (M + 15) / 16, m32 = (M + 31) / 32, m64 = (M + 63) / 64;
    const int chunks = (K + GF_KB - 1) / GF_KB, per = (chunks + GF_PARTS - 1) / GF_PARTS;
    if (M <= 8) return (N + 7) / 8 > cus && per <= GF_HELD_CHUNKS ? GF_HELD_PAIRS : GF_PAIRS;
    if (M <= 16 && n16 > cus && per <= GF_HELD_CHUNKS / 2) return GF_HELD_ROWS16;
    if (M <= 16) return (N + 7) / 8 * 2 <= cus ? GF_PAIRS : GF_ROWS16;
    if (n16 * m16 <= cus) return GF_ROWS16;
    if (M <= 32 || n16 * m32 <= cus) return GF_ROWS32;
    const int64_t n64 = (N + 63) / 64, n96 = (N + 95) / 96, n128 = (N + 127) / 128;
    auto shared = [&](int64_t tiles, float start, float chunk) { return (float)((tiles + cus - 1) / cus) * (start + chunk * chunks); };
    auto rounds = [&](int64_t tiles, int places, float start, float one, float two, float all) {      // `places` workgroups a unit at a time
        const int64_t full = tiles / (places * cus), rest = tiles % (places * cus);
        return start + (float)chunks * ((float)full * all + (rest == 0 ? 0.f : rest <= cus ? one : rest <= 2 * cus ? two : all));
    };
    gf_kernel best = GF_TILE_32_HALVES;
    float us = shared(m32 * n64, 3.82f, 0.63f);
    auto consider = [&](gf_kernel kernel, float takes) {
        if (takes < us) {
            best = kernel;
            us = takes;
        }
    };
    consider(GF_TILE_96_HALVES, shared(m32 * n96, 4.68f, 0.788f));
    consider(GF_TILE_64_QUARTERS, shared(m64 * n64, 5.73f, 0.938f));
    consider(GF_TILE_32, rounds(m32 * n128, 3, 7.39f, 1.52f, 2.19f, 2.89f));
    consider(GF_TILE_64, rounds(m64 * n128, 2, 8.83f, 1.65f, 2.94f, 2.94f));
    *tiles_us = us;
    return best;
}

gf_kernel zi_gemm_f32_split_kernel(int M, int64_t N, int K) {
    float us;
    return gf_choose(M, N, K, &us);
}

template <bool GATED>
static int gs_launch(float* out, const float* x, const float* w, const float* bias, int M, int N, int K, int64_t ldx, int64_t ldw,
                     int64_t ldo, hipStream_t stream) {
    const int chunks = (K + GF_KB - 1) / GF_KB, per = (chunks + GF_PARTS - 1) / GF_PARTS;
    const int vec_out = ldo % 4 == 0 && (uintptr_t)out % 16 == 0;
#define ZI_GF_STREAM(MT, PAIR, RING, XV)                                                                                                 \
    gemm_f32_split_stream_kernel<MT, PAIR, RING, XV><<<dim3((N + (PAIR ? 7 : 15)) / (PAIR ? 8 : 16), (M + (PAIR ? 8 : 16 * MT) - 1) / (PAIR ? 8 : 16 * MT)), \
                                             GF_PARTS * ZI_WAVE, 0, stream>>>(out, x, w, bias, M, N, K, ldx, ldw, ldo, per, vec_out)
    // two workgroups a unit while a lane has registers for that (128), else one
#define ZI_GF_HELD_PAIRS(PER)                                                                                                            \
    do {                                                                                                                                 \
        if (M <= 2) ZI_GF_HELD(true, PER, 2);                                                                                             \
        else if (M <= 4) ZI_GF_HELD(true, PER, 4);                                                                                        \
        else ZI_GF_HELD(true, PER, 8);                                                                                                    \
    } while (0)
#define ZI_GF_HELD(PAIR, PER, XV)                                                                                                        \
    do {                                                                                                                                 \
        const int nc = (PAIR ? 8 : 16) / (GATED ? 2 : 1), groups = (N + nc - 1) / nc;                                                        \
        const int places = zi_compute_units() * ((PAIR ? 1 : 2) * PER <= 3 ? 2 : 1);                                                         \
        gemm_f32_split_held_kernel<PAIR, PER, GATED, XV><<<groups < places ? groups : places, GF_PARTS * ZI_WAVE, 0, stream>>>(                         \
            out, x, w, bias, M, N, K, ldx, ldw, ldo, per, vec_out, groups);                                                               \
    } while (0)
    // (rows in as many launches as 2^32 threads of one make necessary: a row's result does not depend on them)
#define ZI_GF_TILE(MT, NT, WAVES, G)                                                                                                       \
    do {                                                                                                                                  \
        const int tm = 16 * MT, nc = 16 * NT * WAVES / (GATED ? 2 : 1);                                                                      \
        const int64_t nt = (N + nc - 1) / nc, most = ((1ll << 31) / (ZI_WAVE * WAVES * G)) / nt * tm;                                        \
        for (int64_t m = 0; m < M; m += most) {                                                                                           \
            const int rows = (int)(M - m < most ? M - m : most), mt = (rows + tm - 1) / tm, tiles = (int)(mt * nt);                          \
            gemm_f32_split_tile_kernel<MT, NT, WAVES, G, GATED><<<(tiles + 7) / 8 * 8, ZI_WAVE * WAVES * G, 0, stream>>>(                          \
                out + m * ldo, x + m * ldx, w, bias, rows, N, K, ldx, ldw, ldo, per, vec_out, mt, tiles);                                  \
        }                                                                                                                                 \
    } while (0)
    switch (zi_gemm_f32_split_kernel(M, (int64_t)N * (GATED ? 2 : 1), K)) {
        case GF_HELD_PAIRS:
            if (per <= 3) ZI_GF_HELD_PAIRS(3);
            else if (per <= 4) ZI_GF_HELD_PAIRS(4);
            else if (per <= 6) ZI_GF_HELD_PAIRS(6);
            else if (per <= 7) ZI_GF_HELD_PAIRS(7);
            else ZI_GF_HELD_PAIRS(8);
            break;
        case GF_HELD_ROWS16:
            if (per <= 3) ZI_GF_HELD(false, 3, 8);
            else ZI_GF_HELD(false, 4, 8);
            break;
        case GF_TILE_64: ZI_GF_TILE(4, 2, 4, 1); break;
        case GF_TILE_32: ZI_GF_TILE(2, 2, 4, 1); break;
        case GF_TILE_32_HALVES: ZI_GF_TILE(2, 2, 2, 4); break;
        case GF_TILE_64_QUARTERS: ZI_GF_TILE(4, 2, 2, 4); break;
        case GF_TILE_96_HALVES: ZI_GF_TILE(2, 2, 3, 4); break;
        default:
            if constexpr (GATED) {
                return zi_fail("gemm_f32: no gated kernel for %d rows of %d x %d", M, N, K);      // (zi_gemm_f32_swiglu_takes says so)
            } else {
                switch (zi_gemm_f32_split_kernel(M, N, K)) {
                    case GF_PAIRS:
                        if (M <= 2) ZI_GF_STREAM(1, true, 3, 2);
                        else if (M <= 4) ZI_GF_STREAM(1, true, 3, 4);
                        else ZI_GF_STREAM(1, true, 3, 8);
                        break;
                    case GF_ROWS16: ZI_GF_STREAM(1, false, 2, 8); break;
                    default: ZI_GF_STREAM(2, false, 1, 8); break;
                }
            }
    }
#undef ZI_GF_STREAM
#undef ZI_GF_HELD
#undef ZI_GF_HELD_PAIRS
#undef ZI_GF_TILE
    return zi_check_launch("gemm_f32_split");
}

int zi_gemm_f32_split_launch(bool gated, float* out, const float* x, const float* w, const float* bias, int M, int N, int K, int64_t ldx,
                             int64_t ldw, int64_t ldo, hipStream_t stream) {
    return gated ? gs_launch<true>(out, x, w, nullptr, M, N, K, ldx, ldw, ldo, stream) : gs_launch<false>(out, x, w, bias, M, N, K, ldx, ldw, ldo, stream);
}

// ---- many rows ------------------------------------------------------------------------------------------------------------
// The tiles above split x again in every workgroup of a row of tiles (140 times at 17,920 weight rows) and every weight once for 64 rows of x,
// thirteen vector instructions for two values that the matrix cores mostly wait for.  Here x is split once, by a launch of its own
// (gf_parts_kernel), into a workspace that holds the parts as the tiles' LDS does, and a wavefront multiplies each weight that it has split
// with up to 128 rows.  That takes most of a SIMD's registers, so one wavefront a SIMD has to hide its own waits: parts of x go straight into
// LDS three steps ahead, weights into registers two steps ahead, and a weight's split, 1.1 to 2.2 vector instructions a product, stands between
// products of four different sums.  The chains, the runs and their order are the same as everywhere in this file, and so are the bits.

// The parts of x times 2^24, the second chain's negative: [block of 16 rows][chunk][chain][part][a KB as LDS holds it].  Rows past M and
// columns past K are zeros.  A wavefront a chain.
__global__ void __launch_bounds__(4 * ZI_WAVE) gf_parts_kernel(gf_u32x4_t* __restrict__ parts, const float* __restrict__ x, int M, int K,
                                                                     int64_t ldx, int chunks, int per) {
    const int lane = threadIdx.x & (ZI_WAVE - 1), s = blockIdx.x * 4 + (int)(threadIdx.x / ZI_WAVE), c = s >> 1, h = s & 1;
    if (c >= chunks) return;
    const int q = lane >> 2, g = (lane ^ -(q >> 2)) & 3;
    const int k = c * GF_KB + (h ^ ((c / per) & 1)) * 32 + g * 4;
    const int64_t row = (int64_t)blockIdx.y * 16 + q;
    gf_f32x4_t v[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = row < M && k + 16 * i < K ? *reinterpret_cast<const gf_f32x4_t*>(x + row * ldx + k + 16 * i) : gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
    const gf_parts p = gf_split(v[0], v[1], h ? -GF_UP : GF_UP);
    gf_u32x4_t* to = parts + (((int64_t)blockIdx.y * chunks + c) * 2 + h) * (3 * ZI_WAVE) + lane;
#pragma unroll
    for (int i = 0; i < 3; ++i) to[i * ZI_WAVE] = p.p[i].u;
}

#define GF_STAGES 4

// The sums stay in the accumulation registers over the loop: without this the compiler moves all of them to other registers and back.
#ifdef __HIP_DEVICE_COMPILE__
#define GF_KEEP(v) asm volatile("" : "+a"(v))
#else
#define GF_KEEP(v)
#endif

struct gf_many_args {
    float* out;                  // (RUNS: the sums of the runs, [8][M][N], gated [8][M][2 N], the gates' first)
    const gf_u32x4_t* parts;
    const float *x, *w, *bias;
    int M, N, K;
    int64_t ldx, ldw, ldo;
    int chunks, per, vec_out, m_tiles, tiles, runs;     // runs: of a workgroup (RUNS), an even number
    int up_at;                   // (gated: the up rows' place behind the gate rows)
};

// 16 MT rows of x by 128 weight rows a workgroup of four wavefronts, 32 weight rows a wavefront.  A step is one chain of a chunk, 32 k.
// GATED as above.  RUNS: blockIdx.y takes `runs` of the eight runs of k and leaves their sums.
template <int MT, bool GATED, bool RUNS>
__global__ void __launch_bounds__(4 * ZI_WAVE, 1) gemm_f32_split_many_kernel(gf_many_args a) {
    constexpr int NT = 2, WAVES = 4, TM = 16 * MT, NC = GATED ? 64 : 128, NW = NC / WAVES;
    constexpr int LOADS = 3 * MT, PW = (LOADS + WAVES - 1) / WAVES, PIECES = LOADS * ZI_WAVE, STEP_LOADS = PW + 2 * NT;
    static_assert(MT % 2 == 0 && GF_STAGES * PIECES >= WAVES * MT * NT * ZI_WAVE, "rows in pairs of blocks; the sums fit where x was");
    // (spare: where loads go that nobody needs)
    __shared__ __attribute__((aligned(16))) gf_u32x4_t all[GF_STAGES * PIECES], spare[ZI_WAVE];
    __shared__ __attribute__((aligned(16))) gf_f32x4_t turns[WAVES][NT * 128];
    const int per_xcd = (a.tiles + 7) / 8, tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (tile >= a.tiles) return;
    const int m_tile = tile % a.m_tiles, m0 = m_tile * TM, n0 = tile / a.m_tiles * NC;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE), lane = threadIdx.x & (ZI_WAVE - 1), r = lane & 15, g = lane >> 4;
    const int M = a.M, N = a.N, K = a.K, per = a.per, chunks = a.chunks;
    const int rows_w = N - n0 < NC ? N - n0 : NC;
    const __amdgpu_buffer_rsrc_t wb = gf_rows(a.w + (int64_t)n0 * a.ldw, a.ldw, (GATED ? a.up_at : 0) + rows_w, K);
    const int block_bytes = chunks * 6 * 1024, blocks = (M + 15) / 16 - m_tile * MT;
    const char* const parts = reinterpret_cast<const char*>(a.parts) + (int64_t)m_tile * MT * block_bytes;
    const int parts_bytes = (blocks < MT ? blocks : MT) * block_bytes;
    int x_at[PW], w_row[NT][2];
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int L = i * WAVES + wave;
        x_at[i] = L < LOADS && L / 3 < blocks ? L / 3 * block_bytes + L % 3 * 1024 + lane * 16 : GF_OUT;
    }
    const int w_lane = (lane & 7) * 16;
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int q = wave * NW + (GATED ? 0 : u) * 16 + i * 8 + (lane >> 3);
            w_row[u][i] = q < rows_w ? (int)((q + (GATED && (u & 1) ? a.up_at : 0)) * a.ldw * 4) + w_lane : GF_OUT;
        }
    gf_f32x4_t* const turn = turns[wave];
    const int c0 = RUNS ? (int)blockIdx.y * a.runs * per : 0, end = RUNS && c0 + a.runs * per < chunks ? c0 + a.runs * per : chunks;
    int parts_done = 0, in_part = 0;      // runs done (the first is of even number), the chunk's place in its run
    auto fetch_w = [&](gf_f32x4_t (&to)[NT][2], int h, int c, int ahead) __attribute__((always_inline)) {      // as in the tiles above
        const int at = c * (GF_KB * 4) + (h ^ ((parts_done + (in_part + ahead >= per)) & 1)) * 128, rest = c < end ? K * 4 - at : 0;
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) to[u][i] = gf_load<0>(wb, w_lane < rest ? w_row[u][i] : GF_OUT, at);
    };
    // (a step's place is in the buffer it is loaded from: the range is sure to be held against the lane's offset alone)
    auto load_x = [&](__amdgpu_buffer_rsrc_t from, int buf, const int i) __attribute__((always_inline)) {
        const int L = i * WAVES + wave;
#ifdef __HIP_DEVICE_COMPILE__       // (the host's pass knows loads of this size for no target)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(from, L < LOADS ? all + buf + L * ZI_WAVE : spare, 16, x_at[i], 0, 0, 0);
#endif
    };
    gf_f32x4_t acc[2][MT][NT], sum[MT][NT], first[MT][NT], wr[2][NT][2];
    const gf_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) sum[t][u] = first[t][u] = zero;
    gf_parts ws[2][NT], xs[2][2];         // xs: of a pair of blocks, and of the next pair
    gf_f32x4_t lines[NT][2];
    const int read_at = r * 4 + ((g ^ -(r >> 2)) & 3), q8 = lane >> 3, c8 = lane & 7;
    int cur = 0;      // the step's buffer
    auto put_w = [&](const gf_f32x4_t (&from)[NT][2], const int u) __attribute__((always_inline)) {       // gf_turn in its pieces
        turn[u * 128 + q8 * 8 + (c8 ^ (q8 >> 1))] = from[u][0];
        turn[u * 128 + (8 + q8) * 8 + (c8 ^ (4 + (q8 >> 1)))] = from[u][1];
    };
    auto get_w = [&](const int u, const int i) __attribute__((always_inline)) { lines[u][i] = turn[u * 128 + r * 8 + ((4 * i + g) ^ (r >> 1))]; };
    auto split_w = [&](gf_parts (&to)[NT], const int j) __attribute__((always_inline)) {       // two values of the eight of block j / 4
        const int u = j / 4, i = j % 4;
        gf_split_two(lines[u][i / 2][i % 2 * 2], lines[u][i / 2][i % 2 * 2 + 1], GF_UP, [&](int p, uint32_t v) {
            asm volatile("" ::"v"(v));       // (here, not where it is used)
            to[u].p[p].u[i] = v;
        });
    };
    auto read_x = [&](gf_parts (&to)[2], int buf, const int t, const int i) __attribute__((always_inline)) {      // operand i of six
        to[i / 3].p[i % 3].u = all[buf + ((t + i / 3) * 3 + i % 3) * ZI_WAVE + read_at];
    };
    // Chain h of chunk c: its weights' parts lie in ws[h], its x in LDS at `cur`, the first two blocks of that in xs of the step's first pair.
    // Three groups of eight products for every two blocks of rows, two for each of four sums, and beside each group a share of the rest: the next
    // operands of x, the next step's weights through LDS and split, the loads.  Two vector instructions a product cost nothing, a third as much as
    // half a product (8.4, 9.0 and 12.6 ns), and left to itself the compiler puts products of one sum behind each other, so the order is given here.
    constexpr int GROUPS = 3 * MT / 2, LAST = GROUPS - 3;
    const char* x_next = parts + (int64_t)c0 * 6144;          // the parts of the step that is asked for next, and their buffer's bytes from there on
    int x_left = parts_bytes - c0 * 6144;
    auto x_step = [&]() __attribute__((always_inline)) {      // (past the last step: other rows' parts or nothing, never used)
        const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(x_next), 0, x_left > 0 ? x_left : 0, 0x00020000);
        x_next += 3072;
        x_left -= 3072;
        return xb;
    };
    auto step = [&](const int h, int c, const bool fresh) __attribute__((always_inline)) {
        const int next = cur == (GF_STAGES - 1) * PIECES ? 0 : cur + PIECES;
        static const int order[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};      // parts of w and x, gf_multiply's order
        const __amdgpu_buffer_rsrc_t xb = x_step();
#pragma unroll
        for (int k = 0; k < GROUPS; ++k) {
            const int pair = k / 3, in_pair = k % 3, now = (h * (MT / 2) + pair) & 1;
            if (k == LAST) {
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("" ::: "memory");
                // the next step's x is there, all wavefronts have read this step's
                zi_wait_loads<2 * STEP_LOADS, true>();
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
            __builtin_amdgcn_sched_barrier(0);
            // (reads of LDS spread, of four wavefronts at a time it serves one in 32 cycles; none right in front of the barrier)
            const int read_from = k < LAST ? cur : next, read_t = k < LAST ? 2 * pair + 2 : 0, reads = pair == MT / 2 - 2 ? 3 : 2;
#pragma unroll
            for (int i = 0; i < 6; ++i)
                if (i / reads == in_pair) read_x(xs[now ^ 1], read_from, read_t, i);
            if (k == 0) get_w(0, 0), get_w(0, 1);
            if (k == 2) get_w(1, 0);
            if (k == 3) get_w(1, 1);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (k == (MT >= 6 ? 1 + j : 1 + j * 5 / 8)) split_w(ws[h ^ 1], j);
            if (k == LAST + 1) put_w(wr[h], 0);
            if (k == LAST + 2) {
                put_w(wr[h], 1);
                fetch_w(wr[h], h, c + 2, 2);
            }
#pragma unroll
            for (int i = 0; i < PW; ++i)
                if (k >= LAST && i % 3 == in_pair) load_x(xb, cur, i);
#pragma unroll
            for (int o = 2 * in_pair; o < 2 * in_pair + 2; ++o)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int u = 0; u < NT; ++u)
                        acc[h][2 * pair + q][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ws[h][u].p[order[o][0]].b, xs[now][q].p[order[o][1]].b,
                                                                                          fresh && o == 0 ? zero : acc[h][2 * pair + q][u], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, MT >= 6 ? 2 : 4, 0);
                if (i % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x300, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        cur = next;
    };
    fetch_w(wr[0], 0, c0, 0);
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(wr[1], 1, c0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < GF_STAGES; ++i) {
        const __amdgpu_buffer_rsrc_t xb = x_step();
#pragma unroll
        for (int k = 0; k < PW; ++k) load_x(xb, i * PIECES, k);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int u = 0; u < NT; ++u) put_w(wr[h], u);
        if (h == 0) {
#pragma unroll
            for (int i = 0; i < 2 * NT; ++i) get_w(i / 2, i % 2);
#pragma unroll
            for (int j = 0; j < 8; ++j) split_w(ws[0], j);
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch_w(wr[h], h, c0 + 1, 1);
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("" ::: "memory");
    zi_wait_loads<(GF_STAGES - 1) * PW + 4 * NT, true>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 6; ++i) read_x(xs[0], 0, 0, i);
    for (int c = c0; c < end;) {         // the runs
        in_part = 0;
        step(0, c, true);
        step(1, c, true);
        ++c;
        for (in_part = 1; in_part < per && c < end; ++in_part, ++c) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    GF_KEEP(acc[0][t][u]);
                    GF_KEEP(acc[1][t][u]);
                }
            step(0, c, false);
            step(1, c, false);
        }
        if (!RUNS && parts_done == GF_PARTS / 2) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    first[t][u] = sum[t][u];
                    sum[t][u] = zero;
                }
        }
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int u = 0; u < NT; ++u) {
                const gf_f32x4_t run = acc[0][t][u] - acc[1][t][u];
                if (RUNS) {
                    const int m = m0 + t * 16 + r, n = n0 + wave * NW + (GATED ? 0 : u) * 16 + g * 4;      // (N a multiple of four)
                    if (m < M && n < N)
                        *reinterpret_cast<gf_f32x4_t*>(a.out + ((int64_t)(blockIdx.y * a.runs + parts_done) * M + m) * (GATED ? 2 * N : N) + (GATED && (u & 1) ? N : 0) + n) = run;
                } else {
                    sum[t][u] += run;
                }
            }
        ++parts_done;
    }
    zi_wait_loads<0, true>();       // (no load may arrive after the workgroup's LDS is another's)
    if (RUNS) return;
    // (through this thread's own places in LDS, where x was, so that what checks and stores them is there once)
    gf_f32x4_t* const mine = reinterpret_cast<gf_f32x4_t*>(all) + wave * MT * NT * ZI_WAVE + lane;
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) mine[(t * NT + u) * ZI_WAVE] = parts_done > GF_PARTS / 2 ? first[t][u] + sum[t][u] : sum[t][u];
    constexpr int STEP = GATED ? 2 : 1;
    uint64_t nan_rows[2] = {0, 0};       // of the tile's first and last 64 rows
#pragma unroll 1
    for (int b = 0; b < MT * NT; b += STEP) {
        const int t = b / NT, m = m0 + t * 16 + r, n = n0 + wave * NW + (GATED ? 0 : b % NT) * 16 + g * 4, m64 = t / 4 * 64;
        gf_f32x4_t s[STEP];
#pragma unroll
        for (int i = 0; i < STEP; ++i) {
            s[i] = mine[(b + i) * ZI_WAVE];
            uint64_t nans = t < 4 ? nan_rows[0] : nan_rows[1];
            gf_finite(s[i], t % 4 * 16 + r, [&](int e) { return m < M && n + e < N; }, [&](int e) { return n + e + (i ? a.up_at : 0); }, a.x + (int64_t)(m0 + m64) * a.ldx,
                      a.ldx, a.w, a.ldw, K, nans);
            if (t < 4) nan_rows[0] = nans;
            else nan_rows[1] = nans;
        }
        if (m < M && n < N) {
            if (GATED) {
#pragma unroll
                for (int e = 0; e < 4; ++e) s[0][e] = gf_gate(s[0][e], s[GATED][e]);
            }
            gf_store4(a.out + (int64_t)m * a.ldo, GATED ? nullptr : a.bias, s[0], n, N, a.vec_out);
        }
    }
}

// The runs' sums added in the order of this file: a wavefront 256 outputs of a row.
template <bool GATED>
__global__ void __launch_bounds__(4 * ZI_WAVE) gf_add_runs_kernel(const float* __restrict__ sums, gf_many_args a, int runs) {
    const int m = blockIdx.y, n = (blockIdx.x * 4 * ZI_WAVE + threadIdx.x) * 4;
    const int64_t row = GATED ? 2 * a.N : a.N;
    const float* const x = a.x + m * a.ldx;
    gf_f32x4_t s[GATED ? 2 : 1];
    uint64_t nan_rows = 0;
#pragma unroll
    for (int i = 0; i < (GATED ? 2 : 1); ++i) {
        const float* at = sums + m * row + i * a.N + (n < a.N ? n : 0);
        gf_f32x4_t v[GF_PARTS];
#pragma unroll
        for (int p = 0; p < GF_PARTS; ++p) v[p] = p < runs ? *reinterpret_cast<const gf_f32x4_t*>(at + p * a.M * row) : gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
        s[i] = v[0];
        gf_f32x4_t s2 = v[GF_PARTS / 2];
#pragma unroll
        for (int p = 1; p < GF_PARTS / 2; ++p) {
            s[i] += v[p];
            s2 += v[GF_PARTS / 2 + p];
        }
        s[i] += s2;
        gf_finite(s[i], 0, [&](int) { return n < a.N; }, [&](int e) { return n + e + (i ? a.up_at : 0); }, x, a.ldx, a.w, a.ldw, a.K, nan_rows);
    }
    if (n >= a.N) return;
    if (GATED) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[0][e] = gf_gate(s[0][e], s[GATED][e]);
    }
    gf_store4(a.out + m * a.ldo, GATED ? nullptr : a.bias, s[0], n, a.N, a.vec_out);
}

// What the parts of the rows of x that are split at a time may take, and half of what the runs' sums may: the workspace is both.  A tile's parts lie
// within 2^31 bytes for every k up to the longest.
#define GF_MANY_BYTES (256ll << 20)
#define GF_MANY_LONGEST 65536

// Columns up to `whole` by workgroups that take all of k, in tiles of 16 mt rows; the others by workgroups that take `runs` of its eight runs.
struct gf_many_plan {
    int mt, whole, rest_mt, runs;      // (mt 0: columns that are all of the other kind; both 0: not by these kernels)
    int64_t rows;                      // of x at a time
    float us;
};

// us: a start, rounds of workgroups (two a unit at a time where they have the registers) with a time for a step, more of it where all
// units work, and for the end of a run, and the results' way (a million of them; `runs` < 8: to memory, back, and out).  A fit to 12,000 timed
// launches, all tiles and cuts of 4,900 products of 33 to 3,000 rows, 512 to 38,000 weight rows, k to 19,000: off by 2 to 6 % in the mean.
static float gf_many_us(int64_t M, int64_t weight_rows, int chunks, int mt, int runs) {
    static const struct {
        float start, step, full, run, out;
    } fit[2][3] = {{{12.5f, 0.612f, 0.156f, 0.188f, 2.7f}, {13.4f, 0.796f, 0.192f, 0.434f, 1.9f}, {13.3f, 0.914f, 0.213f, 0.585f, 1.8f}},
                   {{12.2f, 0.511f, 0.809f, 0.62f, 8.6f}, {12.7f, 0.795f, 0.158f, 0.75f, 9.0f}, {12.3f, 0.907f, 0.192f, 1.1f, 9.0f}}};
    const bool whole = runs == GF_PARTS;
    const auto& f = fit[!whole][mt / 2 - 2];
    const int per = (chunks + GF_PARTS - 1) / GF_PARTS, steps = 2 * (runs * per > chunks ? chunks : runs * per);
    const int64_t places = (!whole && mt == 4 ? 2 : 1) * zi_compute_units();
    const int64_t units = (M + 16 * mt - 1) / (16 * mt) * ((weight_rows + 127) / 128) * (GF_PARTS / runs), rounds = (units + places - 1) / places;
    return f.start + (float)rounds * (steps * (f.step + f.full * units / (rounds * places)) + runs * f.run) + f.out * 1e-6f * M * weight_rows;
}

static bool gf_many_fits(gf_many_plan* p, int M, int N, int K, bool gated) {
    const int chunks = (K + GF_KB - 1) / GF_KB;
    if ((p->whole < N && (N % 4 || p->whole % 4 || (p->runs != 4 && p->runs != 2))) || p->whole < 0 || p->whole > N) return false;
    const int64_t most = GF_MANY_BYTES / ((int64_t)chunks * 384) / 384 * 384, passes = (M + most - 1) / most;      // (whole tiles of every kind)
    p->rows = passes == 1 ? M : (M + passes * 384 - 1) / (passes * 384) * 384;
    return (p->rows + 63) / 64 * ((N + 63) / 64) < (1 << 23) && GF_PARTS * p->rows * (N - p->whole) * (gated ? 8 : 4) <= 2 * GF_MANY_BYTES;
}

// All columns in one cut, or whole rounds of the chip in the first and what would leave most of it idle in the second.
static gf_many_plan gf_many_best(int M, int N, int K, bool gated) {
    gf_many_plan best{0, 0, 0, 0, 0, 0.f};
    const int chunks = (K + GF_KB - 1) / GF_KB, nc = gated ? 64 : 128, twice = gated ? 2 : 1, cus = zi_compute_units();
    auto consider = [&](gf_many_plan p) {
        if (gf_many_fits(&p, M, N, K, gated) && (!best.us || p.us < best.us)) best = p;
    };
    gf_many_plan all{0, N, 0, 0, 0, 0.f};
    gf_many_fits(&all, M, N, K, gated);
    const int64_t rows = all.rows, passes = (M + rows - 1) / rows;
    const float split = 1e-6f * rows * K;
    for (int mt = 4; mt <= 8; mt += 2) {
        const int64_t m_tiles = (rows + 16 * mt - 1) / (16 * mt), col_tiles = (N + nc - 1) / nc;
        consider({mt, N, 0, 0, 0, passes * (split + gf_many_us(rows, (int64_t)N * twice, chunks, mt, GF_PARTS))});
        for (int runs = 2; runs < GF_PARTS; runs *= 2) consider({0, 0, mt, runs, 0, passes * (split + gf_many_us(rows, (int64_t)N * twice, chunks, mt, runs))});
        const int64_t full = m_tiles * col_tiles / cus * cus / m_tiles;      // tiles of columns in whole rounds
        if (full == 0 || full >= col_tiles) continue;
        const int whole = (int)full * nc;
        const float us = split + gf_many_us(rows, (int64_t)whole * twice, chunks, mt, GF_PARTS);
        for (int rest = 4; rest <= 8; rest += 2)
            for (int runs = 2; runs < GF_PARTS; runs *= 2)
                consider({mt, whole, rest, runs, 0, passes * (us + gf_many_us(rows, (int64_t)(N - whole) * twice, chunks, rest, runs) - 4.f)});      // (the split is launched once)
    }
    return best;
}

static gf_many_plan gf_many_as_told(int M, int N, int K, bool gated, int mt, int runs, int whole) {
    gf_many_plan p{mt, runs == GF_PARTS ? N : whole, mt, runs, 0, 0.f};
    if ((mt != 4 && mt != 6 && mt != 8) || !gf_many_fits(&p, M, N, K, gated)) p.mt = p.rest_mt = 0;
    return p;
}

static int64_t gf_many_bytes(const gf_many_plan& p, int64_t N, int chunks, bool gated) {
    return (p.rows + 15) / 16 * chunks * 6144 + GF_PARTS * p.rows * (N - p.whole) * (gated ? 8 : 4);
}

// Whether these kernels can make the product: operands that the others here take, in tiles that a launch can hold.
static bool gf_many_sizes(int M, int N, int K, int64_t ldx, int64_t ldw, int gated) {
    return M > 0 && N > 0 && K > GF_SPLIT_ABOVE && K <= GF_MANY_LONGEST && ldx >= K && ldw >= K && (int64_t)M * N < (1ll << 36) &&
           (gated ? zi_gemm_f32_swiglu_takes(nullptr, nullptr, M, N, K, ldx, ldw) : zi_gemm_f32_takes(nullptr, nullptr, N, K, ldx, ldw));
}

// Bytes of workspace with which zi_gemm_f32_many makes the product of M rows of x and N (gated: 2 N) weight rows, mt, runs and whole as
// there; 0 where it does not, or (mt 0) where it is not the faster way by both fits: of 5,000 products of 33 to 3,000 rows and sizes as above 3,500
// were given to these kernels and took 0.78 of the time in the mean, eleven of them more than 1.03 of it and 1.11 at worst.
// us, without and with the workspace, the split included, weights from memory: 17,920 x 1,536 with the activation at 256 / 512 / 2,048 rows 129 and 98,
// 200 and 170, 775 and 640; 1,536 x 8,960 89 and 67, 114 and 101, 457 and 331; 37,888 x 3,584 with it 465 and 375, 881 and 700, 3,447 and 2,827;
// 3,584 x 18,944 289 and 195, 531 and 376, 1,830 and 1,420.  Left to the others: few tiles or short runs, 2,048 x 1,536 at 450 rows 30 and 35, and some
// 60 rows and fewer (two more launches).
extern "C" int64_t zi_gemm_f32_many_workspace(int M, int N, int K, int64_t ldx, int64_t ldw, int gated, int mt, int runs, int whole) {
    if (!gf_many_sizes(M, N, K, ldx, ldw, gated)) return 0;
    const gf_many_plan p = mt ? gf_many_as_told(M, N, K, gated, mt, runs, whole) : gf_many_best(M, N, K, gated);
    if (!p.mt && !p.rest_mt) return 0;
    float tiles_us = 0.f;      // of the tiles without a workspace; 0 where other kernels make the product
    gf_choose(M, (int64_t)N * (gated ? 2 : 1), K, &tiles_us);
    tiles_us *= M > 512 ? 1.05f : 0.98f;      // (their fit is low, by 10 to 16 % with a standard deviation of 8 to 12 up to 512 rows, by 15 to 18 with one of 7 beyond)
    return mt || p.us < tiles_us ? gf_many_bytes(p, N, (K + GF_KB - 1) / GF_KB, gated) : 0;
}

template <int MT, bool GATED>
static void gf_many_launch(gf_many_args a, int runs, float* sums, hipStream_t stream) {
    constexpr int TM = 16 * MT, NC = GATED ? 64 : 128;
    a.m_tiles = (a.M + TM - 1) / TM;
    a.tiles = a.m_tiles * ((a.N + NC - 1) / NC);
    const int grid = (a.tiles + 7) / 8 * 8;
    if (runs == GF_PARTS) {
        gemm_f32_split_many_kernel<MT, GATED, false><<<grid, 4 * ZI_WAVE, 0, stream>>>(a);
    } else {
        gf_many_args b = a;
        b.out = sums;
        b.runs = runs;
        gemm_f32_split_many_kernel<MT, GATED, true><<<dim3(grid, GF_PARTS / runs), 4 * ZI_WAVE, 0, stream>>>(b);
        gf_add_runs_kernel<GATED><<<dim3((a.N + 1023) / 1024, a.M), 4 * ZI_WAVE, 0, stream>>>(sums, a, (a.chunks + a.per - 1) / a.per);
    }
}

// out[M,N] = x . w^T + bias, or (gated) up * silu(gate) of the first and the last N rows of w, through a workspace of
// zi_gemm_f32_many_workspace bytes; the bits of the kernels without one.  mt 0: as these sizes are made fastest; else blocks of 16 rows of x a
// tile (4, 6, 8), runs of k a workgroup of the columns from `whole` on (4 or 2, N and whole multiples of four), or 8: all columns whole.
extern "C" int zi_gemm_f32_many(float* out, const float* x, const float* w, const float* bias, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo,
                                int gated, int mt, int runs, int whole, void* workspace, int64_t bytes, hipStream_t stream) {
    ZI_REQUIRE(out && x && w && workspace, "gemm_f32_many: null operand");
    ZI_REQUIRE(gf_many_sizes(M, N, K, ldx, ldw, gated) && ldo >= N && ((uintptr_t)x | (uintptr_t)w | (uintptr_t)workspace) % 16 == 0 && !(gated && bias),
               "gemm_f32_many: M=%d N=%d K=%d is not taken, or not with these strides, alignment or bias", M, N, K);
    const gf_many_plan p = mt ? gf_many_as_told(M, N, K, gated, mt, runs, whole) : gf_many_best(M, N, K, gated);
    const int chunks = (K + GF_KB - 1) / GF_KB, per = (chunks + GF_PARTS - 1) / GF_PARTS;
    ZI_REQUIRE(p.mt || p.rest_mt, "gemm_f32_many: no tiles of %d blocks with %d runs from column %d on", mt, runs, whole);
    ZI_REQUIRE(bytes >= gf_many_bytes(p, N, chunks, gated), "gemm_f32_many: the workspace is too small");
    for (int64_t m = 0; m < M; m += p.rows) {
        const int rows = (int)(M - m < p.rows ? M - m : p.rows), blocks = (rows + 15) / 16;
        gf_many_args a{out + m * ldo, (const gf_u32x4_t*)workspace, x + m * ldx, w, bias, rows, p.whole, K, ldx, ldw, ldo, chunks, per,
                       ldo % 4 == 0 && (uintptr_t)out % 16 == 0, 0, 0, 0, N};
        float* const sums = (float*)((char*)workspace + (int64_t)blocks * chunks * 6144);
        gf_parts_kernel<<<dim3((2 * chunks + 3) / 4, blocks), 4 * ZI_WAVE, 0, stream>>>((gf_u32x4_t*)workspace, a.x, rows, K, ldx, chunks, per);
        auto go = [&](int blocks_of_rows, int runs_a_group) {
#define GF_GO(MT)                                                                  \
    if (blocks_of_rows == MT) {                                                    \
        if (gated) gf_many_launch<MT, true>(a, runs_a_group, sums, stream);        \
        else gf_many_launch<MT, false>(a, runs_a_group, sums, stream);             \
    }
            GF_GO(4) GF_GO(6) GF_GO(8)
#undef GF_GO
        };
        if (p.whole > 0) go(p.mt, GF_PARTS);
        if (p.whole < N) {
            a.N = N - p.whole;
            a.out += p.whole;
            a.w += p.whole * ldw;
            if (bias) a.bias += p.whole;
            go(p.rest_mt, p.runs);
        }
    }
    return zi_check_launch("gemm_f32_many");
}
