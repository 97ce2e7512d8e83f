// out[M,N] = x[M,K] . w[N,K]^T for many rows of x in bfloat16 (a prompt's products), on v_mfma_f32_16x16x32_bf16 with float32 sums,
// and what follows the product where that is one value of one or two columns: a bias, an activation, gate and up.
//
// A workgroup makes a tile of 16 WM MW rows by 32 NW columns, its wavefronts WM along the rows and two along the columns, MW x NW blocks
// of 16 x 16 each.  Both operands go straight into LDS (buffer_load_dwordx4 ... lds, 1 KB an instruction, rows of 128 bytes with piece c
// of row q at place c xor (q / 2 mod 8)), k in steps of 64 through as many buffers as LDS holds, up to five.  A step is two halves:
// while the matrix instructions of one half run, the operands of the next are read from LDS and a share of a later step's loads is issued,
// so that neither the reads nor the loads come in a burst.  The step's one barrier stands between the halves: behind it the buffer
// is free whose last operands were read in the first half, and the next step's, whose loads every wavefront has waited for by count, may
// be read.  Workgroups are resident and take several tiles; the steps of a workgroup's tiles follow each other without a gap, so
// that the next tile's operands are on their way during a tile's last steps and its epilogue.
//
// Which row of the weights stands where in LDS is free, and so chosen that a lane's outputs follow each other in memory (gt_row_of):
// 16-byte stores, and gate and up of one column in one lane.
//
// What bounds it: LDS, which takes a step's loads at 64 bytes a cycle and gives 128 (256 x 256 tiles: 2,560 cycles a step for 2,048 of
// matrix instructions, 192 x 192 1,920 for 1,152), the loads in flight where only two buffers fit, and rows of a tile that the XCD's cache has to fetch (tiles
// that run at a time on an XCD are neighbours).
#include "zi_common.h"
#include "zi_activation.h"
#include "zi_api.h"

typedef __attribute__((ext_vector_type(8))) __bf16 gt_bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float gt_f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned gt_u32x4_t;
typedef __attribute__((ext_vector_type(2))) unsigned gt_u32x2_t;

union gt_pack {
    gt_u32x4_t u;
    gt_bf16x8_t b;
};

#define GT_KB 64
#define GT_LDS 160         // KB
#define GT_XCDS 8
#define GT_GROUP 4         // tiles of rows that are worked on together (gt_place)

// what the kernel ends with
#define GT_BF16 0          // bfloat16 results, with a bias
#define GT_F32 1           // float32 results, with a bias
#define GT_SWIGLU 2        // gate and up rows of the weights alternate in blocks of 8; bfloat16
#define GT_GATED 3         // the gate rows come first, the up rows from row `up_at` on; an activation by its code; bfloat16
#define GT_ERF 4           // the same with the error function's GELU (a kernel of its own: the function is 40 instructions)

__device__ __forceinline__ void gt_to_lds(__amdgpu_buffer_rsrc_t from, gt_u32x4_t* to, int lane_at) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host's pass knows loads of this size for no target)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(from, to, 16, lane_at, 0, 0, 0);
#endif
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t gt_buffer(const zi_bf16* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<zi_bf16*>(p), 0, bytes, 0x00020000);
}

// The sums stay in the accumulation registers over the loop and its ends: without this the compiler moves all of them to other
// registers and back once a step.
#ifdef __HIP_DEVICE_COMPILE__
#define GT_KEEP(v) asm volatile("" : "+a"(v))
#else
#define GT_KEEP(v)
#endif

struct gt_args {
    void* out;
    const zi_bf16 *x, *w, *bias;
    int M, N, K;                   // N: columns of the result (gate and up make one)
    int64_t ldx, ldw, ldo;
    int up_at, act;
    int row_tiles, col_tiles, steps, units;      // units: tiles
};

// Where row q of a wavefront's 16 NW rows of LDS comes from, as (column of the result, gate or up).  Blocks of 16 go to the matrix
// cores one by one and a lane gets four rows of each, 4 j .. 4 j + 3.
template <int NW, bool GATES>
__device__ __forceinline__ int gt_row_of(int q, int* up) {
    const int b = q / 16, r = q % 16, j = r / 4, e = r % 4;
    *up = GATES ? b % 2 : 0;
    if (GATES) return b / 4 * 4 + 4 <= NW ? b / 4 * 32 + j * 8 + b / 2 % 2 * 4 + e : b / 2 * 16 + r;
    return b / 2 * 2 + 2 <= NW ? b / 2 * 32 + j * 8 + b % 2 * 4 + e : q;
}

// Unit of workgroup b in its round i, or -1.  Workgroups go to the XCDs in turn; units that run at a time on one XCD are neighbours.
__device__ __forceinline__ int gt_unit(const gt_args& g, int b, int i) {
    const int grid = gridDim.x, base = i * grid, count = g.units - base < grid ? g.units - base : grid;
    const int share = (count + GT_XCDS - 1) / GT_XCDS, id = b % GT_XCDS * share + b / GT_XCDS;
    return count > 0 && b / GT_XCDS < share && id < count ? base + id : -1;
}

// A unit's place: GT_GROUP tiles of rows at a time, the rows fastest, so that 32 units are about a square of tiles.
__device__ __forceinline__ void gt_place(const gt_args& g, int unit, int* m, int* n) {
    const int per = GT_GROUP * g.col_tiles, group = unit / per, in = unit - group * per;
    const int rows = g.row_tiles - group * GT_GROUP < GT_GROUP ? g.row_tiles - group * GT_GROUP : GT_GROUP;
    *n = in / rows;
    *m = group * GT_GROUP + in - *n * rows;
}

// up * z sigmoid(s).  exp(-s) is 2^t (1 + rest): the rounding of t, which the chip's exponential would make large for large s, is put
// back; then the chip's reciprocal.  (The library's exponential and quotient are 30 instructions a value, which nothing overlaps with
// at a tile's end.)
__device__ __forceinline__ float gt_sigmoid_mul(float z, float s, float up) {
    const float t = s * -1.44269504f, rest = __builtin_fmaf(s, -1.44269504f, -t) + s * -1.92596303e-8f;
    const float e = __builtin_amdgcn_exp2f(t);
    return up * (z * __builtin_amdgcn_rcpf(1.f + (fabsf(t) < 126.f ? __builtin_fmaf(e, rest * 0.693147182f, e) : e)));      // (beyond, e or rest may be infinite)
}

// up times the activation of z: SiLU, GELU in its tanh form, which is z sigmoid(2 u), u = sqrt(2 / pi) (z + 0.044715 z^3), or with the
// error function.
template <int EPI>
__device__ __forceinline__ float gt_gate(float z, float up, int act) {
    if (EPI == GT_ERF) return zi_activation(z, ZI_ACT_GELU_ERF) * up;
    if (EPI == GT_SWIGLU) return gt_sigmoid_mul(z, z, up);
    const float u = z * __builtin_fmaf(0.044715f * 2.f * 0.7978845608028654f * z, z, 2.f * 0.7978845608028654f);
    return gt_sigmoid_mul(z, act == ZI_ACT_GELU_TANH ? u : z, up);
}

template <int WM, int MW, int NW>
struct gt_shape {
    static constexpr int WAVES = 2 * WM, ROWS = 16 * WM * MW, WROWS = 32 * NW, LOADS = (ROWS + WROWS) / 8, FIT = GT_LDS / LOADS,
                         STAGES = FIT < 5 ? FIT : 5;
};

template <int WM, int MW, int NW, int EPI>
__global__ void __launch_bounds__(128 * WM, 1) gemm_tiles_kernel(gt_args g) {
    typedef gt_shape<WM, MW, NW> Z;
    constexpr int S = Z::STAGES, WAVES = Z::WAVES, BM = Z::ROWS, BN = Z::WROWS, XI = BM / 8, PW = Z::LOADS / WAVES, PIECES = Z::LOADS * ZI_WAVE;
    constexpr bool GATES = EPI >= GT_SWIGLU, HALVES = EPI >= GT_GATED;
    constexpr int COLS = GATES ? BN / 2 : BN;
    static_assert(XI % WAVES == 0 && Z::LOADS % WAVES == 0 && S >= 2 && (!GATES || NW % 2 == 0), "whole shares, gates and ups in pairs");
    __shared__ __attribute__((aligned(16))) gt_u32x4_t all[PIECES * S];
    const int tid = threadIdx.x, lane = tid & (ZI_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / ZI_WAVE);
    const int r = lane & 15, j = lane >> 4, sw = (r >> 1) & 7;
    // Load i of a wavefront takes rows of LDS 8 (i WAVES + wave) .. + 7: lane l row l / 8 of them, the piece that belongs at place l % 8.
    // Rows past M, and of the weights past the last, lie past the buffers' ends and are zeros; other weight rows that belong to no column of the
    // result (gates past the last one) are read and their products not stored.
    int lane_at[PW];
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int L = i * WAVES + wave, q = (L < XI ? L : L - XI) * 8 + lane / 8;
        int row = q;
        if (L >= XI) {
            int up;
            const int c = q / (16 * NW) * (GATES ? 8 * NW : 16 * NW) + gt_row_of<NW, GATES>(q % (16 * NW), &up);
            row = EPI == GT_SWIGLU ? c / 8 * 16 + up * 8 + c % 8 : HALVES ? c + up * g.up_at : c;
        }
        lane_at[i] = (int)(row * (L < XI ? g.ldx : g.ldw) * 2) + ((lane & 7) ^ ((q >> 1) & 7)) * 16;
    }
    struct work {
        const zi_bf16 *x, *w;      // of the tile's first rows, at its first column
        int x_bytes, w_bytes, steps;
    };
    const int last_row = EPI == GT_SWIGLU ? 2 * g.N : HALVES ? g.up_at + g.N : g.N;
    auto work_of = [&](int round) {
        work f{g.x, g.w, 0, 0, 64};
        const int unit = gt_unit(g, blockIdx.x, round);
        if (unit >= 0) {
            int m, n;
            gt_place(g, unit, &m, &n);
            const int row = n * (EPI == GT_SWIGLU ? BN : COLS);
            f.steps = g.steps;
            f.x = g.x + (int64_t)m * BM * g.ldx;
            f.w = g.w + (int64_t)row * g.ldw;
            f.x_bytes = (int)(((int64_t)((g.M - m * BM < BM ? g.M - m * BM : BM) - 1) * g.ldx + g.K) * 2);
            f.w_bytes = (int)(((int64_t)(last_row - row - 1) * g.ldw + g.K) * 2);
        }
        return f;
    };
    work now = work_of(0), next = now;
    __amdgpu_buffer_rsrc_t xb = gt_buffer(g.x, 0), wb = gt_buffer(g.w, 0);
    // step t of this tile, or, past its end, of the next one (there is always room for that: no tile has fewer steps than buffers)
    auto aim = [&](int t) __attribute__((always_inline)) {
        const bool over = t >= now.steps;
        const int k = (over ? t - now.steps : t) * GT_KB;
        const int x_bytes = (over ? next.x_bytes : now.x_bytes) - k * 2, w_bytes = (over ? next.w_bytes : now.w_bytes) - k * 2;
        xb = gt_buffer((over ? next.x : now.x) + k, x_bytes > 0 ? x_bytes : 0);
        wb = gt_buffer((over ? next.w : now.w) + k, w_bytes > 0 ? w_bytes : 0);
    };
    auto issue = [&](gt_u32x4_t* buf, int lo, int hi) __attribute__((always_inline)) {
#pragma unroll
        for (int i = lo; i < hi; ++i) gt_to_lds(i * WAVES < XI ? xb : wb, buf + (i * WAVES + wave) * ZI_WAVE, lane_at[i]);
    };
    const int wm = wave % WM, wn = wave / WM;
    const int x_at = (wm * MW * 16 + r) * 8, w_at = BM * 8 + (wn * NW * 16 + r) * 8;
    gt_f32x4_t acc[NW][MW];
    gt_pack a0[NW], b0[MW], a1[NW], b1[MW];        // the operands of a step's halves
    auto read = [&](const gt_u32x4_t* buf, int half, gt_pack (&a)[NW], gt_pack (&b)[MW]) __attribute__((always_inline)) {
        const int p = (half * 4 + j) ^ sw;
#pragma unroll
        for (int m = 0; m < MW; ++m) b[m].u = buf[x_at + m * 128 + p];
#pragma unroll
        for (int n = 0; n < NW; ++n) a[n].u = buf[w_at + n * 128 + p];
    };
    auto multiply = [&](gt_pack (&a)[NW], gt_pack (&b)[MW]) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NW; ++n)
#pragma unroll
            for (int m = 0; m < MW; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[n].b, b[m].b, acc[n][m], 0, 0, 0);
    };
    // products between two reads; fewer in front of the barrier, whose wait for the reads is then shorter
    constexpr int PER = MW * NW / (MW + NW) > 1 ? MW * NW / (MW + NW) : 1, FEWER = PER > 1 ? PER - 1 : 1;
    constexpr int EARLY = S > 2 ? (PW + 1) / 2 : PW;       // loads behind the barrier; the others come before the next one
    int cur = 0, free = (S - 1) * PIECES;                    // the step's buffer, the one that loads go to
    auto step = [&](int t) __attribute__((always_inline)) {
        issue(all + free, EARLY, PW);
        read(all + cur, 1, a1, b1);
        multiply(a0, b0);
#pragma unroll
        for (int i = 0; i < MW + NW; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (i < PW - EARLY) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, FEWER, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        zi_wait_loads<(S - 2) * PW, true>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        free = cur;
        cur = cur == (S - 1) * PIECES ? 0 : cur + PIECES;
        aim(t + S);
        issue(all + free, 0, EARLY);
        read(all + cur, 0, a0, b0);
        multiply(a1, b1);
#pragma unroll
        for (int i = 0; i < MW + NW; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (i < EARLY) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < S; ++i) {
        aim(i);
        issue(all + i * PIECES, 0, i < S - 1 ? PW : EARLY);
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("" ::: "memory");
    zi_wait_loads<(S - 2) * PW + EARLY, true>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    read(all, 0, a0, b0);
    for (int round = 0;; ++round) {
        const int unit = gt_unit(g, blockIdx.x, round);
        if (unit < 0) break;
        next = work_of(round + 1);
#pragma unroll
        for (int n = 0; n < NW; ++n)
#pragma unroll
            for (int m = 0; m < MW; ++m) {
                acc[n][m] = gt_f32x4_t{0.f, 0.f, 0.f, 0.f};
                GT_KEEP(acc[n][m]);
            }
        for (int t = 0; t < now.steps; ++t) step(t);
#pragma unroll
        for (int n = 0; n < NW; ++n)
#pragma unroll
            for (int m = 0; m < MW; ++m) GT_KEEP(acc[n][m]);
        // C[n][m] of a block: row 4 j + e of the weights, row r of x.  Stores are counted like loads and in the same order: they only
        // make the next steps' waits for loads that are older longer.
        int tm, tn;
        gt_place(g, unit, &tm, &tn);
        const int col0 = tn * COLS + wn * (GATES ? 8 * NW : 16 * NW), row0 = tm * BM + wm * MW * 16 + r;
        constexpr int BLOCKS = GATES ? 4 : 2;         // of which a lane's outputs are eight columns; fewer blocks left make four
#pragma unroll
        for (int n = 0; n < NW; n += BLOCKS) {
            const bool eight = n + BLOCKS <= NW;
            const int col = col0 + (GATES ? n * 8 : n * 16) + j * (eight ? 8 : 4);
            float bias[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (!GATES && g.bias && col < g.N) {
#pragma unroll
                for (int e = 0; e < (eight ? 8 : 4); ++e) bias[e] = zi_load(g.bias + col + e);
            }
#pragma unroll
            for (int m = 0; m < MW; ++m) {
                const int row = row0 + m * 16;
                float v[8];
#pragma unroll
                for (int h = 0; h < (eight ? 2 : 1); ++h)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int up = n + 2 * h + 1 < NW ? n + 2 * h + 1 : 0;
                        if (GATES) v[h * 4 + e] = gt_gate<EPI>(acc[n + 2 * h][m][e], acc[up][m][e], g.act);
                        else v[h * 4 + e] = acc[n + h][m][e] + bias[h * 4 + e];
                    }
                if (row < g.M && col < g.N) {
                    if (EPI == GT_F32) {
                        float* to = (float*)g.out + (int64_t)row * g.ldo + col;
                        *reinterpret_cast<gt_f32x4_t*>(to) = gt_f32x4_t{v[0], v[1], v[2], v[3]};
                        if (eight) *reinterpret_cast<gt_f32x4_t*>(to + 4) = gt_f32x4_t{v[4], v[5], v[6], v[7]};
                    } else {
                        zi_bf16* to = (zi_bf16*)g.out + (int64_t)row * g.ldo + col;
                        const uint32_t p0 = zi_pack_bf16x2(v[0], v[1]), p1 = zi_pack_bf16x2(v[2], v[3]);
                        if (eight) *reinterpret_cast<gt_u32x4_t*>(to) = gt_u32x4_t{p0, p1, zi_pack_bf16x2(v[4], v[5]), zi_pack_bf16x2(v[6], v[7])};
                        else *reinterpret_cast<gt_u32x2_t*>(to) = gt_u32x2_t{p0, p1};
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        now = next;
    }
    zi_wait_loads<0, true>();       // (no load may arrive after the workgroup's LDS is another's)
}

// ---- the tile of a product ------------------------------------------------------------------------------------------------
// WM, MW, NW, and what a step of 64 columns takes in ns: c0 where few workgroups run, c0 + c1 where the chip is full of them.
struct gt_tile {
    int wm, mw, nw, c0, c1;
};
#define GT_TILES(X) X(2, 2, 2, 173, 63) X(2, 4, 2, 248, 88) X(2, 4, 3, 304, 115) X(2, 4, 4, 363, 160) X(2, 4, 6, 532, 157) \
    X(2, 6, 5, 584, 168) X(2, 6, 7, 803, 196) X(4, 2, 8, 608, 254) X(4, 3, 6, 638, 252) X(4, 4, 8, 1172, 303)
static const gt_tile gt_tiles[] = {
#define GT_ROW(WM, MW, NW, C0, C1) {WM, MW, NW, C0, C1},
    GT_TILES(GT_ROW)
#undef GT_ROW
};
#define GT_TILE_COUNT ((int)(sizeof(gt_tiles) / sizeof(gt_tiles[0])))
#define GT_FEWEST_STEPS 5       // no fewer than a kernel has buffers
#define GT_ABOVE 256            // rows of x up to which products are the few-rows kernels' or the library's

#define GT_NARROW 512           // columns of the result and of x up to which they are as well: launches, whoever makes them

enum gt_kind { GT_PLAIN, GT_GATES };      // what is made of a product

struct gt_plan {
    int tile;
    double ns;
};

// The tile by the time it takes: a launch, for each round of workgroups its steps and its epilogue, the results' way to memory.  The constants
// are a fit to 9,000 timed launches (10 tiles and, of products in up to 8 cuts of k that no kernel here makes any more, each cut; 500 products, 129 to
// 9,000 rows, 512 to 49,888 columns, k 512 to 27,648, weights from memory): off by 6 % in the mean, and the choice by them is within 0.3 % of the
// best in the mean, 9 % at worst.
static gt_plan gt_best(int M, int64_t N, int K, int kind) {
    gt_plan best{-1, 0.0};
    const int cus = zi_compute_units(), steps = K / GT_KB;
    for (int i = 0; i < GT_TILE_COUNT; ++i) {
        const gt_tile& t = gt_tiles[i];
        if (kind == GT_GATES && t.nw % 2) continue;
        const int rows = 16 * t.wm * t.mw, wrows = 32 * t.nw, cols = kind == GT_GATES ? wrows / 2 : wrows;
        const int64_t tiles = (int64_t)((M + rows - 1) / rows) * ((N + cols - 1) / cols), rounds = (tiles + cus - 1) / cus;
        if (tiles > (1 << 24)) continue;
        const double fill = (double)tiles / (double)(rounds * cus);
        const double ns = 4300.0 + rounds * (steps * (t.c0 + t.c1 * fill) + 0.084 * rows * wrows) + (double)M * (double)N * 0.000232;
        if (best.tile < 0 || ns < best.ns) best = gt_plan{i, ns};
    }
    return best;
}

static bool gt_sizes(int64_t M, int64_t N, int64_t K) {
    return M >= 1 && N >= 8 && N % 8 == 0 && K % GT_KB == 0 && K >= GT_KB * GT_FEWEST_STEPS && M * N < ((int64_t)1 << 40);
}

// The kernel here or the library's product (with the launch of the activation, for gate and up) for more than 256 rows.  0: not taken here;
// 1: taken, but the library is the faster by the rule; 2: the kernel here is; 3: and surely (a gate/up product).  The rule holds the time by the fit
// against 16 us, 10 more from 10 GFLOP on, and 1.3 PFLOP/s, and says 2 up to 100 GFLOP of a plain product and 3 TFLOP of a gate/up product, 3 from
// 0.7 of the library's time down.  7,143 products timed both ways, the library's the fastest of its proposals, and 9,027 with its first one (which runs
// where nothing was measured), weights from memory, 257 to 20,000 rows, 520 to 30,000 columns, k 576 to 27,648, up to 10 TFLOP.  Own time of the
// library's, geometric mean and one in twenty, where the rule says 2:
//                        up to 10 GFLOP     30             100            1,000          3,000          beyond, all of them
//   plain, first         0.83 and 1.02      0.91 and 1.06  0.97 and 1.17                                0.94 and 1.16
//   plain, fastest       0.88 and 1.10      0.94 and 1.08  1.00 and 1.17                                1.02 and 1.16
//   gate/up, first       0.64 and 0.87      0.76 and 1.02  0.79 and 0.97  0.85 and 1.06  0.94 and 1.03  0.99 and 1.08
//   gate/up, fastest     0.64 and 0.87      0.79 and 1.06  0.82 and 0.99  0.89 and 1.09  0.97 and 1.06  1.01 and 1.08
// Beyond the bounds single sizes are up to 1.25 times as fast either way, the library 0.9 to 1.4 PFLOP/s by how its tiles come out, which no rule on the
// sizes that was tried tells apart, so an engine times both (the faster one takes 0.945 of the time of the library's fastest in the mean, plain, and 0.874),
// and where nothing was measured the library keeps them.  Where the rule says 3, 0.72, above 1 in one of eighty and 1.09 at most.  us, own and the library's
// fastest: gate/up with SwiGLU of 8,960 columns x 1,536 at 320 / 512 / 1,024 / 2,048 rows 27 and 34, 43 and 39, 62 and 76, 115 and 122, of 18,944 x
// 3,584 105 and 118, 161 and 134, 270 and 260, 465 and 530, of 27,648 x 5,120 at 2,048 / 4,096 950 and 980, 1,980 and 2,020; 1,536 x 8,960 at 320 / 1,024 / 2,048 /
// 8,192 rows 41 and 31, 54 and 49, 66 and 71, 215 and 171.
#define GT_PLAIN_MOST 1e11
#define GT_GATES_MOST 3e12

extern "C" int zi_gemm_tiles_pays(int M, int N, int K, int kind) {
    if (M <= GT_ABOVE || N <= GT_NARROW || K <= GT_NARROW || kind < GT_PLAIN || kind > GT_GATES || !gt_sizes(M, N, K)) return 0;
    const gt_plan p = gt_best(M, N, K, kind);
    if (p.tile < 0) return 0;
    const double flops = 2.0 * M * (kind == GT_GATES ? 2.0 : 1.0) * N * K;
    double library = 16000.0 + 10000.0 * (flops < 1e10 ? flops / 1e10 : 1.0) + flops / 1.3e6;
    if (kind == GT_GATES) library += 4000.0 + 6.0 * M * N / 4500.0;
    if (p.ns >= library || flops > (kind == GT_GATES ? GT_GATES_MOST : GT_PLAIN_MOST)) return 1;
    return kind == GT_GATES && p.ns < 0.7 * library ? 3 : 2;
}

extern "C" int zi_gemm_tiles_count() { return GT_TILE_COUNT; }

template <int WM, int MW, int NW>
static int gt_launch(gt_args g, int epi, hipStream_t stream) {
    typedef gt_shape<WM, MW, NW> Z;
    const int cols = epi >= GT_SWIGLU ? Z::WROWS / 2 : Z::WROWS, cus = zi_compute_units();
    g.row_tiles = (g.M + Z::ROWS - 1) / Z::ROWS;
    g.col_tiles = (g.N + cols - 1) / cols;
    const int64_t units = (int64_t)g.row_tiles * g.col_tiles;
    ZI_REQUIRE(units <= (1 << 24), "gemm_tiles: too many tiles");
    g.units = (int)units;
    const int most = cus / GT_XCDS * GT_XCDS > 0 ? cus / GT_XCDS * GT_XCDS : GT_XCDS;
    const int grid = g.units < most ? (g.units + GT_XCDS - 1) / GT_XCDS * GT_XCDS : most;
    if (epi == GT_BF16) gemm_tiles_kernel<WM, MW, NW, GT_BF16><<<grid, 128 * WM, 0, stream>>>(g);
    else if (epi == GT_F32) gemm_tiles_kernel<WM, MW, NW, GT_F32><<<grid, 128 * WM, 0, stream>>>(g);
    else if constexpr (NW % 2 == 0) {
        if (epi == GT_SWIGLU) gemm_tiles_kernel<WM, MW, NW, GT_SWIGLU><<<grid, 128 * WM, 0, stream>>>(g);
        else if (g.act == ZI_ACT_GELU_ERF) gemm_tiles_kernel<WM, MW, NW, GT_ERF><<<grid, 128 * WM, 0, stream>>>(g);
        else gemm_tiles_kernel<WM, MW, NW, GT_GATED><<<grid, 128 * WM, 0, stream>>>(g);
    } else {
        return zi_fail("gemm_tiles: gate and up take a tile of an even number of blocks");
    }
    return zi_check_launch("gemm_tiles");
}

// epi 0: out [M,N] bfloat16, bias (bfloat16 [N] or null); 1: the same in float32; 2: w [2 N, K] holds gate and up rows in turn, 8 each, out = up * silu(gate); 3: w holds the gate rows, then from
// row up_at >= N on the up rows, out = act(gate) * up, act 0 SiLU, 1 GELU in its tanh form, 2 with the error function.
// tile: a number below zi_gemm_tiles_count(), or -1 for the one that is taken for these sizes.
extern "C" int zi_gemm_tiles(void* out, int epi, const void* x, const void* w, const void* bias, int M, int N, int K, int64_t ldx,
                             int64_t ldw, int64_t ldo, int up_at, int act, int tile, hipStream_t stream) {
    ZI_REQUIRE(out && x && w, "gemm_tiles: null operand");
    ZI_REQUIRE(epi >= GT_BF16 && epi <= GT_GATED, "gemm_tiles: unknown epilogue %d", epi);
    ZI_REQUIRE(gt_sizes(M, N, K), "gemm_tiles: unsupported sizes M=%d N=%d K=%d (N a multiple of 8, K of 64 and at least %d)", M, N, K,
               GT_KB * GT_FEWEST_STEPS);
    // a tile's rows have to lie within 2^31 bytes, the weights from a tile's first row on too
    const int64_t wrows = epi == GT_SWIGLU ? 2 * (int64_t)N : epi == GT_GATED ? (int64_t)up_at + N : N;
    ZI_REQUIRE(ldx >= K && ldw >= K && ldo >= N && ldx % 8 == 0 && ldw % 8 == 0 && ldx <= (1 << 21) && wrows * ldw < (1 << 30),
               "gemm_tiles: a row stride is too short, too long or no multiple of 8, or the weights are too large");
    ZI_REQUIRE(((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16 == 0 && ldo % (epi == GT_F32 ? 4 : 8) == 0,
               "gemm_tiles: x, w and the rows of out must be 16-byte aligned");
    ZI_REQUIRE(epi != GT_GATED || (up_at >= N && act >= ZI_ACT_SILU && act <= ZI_ACT_GELU_ERF), "gemm_tiles: bad rows of up or activation %d", act);
    ZI_REQUIRE(epi < GT_SWIGLU || !bias, "gemm_tiles: gate and up take no bias");
    ZI_REQUIRE(tile >= -1 && tile < GT_TILE_COUNT, "gemm_tiles: no tile %d", tile);
    if (tile < 0) tile = gt_best(M, N, K, epi >= GT_SWIGLU ? GT_GATES : GT_PLAIN).tile;
    gt_args g{out, (const zi_bf16*)x, (const zi_bf16*)w, (const zi_bf16*)bias, M, N, K, ldx, ldw, ldo, up_at, act, 0, 0, K / GT_KB, 0};
    int at = 0;
#define GT_GO(WM, MW, NW, C0, C1) \
    if (tile == at++) return gt_launch<WM, MW, NW>(g, epi, stream);
    GT_TILES(GT_GO)
#undef GT_GO
    return zi_fail("gemm_tiles: no tile %d", tile);
}
