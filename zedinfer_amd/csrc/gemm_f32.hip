// out[M,N] = x[M,K] . w[N,K]^T (+ bias[N]), everything float32: the entry points, and the products of up to GF_SPLIT_ABOVE columns, on the
// matrix cores' float32 instruction (v_mfma_f32_16x16x4_f32: float32 products and float32 accumulation, no reduced precision).  Longer k
// goes to gemm_f32_split.hip, which adds up products of bfloat16 parts at up to 1.5 times the speed and with smaller errors; its start,
// turning and splitting operands, costs a short k more than it gains (8 and 24 rows, us, here and there: 1,000 x 500 4.7 and 5.2, 5.5 and 6.1;
// 5,000 x 1,100 9.9 and 9.6, 14.1 and 19.2; 9,000 x 128 5.7 and 6.3, 8.1 and 11.2).  Figures of longer k below are of these kernels too.
//
// One order of the sums, the same in every kernel here, so that a row's result does not depend on M, on the tile it
// falls in or on the rest of the batch: k is cut into GF_PARTS runs of whole chunks of 32 (a function of K alone); within
// a run the first and the second 16 of every chunk are two chains, each 16 summed as four instructions whose lanes hold
// k = 4 g + j (instruction j, lane group g); a run's sum is first + second chain; the sums of each half of the runs
// are added in rising order, then the two halves, then the bias.
//
// gemm_f32_stream_kernel, for few rows, is bound by the one pass over the weights.  A workgroup owns 16 weight rows (8 for up
// to 8 rows of x) and its eight wavefronts take a run of k each, so N / 16 workgroups of eight wavefronts share the stream
// however few rows the matrix has, with nothing left to add outside the workgroup.  Operands come straight from memory in
// the matrix cores' layout, several chunks ahead in registers; loads past the end are out of the buffer's range and give
// zeros without a branch.  For up to 8 rows the 16 x 16 instruction holds 8 weight rows twice, at the two halves of a
// chunk, beside the 8 rows of x twice: an instruction's load takes eight whole 128-byte lines, and two of the result's
// four quadrants are the two chains.
// gemm_f32_tile_kernel, for many rows, is bound by the instruction's rate (152 TFLOP/s in a large library product): tiles
// through LDS (three buffers, one barrier a chunk of 32 k, three more chunks on their way in registers), the operands of the next
// half of a chunk on their way from LDS while one half is multiplied; with two buffers, and a chunk's operands asked for after
// its barrier, 448 rows of 1,536 x 8,960 took 144 us where they take 123 now, 512 rows of 17,920 x 1,536 244 and 231, 256 rows of
// 4,608 x 3,584 102 and 97.  The scheduling barriers keep the loads ahead of the products: without them the compiler moves a loop's
// loads to its end and waits for all of them at its head.
//
// Measured, weights from memory, us, launch included: 8 rows of 5,000 x 300 (N x K) 5.0, 1,000 x 500 4.7; 450 rows 22.5 and 10.5; 4,000 rows of
// 4,000 x 512 160 (102 TFLOP/s).
#include "zi_gemm_f32.h"

#define GF_KB 32             // k of a chunk
#define GF_HELD_CHUNKS 6      // chunks of a run that a wavefront may have to hold of x
#define GF_BUFFERS 3         // chunks that the tile kernel holds in LDS, and as many on their way in registers

// PAIR: 8 weight rows and up to 8 rows of x; else 16 weight rows and up to 16 * MT rows of x a workgroup.  RING chunks are
// on their way while one is worked on.
template <int MT, bool PAIR, int RING>
__global__ void __launch_bounds__(GF_PARTS* ZI_WAVE)
gemm_f32_stream_kernel(float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w,
                       const float* __restrict__ bias, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, int per, int vec_out) {
    constexpr int NR = PAIR ? 8 : 16, MR = PAIR ? 8 : 16 * MT, H = PAIR ? 1 : 2;
    __shared__ __attribute__((aligned(16))) gf_f32x4_t part[GF_PARTS][MT][ZI_WAVE];
    const int lane = threadIdx.x & (ZI_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE);
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * NR, m0 = blockIdx.y * MR;
    const int rows_w = N - n0 < NR ? N - n0 : NR, rows_x = M - m0 < MR ? M - m0 : MR;
    const __amdgpu_buffer_rsrc_t wb = gf_rows(w + (int64_t)n0 * ldw, ldw, rows_w, K), xb = gf_rows(x + (int64_t)m0 * ldx, ldx, rows_x, K);
    const int row = PAIR ? r & 7 : r;
    const int k_lane = (PAIR ? (r >> 3) * 64 : 0) + g * 16;       // byte of a chunk that this lane starts at
    const int w_row = row < rows_w ? (int)(row * ldw * 4) : GF_OUT;
    int x_row[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) x_row[t] = t * 16 + row < rows_x ? (int)((t * 16 + row) * ldx * 4) : GF_OUT;
    const int chunks = (K + GF_KB - 1) / GF_KB;
    const int c0 = wave * per, c1 = c0 + per < chunks ? c0 + per : chunks;

    gf_f32x4_t wr[RING][H], xr[RING][H][MT];
    auto fetch = [&](const int slot, int c) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const int k = c * (GF_KB * 4) + h * 64 + k_lane;
            const bool in = c < c1 && k < K * 4;
#pragma unroll
            for (int t = 0; t < MT; ++t) xr[slot][h][t] = gf_load<0>(xb, in && x_row[t] != GF_OUT ? x_row[t] + k : GF_OUT);
            // a weight is read once by one workgroup: past L2, where an instruction takes whole lines
            wr[slot][h] = gf_load<PAIR ? 2 : 0>(wb, in && w_row != GF_OUT ? w_row + k : GF_OUT);
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
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int h = 0; h < H; ++h)
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        acc[h][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wr[s][h][j], xr[s][h][t][j], acc[h][t], 0, 0, 0);
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
            for (int e = 0; e < 4; ++e) s[e] += __shfl(acc[0][t][e], (lane + 40) & 63, ZI_WAVE);
        } else {
            s += acc[H - 1][t];
        }
        part[wave][t][lane] = s;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < MT * ZI_WAVE; i += GF_PARTS * ZI_WAVE) {
        const int t = i / ZI_WAVE, l = i % ZI_WAVE, m = t * 16 + (l & 15), n = (l >> 4) * 4;
        gf_f32x4_t s = part[0][t][l], s2 = part[GF_PARTS / 2][t][l];
#pragma unroll
        for (int p = 1; p < GF_PARTS / 2; ++p) {
            s += part[p][t][l];
            s2 += part[GF_PARTS / 2 + p][t][l];
        }
        s += s2;
        if (m < rows_x && n < rows_w) gf_store4(out + (int64_t)(m0 + m) * ldo, bias, s, n0 + n, N, vec_out);
    }
}

// The same for up to 16 rows of x and more groups of weight rows than there are compute units: a workgroup keeps its wavefronts' runs
// of x in registers (PER chunks a wavefront, at most) and walks over groups of 8 (PAIR) or 16 weight rows, gridDim.x apart.  As
// soon as a chunk of weights has been used, its registers are filled with the same chunk of the next group: PER chunks are always
// on their way, x passes the loads once a workgroup instead of once a group, as many bytes again as the weights' for 8 rows, and a
// workgroup's start and end come once.  The eight runs' sums meet in one of two LDS buffers, so a group costs one barrier, which
// does not wait for loads; the wavefronts take the adding and storing in turn.  GATED: a group is as many gate rows as up rows (row
// n and row N + n of w) and the outputs are up * silu(gate).
//
// Bound by the stream of the weights.  Measured against the stream kernel above (weights from memory, us, launch
// included), 1 and 8 rows: 17,920 x 1,536 29.0 to 20.6 and 35.0 to 23.8 (4.6 TB/s), 151,936 x 1,536 206 to 143 and 261 to 163 (5.7), 37,888
// x 3,584 115 to 88 and 151 to 90 (6.0), 3,000 x 512 6.1 to 3.8 and 6.6 to 4.4; 16 rows 17,920 x 1,536 37.7 to 25.3, 151,936 x 1,536
// 264 to 177, 5,000 x 1,000 11.7 to 11.3.  With the activation 8 rows of 17,920 x 1,536 take 23.8 us, the product and the activation's
// launch 37.3 before.
template <bool PAIR, int PER, bool GATED>
__global__ void __launch_bounds__(GF_PARTS* ZI_WAVE, (PAIR ? 1 : 2) * PER <= 8 ? 4 : 2)
gemm_f32_held_kernel(float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                     int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, int per, int vec_out, int groups) {
    constexpr int NR = PAIR ? 8 : 16, NC = GATED ? NR / 2 : NR, H = PAIR ? 1 : 2;
    __shared__ __attribute__((aligned(16))) gf_f32x4_t part[2][GF_PARTS][ZI_WAVE];
    const int lane = threadIdx.x & (ZI_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE);
    const int r = lane & 15, g = lane >> 4, row = PAIR ? r & 7 : r;
    const int chunks = (K + GF_KB - 1) / GF_KB, c0 = wave * per;
    const int mine = chunks - c0 < per ? chunks - c0 : per;       // chunks of this wavefront's run (none or fewer at the end of k)
    const int k0 = c0 * (GF_KB * 4) + (PAIR ? (r >> 3) * 64 : 0) + g * 16;      // the first byte of a row that this lane loads
    const __amdgpu_buffer_rsrc_t xb = gf_rows(x, ldx, M, K);
    const int x_row = row < M ? (int)(row * ldx * 4) : GF_OUT;
    const int w_row = (int)((GATED && row >= NC ? N + row - NC : row) * ldw * 4);
    // the weight rows of a group: what lies past the last one gives zeros (or, of a gate row past the last, an output that is not stored)
    auto weights = [&](int group) {
        const int64_t n0 = (int64_t)group * NC;
        const int rows = group >= groups ? 0 : (GATED ? N : 0) + (int)(N - n0 < NC ? N - n0 : NC);
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(w + (rows ? n0 * ldw : 0)), 0,
                                                 rows ? (int)(((int64_t)(rows - 1) * ldw + K) * 4) : 0, 0x00020000);
    };
    auto in = [&](int s, int h) { return s < mine && k0 + s * (GF_KB * 4) + h * 64 < K * 4; };
    gf_f32x4_t xr[PER][H], wr[PER][H];
    __amdgpu_buffer_rsrc_t wb = weights(blockIdx.x);
    auto fetch = [&](const int s) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < H; ++h)
            wr[s][h] = gf_load<PAIR ? 2 : 0>(wb, in(s, h) ? w_row + k0 + s * (GF_KB * 4) + h * 64 : GF_OUT);
    };
#pragma unroll
    for (int s = 0; s < PER; ++s) {
#pragma unroll
        for (int h = 0; h < H; ++h)
            xr[s][h] = gf_load<0>(xb, in(s, h) && x_row != GF_OUT ? x_row + k0 + s * (GF_KB * 4) + h * 64 : GF_OUT);
        fetch(s);
        __builtin_amdgcn_sched_barrier(0);
    }
    int b = 0, turn = 0;
    for (int group = blockIdx.x; group < groups; group += gridDim.x, b ^= 1, turn = (turn + 1) % GF_PARTS) {
        wb = weights(group + (int)gridDim.x);
        gf_f32x4_t acc[H];
#pragma unroll
        for (int h = 0; h < H; ++h) acc[h] = gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < PER; ++s) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int h = 0; h < H; ++h) acc[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(wr[s][h][j], xr[s][h][j], acc[h], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            fetch(s);
            __builtin_amdgcn_sched_barrier(0);
        }
        gf_f32x4_t sum = acc[0];
        if (PAIR) {
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] += __shfl(acc[0][e], (lane + 40) & 63, ZI_WAVE);
        } else {
            sum += acc[H - 1];
        }
        part[b][wave][lane] = sum;
        // all sums are in LDS (and the buffer's reader of two groups ago is past the barrier of the last one); loads travel on
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        if (wave != turn) continue;
        gf_f32x4_t s = part[b][0][lane], s2 = part[b][GF_PARTS / 2][lane];
#pragma unroll
        for (int p = 1; p < GF_PARTS / 2; ++p) {
            s += part[b][p][lane];
            s2 += part[b][GF_PARTS / 2 + p][lane];
        }
        s += s2;
        if (GATED) {
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = gf_gate(s[e], __shfl(s[e], lane + (PAIR ? 16 : 32), ZI_WAVE));
        }
        const int64_t n = (int64_t)group * NC + g * 4;
        if (r < M && g * 4 < NC && n < N) gf_store4(out + (int64_t)r * ldo, bias, s, (int)n, N, vec_out);
    }
}

// TM x 32 NT outputs a workgroup; GROUPS (1 or 2) groups of four wavefronts, each over half of the runs of k when there are
// two; TM/2 x 16 NT outputs a wavefront.  GATED (NT = 2): of a wavefront's two
// blocks of 16 weight rows one are gate rows and one the up rows of the same outputs (rows n and N + n of w), and TM x 32 outputs
// up * silu(gate) are what the tile leaves.
template <int TM, int NT, int GROUPS, bool GATED, bool SHORT>
__global__ void __launch_bounds__(256 * GROUPS, GROUPS == 1 ? 3 : 2)
gemm_f32_tile_kernel(float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w,
                     const float* __restrict__ bias, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, int per, int vec_out,
                     int m_tiles, int tiles) {
    constexpr int TN = 32 * NT, XP = TM / 32, WP = TN / 32, MT = TM / 32;     // pieces a thread loads; 16 x 16 tiles a wavefront
    __shared__ __attribute__((aligned(16))) gf_f32x4_t lds[GROUPS][GF_BUFFERS][(TM + TN) * 8];
    // the tiles that share weight rows follow each other on one XCD (workgroup i runs on XCD i mod 8)
    const int per_xcd = (tiles + 7) / 8, tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (tile >= tiles) return;
    static_assert(!GATED || NT == 2, "a gate and an up block a wavefront");
    constexpr int NC = GATED ? TN / 2 : TN;
    const int m0 = (tile % m_tiles) * TM, n0 = (tile / m_tiles) * NC;
    const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE), group = wave_all / 4, wave = wave_all & 3;
    const int tid = threadIdx.x & 255, lane = tid & (ZI_WAVE - 1);
    const int r = lane & 15, g = lane >> 4;
    const int rows_w = N - n0 < NC ? N - n0 : NC, rows_x = M - m0 < TM ? M - m0 : TM;
    const __amdgpu_buffer_rsrc_t wb = gf_rows(w + (int64_t)n0 * ldw, ldw, (GATED ? N : 0) + rows_w, K), xb = gf_rows(x + (int64_t)m0 * ldx, ldx, rows_x, K);
    // a thread loads piece tid % 8 (16 bytes) of rows tid / 8, + 32, ...; piece c of row q lies at place c xor (q / 2 mod 8)
    const int pc = tid & 7, pr = tid >> 3;
    const int place = pc ^ ((pr >> 1) & 7);            // the same for rows 32 apart
    int x_row[XP], w_row[WP];
#pragma unroll
    for (int p = 0; p < XP; ++p) x_row[p] = pr + 32 * p < rows_x ? (int)((pr + 32 * p) * ldx * 4) : GF_OUT;
#pragma unroll
    for (int p = 0; p < WP; ++p) {
        // GATED: row q of the tile is row q % 16 + 16 (q / 32) of the gate rows, of the up rows if q / 16 is odd
        const int q = GATED ? 16 * p + (pr & 15) : pr + 32 * p;
        w_row[p] = q < rows_w ? (int)((q + (GATED && (pr & 16) ? N : 0)) * ldw * 4) : GF_OUT;
    }
    const int chunks = (K + GF_KB - 1) / GF_KB, half = per * (GF_PARTS / 2);
    const int c0 = group * half, c1 = GROUPS == 2 && c0 + half < chunks ? c0 + half : chunks;
    const int steps = GROUPS == 2 ? half : chunks;      // the same for both groups: they share the barriers
    gf_f32x4_t xr[GF_BUFFERS][XP], wr[GF_BUFFERS][WP];
    auto fetch = [&](const int slot, int c) __attribute__((always_inline)) {
        const int k = c * (GF_KB * 4) + pc * 16;
        const bool in = c < c1 && k < K * 4;
#pragma unroll
        for (int p = 0; p < XP; ++p) xr[slot][p] = gf_load<0>(xb, in && x_row[p] != GF_OUT ? x_row[p] + k : GF_OUT);
#pragma unroll
        for (int p = 0; p < WP; ++p) wr[slot][p] = gf_load<0>(wb, in && w_row[p] != GF_OUT ? w_row[p] + k : GF_OUT);
    };
    auto stash = [&](const int slot) __attribute__((always_inline)) {
        gf_f32x4_t* xs = lds[group][slot], *ws = xs + TM * 8;
#pragma unroll
        for (int p = 0; p < XP; ++p) xs[(pr + 32 * p) * 8 + place] = xr[slot][p];
#pragma unroll
        for (int p = 0; p < WP; ++p) ws[(pr + 32 * p) * 8 + place] = wr[slot][p];
    };
    const int wm = (wave & 1) * (TM / 2), wn = (wave >> 1) * (TN / 2);
    const gf_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    gf_f32x4_t acc[2][MT][NT], sum[MT][NT], first[MT][NT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) acc[0][t][u] = acc[1][t][u] = sum[t][u] = first[t][u] = zero;
    int in_part = 0, parts = 0;
    gf_f32x4_t va[2][NT], vb[2][MT];
    const int sw = (r >> 1) & 7;
    auto read = [&](const int b, const int h) __attribute__((always_inline)) {      // the operands of a half of the chunk in buffer b
        const gf_f32x4_t* xs = lds[group][b], *ws = xs + TM * 8;
#pragma unroll
        for (int u = 0; u < NT; ++u) va[h][u] = ws[(wn + u * 16 + r) * 8 + ((h * 4 + g) ^ sw)];
#pragma unroll
        for (int t = 0; t < MT; ++t) vb[h][t] = xs[(wm + t * 16 + r) * 8 + ((h * 4 + g) ^ sw)];
    };
    auto multiply = [&](const int h) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int u = 0; u < NT; ++u)
                    acc[h][t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[h][u][j], vb[h][t][j], acc[h][t][u], 0, 0, 0);
    };
    // Chunk c lies in buffer and slot c mod 3.  While a half is multiplied the next one's operands are on their way from LDS; between
    // the halves the chunk after the next goes into LDS (its buffer was last read a step ago) and its registers are asked for anew.
    auto step = [&](const int s, int c) __attribute__((always_inline)) {
        constexpr int B = GF_BUFFERS;
        read(s, 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0);
        __builtin_amdgcn_sched_barrier(0);
        read((s + 1) % B, 0);
        stash((s + 2) % B);
        __builtin_amdgcn_sched_barrier(0);
        fetch((s + 2) % B, c + 2 + B);
        __builtin_amdgcn_sched_barrier(0);
        multiply(1);
        if (++in_part == per) {                         // a run of k ends
            in_part = 0;
            ++parts;
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    sum[t][u] += acc[0][t][u] + acc[1][t][u];
                    acc[0][t][u] = acc[1][t][u] = zero;
                    if (GROUPS == 1 && parts == GF_PARTS / 2) {
                        first[t][u] = sum[t][u];
                        sum[t][u] = zero;
                    }
                }
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };
#pragma unroll
    for (int s = 0; s < GF_BUFFERS; ++s) {
        fetch(s, c0 + s);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        stash(s);
        __builtin_amdgcn_sched_barrier(0);
        fetch(s, c0 + GF_BUFFERS + s);
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    read(0, 0);
    // (the large tiles have no registers for an ending of their own, 240 against 207 us: steps past the end add zeros; SHORT: at most two
    // steps, 9,000 x 64 at 1,024 rows 28 us with three)
    int c = 0;
    for (; !SHORT && c + (TM == 64 ? 1 : GF_BUFFERS) <= steps; c += GF_BUFFERS) {
#pragma unroll
        for (int s = 0; s < GF_BUFFERS; ++s) step(s, c0 + c + s);
    }
    if (SHORT || TM < 64) {
        if (c < steps) step(0, c0 + c);
        if (c + 1 < steps) step(1, c0 + c + 1);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) sum[t][u] += acc[0][t][u] + acc[1][t][u];       // (zeros where the last run ended)
    if (GROUPS == 2) {
        // the second half's sums go through LDS to the first group's wavefronts
        gf_f32x4_t* hand = lds[0][0];
        static_assert(GROUPS == 1 || (int)(sizeof(lds) / 16) >= 4 * MT * NT * ZI_WAVE, "the sums of four wavefronts fit");
        if (group == 1) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int u = 0; u < NT; ++u) hand[((wave * MT + t) * NT + u) * ZI_WAVE + lane] = sum[t][u];
        }
        __syncthreads();
        if (group == 1) return;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int u = 0; u < NT; ++u) {
                first[t][u] = sum[t][u];
                sum[t][u] = hand[((wave * MT + t) * NT + u) * ZI_WAVE + lane];
            }
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int m = m0 + wm + t * 16 + r;
        if (m >= M) continue;
        if (GATED) {
            const int n = n0 + wn / 2 + g * 4;
            const gf_f32x4_t gate = first[t][0] + sum[t][0], up = first[t][NT - 1] + sum[t][NT - 1];
            gf_f32x4_t s;
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = gf_gate(gate[e], up[e]);
            if (n < N) gf_store4(out + (int64_t)m * ldo, nullptr, s, n, N, vec_out);
            continue;
        }
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            const int n = n0 + wn + u * 16 + g * 4;
            if (n < N) gf_store4(out + (int64_t)m * ldo, bias, first[t][u] + sum[t][u], n, N, vec_out);
        }
    }
}

// Whether these kernels take the operands (all float32): whole 16-byte pieces of every row, rows of a tile within a buffer's
// range, and weight rows whose workgroups fit a launch of one dimension (2^32 threads; 64 a row for up to 8 rows of x).
bool zi_gemm_f32_takes(const void* x, const void* w, int N, int K, int64_t ldx, int64_t ldw) {
    return K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0 && ldx < (1 << 21) && ldw < (1 << 21) &&
           N <= (1 << 25);
}

// Which kernel M rows of x and N weight rows take is a matter of filling the compute units only.  Up to 16 rows a stream of the
// weights, 8 or 16 of them a workgroup (one row of a 151,936-row head 190 in pairs, 233 us without), with x held in registers once
// there are more such groups than units and k is not too long for it (see there).  9 to 16 rows go twice over groups of 8 weight rows
// while both passes are one round of workgroups, 1,024 weight rows (us, twice over 8 against once over 16, 9 and 16 rows: 896 x 4,864
// 13.2 and 12.8 against 17.3 and 20.3, 1,024 x 1,024 5.9 and 6.0 against 6.7 and 7.3; with two workgroups a unit 2,048 x 2,048 12.0
// and 12.9 against 9.5 and 10.7, 1,536 x 8,960 32.6 and 37.2 against 29.1 and 34.8, 2,000 x 256 5.8 and 6.0 against 4.0 and 4.2; twelve
// chunks on their way instead of six gained nothing, 21.4 against 20.9 us at 8 rows).  16 rows a workgroup while that gives no unit a
// second workgroup (32 rows, 1,536 x 8,960: 34 against 52 us), 32 rows up to 32 rows and then while the same holds (64 rows:
// 52 against 84 us for the tiles).  Beyond, tiles of 32 x 64 in two halves of k while they are one round of workgroups
// (256 rows, 1,536 x 8,960: 85 us, one group 110, tiles of 64 x 64 184), of 32 x 96 where those make one round of what
// would be two (448 rows: 122 against 148, 2,560 x 2,560 at 288 rows 39 against 46, 2,816 x 1,024 at 256 18.6 against 22.1, 6,144 x
// 2,048 at 128 34 against 40); from six rounds of 64 x 64 tiles on those (17,920 x 1,536 at 448 rows 206
// against 215 us, at 256 rows, 4.4 rounds, 131 against 129); else 32 x 64, in two halves up to three rounds (448
// rows, 2,048 x 1,536: 30 against 33; 1,024 rows, four rounds: 59 against 58).  The large tiles work a multiple of three chunks, so not
// for a short k that is none, where those past its end count (us, 64 x 64 against 32 x 64: 4,000 rows 4,000 x 128 71 and 53, x 320 120 and
// 107, x 512 171 and 161, but 1,024 rows 9,000 x 384 71 and 74, 4,000 rows 4,000 x 896 266 and 282).
// Up to K = 128 the second half of the runs is empty, so one group (4,000 rows, 128 x 128: 5.7 against 6.8 us), and up to K = 192 while two
// halves would be more than a round (6,144 x 132 at 128 rows 7.3 against 8.4 in tiles of 32 x 96, x 192 8.4 and 8.6; 2,000 x 192 at 320 rows
// 7.7 and 7.9).  Up to K = 64 a workgroup is little more than its start, so the
// larger tiles (1,024 rows, 9,000 x 64: 20.4 against 22.8, in halves 59), after 32 rows a workgroup up to two a unit (320 rows, 256 x 32:
// 3.3 against 3.6 us).
static gf_kernel gf_kernel_for(int M, int64_t N, int K) {
    if (K > GF_SPLIT_ABOVE) return zi_gemm_f32_split_kernel(M, N, K);
    const int chunks = (K + GF_KB - 1) / GF_KB;
    const int64_t cus = zi_compute_units(), n16 = (N + 15) / 16, m32 = (M + 31) / 32;
    const int64_t t32 = m32 * ((N + 63) / 64), t96 = m32 * ((N + 95) / 96), t64 = (int64_t)((M + 63) / 64) * ((N + 63) / 64);
    if (M <= 8) return (N + 7) / 8 > cus ? GF_HELD_PAIRS : GF_PAIRS;
    if (M <= 16 && n16 > cus) return GF_HELD_ROWS16;
    if (M <= 16) return (N + 7) / 8 * 2 <= cus ? GF_PAIRS : GF_ROWS16;
    if (n16 * ((M + 15) / 16) <= cus) return GF_ROWS16;
    if (M <= 32 || n16 * m32 <= (chunks <= 2 ? 2 : 1) * cus) return GF_ROWS32;
    if (chunks <= 2) return GF_TILE_64;
    if (chunks <= GF_PARTS / 2 || (chunks <= 6 && t32 > cus)) return GF_TILE_32;
    if (t32 <= cus) return GF_TILE_32_HALVES;
    if (t96 <= cus) return GF_TILE_96_HALVES;
    if (t64 >= 6 * cus && (chunks > 16 || chunks % 3 == 0)) return GF_TILE_64;
    return t32 <= 3 * cus ? GF_TILE_32_HALVES : GF_TILE_32;
}

// (for tests: the kernel by its place in the list above)
extern "C" int zi_gemm_f32_kernel(int M, int N, int K) {
    return gf_kernel_for(M, N, K);
}

static_assert((GF_SPLIT_ABOVE + GF_KB - 1) / GF_KB <= GF_PARTS * GF_HELD_CHUNKS, "the longest k's runs fit the kernels that hold x");

template <bool GATED>
static int gf_launch(float* out, const float* x, const float* w, const float* bias, int M, int N, int K, int64_t ldx, int64_t ldw,
                     int64_t ldo, hipStream_t stream) {
    if (K > GF_SPLIT_ABOVE) return zi_gemm_f32_split_launch(GATED, out, x, w, bias, M, N, K, ldx, ldw, ldo, stream);
    const int chunks = (K + GF_KB - 1) / GF_KB, per = (chunks + GF_PARTS - 1) / GF_PARTS;
    const int vec_out = ldo % 4 == 0 && (uintptr_t)out % 16 == 0;
#define ZI_GF_STREAM(MT, PAIR, RING)                                                                                                     \
    gemm_f32_stream_kernel<MT, PAIR, RING><<<dim3((N + (PAIR ? 7 : 15)) / (PAIR ? 8 : 16), (M + (PAIR ? 8 : 16 * MT) - 1) / (PAIR ? 8 : 16 * MT)), \
                                             GF_PARTS * ZI_WAVE, 0, stream>>>(out, x, w, bias, M, N, K, ldx, ldw, ldo, per, vec_out)
    // two workgroups a unit while a lane has registers for that (128), else one
#define ZI_GF_HELD(PAIR, PER)                                                                                                            \
    do {                                                                                                                                 \
        const int nc = (PAIR ? 8 : 16) / (GATED ? 2 : 1), groups = (N + nc - 1) / nc;                                                        \
        const int places = zi_compute_units() * ((PAIR ? 1 : 2) * PER <= 8 ? 2 : 1);                                                         \
        gemm_f32_held_kernel<PAIR, PER, GATED><<<groups < places ? groups : places, GF_PARTS * ZI_WAVE, 0, stream>>>(                         \
            out, x, w, bias, M, N, K, ldx, ldw, ldo, per, vec_out, groups);                                                               \
    } while (0)
    // (rows in as many launches as 2^32 threads of one make necessary: a row's result does not depend on them)
#define ZI_GF_TILE(TM, NT, G, SHORT)                                                                                                              \
    do {                                                                                                                                  \
        const int nc = 32 * NT / (GATED ? 2 : 1);                                                                                              \
        const int64_t nt = (N + nc - 1) / nc, most = ((1ll << 31) / (256 * G)) / nt * TM;                                                      \
        for (int64_t m = 0; m < M; m += most) {                                                                                           \
            const int rows = (int)(M - m < most ? M - m : most), mt = (rows + TM - 1) / TM, tiles = (int)(mt * nt);                              \
            gemm_f32_tile_kernel<TM, NT, G, GATED, SHORT><<<(tiles + 7) / 8 * 8, 256 * G, 0, stream>>>(out + m * ldo, x + m * ldx, w, bias, rows, N, \
                                                                                                   K, ldx, ldw, ldo, per, vec_out, mt, tiles);  \
        }                                                                                                                                 \
    } while (0)
    switch (gf_kernel_for(M, (int64_t)N * (GATED ? 2 : 1), K)) {
        case GF_HELD_PAIRS:
            if (per <= 2) ZI_GF_HELD(true, 2);
            else if (per <= 4) ZI_GF_HELD(true, 4);
            else ZI_GF_HELD(true, 6);
            break;
        case GF_HELD_ROWS16:
            if (per <= 2) ZI_GF_HELD(false, 2);
            else if (per <= 4) ZI_GF_HELD(false, 4);
            else ZI_GF_HELD(false, 6);
            break;
        case GF_TILE_64:
            if (chunks <= 2) ZI_GF_TILE(64, 2, 1, true);
            else ZI_GF_TILE(64, 2, 1, false);
            break;
        case GF_TILE_32: ZI_GF_TILE(32, 2, 1, false); break;
        case GF_TILE_32_HALVES: ZI_GF_TILE(32, 2, 2, false); break;
        default:
            if constexpr (GATED) {
                return zi_fail("gemm_f32: no gated kernel for %d rows of %d x %d", M, N, K);      // (zi_gemm_f32_swiglu_takes says so)
            } else {
                switch (gf_kernel_for(M, N, K)) {
                    case GF_PAIRS: ZI_GF_STREAM(1, true, 6); break;
                    case GF_ROWS16: ZI_GF_STREAM(1, false, 4); break;
                    case GF_ROWS32: ZI_GF_STREAM(2, false, 3); break;
                    default: ZI_GF_TILE(32, 3, 2, false); break;
                }
            }
    }
#undef ZI_GF_STREAM
#undef ZI_GF_HELD
#undef ZI_GF_TILE
    return zi_check_launch("gemm_f32");
}

// The launch; the sizes are checked by the caller (zi_gemm_generic).
int zi_gemm_f32_launch(float* out, const float* x, const float* w, const float* bias, int M, int N, int K, int64_t ldx, int64_t ldw,
                       int64_t ldo, hipStream_t stream) {
    return gf_launch<false>(out, x, w, bias, M, N, K, ldx, ldw, ldo, stream);
}

// Whether zi_gemm_f32_swiglu takes M rows of x and the [2 inter, K] weights: what the product's own kernels take, with the up rows within
// 2^31 bytes of the gate rows they belong to, where the kernel that the product would take has the activation in its end.
extern "C" int zi_gemm_f32_swiglu_takes(const void* x, const void* w, int M, int inter, int K, int64_t ldx, int64_t ldw) {
    if (M < 1 || M > 65535 * 64 || inter < 1 || K < 1 || inter > (1 << 24) || ldx < K || ldw < K || !zi_gemm_f32_takes(x, w, 2 * inter, K, ldx, ldw)) return 0;
    if (((int64_t)inter + 64) * ldw * 4 >= (1ll << 31) - 64) return 0;
    const gf_kernel k = gf_kernel_for(M, 2ll * inter, K);
    if (k == GF_TILE_96_HALVES) return K > GF_SPLIT_ABOVE;      // (three blocks of weight rows a wavefront here, two there)
    return k == GF_HELD_PAIRS || k == GF_HELD_ROWS16 || k == GF_TILE_64 || k == GF_TILE_32 || k == GF_TILE_32_HALVES || k == GF_TILE_64_QUARTERS;
}

// out[M, inter] = up * silu(gate), gate and up the products of x with the first and the last inter rows of w: the bits of the product
// and the activation one after the other.
extern "C" int zi_gemm_f32_swiglu(float* out, const float* x, const float* w, int M, int inter, int K, int64_t ldx, int64_t ldw, int64_t ldo,
                                  hipStream_t stream) {
    ZI_REQUIRE(zi_gemm_f32_swiglu_takes(x, w, M, inter, K, ldx, ldw), "gemm_f32_swiglu: M=%d inter=%d K=%d is not taken", M, inter, K);
    ZI_REQUIRE(ldo >= inter, "gemm_f32_swiglu: leading dimension too small");
    return gf_launch<true>(out, x, w, nullptr, M, inter, K, ldx, ldw, ldo, stream);
}
