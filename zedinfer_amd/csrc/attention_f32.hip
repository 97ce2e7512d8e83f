// Causal grouped-query attention over the paged cache in float32 on the matrix cores (v_mfma_f32_16x16x4_f32: float32
// products and sums), for head sizes that are multiples of 16 up to 128 and pages of a multiple of 16 positions.
// attention_generic.hip is the same function for every other shape and for scores with caps, biases or distances.
//
// A workgroup owns 16 columns, (token, head) pairs that share a key/value head: 16 listed tokens of one head, or the
// heads of one token's group (a decoded token).  Its eight wavefronts share the keys: blocks of 16 positions, block b of
// the sequence to wavefront b mod 8, and their running maxima and sums meet in LDS at the end, in the wavefronts' order.
// So a column's result depends on its position and its keys alone, not on the columns beside it, nor on which of the
// two ways it came.  Scores are K . Q^T with keys as the instruction's rows, 16 bytes a lane straight from the cache
// (queries stay in registers); the layout of the result, four keys of one column a lane, is the layout the second
// product wants its probabilities in, and the transposed value cache gives the other operand in 16-byte pieces, so
// nothing passes through LDS in between.  The next block's keys travel during the softmax and the second product, its
// values during the next scores.
//
// Tokens of several sequences among the 16 are done sequence by sequence.  A masked probability is zero, but zero times
// an infinity or a NaN is not: where a block is not seen whole by all columns and one of its values is not finite, the
// second product is made with zeros in the place of such values, and their terms are added afterwards to the columns that
// see them.  A column that sees none keeps its bits, whatever lies in masked cells.
//
// Bound, for prompts, by the instruction's rate and the trips to the cache (16 queries share a pass over the keys); for
// decoded tokens by the trips that follow each other, one a block and wavefront.  Measured against the plain kernel
// (12 heads of 128, 2 key/value heads): a prompt of 450 tokens 585 to 39 us, 8 decoded tokens of 400 keys 176 to 13 us.
#include "zi_common.h"

typedef __attribute__((ext_vector_type(4))) float af_f32x4_t;

#define AF_WAVES 8
#define AF_COLS 16

// DT: head size / 16; DV: how many 16 dims of the values a workgroup makes, from blockIdx.z * DV on.
template <int DT, int DV>
__global__ void __launch_bounds__(AF_WAVES* ZI_WAVE)
attention_f32_kernel(float* __restrict__ out, const float* __restrict__ q, int64_t ldq, int64_t ldo, const float* __restrict__ kcache,
                     const float* __restrict__ vcache, const int32_t* __restrict__ tok_index, const int32_t* __restrict__ tok_seq,
                     const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ block_tables, int max_pages, int num_pages, int n,
                     int nh, int nkv, int page_size, int window, float scale, const float* __restrict__ sinks, int by_heads) {
    constexpr int D = DT * 16;
    const int d0 = DV == DT ? 0 : blockIdx.z * DV * 16;
    __shared__ __attribute__((aligned(16))) af_f32x4_t os[AF_WAVES][DV][ZI_WAVE];
    __shared__ float ms[AF_WAVES][AF_COLS], ls[AF_WAVES][AF_COLS];
    const int lane = threadIdx.x & (ZI_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE);
    const int c = lane & 15, g = lane >> 4;
    const int group = nh / nkv;
    // this lane's column: token t, head h
    const int at = by_heads ? blockIdx.x : blockIdx.x * AF_COLS + c;
    const int slices = (group + AF_COLS - 1) / AF_COLS, in_group = by_heads ? blockIdx.y % slices * AF_COLS + c : 0;
    const bool real = by_heads ? in_group < group : at < n;
    const int place = at < n ? at : n - 1;
    const int t = tok_index ? tok_index[place] : place;
    const int kvh = by_heads ? blockIdx.y / slices : blockIdx.y / group;
    const int h = by_heads ? kvh * group + (real ? in_group : 0) : blockIdx.y;
    const int p = tok_pos[t], seq = tok_seq[t];
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    const af_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    af_f32x4_t qr[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i) qr[i] = *reinterpret_cast<const af_f32x4_t*>(q + (int64_t)t * ldq + (int64_t)h * D + i * 16 + g * 4);

    uint64_t todo = __ballot(real);
    while (todo) {
        const int s = __builtin_amdgcn_readlane(seq, __builtin_ctzll(todo));
        const bool mine = real && seq == s;
        todo &= ~__ballot(mine);
        int hi_all = mine ? p : -1, lo_all = mine ? lo : 0x7fffffff;
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) {
            const int a = __shfl_xor(hi_all, o, ZI_WAVE), b = __shfl_xor(lo_all, o, ZI_WAVE);
            hi_all = a > hi_all ? a : hi_all;
            lo_all = b < lo_all ? b : lo_all;
        }
        hi_all = __builtin_amdgcn_readfirstlane(hi_all);
        lo_all = __builtin_amdgcn_readfirstlane(lo_all);
        const int32_t* bt = block_tables + (int64_t)s * max_pages;
        const int b0 = lo_all / 16, first = b0 + ((wave - b0) & (AF_WAVES - 1)), last = hi_all / 16;

        // the 16 positions of block b: their page (-1: none is held) and the addresses of this lane's pieces
        auto page_of = [&](int b) -> int {
            const int pi = (b < last ? b : last) * 16 / page_size;
            const int page = pi < max_pages ? bt[pi] : -1;
            return __builtin_amdgcn_readfirstlane(page < num_pages ? page : -1);
        };
        auto cell = [&](int page) -> int64_t { return ((int64_t)(page < 0 ? 0 : page) * nkv + kvh) * page_size * D; };
        af_f32x4_t kr[DT], vr[DV];
        auto fetch_k = [&](int b, int page) __attribute__((always_inline)) {
            const float* k = kcache + cell(page) + (int64_t)((b * 16) % page_size + c) * D + g * 4;
#pragma unroll
            for (int i = 0; i < DT; ++i) kr[i] = *reinterpret_cast<const af_f32x4_t*>(k + i * 16);
        };
        auto fetch_v = [&](int b, int page) __attribute__((always_inline)) {
            const float* v = vcache + cell(page) + (int64_t)(d0 + c) * page_size + (b * 16) % page_size + g * 4;
#pragma unroll
            for (int i = 0; i < DV; ++i) vr[i] = *reinterpret_cast<const af_f32x4_t*>(v + (int64_t)i * 16 * page_size);
        };
        float m = -INFINITY, l = 0.f;
        bool any = false;      // this column saw a key
        af_f32x4_t acc[DV];
#pragma unroll
        for (int i = 0; i < DV; ++i) acc[i] = zero;
        int page = page_of(first), page_next = page_of(first + AF_WAVES);
        fetch_k(first <= last ? first : last, page);
        fetch_v(first <= last ? first : last, page);
        for (int b = first; b <= last; b += AF_WAVES) {
            const int next = b + AF_WAVES <= last ? b + AF_WAVES : last;
            const int page_after = page_of(b + 2 * AF_WAVES);
            af_f32x4_t s0 = zero, s1 = zero;
#pragma unroll
            for (int i = 0; i < DT; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    af_f32x4_t& sc = i % 2 ? s1 : s0;
                    sc = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[i][j], qr[i][j], sc, 0, 0, 0);
                }
            s0 += s1;
            __builtin_amdgcn_sched_barrier(0);
            fetch_k(next, page_next);
            __builtin_amdgcn_sched_barrier(0);
            const int key = b * 16 + g * 4;
            bool seen[4];
            float top = -INFINITY;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                seen[e] = mine && page >= 0 && key + e <= p && key + e >= lo;
                any |= seen[e];
                s0[e] = seen[e] ? s0[e] * scale : -INFINITY;
                top = fmaxf(top, s0[e]);
            }
            top = fmaxf(top, __shfl_xor(top, 16, ZI_WAVE));
            top = fmaxf(top, __shfl_xor(top, 32, ZI_WAVE));
            const float m_new = fmaxf(m, top), corr = m == -INFINITY ? 0.f : expf(m - m_new);
            m = m_new;
            // (where all that was seen scores minus infinity, its weight is zero; a NaN stays one)
            const float from = m_new == -INFINITY ? 0.f : m_new;
            float sum = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s0[e] = seen[e] ? expf(s0[e] - from) : 0.f;
                sum += s0[e];
            }
            l = l * corr + sum;
#pragma unroll
            for (int i = 0; i < DV; ++i) acc[i] *= corr;
            bool by_key = false;
            if (__ballot(mine && !(seen[0] && seen[3]))) {      // (what a column sees of a block has no gaps)
                bool odd = false;
#pragma unroll
                for (int i = 0; i < DV; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) odd |= !(fabsf(vr[i][e]) < INFINITY);
                by_key = __ballot(odd) != 0;
            }
            if (by_key) {
#pragma unroll
                for (int i = 0; i < DV; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) vr[i][e] = fabsf(vr[i][e]) < INFINITY ? vr[i][e] : 0.f;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < DV; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[i][j], s0[j], acc[i], 0, 0, 0);
            if (by_key) {
                const float* v = vcache + cell(page) + (b * 16) % page_size + (int64_t)(d0 + g * 4) * page_size;
#pragma unroll 1
                for (int kk = 0; kk < 16; ++kk) {
                    const int e = kk & 3, from = (kk >> 2) * 16 + c;
                    const float pe = e == 0 ? s0[0] : e == 1 ? s0[1] : e == 2 ? s0[2] : s0[3];
                    const bool se = e == 0 ? seen[0] : e == 1 ? seen[1] : e == 2 ? seen[2] : seen[3];
                    const float pk = __shfl(pe, from, ZI_WAVE);
                    const bool sk = __shfl((int)se, from, ZI_WAVE) != 0;
                    const float* vk = v + kk;
#pragma unroll
                    for (int i = 0; i < DV; ++i) {
#pragma unroll
                        for (int x = 0; x < 4; ++x) {
                            const float val = *vk;
                            acc[i][x] += sk && !(fabsf(val) < INFINITY) ? pk * val : 0.f;
                            vk += x < 3 ? page_size : 13 * page_size;
                            asm volatile("" : "+v"(vk));      // (32 addresses held for a path hardly ever taken cost registers)
                        }
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            fetch_v(next, page_next);
            page = page_next;
            page_next = page_after;
        }
        l += __shfl_xor(l, 16, ZI_WAVE);
        l += __shfl_xor(l, 32, ZI_WAVE);
        const uint64_t who = __ballot(any);
        if (g == 0) {
            ms[wave][c] = m;
            ls[wave][c] = (who | who >> 16 | who >> 32 | who >> 48) >> c & 1 ? l : -1.f;      // (below zero: saw none)
        }
#pragma unroll
        for (int i = 0; i < DV; ++i) os[wave][i][lane] = acc[i];
        __syncthreads();
        float top = ms[0][c];
#pragma unroll
        for (int u = 1; u < AF_WAVES; ++u) top = fmaxf(top, ms[u][c]);
        float part[AF_WAVES], total = 0.f;
        bool none = true;
#pragma unroll
        for (int u = 0; u < AF_WAVES; ++u) {
            none &= ls[u][c] < 0.f;
            part[u] = ms[u][c] == -INFINITY ? 0.f : expf(ms[u][c] - top);
            total += ls[u][c] * part[u];
        }
        if (sinks) total += expf(sinks[h] - top);
        // (a token that sees no key, as one that stands behind a step's requests to fill it up, has zeros, not 0 / 0: sums over it
        // that are no numbers would be made again in the products that follow)
        const float inv = none ? 0.f : 1.f / total;
        for (int i = wave; i < DV; i += AF_WAVES) {
            af_f32x4_t o = os[0][i][lane] * part[0];
#pragma unroll
            for (int u = 1; u < AF_WAVES; ++u) o += os[u][i][lane] * part[u];
            if (mine) {
                float* dst = out + (int64_t)t * ldo + (int64_t)h * D + d0 + i * 16 + g * 4;
#pragma unroll
                for (int e = 0; e < 4; ++e) dst[e] = o[e] * inv;
            }
        }
        __syncthreads();
    }
}

extern "C" int zi_attention_f32_supported(int nh, int nkv, int d, int page_size) {
    return nkv > 0 && nh % nkv == 0 && d >= 16 && d <= 128 && d % 16 == 0 && page_size >= 16 && page_size % 16 == 0;
}

// Whether n tokens of so many sequences are the faster taken by heads than in tiles of 16 tokens.  A tile does the sequences among
// its tokens one after the other (on average 1 + 15 / (tokens a sequence) of them), while a token by heads is a workgroup for
// every key/value head; a launch past one workgroup a compute unit takes so many times longer.  From 16 tokens a sequence on, tiles.
// Measured, us, by heads against tiles: 12 heads, 2 key/value heads of 128, 20 sequences of 5 tokens 6.5 against 18, 64 of 3 tokens
// after 30 14 against 33, 16 of 8 after 1,000 53 against 74; 16 heads of 32 that share nothing, 64 sequences of 2 tokens 14 against 20,
// of 4 tokens 26 against 11 (tiles); 28 heads, 4 key/value heads, 20 sequences of 16 tokens 29 against 20 (tiles).
extern "C" int zi_attention_f32_by_heads(int n, int sequences, int nh, int nkv) {
    if (n < 1 || nkv < 1 || nh < nkv || n >= 16 * (int64_t)sequences) return 0;
    const double units = zi_compute_units();
    const double heads = (double)n * nkv * ((nh / nkv + AF_COLS - 1) / AF_COLS) / units, tiles = (double)((n + AF_COLS - 1) / AF_COLS) * nh / units;
    return (heads > 1 ? heads : 1) <= (tiles > 1 ? tiles : 1) * (1 + 15. * sequences / n);
}

// `by_heads`: a workgroup takes up to 16 heads of one token's group (decoded tokens), else 16 listed tokens of one head.  The
// results are the same.
extern "C" int zi_attention_f32(void* out, const void* q, int n, int64_t ldq, int64_t ldo, const void* kcache, const void* vcache,
                                const int32_t* tok_index, const int32_t* tok_seq, const int32_t* tok_pos, const int32_t* block_tables,
                                int max_pages, int num_pages, int nh, int nkv, int d, int page_size, int window, float scale,
                                const float* sinks, int by_heads, hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && max_pages > 0 && num_pages > 0 && window >= 0, "attention: bad sizes");
    ZI_REQUIRE(zi_attention_f32_supported(nh, nkv, d, page_size), "attention: unsupported heads (%d, %d), head_dim %d or page size %d", nh, nkv, d, page_size);
    ZI_REQUIRE(nh <= 65535, "attention: too many heads (%d)", nh);
    ZI_REQUIRE(ldq >= (int64_t)nh * d && ldo >= (int64_t)nh * d, "attention: row stride too small");
    ZI_REQUIRE(ldq % 4 == 0 && ((uintptr_t)q | (uintptr_t)kcache | (uintptr_t)vcache) % 16 == 0, "attention: rows must be 16-byte aligned");
    if (n == 0) return 0;
    const dim3 grid(by_heads ? n : (n + AF_COLS - 1) / AF_COLS, by_heads ? nkv * ((nh / nkv + AF_COLS - 1) / AF_COLS) : nh);
    // Few workgroups leave most units idle, and a wavefront's time is its matrix instructions (32 a block of 16 keys for the scores, 32
    // for the values at head size 128, two wavefronts a SIMD): then four workgroups make the scores each and a quarter of the dims,
    // the same sums of each.  us, one workgroup against four: 8 tokens of
    // 400 keys, 12 heads of 128 on 2 key/value heads, 16.6 to 12.9, of 900 28.0 to 21.2, of 100 9.2 to 8.0; 14 heads of 64 10.6 to 9.2.
    // (Two or four blocks of keys on their way a wavefront instead of one: 16.6 and 19.3 us at 400 keys, with the waits counted
    // exactly; the blocks' loads are not what a wavefront waits for.)
    const bool quarters = by_heads && d % 64 == 0 && (int64_t)grid.x * grid.y * 4 <= zi_compute_units();
#define ZI_AF_LAUNCH(DT, DV)                                                                                                       \
    attention_f32_kernel<DT, DV><<<dim3(grid.x, grid.y, DT / DV), AF_WAVES * ZI_WAVE, 0, stream>>>(                                 \
        (float*)out, (const float*)q, ldq, ldo, (const float*)kcache, (const float*)vcache, tok_index, tok_seq, tok_pos, block_tables, \
        max_pages, num_pages, n, nh, nkv, page_size, window, scale, sinks, by_heads)
#define ZI_AF(DT)                     \
    case DT: ZI_AF_LAUNCH(DT, DT); break
    if (quarters && d == 64) ZI_AF_LAUNCH(4, 1);
    else if (quarters) ZI_AF_LAUNCH(8, 2);
    else switch (d / 16) {
        ZI_AF(1); ZI_AF(2); ZI_AF(3); ZI_AF(4); ZI_AF(5); ZI_AF(6); ZI_AF(7); ZI_AF(8);
    }
#undef ZI_AF
#undef ZI_AF_LAUNCH
    return zi_check_launch("attention_f32");
}
