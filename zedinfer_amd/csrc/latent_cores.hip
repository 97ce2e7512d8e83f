// Latent attention on the matrix cores (bfloat16 cache, float32 scores and sums; see latent.hip for what is
// computed).  A row is one (token, head); all heads of a token meet the same latents, and neighbouring tokens
// nearly the same, so a workgroup takes 16 rows a wavefront of ONE entry (rows in the order token, head) and walks
// the keys its rows see in blocks of 32:
//
//   stage    the block's latents and key parts, [32][rank + rot], from the pages straight into LDS
//            (global_load_lds_dwordx4), one block ahead, in one of two buffers; where its keys lie in the pool is asked for
//            two blocks ahead, a lane a key, and traded between lanes.  Rows are not padded but swizzled: the 16-byte
//            piece c of row k sits at place c xor la_swizzle(k), so that neither product's reads meet in a bank: sixteen
//            rows' piece c and eight rows' pieces c, c + 1 (c even) lie in different banks
//   scores   S[key][row] = K . Q^T   v_mfma_f32_16x16x32_bf16: first operand the keys' rows from LDS, second the
//            queries, held in registers for the whole walk (KS operands a lane)
//   softmax  a lane holds 8 of a row's 32 scores, the row's other 24 are in 3 lanes: two lane exchanges; running
//            maximum and sum in float32, base 2; a block that all rows of the wavefront see whole needs no mask
//   values   O[dim][row] += C^T . P   the same instruction, contraction over the block's keys in the order in
//            which the lanes hold P (keys 4j..4j+3 and 16+4j..16+4j+3 for lane group j): the latents are read
//            transposed from the same rows (ds_read_b64_tr_b16: sixteen lanes read four keys x sixteen dims and each
//            gets one dim of the four keys), so no second copy of them is made
//
// (Staged through registers, with a transposed copy of the latents written by 2-byte stores, the same walk took 381 us
// for the 2,048 tokens of a layer with 12 heads, rank 512 and a window of 1,024 keys.)
//
// Bound by LDS (68 KB a wavefront and block of rank 512 in about 540 cycles) and, where the tiles are no two for every unit, by the
// units with one.  A wavefront's turn was 11,000 cycles: a read's wait for each of 68 products, a branch for each tile of the second,
// and the loads of the next block waited for as soon as they were issued, together with a page number asked for behind them.  us, then
// and now, rank 512, rot 64, window 1,024: 2,000 tokens of 12 heads 178 to 121, without a window 295 to 193; 2,048 of 28 heads
// behind 3,000 cached 338 to 241; 31 decoded beside 700 prompt tokens 158 to 101; 32 decoded of 12 heads 25.5 to 23.6; rank 256, 16 heads,
// 2,048 tokens 104 to 83, rank 128 67 to 59.
//
// A tile's keys can be cut into chunks over blockIdx.y (decoded tokens: few rows, many keys); the chunks leave
// (maximum, sum, unnormalised O) per row and a second kernel merges them.  The cut is a launch parameter that
// depends on the window and the head count only.  Which tile a workgroup owns it finds itself from the step's
// entry lengths, so the launch is sized by tokens and entries alone.
#include "zi_common.h"
#include "zi_api.h"

typedef __attribute__((ext_vector_type(8))) __bf16 la_bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float la_f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned la_u32x4_t;
typedef __attribute__((ext_vector_type(4))) short la_s16x4_t;
union la_pack {
    la_u32x4_t u;
    la_bf16x8_t b;
    la_s16x4_t h[2];
    unsigned w[4];
};

#define LA_BK 32      // keys a block
#define LA_EMPTY -1e30f
#define LA_LOG2E 1.4426950408889634f

__device__ __attribute__((aligned(16))) const unsigned la_zero16[4] = {0u, 0u, 0u, 0u};

// of row k (rows k and k + 16 alike): a permutation of 0 .. 7 over eight rows of one parity, its upper two bits one of 0 .. 3
// over four of them
__device__ __forceinline__ int la_swizzle(int k) { return ((k & 6)) | ((k >> 3) & 1); }

// four keys of one dim from rows of LDS: see above
__device__ __forceinline__ la_s16x4_t la_read_transposed(const char* at) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) la_s16x4_t*)at);
}

// COUNT products, the operands of BATCH of them read from LDS together: left to itself, with nearly all registers taken, the compiler
// reads one, waits for it and makes its product, and a read's wait is ten times the product.  (Four are what the registers have room for
// at rank 512.)
template <int BATCH, int COUNT, typename Read, typename Make>
__device__ __forceinline__ void la_products(Read read, Make make) {
    static_assert(COUNT % BATCH == 0, "whole batches");
#pragma unroll
    for (int b = 0; b < COUNT; b += BATCH) {
        la_pack a[BATCH];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < BATCH; ++i) a[i] = read(b + i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < BATCH; ++i) make(b + i, a[i]);
    }
    __builtin_amdgcn_sched_barrier(0);
}
#define LA_BATCH 4

// SPLIT: all WAVES wavefronts share one tile of 16 rows (decoded tokens): they stage together, each makes the
// scores again (cheap) and every WAVES-th tile of 16 latent dims of the second product.
template <int WAVES, int NT, int KS, bool SPLIT>      // rank <= 16 NT, rank + rot <= 32 KS
__global__ void __launch_bounds__(WAVES* ZI_WAVE, 2)
latent_attention_cores_kernel(void* __restrict__ out, int out_f32, float* __restrict__ partial, const void* __restrict__ qa, int qa_f32,
                              const zi_bf16* __restrict__ c_cache, const zi_bf16* __restrict__ kr_cache,
                              const int32_t* __restrict__ entry_start, const int32_t* __restrict__ entry_len,
                              const int32_t* __restrict__ entry_past, const int32_t* __restrict__ block_tables,
                              int entries, int max_pages, int num_pages, int heads, int rank, int rot, int page_size,
                              int window, float scale, int chunk_keys, int total_rows) {
    constexpr int ROWS = SPLIT ? 16 : WAVES * 16, OT = SPLIT ? (NT + WAVES - 1) / WAVES : NT;
    constexpr int P = KS * 4;                                  // 16-byte pieces of a staged key
    constexpr int KI = LA_BK * P / (WAVES * ZI_WAVE);          // load instructions a wavefront issues per block
    static_assert(P % 8 == 0 && (P * 16) % 256 == 128 && KI * WAVES * ZI_WAVE == LA_BK * P, "whole loads, rows half the banks apart");
    __shared__ __attribute__((aligned(16))) la_u32x4_t buf_a[LA_BK * P];
    __shared__ __attribute__((aligned(16))) la_u32x4_t buf_b[LA_BK * P];
    const int lane = threadIdx.x % ZI_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / ZI_WAVE), r = lane % 16, j = lane / 16;
    // the entry whose tiles this one is among: 64 entries at a time, a lane each, their tiles summed up over the lanes
    int tile = blockIdx.x, e = entries;
    for (int e0 = 0; e0 < entries; e0 += ZI_WAVE) {
        const int mine = e0 + lane < entries ? (entry_len[e0 + lane] * heads + ROWS - 1) / ROWS : 0;
        int upto = mine;
#pragma unroll
        for (int d = 1; d < ZI_WAVE; d *= 2) {
            const int below = __shfl_up(upto, d, ZI_WAVE);
            if (lane >= d) upto += below;
        }
        const uint64_t past_it = __ballot(upto > tile);
        if (past_it) {
            const int at = __builtin_ctzll(past_it);
            e = e0 + at;
            tile -= __builtin_amdgcn_readlane(upto - mine, at);
            break;
        }
        tile -= __builtin_amdgcn_readlane(upto, ZI_WAVE - 1);
    }
    if (e >= entries) return;      // the launch is sized for the worst case: the whole workgroup leaves
    const int len = entry_len[e], past = entry_past[e], start = entry_start[e];
    const int erows = len * heads, row0 = tile * ROWS;
    const int32_t* bt = block_tables + (int64_t)e * max_pages;
    const int qw = rank + rot;

    // the tile's keys, and this workgroup's chunk of them
    const int last_row = (row0 + ROWS < erows ? row0 + ROWS : erows) - 1;
    const int pos_first = past + row0 / heads, pos_last = past + last_row / heads;
    const int kmin = (window > 0 && pos_first - window + 1 > 0) ? pos_first - window + 1 : 0;
    int k_lo = kmin, k_hi = pos_last;
    if (chunk_keys > 0) {
        k_lo = kmin + (int)blockIdx.y * chunk_keys;
        if (k_lo + chunk_keys - 1 < k_hi) k_hi = k_lo + chunk_keys - 1;
    }

    // this lane's row; the keys that all rows of the wavefront see are [all_lo, all_hi]
    const int wave_row0 = row0 + (SPLIT ? 0 : wave * 16);
    const int row = wave_row0 + r;
    const bool row_ok = row < erows;
    const int rc = row_ok ? row : last_row;
    const int tok = start + rc / heads, head = rc % heads, pos = past + rc / heads;
    const int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    const int wave_last = wave_row0 + 15 < last_row ? wave_row0 + 15 : last_row;
    const int all_hi = past + (wave_row0 < last_row ? wave_row0 : last_row) / heads, all_pos = past + wave_last / heads;
    const int all_lo = (window > 0 && all_pos - window + 1 > 0) ? all_pos - window + 1 : 0;
    const int64_t grow = (int64_t)tok * heads + head;

    la_pack q[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int d = ks * 32 + 8 * j;
        q[ks].u = (la_u32x4_t){0u, 0u, 0u, 0u};
        if (d >= qw) continue;      // rank + rot is a multiple of 8: a piece of eight lies inside or outside
        if (qa_f32) {
            const float* qr = (const float*)qa + grow * qw + d;
            const float4 a = *reinterpret_cast<const float4*>(qr), b = *reinterpret_cast<const float4*>(qr + 4);
            q[ks].w[0] = zi_pack_bf16x2(a.x, a.y);
            q[ks].w[1] = zi_pack_bf16x2(a.z, a.w);
            q[ks].w[2] = zi_pack_bf16x2(b.x, b.y);
            q[ks].w[3] = zi_pack_bf16x2(b.z, b.w);
        } else {
            q[ks].u = *reinterpret_cast<const la_u32x4_t*>((const zi_bf16*)qa + grow * qw + d);
        }
    }

    float m = LA_EMPTY, l = 0.f;
    la_f32x4_t o[OT];      // tile tq of this wavefront is the latent dims 16 t ..., t = tq (SPLIT: tq WAVES + wave)
#pragma unroll
    for (int t = 0; t < OT; ++t) o[t] = (la_f32x4_t){0.f, 0.f, 0.f, 0.f};

    // the page of key kb + lane % 32, and from it its place in the pool, or -1: past the end, or a page that is not held.  Asked for
    // in one turn and used in the next: to wait for it is to wait for the loads into LDS that were issued before it.
    auto ask = [&](int kb) {
        const int kp = kb + (lane & (LA_BK - 1)), pi = (kp <= k_hi ? kp : k_hi) / page_size;
        return bt[pi < max_pages ? pi : max_pages - 1];
    };
    auto places = [&](int kb, int page) {
        const int kp = kb + (lane & (LA_BK - 1)), kc = kp <= k_hi ? kp : k_hi;
        return (kp <= k_hi) & ((unsigned)page < (unsigned)num_pages) ? page * page_size + kc % page_size : -1;
    };
    auto issue = [&](int slots, la_u32x4_t* dst) {
        int ln = lane;      // (what a lane loads is worked out anew every block: kept, it takes the registers of the sums)
        asm volatile("" : "+v"(ln));
#pragma unroll
        for (int i = 0; i < KI; ++i) {
            const int L = (wave * KI + i) * ZI_WAVE + ln, key = L / P, d = ((L % P) ^ la_swizzle(key)) * 8;
            const int slot = __shfl(slots, key, ZI_WAVE);
            const bool latent = d < rank;
            const zi_bf16* src = (latent ? c_cache : kr_cache) + ((int64_t)slot * (latent ? rank : rot) + (latent ? d : d - rank));
            if ((slot < 0) | (d >= qw)) src = reinterpret_cast<const zi_bf16*>(la_zero16);
            __builtin_amdgcn_global_load_lds(src, dst + (wave * KI + i) * ZI_WAVE, 16, 0, 0);
        }
    };
    // where this lane reads in a buffer, in bytes: the keys' rows (k-steps even and odd), and four keys x sixteen dims
    const int sw = la_swizzle(r);      // of rows r and 16 + r
    const int s_even = (r * P + (j ^ sw)) * 16, s_odd = (r * P + ((4 + j) ^ sw)) * 16;
    const int vrow = 4 * j + (r >> 2), vsw = la_swizzle(vrow);
    int v_at[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) v_at[t] = (vrow * P + ((t * 2 + ((r & 3) >> 1)) ^ vsw)) * 16 + (r & 1) * 8;
    const float scale2 = scale * LA_LOG2E;

    auto work = [&](int kb, const la_u32x4_t* buf) {
        const char* base = reinterpret_cast<const char*>(buf);
        la_f32x4_t s[2];
        s[0] = s[1] = (la_f32x4_t){0.f, 0.f, 0.f, 0.f};
        la_products<LA_BATCH, 2 * KS>(
            [&](int i) {
                const int ks = i / 2, h = i % 2;
                la_pack a;
                a.u = *reinterpret_cast<const la_u32x4_t*>(base + ((ks & 1) ? s_odd : s_even) + h * (16 * P * 16) + (ks / 2) * 128);
                return a;
            },
            [&](int i, const la_pack& a) { s[i % 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.b, q[i / 2].b, s[i % 2], 0, 0, 0); });
        // lane (r, j) holds, of row r, the keys kb + 16 h + 4 j + x; in base-2 units from here on
        float mb = LA_EMPTY;
        const bool whole = kb >= all_lo && kb + LA_BK - 1 <= all_hi && kb + LA_BK - 1 <= k_hi;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const int kp = kb + 16 * h + 4 * j + x;
                const bool seen = whole || (row_ok && kp >= lo && kp <= pos && kp <= k_hi);
                s[h][x] = seen ? s[h][x] * scale2 : -INFINITY;
                mb = fmaxf(mb, s[h][x]);
            }
        mb = fmaxf(mb, __shfl_xor(mb, 16, ZI_WAVE));
        mb = fmaxf(mb, __shfl_xor(mb, 32, ZI_WAVE));
        const float m_new = fmaxf(m, mb);      // (never below LA_EMPTY, so a key that is not seen weighs 2^-inf = 0)
        const float corr = __builtin_amdgcn_exp2f(m - m_new);
        float sum = 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                s[h][x] = __builtin_amdgcn_exp2f(s[h][x] - m_new);
                sum += s[h][x];
            }
        l = l * corr + sum;      // this lane's keys; the row's four lanes are added up at the end
        m = m_new;
        la_pack pb;
        pb.w[0] = zi_pack_bf16x2(s[0][0], s[0][1]);
        pb.w[1] = zi_pack_bf16x2(s[0][2], s[0][3]);
        pb.w[2] = zi_pack_bf16x2(s[1][0], s[1][1]);
        pb.w[3] = zi_pack_bf16x2(s[1][2], s[1][3]);
        if (__any(corr != 1.f)) {      // the running maximum seldom moves after the first blocks
#pragma unroll
            for (int tq = 0; tq < OT; ++tq) o[tq] *= corr;
        }
        // groups of tiles, each either whole or left out: what lies behind the rank is staged too, and is not stored
        constexpr int G = OT < 16 ? OT : 16;
#pragma unroll
        for (int g = 0; g < OT; g += G) {
            if (g * (SPLIT ? WAVES : 1) * 16 >= rank) break;
            la_products<(G < LA_BATCH ? G : LA_BATCH), G>(
                [&](int i) {
                    const int tq = g + i, t = tq * WAVES + wave;
                    const char* at = SPLIT ? base + (vrow * P + ((t * 2 + ((r & 3) >> 1)) ^ vsw)) * 16 + (r & 1) * 8
                                           : base + v_at[tq & 3] + (tq / 4) * 128;
                    la_pack a;
                    a.h[0] = la_read_transposed(at);
                    a.h[1] = la_read_transposed(at + 16 * P * 16);
                    return a;
                },
                [&](int i, const la_pack& a) { o[g + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.b, pb.b, o[g + i], 0, 0, 0); });
        }
    };
    // Two blocks a turn, buffer a then b.  At each barrier the block about to be worked on has arrived and everyone has finished with
    // the other buffer.
    if (k_lo <= k_hi) {
        issue(places(k_lo, ask(k_lo)), buf_a);
        int page = ask(k_lo + LA_BK), kb = k_lo;
        auto ahead = [&](la_u32x4_t* dst) {
            asm volatile("" : "+v"(page));      // (here, behind the barrier)
            if (kb + LA_BK > k_hi) return;
            const int slots = places(kb + LA_BK, page);
            page = ask(kb + 2 * LA_BK);
            issue(slots, dst);
        };
        while (true) {
            zi_barrier_loaded();
            ahead(buf_b);
            work(kb, buf_a);
            if (kb + LA_BK > k_hi) break;
            kb += LA_BK;
            zi_barrier_loaded();
            ahead(buf_a);
            work(kb, buf_b);
            if (kb + LA_BK > k_hi) break;
            kb += LA_BK;
        }
    }
    l += __shfl_xor(l, 16, ZI_WAVE);
    l += __shfl_xor(l, 32, ZI_WAVE);
    // lane (r, j) holds, of row r, the dims 16 t + 4 j + x (rank is a multiple of 8: four dims lie inside or outside)
    if (!row_ok) return;
    const bool parts = gridDim.y > 1;
    const float inv = parts ? 1.f : 1.f / l;
    const int64_t prow = ((int64_t)blockIdx.y * total_rows + grow) * (rank + 4);      // maximum, sum, two unused, then O
    if (parts && j == 0 && (!SPLIT || wave == 0)) {
        partial[prow] = m;
        partial[prow + 1] = l;
    }
#pragma unroll
    for (int tq = 0; tq < OT; ++tq) {
        const int d = 16 * (SPLIT ? tq * WAVES + wave : tq) + 4 * j;
        if (d >= rank) continue;
        const la_f32x4_t v = o[tq] * inv;
        if (parts) {
            *reinterpret_cast<la_f32x4_t*>(partial + prow + 4 + d) = v;
        } else if (out_f32) {
            *reinterpret_cast<la_f32x4_t*>((float*)out + grow * rank + d) = v;
        } else {
            uint2 w;
            w.x = zi_pack_bf16x2(v[0], v[1]);
            w.y = zi_pack_bf16x2(v[2], v[3]);
            *reinterpret_cast<uint2*>((zi_bf16*)out + grow * rank + d) = w;
        }
    }
}

// out[row] = sum_c O_c 2^(m_c - M) / sum_c l_c 2^(m_c - M), chunks in rising order.  A thread owns four dims; the loads of
// eight chunks travel together.
#define LA_MAX_CHUNKS 4096
__global__ void __launch_bounds__(128)
latent_attention_merge_kernel(void* __restrict__ out, int out_f32, const float* __restrict__ partial, int chunks, int total_rows,
                              int rank) {
    __shared__ float weight[128];
    const int64_t row = blockIdx.x, stride = (int64_t)total_rows * (rank + 4);
    const float* p0 = partial + row * (rank + 4);
    const int tid = threadIdx.x, lane = tid & (ZI_WAVE - 1);
    const int d = tid * 4;
    // every wavefront makes the maximum and the sum: lane c takes chunks c, c + 64, ...
    float M = LA_EMPTY;
    for (int c = lane; c < chunks; c += ZI_WAVE) M = fmaxf(M, p0[c * stride]);
    M = zi_wave_max(M);
    float L = 0.f;
    for (int c = lane; c < chunks; c += ZI_WAVE) L += p0[c * stride + 1] * __builtin_amdgcn_exp2f(p0[c * stride] - M);
    const float inv = 1.f / zi_wave_sum(L);
    la_f32x4_t acc = (la_f32x4_t){0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < chunks; c0 += 128) {
        __syncthreads();
        if (c0 + tid < chunks) weight[tid] = __builtin_amdgcn_exp2f(p0[(c0 + tid) * stride] - M);
        __syncthreads();
        const int count = chunks - c0 < 128 ? chunks - c0 : 128;
        if (d >= rank) continue;
        for (int c = 0; c < count; c += 8) {
            la_f32x4_t v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const la_f32x4_t*>(p0 + (c0 + (c + u < count ? c + u : c)) * stride + 4 + d);
#pragma unroll
            for (int u = 0; u < 8; ++u) acc += v[u] * (c + u < count ? weight[c + u] : 0.f);
        }
    }
    if (d >= rank) return;
    acc *= inv;
    if (out_f32) {
        *reinterpret_cast<la_f32x4_t*>((float*)out + row * rank + d) = acc;
    } else {
        uint2 w;
        w.x = zi_pack_bf16x2(acc[0], acc[1]);
        w.y = zi_pack_bf16x2(acc[2], acc[3]);
        *reinterpret_cast<uint2*>((zi_bf16*)out + row * rank + d) = w;
    }
}

extern "C" int zi_latent_attention_cores_supported(int dt, int rank, int rot) {
    return dt == ZI_BF16 && rank > 0 && rank % 8 == 0 && rot >= 0 && rot % 8 == 0 && rank <= 512 && rank + rot <= 576;
}

// Rows of a tile for `waves` wavefronts, and the most tiles a step of n tokens in `entries` entries has.
extern "C" int zi_latent_attention_cores_tiles(int n, int entries, int heads, int waves) {
    const int64_t rows = 16 * waves;
    const int64_t by_entry = ((int64_t)n * heads + rows - 1) / rows + entries, by_token = (int64_t)n * ((heads + rows - 1) / rows);
    return (int)(by_entry < by_token ? by_entry : by_token);
}

// qa [n][heads][rank + rot] and out [n][heads][rank], each float32 or bfloat16; partial: chunks * n * heads * (rank + 4) floats.
extern "C" int zi_latent_attention_cores(void* out, int out_dt, float* partial, int64_t partial_floats, const void* qa, int qa_dt,
                                         const void* c_cache, const void* kr_cache, const int32_t* entry_start,
                                         const int32_t* entry_len, const int32_t* entry_past, const int32_t* block_tables,
                                         int entries, int n, int max_pages, int num_pages, int heads, int rank, int rot,
                                         int page_size, int window, float scale, int waves, int chunk_keys, int chunks,
                                         hipStream_t stream) {
    ZI_REQUIRE(zi_latent_attention_cores_supported(ZI_BF16, rank, rot), "latent_attention_cores: rank %d, rot %d not taken",
               rank, rot);
    ZI_REQUIRE(n >= 0 && entries > 0 && heads > 0 && page_size > 0 && max_pages > 0 && num_pages > 0 && window >= 0 &&
                   (int64_t)num_pages * page_size < (1ll << 31), "latent_attention_cores: bad sizes");
    ZI_REQUIRE((out_dt == ZI_F32 || out_dt == ZI_BF16) && (qa_dt == ZI_F32 || qa_dt == ZI_BF16) && ((uintptr_t)qa % 16) == 0 &&
                   ((uintptr_t)out % 16) == 0 && ((uintptr_t)partial % 16) == 0 && ((uintptr_t)c_cache % 16) == 0 && ((uintptr_t)kr_cache % 16) == 0,
               "latent_attention_cores: unknown types, or addresses that are not aligned to 16 bytes");
    ZI_REQUIRE(waves == 1 || waves == 4, "latent_attention_cores: 1 or 4 wavefronts a workgroup");
    ZI_REQUIRE(chunks >= 1 && chunks <= LA_MAX_CHUNKS && (chunks == 1) == (chunk_keys == 0) && chunk_keys >= 0,
               "latent_attention_cores: bad cut (%d chunks of %d keys)", chunks, chunk_keys);
    if (chunks > 1) {
        // every key a tile's rows see lies in one of the chunks
        const int tokens_in_tile = (16 * waves + heads - 1) / heads + 1;
        // (without a window the caller sees to it that the chunks reach the last key of every entry)
        ZI_REQUIRE(window == 0 || (int64_t)chunks * chunk_keys >= (int64_t)window + tokens_in_tile,
                   "latent_attention_cores: %d chunks of %d keys do not cover a window of %d", chunks, chunk_keys, window);
        ZI_REQUIRE(partial && partial_floats >= (int64_t)chunks * n * heads * (rank + 4),
                   "latent_attention_cores: the workspace is too small");
    }
    if (n == 0) return 0;
    const int total_rows = n * heads;
    const dim3 grid(zi_latent_attention_cores_tiles(n, entries, heads, waves), chunks);
#define ZI_LA_LAUNCH(W, NT, KS)                                                                                       \
    latent_attention_cores_kernel<4, NT, KS, W == 1><<<grid, 4 * ZI_WAVE, 0, stream>>>(                                \
        out, out_dt == ZI_F32, partial, qa, qa_dt == ZI_F32, (const zi_bf16*)c_cache, (const zi_bf16*)kr_cache, entry_start, entry_len, \
        entry_past, block_tables, entries, max_pages, num_pages, heads, rank, rot, page_size, window, scale, chunk_keys, total_rows)
#define ZI_LA_SIZES(W)                                                       \
    do {                                                                     \
        if (rank <= 128 && rank + rot <= 192) ZI_LA_LAUNCH(W, 8, 6);         \
        else if (rank <= 256 && rank + rot <= 320) ZI_LA_LAUNCH(W, 16, 10);  \
        else ZI_LA_LAUNCH(W, 32, 18);                                        \
    } while (0)
    if (waves == 1) ZI_LA_SIZES(1);
    else ZI_LA_SIZES(4);
#undef ZI_LA_SIZES
#undef ZI_LA_LAUNCH
    int rc = zi_check_launch("latent_attention_cores");
    if (rc != 0 || chunks == 1) return rc;
    latent_attention_merge_kernel<<<total_rows, 128, 0, stream>>>(out, out_dt == ZI_F32, partial, chunks, total_rows, rank);
    return zi_check_launch("latent_attention_merge");
}

// ---- a product per head on the matrix cores ---------------------------------------------------------------------
// out[t][h][i] = sum_k w[h][i][k] x[t][h][k]: w bfloat16 [heads][N][K] (k runs fastest), x float32 (rounded to bfloat16 as
// it is loaded) or bfloat16 with row stride ldx and head stride xs, out float32 or bfloat16 with row stride ldo and head stride
// os.  It carries the queries through W_uk (w = W_uk of the head, transposed at load) and the attended latents through W_uv.
// GATED: out *= sigmoid(gate[t][h * N + i]), the gate bfloat16 or the sum of `splits` float32 terms.
// Few tokens: 16 x 16 a workgroup, operands straight from memory, k dealt over the four wavefronts in runs of 32 and added up in their
// order.  Many: 64 tokens x 32, 64 or 128 outputs (la_tile_outputs), a wavefront 32 x half of these.  Bound by memory (x once, the results), and
// before by the vector cache: operands loaded as the product wants them lie in a row apiece, 9 to 10 accesses a line of 128 bytes.  So a step's
// rows of 128 bytes are loaded whole, two steps on their way in registers, and turn in LDS in places that neither side's lanes share a bank in;
// the results turn there too and leave in runs of whole rows of the tile; a thread asks for all its gates at once.  us, operands straight from
// memory, tiles of 128 outputs with gates asked for one after the other, now: 12 heads, 512 outputs of k 128, 2,000 tokens 24.5, 12.5, 12.6 (3 TB/s with
// x once), 8,000 82, 38.5, 38.4; 128 of 512 26.4, 14.2, 12.8 and 84, 31.2, 30.9; 128 tokens 5.9, 4.4, 3.9 and 13.4, 8.3, 6.6; with a gate 34.6, 21.4,
// 16.6 (2,000 tokens); 64 outputs of 512 14.6, 11.4, 8.7; 16 of 16 with a gate 4.7, 10.0, 4.7; 64 heads, 64 of 64 with a gate, 8,000 tokens 100, 145, 51.
// One step on its way instead of two: 128 tokens 5.0 and 9.8.  Over 4,780 products 0.68 of the first's time; slower by a tenth or more: gates over 8 or 16
// outputs of a k of up to 128 at 8,000 tokens (12 heads, 16 of 16, three terms 1.29), 33 outputs of up to 16 (1.18).
struct LaGate {
    const void* g;
    int f32, splits;
    int64_t ld, stride;
};

__device__ __forceinline__ la_pack la_load8(const float* p) {
    const float4 lo = *reinterpret_cast<const float4*>(p), hi = *reinterpret_cast<const float4*>(p + 4);
    la_pack b;
    b.w[0] = zi_pack_bf16x2(lo.x, lo.y);
    b.w[1] = zi_pack_bf16x2(lo.z, lo.w);
    b.w[2] = zi_pack_bf16x2(hi.x, hi.y);
    b.w[3] = zi_pack_bf16x2(hi.z, hi.w);
    return b;
}
__device__ __forceinline__ la_pack la_load8(const zi_bf16* p) {
    la_pack b;
    b.u = *reinterpret_cast<const la_u32x4_t*>(p);
    return b;
}

// four gates of one token and head, columns n0 .. n0 + 3 (clamped to the head), stored as T
template <typename T>
__device__ __forceinline__ la_f32x4_t la_gates(const LaGate& gt, int64_t t, int h, int n0, int N) {
    const int64_t at = t * gt.ld + (int64_t)h * N;
    const T* g0 = (const T*)gt.g + at;
    la_f32x4_t g;
#pragma unroll
    for (int i = 0; i < 4; ++i) g[i] = zi_load(g0 + (n0 + i < N ? n0 + i : N - 1));
    if (sizeof(T) == 4) {
        int s = 1;
        for (; s + 3 < gt.splits; s += 4) {      // four terms in flight, added in their order
            la_f32x4_t v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[u][i] = zi_load(g0 + (s + u) * gt.stride + (n0 + i < N ? n0 + i : N - 1));
#pragma unroll
            for (int u = 0; u < 4; ++u) g += v[u];
        }
        for (; s < gt.splits; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) g[i] += zi_load(g0 + s * gt.stride + (n0 + i < N ? n0 + i : N - 1));
    }
    return g;
}
template <typename TO>
__device__ __forceinline__ void la_store4(TO* orow, la_f32x4_t v, int left) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < left) zi_store(orow + i, v[i]);
}
__device__ __forceinline__ void la_gate4(la_f32x4_t& v, const la_f32x4_t& g) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.f + expf(-g[i]));
}

template <typename TX, typename TO, bool GATED>
__global__ void __launch_bounds__(4 * ZI_WAVE)
headwise_linear_few_kernel(TO* __restrict__ out, int64_t ldo, int os, const TX* __restrict__ x, int64_t ldx, int xs,
                           const zi_bf16* __restrict__ w, int n, int N, int K, LaGate gt) {
    __shared__ la_f32x4_t part[3][ZI_WAVE];
    const int t0 = blockIdx.x * 16, h = blockIdx.y, n0 = blockIdx.z * 16;
    const int lane = threadIdx.x % ZI_WAVE, wave = threadIdx.x / ZI_WAVE, r = lane % 16, j = lane / 16;
    const zi_bf16* wrow = w + ((int64_t)h * N + (n0 + r < N ? n0 + r : N - 1)) * K;
    const int64_t t = t0 + r < n ? t0 + r : n - 1;
    const TX* xrow = x + t * ldx + (int64_t)h * xs;
    la_f32x4_t acc = (la_f32x4_t){0.f, 0.f, 0.f, 0.f}, gate = acc;
    if (GATED && wave == 0) gate = gt.f32 ? la_gates<float>(gt, t, h, n0 + 4 * j, N) : la_gates<zi_bf16>(gt, t, h, n0 + 4 * j, N);      // asked for before the product, used after it
#pragma unroll 4
    for (int k0 = wave * 32; k0 < K; k0 += 128) {
        const int k = k0 + 8 * j, kc = k < K ? k : 0;      // K is a multiple of 8
        const unsigned mask = 0u - (unsigned)(k < K);
        la_pack a = la_load8(wrow + kc), b = la_load8(xrow + kc);
        a.u &= mask;
        b.u &= mask;
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.b, b.b, acc, 0, 0, 0);
    }
    if (wave > 0) part[wave - 1][lane] = acc;
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int u = 0; u < 3; ++u) acc += part[u][lane];
    if (t0 + r >= n || n0 + 4 * j >= N) return;
    if constexpr (GATED) la_gate4(acc, gate);
    la_store4(out + t * ldo + (int64_t)h * os + n0 + 4 * j, acc, N - n0 - 4 * j);
}

#define LA_HT 64       // tokens
#define LA_HK 64       // k a step: rows of 128 bytes
template <typename TX, typename TO, bool GATED, int TN>
__global__ void __launch_bounds__(4 * ZI_WAVE, 3)
headwise_linear_many_kernel(TO* __restrict__ out, int64_t ldo, int os, const TX* __restrict__ x, int64_t ldx, int xs,
                            const zi_bf16* __restrict__ w, int n, int N, int K, LaGate gt) {
    constexpr int TM = 2, HN = 32 * TN, HROW = HN + 4;      // a wavefront's tiles of 16 tokens; outputs, a row of results
    constexpr int PX = LA_HT / 32, PW = HN / 32;     // a thread's pieces of 16 bytes a step
    constexpr int STEP = (LA_HT + HN) * 8;           // pieces a step
    __shared__ la_u32x4_t lds[2 * STEP];
    static_assert(LA_HT * HROW * sizeof(float) <= sizeof(lds), "the results turn in the operands' place");
    const int tid = threadIdx.x, lane = tid % ZI_WAVE, wave = tid / ZI_WAVE, r = lane % 16, j = lane / 16;
    const int t0 = blockIdx.x * LA_HT, h = blockIdx.y, n0 = blockIdx.z * HN;
    const int q = tid / 8, c8 = tid % 8;                // rows q, q + 32, ..; (q + 32 i) / 2 keeps its last three bits
    const int at = q * 8 + (c8 ^ (q / 2 & 7));
    const TX* xr[PX];
    const zi_bf16* wr[PW];
#pragma unroll
    for (int i = 0; i < PX; ++i) {
        const int t = t0 + q + 32 * i;
        xr[i] = x + (int64_t)(t < n ? t : n - 1) * ldx + (int64_t)h * xs;
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int o = n0 + q + 32 * i;
        wr[i] = w + ((int64_t)h * N + (o < N ? o : N - 1)) * K;
    }
    struct Pieces { la_pack x[PX], w[PW]; };
    auto load = [&](Pieces& to, int k0) {
        const int k = k0 + 8 * c8, kc = k < K ? k : 0;      // K is a multiple of 8
        const unsigned mask = 0u - (unsigned)(k < K);
#pragma unroll
        for (int i = 0; i < PX; ++i) to.x[i] = la_load8(xr[i] + kc);
#pragma unroll
        for (int i = 0; i < PW; ++i) to.w[i] = la_load8(wr[i] + kc);
#pragma unroll
        for (int i = 0; i < PX; ++i) to.x[i].u &= mask;
#pragma unroll
        for (int i = 0; i < PW; ++i) to.w[i].u &= mask;
    };
    auto stash = [&](const Pieces& p, la_u32x4_t* to) {
#pragma unroll
        for (int i = 0; i < PX; ++i) to[at + 32 * 8 * i] = p.x[i].u;
#pragma unroll
        for (int i = 0; i < PW; ++i) to[LA_HT * 8 + at + 32 * 8 * i] = p.w[i].u;
    };
    const int tw = (wave % 2) * (16 * TM), ow = (wave / 2) * (16 * TN);
    la_f32x4_t acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int c = 0; c < TN; ++c) acc[a][c] = (la_f32x4_t){0.f, 0.f, 0.f, 0.f};
    // one step on its way in registers, one on its way to memory's answer, one in LDS
    auto step = [&](int k0, Pieces& mine, const Pieces& next, int buf) {
        __syncthreads();
        if (k0 + 2 * LA_HK < K) load(mine, k0 + 2 * LA_HK);
        const la_u32x4_t *lx = lds + buf * STEP + (tw + r) * 8, *lw = lds + buf * STEP + (LA_HT + ow + r) * 8;
#pragma unroll
        for (int s = 0; s < LA_HK / 32; ++s) {
            const int place = (4 * s + j) ^ (r / 2 & 7);
            la_pack a[TN], b[TM];
#pragma unroll
            for (int c = 0; c < TN; ++c) a[c].u = lw[c * 16 * 8 + place];
#pragma unroll
            for (int c = 0; c < TM; ++c) b[c].u = lx[c * 16 * 8 + place];
#pragma unroll
            for (int m = 0; m < TM; ++m)
#pragma unroll
                for (int c = 0; c < TN; ++c) acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c].b, b[m].b, acc[m][c], 0, 0, 0);
        }
        if (k0 + LA_HK < K) stash(next, lds + (buf ^ 1) * STEP);      // read for the last time before this step's barrier
    };
    Pieces even, odd;
    load(even, 0);
    if (LA_HK < K) load(odd, LA_HK);
    stash(even, lds);
    for (int k0 = 0; k0 < K; k0 += 2 * LA_HK) {
        step(k0, even, odd, 0);
        if (k0 + LA_HK < K) step(k0 + LA_HK, odd, even, 1);
    }
    // eight outputs' gates for each of this thread's pieces, all asked for at once
    la_f32x4_t gates[GATED ? TN : 1][2];
    auto piece = [&](int u, int& row, int& o) {
        const int p = tid + u * (4 * ZI_WAVE);
        row = p / (HN / 8);
        o = p % (HN / 8) * 8;
        return t0 + row < n && n0 + o < N;
    };
    if constexpr (GATED) {
        auto ask = [&](auto read) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < TN; ++u) {
                int row, o;
                if (!piece(u, row, o)) continue;
                gates[u][0] = read(t0 + row, n0 + o);
                gates[u][1] = read(t0 + row, n0 + o + 4);
            }
        };
        if (gt.f32) ask([&](int t, int i) { return la_gates<float>(gt, t, h, i, N); });
        else ask([&](int t, int i) { return la_gates<zi_bf16>(gt, t, h, i, N); });
    }
    __syncthreads();
    float* turned = reinterpret_cast<float*>(lds);      // [token][output]
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int c = 0; c < TN; ++c)
            *reinterpret_cast<la_f32x4_t*>(turned + (tw + m * 16 + r) * HROW + ow + c * 16 + 4 * j) = acc[m][c];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TN; ++u) {
        int row, o;
        if (!piece(u, row, o)) continue;
        const int t = t0 + row, i = n0 + o;
        la_f32x4_t lo = *reinterpret_cast<const la_f32x4_t*>(turned + row * HROW + o);
        la_f32x4_t hi = *reinterpret_cast<const la_f32x4_t*>(turned + row * HROW + o + 4);
        if constexpr (GATED) {
            la_gate4(lo, gates[u][0]);
            la_gate4(hi, gates[u][1]);
        }
        TO* dst = out + (int64_t)t * ldo + (int64_t)h * os + i;
        if (sizeof(TO) == 2 && i + 7 < N && ((uintptr_t)dst % 16) == 0) {
            la_pack b;
            b.w[0] = zi_pack_bf16x2(lo[0], lo[1]);
            b.w[1] = zi_pack_bf16x2(lo[2], lo[3]);
            b.w[2] = zi_pack_bf16x2(hi[0], hi[1]);
            b.w[3] = zi_pack_bf16x2(hi[2], hi[3]);
            *reinterpret_cast<la_u32x4_t*>(dst) = b.u;
        } else if (sizeof(TO) == 4 && i + 7 < N && ((uintptr_t)dst % 16) == 0) {
            reinterpret_cast<la_f32x4_t*>(dst)[0] = lo;
            reinterpret_cast<la_f32x4_t*>(dst)[1] = hi;
        } else {
            la_store4(dst, lo, N - i);
            la_store4(dst + 4, hi, N - i - 4);
        }
    }
}

// (either storage type of x)
extern "C" int zi_headwise_linear_supported(int w_dt, int K, int64_t ldx, int xs) {
    return w_dt == ZI_BF16 && K > 0 && K % 8 == 0 && ldx % 8 == 0 && xs % 8 == 0;
}

#define LA_MANY_TOKENS 128      // from this many tokens on the kernel for many

// Outputs of its tiles: 32 for heads that have no more.  Else 64, and 128 without a gate where the tiles of 128 fill the chip, three
// workgroups a unit (two and a half of them, eight where half of a head's last tile is empty): x is read once a tile, but a tile's end is one
// long wait.  Time in tiles of 128 over that in tiles of 64, geometric means by tiles of 128 a unit, 1,087 products of 2 to 64 heads, 65 to 512
// outputs, a k of 16 to 512, 128 to 12,000 tokens:
//   up to 1     1.16   x float32 1.15   a bfloat16 gate 1.35   three terms of a gate 1.46
//   1 to 2.5    1.04             1.01                   1.17                         1.15
//   2.5 to 6    0.93             0.87                   1.03                         1.06
//   from 6 on   0.88             0.80                   0.99                         1.08
// half empty tiles, up to 8 1.03 to 1.15 and 0.99 to 1.13, from there on 0.99 and 0.90.
static int la_tile_outputs(int n, int heads, int N, bool gated) {
    if (N <= 32) return 32;
    if (gated || N <= 64) return 64;
    const int64_t tiles = (int64_t)((n + LA_HT - 1) / LA_HT) * heads * ((N + 127) / 128);
    return tiles >= (int64_t)zi_compute_units() * ((N - 1) % 128 < 64 ? 16 : 5) / 2 ? 128 : 64;
}

extern "C" int zi_headwise_linear_gated(void* out, int out_dt, int64_t ldo, int os, const void* x, int x_dt, int64_t ldx, int xs,
                                        const void* w, int n, int heads, int N, int K, const void* gate, int g_dt,
                                        int64_t ld_gate, int g_splits, int64_t g_stride, hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && heads > 0 && heads <= 65535 && N > 0 && (N + 15) / 16 <= 65535, "headwise_linear: bad sizes");
    ZI_REQUIRE(zi_headwise_linear_supported(ZI_BF16, K, ldx, xs) && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0,
               "headwise_linear: K %d, row stride %lld, head stride %d or an address is not aligned", K, (long long)ldx, xs);
    ZI_REQUIRE(xs >= K && os >= N && ldx >= (int64_t)(heads - 1) * xs + K && ldo >= (int64_t)(heads - 1) * os + N,
               "headwise_linear: strides too small");
    ZI_REQUIRE(!gate || (ld_gate >= (int64_t)heads * N && g_splits >= 1 && (g_dt == ZI_F32 || (g_dt == ZI_BF16 && g_splits == 1))),
               "headwise_linear: bad gate");
    if (n == 0) return 0;
    const bool many = n >= LA_MANY_TOKENS;
    const int wide = la_tile_outputs(n, heads, N, gate) / 32;
    const dim3 grid(many ? (n + LA_HT - 1) / LA_HT : (n + 15) / 16, heads, many ? (N + 32 * wide - 1) / (32 * wide) : (N + 15) / 16);
    const LaGate gt = {gate, g_dt == ZI_F32, g_splits, ld_gate, g_stride};
#define ZI_HW(...) __VA_ARGS__<<<grid, 4 * ZI_WAVE, 0, stream>>>((TO*)out, ldo, os, (const TX*)x, ldx, xs, (const zi_bf16*)w, n, N, K, gt)
#define ZI_HW_MANY(GATED)                                                                 \
    do {                                                                                  \
        if (wide == 1) ZI_HW(headwise_linear_many_kernel<TX, TO, GATED, 1>);              \
        else if (GATED || wide == 2) ZI_HW(headwise_linear_many_kernel<TX, TO, GATED, 2>); \
        else ZI_HW(headwise_linear_many_kernel<TX, TO, GATED, GATED ? 2 : 4>);            \
    } while (0)
    ZI_DISPATCH_DTYPE(x_dt, TX, ZI_DISPATCH_DTYPE(out_dt, TO, {
        if (many && gate) ZI_HW_MANY(true);
        else if (many) ZI_HW_MANY(false);
        else if (gate) ZI_HW(headwise_linear_few_kernel<TX, TO, true>);
        else ZI_HW(headwise_linear_few_kernel<TX, TO, false>);
    }));
#undef ZI_HW_MANY
#undef ZI_HW
    return zi_check_launch("headwise_linear");
}

extern "C" int zi_headwise_linear(void* out, int out_dt, int64_t ldo, int os, const void* x, int x_dt, int64_t ldx, int xs,
                                  const void* w, int n, int heads, int N, int K, hipStream_t stream) {
    return zi_headwise_linear_gated(out, out_dt, ldo, os, x, x_dt, ldx, xs, w, n, heads, N, K, nullptr, ZI_F32, 0, 1, 0, stream);
}

// qa[t][h][rank + ...] = the rotated part of every head's query, turned in neighbouring pairs.
template <typename T, typename TO>
__global__ void latent_query_rot_kernel(TO* __restrict__ qa, const T* __restrict__ q, int64_t ldq,
                                        const float* __restrict__ table, int n, int heads, int dim, int rank, int rot) {
    const int half = rot / 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)n * heads * half) return;
    const int p = (int)(i % half), h = (int)((i / half) % heads);
    const int64_t t = i / ((int64_t)half * heads);
    const T* qr = q + t * ldq + (int64_t)h * (dim + rot) + dim + 2 * p;
    const float u = zi_load(qr), v = zi_load(qr + 1);
    const float c = table[(t * half + p) * 2], s = table[(t * half + p) * 2 + 1];
    TO* o = qa + (t * heads + h) * (rank + rot) + rank + 2 * p;
    zi_store(o, u * c - v * s);
    zi_store(o + 1, v * c + u * s);
}

extern "C" int zi_latent_query_rot(void* qa, int qa_dt, const void* q, int dt, int64_t ldq, const float* table, int n, int heads,
                                   int dim, int rank, int rot, hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && heads > 0 && dim > 0 && rank > 0 && rot >= 0 && rot % 2 == 0 && ldq >= (int64_t)heads * (dim + rot),
               "latent_query_rot: bad sizes");
    const int64_t total = (int64_t)n * heads * (rot / 2);
    if (total == 0) return 0;
    ZI_REQUIRE(table, "latent_query_rot: no table of angles");
    ZI_DISPATCH_DTYPE(dt, T, ZI_DISPATCH_DTYPE(qa_dt, TO, {
        latent_query_rot_kernel<T, TO><<<(unsigned)((total + 255) / 256), 256, 0, stream>>>((TO*)qa, (const T*)q, ldq, table, n, heads,
                                                                                             dim, rank, rot);
    }));
    return zi_check_launch("latent_query_rot");
}

// Few tokens: qa[t][h] = (W_uk[h]^T q_plain, turn(q_rot)) from the query product's float32 partial sums, one launch.
// x [splits][n][heads * (dim + rot)] (row stride ldx); w bfloat16 [heads][rank][dim].  Workgroups as in
// headwise_linear_few_kernel (the terms are added as they are loaded); the last of a head's (blockIdx.z) turns the rotated part.
template <typename TO>
__global__ void __launch_bounds__(4 * ZI_WAVE)
latent_query_sums_kernel(TO* __restrict__ qa, const float* __restrict__ x, int splits, int64_t split_stride, int64_t ldx,
                         const zi_bf16* __restrict__ w, const float* __restrict__ table, int n, int heads, int dim, int rank, int rot) {
    __shared__ la_f32x4_t part[3][ZI_WAVE];
    const int t0 = blockIdx.x * 16, h = blockIdx.y;
    const int out_w = rank + rot, xs = dim + rot;
    if (blockIdx.z == gridDim.z - 1) {
        const int half = rot / 2;
        for (int i = threadIdx.x; i < 16 * half; i += 4 * ZI_WAVE) {
            const int t = t0 + i / half, p = i % half;
            if (t >= n) continue;
            const float* at = x + (int64_t)t * ldx + (int64_t)h * xs + dim + 2 * p;
            float u = at[0], v = at[1];
            for (int s = 1; s < splits; ++s) {
                u += at[s * split_stride];
                v += at[s * split_stride + 1];
            }
            const float c = table[((int64_t)t * half + p) * 2], sn = table[((int64_t)t * half + p) * 2 + 1];
            TO* o = qa + ((int64_t)t * heads + h) * out_w + rank + 2 * p;
            zi_store(o, u * c - v * sn);
            zi_store(o + 1, v * c + u * sn);
        }
        return;
    }
    const int n0 = blockIdx.z * 16;
    const int lane = threadIdx.x % ZI_WAVE, wave = threadIdx.x / ZI_WAVE, r = lane % 16, j = lane / 16;
    const zi_bf16* wrow = w + ((int64_t)h * rank + (n0 + r < rank ? n0 + r : rank - 1)) * dim;
    const int64_t t = t0 + r < n ? t0 + r : n - 1;
    const float* xrow = x + t * ldx + (int64_t)h * xs;
    la_f32x4_t acc = (la_f32x4_t){0.f, 0.f, 0.f, 0.f};
    for (int k0 = wave * 32; k0 < dim; k0 += 128) {
        const int k = k0 + 8 * j, kc = k < dim ? k : 0;
        const unsigned mask = 0u - (unsigned)(k < dim);
        la_pack a = la_load8(wrow + kc), b;
        float4 lo = *reinterpret_cast<const float4*>(xrow + kc), hi = *reinterpret_cast<const float4*>(xrow + kc + 4);
        for (int s0 = 1; s0 < splits; s0 += 4) {      // four terms in flight, added in their order
            float4 l4[4], h4[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float* at = xrow + (int64_t)(s0 + u < splits ? s0 + u : 0) * split_stride + kc;
                l4[u] = *reinterpret_cast<const float4*>(at);
                h4[u] = *reinterpret_cast<const float4*>(at + 4);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (s0 + u >= splits) break;
                lo.x += l4[u].x; lo.y += l4[u].y; lo.z += l4[u].z; lo.w += l4[u].w;
                hi.x += h4[u].x; hi.y += h4[u].y; hi.z += h4[u].z; hi.w += h4[u].w;
            }
        }
        b.w[0] = zi_pack_bf16x2(lo.x, lo.y);
        b.w[1] = zi_pack_bf16x2(lo.z, lo.w);
        b.w[2] = zi_pack_bf16x2(hi.x, hi.y);
        b.w[3] = zi_pack_bf16x2(hi.z, hi.w);
        a.u &= mask;
        b.u &= mask;
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.b, b.b, acc, 0, 0, 0);
    }
    if (wave > 0) part[wave - 1][lane] = acc;
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int u = 0; u < 3; ++u) acc += part[u][lane];
    if (t0 + r >= n || n0 + 4 * j >= rank) return;
    la_store4(qa + (t * heads + h) * out_w + n0 + 4 * j, acc, rank - n0 - 4 * j);
}

extern "C" int zi_latent_query_sums(void* qa, int qa_dt, const float* x, int splits, int64_t split_stride, int64_t ldx, const void* w,
                                    const float* table, int n, int heads, int dim, int rank, int rot, hipStream_t stream) {
    ZI_REQUIRE(n >= 0 && heads > 0 && heads <= 65535 && dim > 0 && rank > 0 && rot >= 0 && rot % 2 == 0 && splits >= 1 &&
                   ldx >= (int64_t)heads * (dim + rot) && (rank + 15) / 16 < 65535, "latent_query_sums: bad sizes");
    ZI_REQUIRE(zi_headwise_linear_supported(ZI_BF16, dim, ldx, dim + rot) && split_stride % 4 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0,
               "latent_query_sums: sizes in eights and aligned rows are needed");
    ZI_REQUIRE(rot == 0 || table, "latent_query_sums: no table of angles");
    if (n == 0) return 0;
    const dim3 grid((n + 15) / 16, heads, (rank + 15) / 16 + 1);
    ZI_DISPATCH_DTYPE(qa_dt, TO, {
        latent_query_sums_kernel<TO><<<grid, 4 * ZI_WAVE, 0, stream>>>((TO*)qa, x, splits, split_stride, ldx, (const zi_bf16*)w, table, n,
                                                                       heads, dim, rank, rot);
    });
    return zi_check_launch("latent_query_sums");
}
