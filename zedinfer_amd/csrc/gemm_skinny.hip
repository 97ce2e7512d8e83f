// out[M,N] = x[M,K] . w[N,K]^T (+ bias) for up to 256 rows of x: the decode-time matrix products, bound by the
// one pass over the weights.  This file holds their entry points, the cut's bookkeeping and the kernel that
// adds partial sums; the product kernels are in gemm_mid.hip (x staged in LDS, a workgroup's wavefronts take 16 weight rows each, or,
// from 65 rows on, share the rows of x, the cut over workgroups balanced over the compute units).
//
// When the weight matrix gives too few workgroups the k dimension is cut over several of them (gridDim.y
// "splits"); those write float32 partial sums [split][M][N] that the consumer adds in rising order (the next
// norm, the rotary kernel, the SwiGLU kernel, or the reduce kernel here).  The cut depends on N and K only,
// so a row's result does not depend on how many rows ride along.
//
// Epilogues: plain (bias, bfloat16 or float32 out), partial sums, and SwiGLU: when the weight rows are gate
// and up rows interleaved in blocks of 8 (tile = 8 gate rows, then the 8 up rows of the same columns), the
// tile's lanes exchange halves and write act = up * gate / (1 + exp(-gate))
// (reference: src/backend/ops/swiglu/cpu/swiglu_cpu.cpp:9-23); and an activation of every output, for products that are made
// whole.
//
// A kernel that kept x in registers and cut k over a workgroup's wavefronts served up to 16 rows before the
// other one's cut was balanced; since then it was slower at every size from one row on (1.5B gate/up at 8 rows
// 12.9 against 11.7 us, 32B gate/up 111 against 95 us) and is gone.
#include "zi_common.h"
#include "zi_activation.h"
#include "zi_api.h"

#define SK_MODE_PLAIN 0
#define SK_MODE_PARTIAL 1
#define SK_MODE_SWIGLU 2
#define SK_MODE_CLAMPED 3
#define SK_MODE_ACT 4              // + the activation's code

// out[m,n] = sum_s partial[s,m,n] + bias[n], splits added in rising order.
__global__ void gemm_skinny_reduce_kernel(void* __restrict__ out, int out_f32, const float* __restrict__ partial,
                                          const zi_bf16* __restrict__ bias, int M, int N, int64_t ldo, int splits) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)M * N) return;
    const int m = (int)(i / N), n = (int)(i % N);
    float s = 0.f;
    for (int k = 0; k < splits; ++k) s += partial[(int64_t)k * M * N + i];
    if (bias) s += zi_load(bias + n);
    if (out_f32) ((float*)out)[(int64_t)m * ldo + n] = s;
    else zi_store((zi_bf16*)out + (int64_t)m * ldo + n, s);
}

// The same, four columns a thread and all of its sums on their way before the first is added: the kernel is a trip to memory that other XCDs
// have just written, and one after the other they were as many trips.  us: 32 rows of
// 1,536 columns and 10 sums 4.7 to 2.6, of 4,632 and 6 3.9 to 2.9, 8 of 4,632 2.9 to 2.35, 64 of 1,536 and 10 to bfloat16 4.6 to 2.9.
template <int SPLITS>
__global__ void __launch_bounds__(64)
gemm_skinny_reduce4_kernel(void* __restrict__ out, int out_f32, const float* __restrict__ partial, const zi_bf16* __restrict__ bias,
                           int N, int64_t total, int64_t ldo) {
    const int64_t i = ((int64_t)blockIdx.x * 64 + threadIdx.x) * 4;
    if (i >= total) return;
    const int64_t m = i / N;
    const int n = (int)(i - m * N);
    float4 p[SPLITS];
#pragma unroll
    for (int k = 0; k < SPLITS; ++k) p[k] = *reinterpret_cast<const float4*>(partial + k * total + i);
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < SPLITS; ++k) {
        s.x += p[k].x;
        s.y += p[k].y;
        s.z += p[k].z;
        s.w += p[k].w;
    }
    if (bias) {
        s.x += zi_load(bias + n);
        s.y += zi_load(bias + n + 1);
        s.z += zi_load(bias + n + 2);
        s.w += zi_load(bias + n + 3);
    }
    if (out_f32) {
        *reinterpret_cast<float4*>((float*)out + m * ldo + n) = s;
    } else {
        uint2 pk;
        pk.x = zi_pack_bf16x2(s.x, s.y);
        pk.y = zi_pack_bf16x2(s.z, s.w);
        *reinterpret_cast<uint2*>((zi_bf16*)out + m * ldo + n) = pk;
    }
}

// The sums added, by the one kernel where every four columns are whole 16-byte pieces (8-byte ones of a bfloat16 result), else by the
// other: the same order, the same bits.
static void sk_reduce(void* out, int out_f32, const float* partial, const zi_bf16* bias, int M, int N, int64_t ldo, int splits,
                      hipStream_t stream) {
    const int64_t total = (int64_t)M * N;
    if (N % 4 == 0 && ldo % 4 == 0 && (uintptr_t)partial % 16 == 0 && (uintptr_t)out % (out_f32 ? 16 : 8) == 0 && splits <= 16) {
#define ZI_SK_REDUCE(S)                                                                                                          \
    case S:                                                                                                                      \
        gemm_skinny_reduce4_kernel<S><<<(unsigned)((total / 4 + 63) / 64), 64, 0, stream>>>(out, out_f32, partial, bias, N, total, ldo); \
        return
        switch (splits) {
            ZI_SK_REDUCE(1); ZI_SK_REDUCE(2); ZI_SK_REDUCE(3); ZI_SK_REDUCE(4); ZI_SK_REDUCE(5); ZI_SK_REDUCE(6); ZI_SK_REDUCE(7); ZI_SK_REDUCE(8);
            ZI_SK_REDUCE(9); ZI_SK_REDUCE(10); ZI_SK_REDUCE(11); ZI_SK_REDUCE(12); ZI_SK_REDUCE(13); ZI_SK_REDUCE(14); ZI_SK_REDUCE(15); ZI_SK_REDUCE(16);
        }
#undef ZI_SK_REDUCE
    }
    gemm_skinny_reduce_kernel<<<(int)((total + 255) / 256), 256, 0, stream>>>(out, out_f32, partial, bias, M, N, ldo, splits);
}

#define SK_MAX_ROWS 256
#define SK_MID_MAX_ROWS 128        // up to here one cut of the weights, beyond it another
#define SK_MAX_ROWS_ACT 64         // ... with the epilogues that only products of few rows have

extern "C" int zi_gemm_skinny_supported(int M, int N, int K, int64_t ldx, int64_t ldw) {
    return M >= 1 && M <= SK_MAX_ROWS && N >= 1 && K >= 8 && K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0;
}

// most rows the products take
extern "C" int zi_gemm_skinny_max_rows() { return SK_MAX_ROWS; }

// 1 when these kernels are the faster way to partial sums than the library's product of the same operands, with what the next kernel's
// reading of the sums costs, as measured: always up to 128 rows; beyond, for weights with at least twice as many columns as
// rows (a down projection) from 2^24 elements on (us at 160 and 256 rows against the library's 36 and 40: 2,048 x 11,008 19 and 23 with
// 8 splits; 1,536 x 8,960 14 and 17 against 23 and 31, of which 10 splits of sums take most back), and for about square ones (q/k/v,
// output) from 2^23 on (3,072 x 3,072 12 and 15 against 17 and 18, 4,096 x 4,096 14 and 18 against 27 and 23; 2,048 x 2,048 8 and 11
// against 9 and 10).  Weights with many more rows than columns are whole products, whose partial sums gain nothing.
extern "C" int zi_gemm_skinny_pays(int M, int N, int K) {
    if (M <= SK_MID_MAX_ROWS) return 1;
    const int64_t n = N, k = K, size = n * k;
    return M <= SK_MAX_ROWS && (k >= 2 * n ? size >= 1 << 24 : n <= 2 * k && size >= 1 << 23);
}

// The product kernels (gemm_mid.hip): their cuts and their launch.
int64_t zi_gemm_mid_plan(int N, int K, int whole, int* splits, int* kb_per_split, int* waves);
int64_t zi_gemm_many_plan(int N, int K, int whole, int* splits, int* kb_per_split, int* tiles);
int zi_gemm_mid_launch(void* out, int out_f32, int mode, const zi_bf16* x, const zi_bf16* w, const zi_bf16* bias, int M,
                       int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, int vec_out, float limit, hipStream_t stream);

static bool sk_many(int M) { return M > SK_MID_MAX_ROWS; }

// Splits of k for a weight matrix [N, K]: the leading dimension of the partial sums.  A function of N and K and
// of whether there are more than 128 rows.
extern "C" int zi_gemm_skinny_splits(int M, int N, int K) {
    int s, per, waves;
    if (sk_many(M)) zi_gemm_many_plan(N, K, 0, &s, &per, &waves);
    else zi_gemm_mid_plan(N, K, 0, &s, &per, &waves);
    return s;
}

// Floats of workspace for the split partials (0 when the product is not split).
extern "C" int64_t zi_gemm_skinny_workspace(int M, int N, int K) {
    const int s = zi_gemm_skinny_splits(M, N, K);
    return s > 1 ? (int64_t)s * M * N : 0;
}

// 1 when a product with an activation in its epilogue, which is made whole, costs no more than one that may be split and the
// activation's launch after it: a launch is worth about as much as this many of the cut's wavefront-blocks.
#define SK_LAUNCH_COST 32
extern "C" int zi_gemm_skinny_act_pays(int M, int N, int K) {
    if (M < 1 || M > SK_MAX_ROWS_ACT) return 0;
    int s, per, waves;
    const int64_t whole = zi_gemm_mid_plan(N, K, 1, &s, &per, &waves);
    return whole <= zi_gemm_mid_plan(N, K, 0, &s, &per, &waves) + SK_LAUNCH_COST;
}

// 1 when the SwiGLU epilogue of 65 to 128 rows beats the library's product and the activation's launch.  It makes the product
// whole, so it does where a cut would gain no more than a launch is worth and where the workgroups are one round on the compute
// units.  Measured with weights from memory, columns I of output x K, epilogue against library and launch, at 65 and at 128 rows: one
// round 8,960 x 1,536 16.8 against 21.4 us and 21.1 against 25.5, 13,824 x 5,120 57 against 62 and 65 against 70, 3,072 x 1,024
// 10.4 against 15.0 and 11.7 against 15.1; two rounds 18,944 x 3,584 60 against 64 but 73 against 65, 27,648 x 5,120 112 against
// 116 but 134 against 124; a product that wants its cut 2,048 x 7,168 39 against 26 and 50 against 30, 512 x 8,192 42 against 15
// and 50 against 17, 4,096 x 4,096 25 against 23 and 31 against 25.
extern "C" int zi_gemm_skinny_swiglu_pays(int M, int N, int K) {
    if (M <= 64 || M > SK_MID_MAX_ROWS) return 0;
    int s, per, waves;
    const int64_t cut = zi_gemm_mid_plan(N, K, 0, &s, &per, &waves), whole = zi_gemm_mid_plan(N, K, 1, &s, &per, &waves);
    return whole <= cut + SK_LAUNCH_COST && ((N + 15) / 16 + waves - 1) / waves <= zi_compute_units();
}

// The same for 129 to 256 rows.  A launch and the sums that a cut leaves are 4 us; the workgroups have to be one round, and of ten
// weight tiles (a slice of x is read for each of them) unless k is short.  us at 160 and 256 rows, epilogue against the library's first
// proposal and the launch: 18,944 columns I x 3,584 63 and 79 against 84 and 88, 8,960 x 1,536 24 and 27 against 30 and 34, 11,008 x
// 2,048 29 and 34 against 35 and 39, 4,864 x 896 13 and 16 against 17 and 20, 20,480 x 7,168 120 and 151 against 155 and 167; left to the
// library: two rounds 27,648 x 5,120 152 and 176 against 137 and 169, seven tiles 13,824 x 5,120 77 and 94 against 79 and 95, half
// a round 4,096 x 4,096 36 and 47 against 32 and 45.
extern "C" int zi_gemm_skinny_swiglu_many_pays(int M, int N, int K) {
    if (M <= SK_MID_MAX_ROWS || M > SK_MAX_ROWS) return 0;
    int s, per, tiles, cut_tiles;
    const int64_t cut = zi_gemm_many_plan(N, K, 0, &s, &per, &cut_tiles), whole = zi_gemm_many_plan(N, K, 1, &s, &per, &tiles);
    return whole <= cut + 4000 && ((N + 15) / 16 + tiles - 1) / tiles <= zi_compute_units() && (tiles == 10 || K < 4096);
}

// mode 0: out[M,N] (+ bias), reduced through `workspace` when the product is split.
// mode 1: out = float32 partial sums [splits][M][N] (splits from zi_gemm_skinny_splits; the bias, if any, is in the first).
// mode 2: w holds gate and up rows interleaved in blocks of 8; out[M, N/2] (bfloat16) =
//         up * silu(gate); only for products that are not split.
// mode 3: the same with g = min(gate + bias, limit), u = clamp(up + bias, -limit, limit), g sigmoid(1.702 g) (u + 1), the
//         bias [N] (or null) interleaved as the rows are; up to 64 rows.
// mode 4 + a: out[M,N] (bfloat16) = activation a (0 SiLU, 1 GELU in its tanh form, 3 relu squared) of the product and the bias
//         [N] (or null); up to 64 rows, the product never split.
extern "C" int zi_gemm_skinny_act(void* out, int out_dt, int mode, const void* x, const void* w, const void* bias, int M,
                                  int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, float* workspace,
                                  int64_t workspace_floats, float limit, hipStream_t stream) {
    ZI_REQUIRE(zi_gemm_skinny_supported(M, N, K, ldx, ldw),
               "gemm_skinny: unsupported sizes M=%d N=%d K=%d (1 <= M <= 256, K and row strides multiples of 8)", M, N, K);
    ZI_REQUIRE(out_dt == ZI_F32 || out_dt == ZI_BF16, "gemm_skinny: unknown output dtype %d", out_dt);
    ZI_REQUIRE(mode >= 0 && mode <= SK_MODE_ACT + ZI_ACT_RELU2 && mode != SK_MODE_ACT + ZI_ACT_GELU_ERF, "gemm_skinny: unknown mode %d", mode);
    ZI_REQUIRE(mode < SK_MODE_ACT || (M <= SK_MAX_ROWS_ACT && out_dt == ZI_BF16 && ldo >= N),
               "gemm_skinny: an activation takes up to %d rows and a bfloat16 out of N columns", SK_MAX_ROWS_ACT);
    ZI_REQUIRE(mode != SK_MODE_CLAMPED || (limit > 0.f && M <= SK_MAX_ROWS_ACT), "gemm_skinny: the clamped epilogue takes up to %d rows and a positive limit", SK_MAX_ROWS_ACT);
    ZI_REQUIRE(ldx >= K && ldw >= K, "gemm_skinny: leading dimension too small");
    ZI_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0, "gemm_skinny: x and w must be 16-byte aligned");
    int splits, per, waves;
    if (sk_many(M)) zi_gemm_many_plan(N, K, mode == SK_MODE_SWIGLU, &splits, &per, &waves);
    else zi_gemm_mid_plan(N, K, mode >= SK_MODE_ACT || (mode == SK_MODE_SWIGLU && M > 64), &splits, &per, &waves);       // (whole from 65 rows on)
    void* dst = out;
    int kmode = mode;
    if (mode == SK_MODE_PLAIN) {
        ZI_REQUIRE(ldo >= N, "gemm_skinny: leading dimension of out too small");
        if (splits > 1) {
            ZI_REQUIRE(workspace && workspace_floats >= (int64_t)splits * M * N,
                       "gemm_skinny: workspace of %lld floats is too small (%lld needed)", (long long)workspace_floats,
                       (long long)splits * M * N);
            dst = workspace;
            kmode = SK_MODE_PARTIAL;
        }
    } else if (mode == SK_MODE_PARTIAL) {
        ZI_REQUIRE(out_dt == ZI_F32, "gemm_skinny: partial sums are float32");
    } else if (mode < SK_MODE_ACT) {
        ZI_REQUIRE(splits == 1, "gemm_skinny: the SwiGLU epilogue needs a product that is not split (N=%d K=%d has %d)",
                   N, K, splits);
        ZI_REQUIRE(N % 16 == 0 && out_dt == ZI_BF16 && ldo >= N / 2,
                   "gemm_skinny: the SwiGLU epilogue needs N %% 16 == 0 and a bfloat16 out of N/2 columns");
    }
    const zi_bf16* b = (kmode == SK_MODE_PLAIN || mode == SK_MODE_PARTIAL || mode >= SK_MODE_CLAMPED) ? (const zi_bf16*)bias : nullptr;
    // four columns go out as one store when every row of the destination keeps them aligned
    int vec_out;
    if (kmode == SK_MODE_PARTIAL) vec_out = N % 4 == 0 && ((uintptr_t)dst % 16) == 0;
    else if (kmode >= SK_MODE_SWIGLU) vec_out = ldo % 4 == 0 && ((uintptr_t)dst % 8) == 0;
    else vec_out = ldo % 4 == 0 && ((uintptr_t)dst % (out_dt == ZI_F32 ? 16 : 8)) == 0;
    const int of32 = out_dt == ZI_F32;
    const int rc = zi_gemm_mid_launch(dst, of32, kmode, (const zi_bf16*)x, (const zi_bf16*)w, b, M, N, K, ldx, ldw, ldo, vec_out, limit, stream);
    if (rc) return rc;
    if (mode == SK_MODE_PLAIN && splits > 1) sk_reduce(out, of32, workspace, (const zi_bf16*)bias, M, N, ldo, splits, stream);
    return zi_check_launch("gemm_skinny");
}

extern "C" int zi_gemm_skinny(void* out, int out_dt, int mode, const void* x, const void* w, const void* bias, int M,
                              int N, int K, int64_t ldx, int64_t ldw, int64_t ldo, float* workspace,
                              int64_t workspace_floats, hipStream_t stream) {
    ZI_REQUIRE(mode >= 0 && mode <= 2, "gemm_skinny: unknown mode %d", mode);
    return zi_gemm_skinny_act(out, out_dt, mode, x, w, bias, M, N, K, ldx, ldw, ldo, workspace, workspace_floats, 0.f, stream);
}

// out[m,n] = sum_s sums[s,m,n] + bias[n] for float32 sums [splits][M][N], added in rising order.
extern "C" int zi_reduce_splits(void* out, int out_dt, const float* sums, const void* bias, int M, int N, int64_t ldo,
                                int splits, hipStream_t stream) {
    ZI_REQUIRE(M >= 0 && N > 0 && splits >= 1 && ldo >= N, "reduce_splits: bad sizes");
    ZI_REQUIRE(out_dt == ZI_F32 || out_dt == ZI_BF16, "reduce_splits: unknown output dtype %d", out_dt);
    if (M == 0) return 0;
    sk_reduce(out, out_dt == ZI_F32, sums, (const zi_bf16*)bias, M, N, ldo, splits, stream);
    return zi_check_launch("reduce_splits");
}
