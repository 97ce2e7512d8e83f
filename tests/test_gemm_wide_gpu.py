"""The products of 65 to 128 rows (csrc/gemm_mid.hip, both operands by buffer loads straight into LDS) where their addressing can
go wrong: rows that lie apart, columns past K, weight rows past a workgroup's, the last row at the end of its memory."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inside(rows, cols, ld, at, g):
    """[rows, cols] bfloat16 of row stride ld in memory that holds NaN wherever it does not lie, and ends with its last value."""
    store = torch.full((at + (rows - 1) * ld + cols,), float("nan"), dtype=torch.bfloat16, device="cuda")
    t = store.as_strided((rows, cols), (ld, 1), at)
    t.copy_(torch.randn(rows, cols, generator=g, device="cuda"))
    return t


def _check(ops, x, w, monkeypatch):
    from zedinfer_amd.ops import functional
    from zedinfer_amd.parts.feed_forward import GATE_UP_BLOCK
    monkeypatch.setattr(functional, "SWIGLU_MAX_ROWS", 128)
    M, K, N = x.shape[0], x.shape[1], w.shape[0]
    sums = ops.linear_sums(x, w)
    ref, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    # exact products, at most K + 16 roundings of running sums that are at most `size`
    bound = (K + 16) * 2.0 ** -24 * size
    assert bool(((sums.double().sum(0) - ref).abs() <= bound).all())
    # the kernel for up to 64 rows: the same sums in the same order
    for rows in (slice(0, 64), slice(M - 33, M)):
        assert torch.equal(ops.linear_sums(x[rows], w), sums[:, rows])
    if N % 16 == 0:
        wide = torch.full((M, N // 2 + 8), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.linear_swiglu(x, w, out=wide[:, :N // 2])
        gu = ref.view(M, -1, 2, GATE_UP_BLOCK)
        want = (gu[:, :, 1] * torch.nn.functional.silu(gu[:, :, 0])).reshape(M, N // 2)
        # gate and up each off by `bound`, and one rounding to bfloat16 (silu's slope is below 1.1)
        off = bound.view(M, -1, 2, GATE_UP_BLOCK)
        slack = 1.1 * off[:, :, 0] * gu[:, :, 1].abs() + off[:, :, 1] * gu[:, :, 0].abs()
        assert bool(((wide[:, :N // 2].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2 * slack.reshape(M, -1) + 1e-30).all())
        assert bool((wide[:, N // 2:] == 7.0).all())


@pytest.mark.parametrize("M", [65, 80, 97, 128])
@pytest.mark.parametrize("N,K,padx,padw", [(1, 8, 0, 0), (16, 72, 8, 16), (130, 200, 24, 8), (304, 1000, 0, 40), (1024, 1544, 56, 0), (7, 4096, 8, 8)])
def test_rows_that_lie_apart(M, N, K, padx, padw, monkeypatch):
    from zedinfer_amd import ops
    g = torch.Generator(device="cuda").manual_seed(M * N + K)
    _check(ops, _inside(M, K, K + padx, padx // 8 * 8, g), _inside(N, K, K + padw, padw // 8 * 8, g), monkeypatch)


@pytest.mark.parametrize("ldx,ldw", [(1 << 22, 1 << 22), ((1 << 22) + 8, 264), (264, (1 << 22) + 8), ((1 << 24) + (1 << 23), 1 << 24)])
def test_rows_further_apart_than_offsets_of_31_bits_reach(ldx, ldw, monkeypatch):
    """128 rows of 2^23 elements and more are 2^31 bytes apart and more: the kernel with addresses of 64 bits takes them."""
    from zedinfer_amd import ops
    g = torch.Generator(device="cuda").manual_seed(ldx % 1000 + ldw % 1000)
    for M, N, K in ((128, 80, 264), (77, 16, 72)):
        _check(ops, _inside(M, K, ldx, 0, g), _inside(N, K, ldw, 0, g), monkeypatch)


@pytest.mark.parametrize("I,K,many", [(8960, 1536, True), (3072, 1024, True), (18944, 3584, False), (2048, 7168, False), (512, 8192, False),
                                      (256, 7168, False), (2048, 2048, False)])
def test_which_products_take_the_swiglu_epilogue_beyond_64_rows(I, K, many):
    """Those that would not be cut for more than a launch is worth and whose workgroups are one round on 256 compute units (up to 64
    rows: those that are never cut)."""
    from zedinfer_amd import ops
    w = torch.empty(2 * I, K, dtype=torch.bfloat16, device="cuda")
    for M in (64, 65, 100, 128, 129):
        x = torch.empty(M, K, dtype=torch.bfloat16, device="cuda")
        if M > 64:
            assert ops.linear_swiglu_pays(x, w) == (many and M <= 128), M
        else:
            assert ops.linear_swiglu_pays(x, w) == ops.linear_swiglu_supported(x, w) == (ops.linear_splits(M, 2 * I, K) == 1)


# ---- 129 to 256 rows: eight wavefronts, four along the rows of x and two along the weight rows -----------------------------------
# (weight rows that make workgroups of 4, 5, 6, 7, 8 and 10 weight tiles on 256 compute units, the last one not whole, and, with the
# rows of x, three buffers of a step or four; columns that end inside a step)
@pytest.mark.parametrize("M", [129, 160, 192, 210, 225, 256])
@pytest.mark.parametrize("N,K", [(16, 8), (16000, 72), (20464, 72), (24544, 200), (28640, 72), (32720, 136), (40944, 72)])
def test_the_epilogue_of_129_to_256_rows(M, N, K, monkeypatch):
    from zedinfer_amd import ops
    from zedinfer_amd.ops import functional
    from zedinfer_amd.parts.feed_forward import GATE_UP_BLOCK
    monkeypatch.setattr(functional, "SWIGLU_MAX_ROWS", 256)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, w = _inside(M, K, K + 24, 8, g), _inside(N, K, K + 8, 0, g)
    wide = torch.full((M, N // 2 + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.linear_swiglu(x, w, out=wide[:, :N // 2])
    gu, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    gu, off = gu.view(M, -1, 2, GATE_UP_BLOCK), (K + 16) * 2.0 ** -24 * size.view(M, -1, 2, GATE_UP_BLOCK)
    want = (gu[:, :, 1] * torch.nn.functional.silu(gu[:, :, 0])).reshape(M, N // 2)
    slack = 1.1 * off[:, :, 0] * gu[:, :, 1].abs() + off[:, :, 1] * gu[:, :, 0].abs()
    assert bool(((wide[:, :N // 2].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2 * slack.reshape(M, -1) + 1e-30).all())
    assert bool((wide[:, N // 2:] == 7.0).all())
    # the kernel for up to 128 rows: the same sums in the same order
    assert torch.equal(ops.linear_swiglu(x[M - 101:], w), wide[M - 101:, :N // 2])
    if ops.linear_swiglu_many_pays(x, w):
        assert torch.equal(ops.linear_swiglu_many(x, w), wide[:, :N // 2])


@pytest.mark.parametrize("M", [129, 150, 200, 256])
@pytest.mark.parametrize("N,K,padx,padw", [(3000, 2800, 8, 16), (2904, 5800, 0, 0), (4608, 3584, 0, 8), (1000, 33560, 24, 0), (80, 209736, 8, 8)])
def test_partial_sums_of_129_to_256_rows(M, N, K, padx, padw):
    from zedinfer_amd import ops
    g = torch.Generator(device="cuda").manual_seed(M * N + K)
    x, w = _inside(M, K, K + padx, padx // 8 * 8, g), _inside(N, K, K + padw, 0, g)
    assert ops.linear_sums_supported(x, w)
    sums = ops.linear_sums(x, w)
    ref, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert bool(((sums.double().sum(0) - ref).abs() <= (K + 16) * 2.0 ** -24 * size).all())
    assert torch.equal(ops.linear_sums(x[:129].contiguous(), w), sums[:, :129])


def test_partial_sums_of_rows_further_apart_than_offsets_of_31_bits_reach():
    from zedinfer_amd import ops
    g = torch.Generator(device="cuda").manual_seed(1)
    N, K = 80, 209736
    near = _inside(256, K, K, 0, g), _inside(N, K, K, 0, g)
    for ldx, ldw in (((1 << 21) + 8, K), (K, (1 << 22) + 8), (1 << 21, 1 << 21)):
        x, w = _inside(256, K, ldx, 0, g), _inside(N, K, ldw, 0, g)
        x.copy_(near[0])
        w.copy_(near[1])
        assert torch.equal(ops.linear_sums(x, w), ops.linear_sums(*near))


@pytest.mark.parametrize("I,K,pays", [(18944, 3584, True), (8960, 1536, True), (4864, 896, True), (3072, 1024, True), (20480, 7168, True),
                                      (27648, 5120, False), (13824, 5120, False), (4096, 4096, False), (512, 8192, False)])
def test_which_products_of_129_to_256_rows_take_the_epilogue(I, K, pays):
    from zedinfer_amd import ops
    w = torch.empty(2 * I, K, dtype=torch.bfloat16, device="cuda")
    for M, here in ((128, False), (129, pays), (256, pays), (257, False)):
        x = torch.empty(M, K, dtype=torch.bfloat16, device="cuda")
        assert ops.linear_swiglu_many_pays(x, w) == here, M
        if not here:
            with pytest.raises(ValueError):
                ops.linear_swiglu_many(x, w)
