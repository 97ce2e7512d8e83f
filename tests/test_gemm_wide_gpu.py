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
