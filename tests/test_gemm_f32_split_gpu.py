"""float32 products of more than 1,408 columns (csrc/gemm_f32_split.hip): products of bfloat16 parts that add up to the float32 product.
What rides on the split itself, beyond what tests/test_gemm_f32_gpu.py asks of every float32 product."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# every kernel: groups of 8 rows, streams of 16 and 32 rows of x, x held for both (3, 4, 6, 8 chunks a run), tiles of every kind with rows,
# weight rows and columns that end within a tile, a chunk and a run
CASES = [(3, 1030, 1412, "pairs"), (8, 700, 9000, "pairs"), (12, 2070, 1412, "rows16"), (12, 300, 4100, "pairs"), (30, 2040, 1420, "rows16"), (40, 2040, 1500, "rows32"),
         (7, 2059, 1536, "held_pairs"), (5, 2054, 1800, "held_pairs"), (8, 3000, 3000, "held_pairs"), (2, 2049, 4096, "held_pairs"),
         (16, 5000, 1532, "held_rows16"), (13, 4098, 2048, "held_rows16"), (100, 2050, 1500, "tile_32_halves"), (500, 1500, 1480, "tile_96_halves"),
         (449, 2047, 1540, "tile_64_quarters"), (700, 4610, 1412, "tile_64"), (450, 4610, 1500, "tile_96_halves"), (449, 8194, 1500, "tile_32")]


def _linear(M, N, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N + seed)
    return tuple(torch.randn(s, generator=g, device="cuda") for s in ((M, K), (N, K), (N,)))


@pytest.mark.parametrize("M,N,K,kernel", CASES)
def test_as_exact_as_float32_sums_and_without_a_bias(M, N, K, kernel):
    from zedinfer_amd import ops
    assert ops.linear_f32_kernel(M, N, K) == kernel
    x, w, b = _linear(M, N, K)
    got = ops.linear(x, w, b).double()
    ref = x.double() @ w.double().t() + b.double()
    # an instruction adds 32 products to the sum with errors of at most three of the sum's last bits, six instructions to 32 columns in
    # each of two chains of an eighth of k (rounded up to chunks of 64), then eleven additions: so many times 2^-23 of at most sum |x w| + |b|
    steps = 2 * 6 * -(-(-(-K // 64)) // 8) + 11
    bound = steps * 2.0 ** -23 * (x.double().abs() @ w.double().abs().t() + b.double().abs())
    assert bool(((got - ref).abs() <= bound).all())
    # the same in the mean: the roundings of one chain's sums times 2^-24 of the result's rms each (the sums grow to it), added as squares
    err = (got - ref).square().mean().sqrt() / ref.square().mean().sqrt()
    assert float(err) <= 2.0 ** -24 * steps ** 0.5, float(err)
    # the instruction rounds small products down: with one sign for both chains the mean error is a fifth of its rms and more
    assert float((got - ref).mean().abs()) <= float((got - ref).square().mean().sqrt()) * (1 / 16 + 6 / (M * N) ** 0.5)
    for rows in (slice(M - 1, M), slice(max(0, M - 11), M), slice(max(0, M - 40), M)):
        assert torch.equal(ops.linear(x[rows].contiguous(), w, b).double(), got[rows])


@pytest.mark.parametrize("half", [0, 1])
@pytest.mark.parametrize("M,N,K,kernel", CASES)
def test_no_bias_where_one_half_of_every_chunk_is_empty(M, N, K, kernel, half):
    """The two chains change places from run to run, so the instruction's rounding down cancels in them too: test_as_exact_...'s bound on the mean."""
    from zedinfer_amd import ops
    assert ops.linear_f32_kernel(M, N, K) == kernel
    x, w, _ = _linear(M, N, K)
    x *= torch.arange(K, device="cuda") // 32 % 2 == half
    err = ops.linear(x, w).double() - x.double() @ w.double().t()
    assert float(err.mean().abs()) <= float(err.square().mean().sqrt()) * (1 / 16 + 6 / (M * N) ** 0.5)


def _mean_bound(K):
    """The mean of the error, 2-norm over 2-norm: the roundings of one chain's sums times 2^-24 of the result's rms each, added as squares."""
    return 2.0 ** -24 * (2 * 6 * -(-(-(-K // 64)) // 8) + 11) ** 0.5


def _error(x, w):
    from zedinfer_amd import ops
    got, ref = ops.linear(x, w).double(), x.double() @ w.double().t()
    return float(((got - ref).square().sum(1) / ref.square().sum(1)).max().sqrt()) if ref.numel() else 0.0


@pytest.mark.parametrize("M,N,K,kernel", CASES)
def test_sums_made_again_from_the_operands(M, N, K, kernel):
    """A row whose values all round to an infinity in bfloat16 is as exact as any other; a row with a NaN is NaNs, all of it; neither touches the others."""
    from zedinfer_amd import ops
    assert ops.linear_f32_kernel(M, N, K) == kernel
    x, w, _ = _linear(M, N, K)
    w *= 2.0 ** -110
    y = ops.linear(x, w)
    x[0] = torch.where(x[0] < 0, -3.4e38, 3.4e38)
    assert _error(x[:1], w) <= _mean_bound(K)
    x[M - 1, K - 1] = float("nan")
    got = ops.linear(x, w)
    ref = x[:1].double() @ w.double().t()
    assert float((got[:1] - ref).norm() / ref.norm()) <= _mean_bound(K)
    assert bool(torch.isnan(got[M - 1]).all()) and torch.equal(got[1:M - 1], y[1:M - 1])
    if N % 2 == 0 and ops.linear_swiglu_halves_supported(x, w):
        assert torch.equal(ops.linear_swiglu_halves(x, w)[:M - 1], ops.swiglu(got[:, :N // 2], got[:, N // 2:])[:M - 1])


@pytest.mark.parametrize("M,N,K,kernel", CASES)
def test_small_and_large_values_keep_their_last_bits(M, N, K, kernel):
    """Values of any mantissa over float32's whole range, on either side: as exact as values around one."""
    from zedinfer_amd import ops
    assert ops.linear_f32_kernel(M, N, K) == kernel
    x, w, _ = _linear(M, N, K)
    for e in (-60, -90, -104, -112, -120, -126, -132, -138, -145):       # (from -126 on subnormal: the reference multiplies what is left of them)
        other = 2.0 ** min(-e - 20, 121)
        small = x * 2.0 ** e if e > -140 else torch.where(x.abs() < 1, torch.ones_like(x), x.round()) * 2.0 ** e
        assert _error(small, w * other) <= _mean_bound(K), e
        small = w * 2.0 ** e if e > -140 else torch.where(w.abs() < 1, torch.ones_like(w), w.round()) * 2.0 ** e
        assert _error(x * other, small) <= _mean_bound(K), e
    for e in (70, 104, 125):
        assert _error(x * 2.0 ** (e - 3), w * 2.0 ** (-e)) <= _mean_bound(K) and _error(x * 2.0 ** (1 - e), w * 2.0 ** (e - 3)) <= _mean_bound(K), e


@pytest.mark.parametrize("M,N", [(3, 300), (3, 2100), (12, 4100), (12, 2070), (40, 2040), (100, 2050), (449, 1500), (449, 2047), (700, 4610)])
def test_values_that_do_not_split(M, N):
    """Infinities, NaNs and values that round to an infinity in bfloat16 give what the float32 sum gives, in their row and column alone."""
    from zedinfer_amd import ops
    K = 1500
    x, w = torch.ones(M, K, device="cuda"), torch.ones(N, K, device="cuda")
    big = torch.finfo(torch.float32).max
    x[0, 3], x[1, 1499], x[2, :] = float("inf"), big, 2.0 ** -130
    w[5, 0], w[6, 7] = float("nan"), float("-inf")
    y = ops.linear(x, w)
    cols = [i for i in range(N) if i not in (5, 6)]
    assert bool((y[0, cols] == float("inf")).all()) and bool(torch.isnan(y[:, 5]).all())
    assert bool(torch.isnan(y[0, 6])) and bool((y[1:, 6] == float("-inf")).all())
    assert bool((y[1, cols] == big).all())                      # (the other ones are far below its last bit)
    assert bool((y[2, cols] == 1500 * 2.0 ** -130).all())
    if M > 3:
        assert bool((y[3:][:, cols] == 1500).all())
    if ops.linear_swiglu_halves_supported(x, torch.cat([w, w])):
        a = ops.linear_swiglu_halves(x, torch.cat([w, w]))
        assert torch.equal(a.nan_to_num(), ops.swiglu(y, y).nan_to_num())


@pytest.mark.parametrize("M,I,K", [(100, 3001, 1500), (129, 4097, 1500), (64, 8960, 1536), (330, 1537, 1412), (600, 1000, 2052)])
def test_tiles_of_32_by_96_take_the_activation(M, I, K):
    """The bits of the product and the activation one after the other; gate and up rows that end within a tile."""
    from zedinfer_amd import ops
    assert ops.linear_f32_kernel(M, 2 * I, K) == "tile_96_halves"
    x, w, _ = _linear(M, 2 * I, K)
    assert ops.linear_swiglu_halves_supported(x, w)
    two = ops.linear(x, w)
    wide = torch.zeros((M, I + 6), device="cuda")
    ops.linear_swiglu_halves(x, w, out=wide[:, 3:I + 3])
    assert torch.equal(wide[:, 3:I + 3], ops.swiglu(two[:, :I], two[:, I:])) and not wide[:, :3].any() and not wide[:, I + 3:].any()


def test_bits_depend_on_k_alone():
    """On both sides of the bound on k every number of rows has the same bits, and whole numbers give whole numbers."""
    from zedinfer_amd import ops
    for K in (1408, 1412):
        x, w, b = _linear(300, 2060, K)
        whole = ops.linear(x, w, b)
        for m in (1, 8, 9, 16, 17, 33, 130):
            assert torch.equal(ops.linear(x[:m].contiguous(), w, b), whole[:m])
    x, w = torch.randint(-8, 9, (40, 2000), device="cuda").float(), torch.randint(-8, 9, (300, 2000), device="cuda").float()
    assert torch.equal(ops.linear(x, w).double(), x.double() @ w.double().t())


@pytest.mark.parametrize("N,K", [(700, 9000), (1030, 1412), (300, 4100), (2059, 1536), (2054, 1800), (3000, 3000), (2049, 4096)])
def test_one_to_eight_rows_alone_and_together(N, K):
    """Up to two and up to four rows of x are loaded and split by all lanes: the bits of eight rows, in the streams and where x is held (3, 4, 6, 8 chunks)."""
    from zedinfer_amd import ops
    x, w, b = _linear(8, N, K)
    x[5, :40] = 0.0
    x[6] *= 2.0 ** -140
    y = ops.linear(x, w, b)
    halves = N % 2 == 0 and ops.linear_swiglu_halves_supported(x, w)
    z = ops.linear_swiglu_halves(x, w) if halves else None
    for rows in range(1, 8):
        for first in (0, 8 - rows):
            part = torch.full((rows + 2, K + 4), float("nan"), device="cuda")      # (what lies beside the rows is no number)
            part[:rows, :K] = x[first:first + rows]
            assert torch.equal(ops.linear(part[:rows, :K], w, b), y[first:first + rows])
            if halves and ops.linear_swiglu_halves_supported(part[:rows, :K], w):
                assert torch.equal(ops.linear_swiglu_halves(part[:rows, :K], w), z[first:first + rows])
    x[2, K - 1] = float("nan")
    got = ops.linear(x[2:4].contiguous(), w, b)
    assert bool(torch.isnan(got[0]).all()) and torch.equal(got[1], y[3])
