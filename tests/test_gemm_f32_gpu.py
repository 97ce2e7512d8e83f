"""The float32 product on the matrix cores (csrc/gemm_f32.hip): every kernel its dispatch can choose, at the edges of tiles,
chunks and runs of k, against a float64 product, and bit for bit the same row whatever rows ride along."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (rows, weight rows, columns): rows on both sides of every bound of the dispatch (8, 16, 32 rows; one round of 16-, 32-row and
# tiled workgroups on 256 compute units, two to three, four, six of the large tiles)
CASES = [(1, 7, 4), (8, 33, 36), (9, 16, 32), (16, 300, 260), (17, 1030, 100), (17, 5000, 68), (33, 2050, 64), (48, 130, 1540),
         (65, 2060, 1500), (130, 1536, 8960), (449, 1500, 320), (450, 2048, 1536), (1025, 2051, 72), (500, 17920, 48)]


@pytest.mark.parametrize("M,N,K", CASES)
def test_float32_product(M, N, K):
    from zedinfer_amd import ops
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N)
    x, w = (torch.randn(s, generator=g, device="cuda") for s in ((M, K), (N, K)))
    b = torch.randn(N, generator=g, device="cuda")
    got = ops.linear(x, w, b)
    ref = x.double() @ w.double().t() + b.double()
    # an output is chains of at most 16 multiply-adds for every chunk of 32 in an eighth of k (rounded up), then ten additions:
    # so many roundings, each at most 2^-24 of a partial sum, which is at most sum |x w| + |b|
    roundings = 16 * -(-(-(-K // 32)) // 8) + 10
    bound = roundings * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs())
    assert bool(((got.double() - ref).abs() <= bound).all()), float(((got.double() - ref).abs() / bound).max())
    # the same bits in other company: alone, among few, from rows that lie apart, into a slice of a wider result
    for rows in (slice(M - 1, M), slice(max(0, M - 11), M), slice(max(0, M - 40), M)):
        assert torch.equal(ops.linear(x[rows].contiguous(), w, b), got[rows])
    apart, wide = torch.full((M, K + 8), float("nan"), device="cuda"), torch.zeros((M, N + 6), device="cuda")
    apart[:, 4:K + 4] = x
    ops.linear(apart[:, 4:K + 4], w, b, out=wide[:, 3:N + 3])
    assert torch.equal(wide[:, 3:N + 3], got) and not wide[:, :3].any() and not wide[:, N + 3:].any()


def test_float32_product_keeps_infinities_and_rows_apart():
    """A row of x with an infinity or a NaN, and a weight row with one, change their own row and column and nothing else; columns
    that are no multiple of a chunk are not read past their end."""
    from zedinfer_amd import ops
    for M in (3, 12, 20, 200):
        x, w = torch.ones(M, 36, device="cuda"), torch.ones(70, 36, device="cuda")
        x[1, 35], w[5, 0], x[2, 3] = float("inf"), float("nan"), 1e-40
        y = ops.linear(x, w)
        cols = [i for i in range(70) if i != 5]
        assert bool(torch.isinf(y[1, cols]).all()) and bool(torch.isnan(y[:, 5]).all())
        rest = [i for i in range(M) if i not in (1, 2)]
        assert bool((y[rest][:, cols] == 36).all()) and bool((y[2, cols] == 35).all())


def test_float32_products_too_large_for_a_launch():
    """More rows than the entry point takes are refused, whichever kernel; more weight rows than a launch of one dimension has
    workgroups for go to the plain kernel."""
    from zedinfer_amd import ops
    x, w = torch.zeros(65535 * 64 + 1, 4, device="cuda"), torch.ones(1, 4, device="cuda")
    with pytest.raises(RuntimeError):
        ops.linear(x, w)
    x[:, 1] = torch.arange(x.shape[0], device="cuda")
    assert torch.equal(ops.linear(x[:-1], w)[:, 0], x[:-1, 1])
    many = torch.zeros((1 << 26) + 9, 4, device="cuda")
    many[:, 0] = torch.arange(many.shape[0], device="cuda") % 1021
    assert torch.equal(ops.linear(torch.full((2, 4), 3.0, device="cuda"), many)[1], 3 * many[:, 0])


# products of few columns: one round and two of 32-row workgroups, tiles of one group (K up to 128), of 64 x 64 (K up to 64)
@pytest.mark.parametrize("M,N,K", [(9000, 4, 4), (1024, 256, 32), (1025, 256, 32), (4100, 70, 20), (513, 250, 64), (1100, 250, 64),
                                   (520, 250, 68), (2070, 130, 100), (4000, 128, 128), (3000, 2060, 96), (520, 250, 132)])
def test_float32_product_of_few_columns(M, N, K):
    test_float32_product(M, N, K)


# x held in registers: every number of chunks a kernel is made for, the last group of weight rows not whole, groups for every place and more
@pytest.mark.parametrize("M,N,K", [(1, 2051, 4), (8, 3000, 512), (3, 2100, 516), (5, 2054, 1000), (8, 4100, 1500), (7, 2059, 2048), (8, 2066, 3000), (2, 2049, 4096),
                                   (9, 4105, 500), (16, 5000, 1000), (12, 4100, 1500), (13, 4098, 2048), (10, 9000, 36)])
def test_float32_product_with_x_held_in_registers(M, N, K):
    """Against float64, and bit for bit what other kernels make of the same rows among more."""
    from zedinfer_amd import ops
    assert ops.linear_f32_kernel(M, N, K) == ("held_pairs" if M <= 8 else "held_rows16") and not ops.linear_f32_kernel(M + 17, N, K).startswith("held")
    test_float32_product(M, N, K)
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N)
    x, w, b = (torch.randn(s, generator=g, device="cuda") for s in ((M + 17, K), (N, K), (N,)))
    among = ops.linear(x, w, b)
    for rows in (slice(0, M), slice(17, 17 + M)):
        assert torch.equal(ops.linear(x[rows].contiguous(), w, b), among[rows])


# tiles of 64 x 64 with more than two chunks: one, two and no chunks past the last multiple of three, runs of k that end in the chunks past
# the end and before, an odd number of weight rows and a last tile of rows that is not whole
@pytest.mark.parametrize("M,N,K", [(450, 17921, 260), (450, 17921, 516), (1025, 6203, 544), (450, 17921, 580), (450, 17921, 576), (1025, 6203, 1540),
                                   (3001, 2050, 612), (450, 17921, 900)])
def test_float32_product_in_large_tiles(M, N, K):
    from zedinfer_amd import ops
    assert ops.linear_f32_kernel(M, N, K) == "tile_64"
    test_float32_product(M, N, K)


# ... and what a short k gives to tiles of 32 x 64: five and six chunks of more than a round of halves, and six rounds of large tiles whose
# chunks are no multiple of three
@pytest.mark.parametrize("M,N,K", [(130, 6147, 132), (129, 6200, 192), (1025, 6203, 388), (450, 17921, 512), (3001, 2050, 228)])
def test_float32_product_of_a_short_k_in_small_tiles(M, N, K):
    from zedinfer_amd import ops
    assert ops.linear_f32_kernel(M, N, K) == "tile_32"
    test_float32_product(M, N, K)


# the activation in the product's end: x held in registers for up to 8 and 16 rows (every number of chunks a kernel is made for, the
# last group of weight rows not whole, groups for every place and more), each kind of tile, and what is left to two launches
@pytest.mark.parametrize("M,I,K", [(450, 8961, 260), (450, 8961, 516), (513, 8961, 576), (1025, 3102, 1540), (1, 1030, 4), (8, 1500, 512), (3, 2050, 1000), (5, 1027, 1536), (8, 1100, 2048), (7, 1029, 3000), (8, 1050, 4096),
                                   (9, 2070, 96), (16, 2053, 1024), (12, 2100, 1500), (13, 2049, 2048), (70, 1000, 60), (70, 5000, 60), (100, 3001, 100),
                                   (200, 530, 1500), (300, 2050, 260), (450, 4480, 200), (8, 64, 260), (40, 100, 260), (8, 5000, 4100)])
def test_float32_product_with_the_activation(M, I, K):
    """The bits of the product and the activation one after the other, whatever rows ride along, and nothing written beside them."""
    from zedinfer_amd import ops
    g = torch.Generator(device="cuda").manual_seed(M * 31 + I)
    x, w = (torch.randn(s, generator=g, device="cuda") for s in ((M, K), (2 * I, K)))
    two = ops.linear(x, w)
    # (the same kernel as the product with the activation takes: so against float64 too, with test_float32_product's bound)
    roundings = 16 * -(-(-(-K // 32)) // 8) + 10
    bound = roundings * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert bool(((two.double() - x.double() @ w.double().t()).abs() <= bound).all())
    ref = two[:, :I].double()
    ref = two[:, I:].double() * ref / (1 + torch.exp(-ref))
    want = ops.swiglu(two[:, :I], two[:, I:])
    assert bool(((want.double() - ref).abs() <= 1e-6 * ref.abs() + 1e-30).all())
    if not ops.linear_swiglu_halves_supported(x, w):
        assert (M, I) in ((70, 1000), (8, 64), (40, 100), (8, 5000))
        return
    wide = torch.zeros((M, I + 6), device="cuda")
    ops.linear_swiglu_halves(x, w, out=wide[:, 3:I + 3])
    assert torch.equal(wide[:, 3:I + 3], want) and not wide[:, :3].any() and not wide[:, I + 3:].any()
    apart = torch.full((M, K + 8), float("nan"), device="cuda")
    apart[:, 4:K + 4] = x
    assert torch.equal(ops.linear_swiglu_halves(apart[:, 4:K + 4], w), want)


@pytest.mark.parametrize("N,K,kernel", [(1024, 4864, "pairs"), (1025, 4864, "rows16"), (2048, 2048, "rows16"), (1536, 8960, "rows16"), (2000, 256, "rows16"),
                                        (5000, 1000, "held_rows16")])
def test_which_products_of_9_to_16_rows_go_twice_over_groups_of_8(N, K, kernel):
    """Only those whose two passes are one round of workgroups."""
    from zedinfer_amd import ops
    for M in (9, 16):
        assert ops.linear_f32_kernel(M, N, K) == kernel


@pytest.mark.parametrize("M,N,K,kernel", [(4000, 4000, 64, "tile_64"), (4000, 4000, 65, "tile_32"), (4000, 4000, 128, "tile_32"), (512, 17920, 320, "tile_32"),
                                          (1024, 9728, 384, "tile_64"), (1024, 9728, 388, "tile_32"), (1024, 9728, 512, "tile_32"), (1024, 9728, 516, "tile_64"), (256, 17920, 1536, "tile_64"),
                                          (128, 6144, 192, "tile_32"), (128, 6144, 193, "tile_96_halves"), (128, 2000, 192, "tile_32_halves"),
                                          (448, 1536, 8960, "tile_96_halves"), (1024, 1536, 8960, "tile_96_halves"),
                                          (992, 1536, 8960, "tile_96_halves"), (1024, 1536, 1536, "tile_96_halves"), (1500, 1536, 8960, "tile_96_halves"), (450, 4608, 3584, "tile_96_halves"),
                                          (2048, 3584, 18944, "tile_64"), (80, 17920, 1536, "tile_32"), (512, 2048, 1536, "tile_64_quarters"), (256, 1536, 8960, "tile_32_halves")])
def test_which_tiles_a_product_takes(M, N, K, kernel):
    """The large tiles of the float32 instruction, which work a multiple of three chunks of 32, only where k is long; of more than 1,408 columns the fastest by measurement."""
    from zedinfer_amd import ops
    assert ops.linear_f32_kernel(M, N, K) == kernel
