"""The experts' products on the matrix cores (csrc/moe.hip) at the sizes where the staging can go wrong: remainders of the k
step, fewer steps than buffers, columns past a workgroup's, ragged tiles, strided operands; against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile_rows", [16, 32, 64])
@pytest.mark.parametrize("N,K", [(1, 8), (60, 64), (130, 72), (257, 128), (515, 200), (64, 264), (768, 1024)])
@pytest.mark.parametrize("out_dtype,pad", [(torch.float32, 0), (torch.bfloat16, 8), (torch.float32, 1)])
def test_products_of_sorted_rows(tile_rows, N, K, out_dtype, pad):
    from zedinfer_amd import ops
    g = torch.Generator().manual_seed(N + K)
    counts, top = [0, 1, 70, 16, 129, 3], 3
    pairs, E = sum(counts), len(counts)
    x = torch.randn(pairs // top, K + 8, generator=g).to(torch.bfloat16).cuda()[:, :K]
    w = torch.randn(E, N, K, generator=g).to(torch.bfloat16).cuda()
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(pairs, generator=g)]
    tiles = ops.moe_max_tiles(pairs, E, tile_rows)
    plan = torch.zeros(1 + 3 * tiles, dtype=torch.int32, device="cuda")
    order, place = (torch.empty(pairs, dtype=torch.int32, device="cuda") for _ in range(2))
    ops.moe_group(idx.to(torch.int32).view(-1, top).cuda(), E, tile_rows, plan, order, place)
    store = torch.full((pairs, N + pad), 7.0, dtype=out_dtype, device="cuda")
    ops.moe_linear(x, w, plan, tile_rows, tiles, out=store[:, :N], source=order, source_div=top)
    o = order.cpu().long()
    xd, wd = x.cpu().double()[o // top], w.cpu().double()
    want, size = torch.empty(pairs, N, dtype=torch.float64), torch.empty(pairs, N, dtype=torch.float64)
    for e in range(E):
        at = idx[o] == e
        want[at], size[at] = xd[at] @ wd[e].t(), xd[at].abs() @ wd[e].abs().t()
    # float32 sums of K exact products: at most K roundings of the running sum; bfloat16 rounds the result once
    bound = K * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if out_dtype == torch.bfloat16 else 0)
    assert bool(((store[:, :N].cpu().double() - want).abs() <= bound).all())
    assert bool((store[:, N:] == 7.0).all())


def test_rows_of_weights_past_the_staged_lengths():
    """More columns than a tile's 31-bit offsets reach: the plain kernel, every 16 rows of a larger tile."""
    from zedinfer_amd import ops
    K, N, rows = (1 << 21) + 8, 3, 40
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randint(-1, 2, (rows, K), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randint(-1, 2, (1, N, K), generator=g, device="cuda").to(torch.bfloat16)
    plan = torch.tensor([1, 0, 0, rows], dtype=torch.int32, device="cuda")
    out = torch.empty(rows, N, dtype=torch.float32, device="cuda")
    ops.moe_linear(x, w, plan, 64, 1, out=out)
    assert torch.equal(out, x.float() @ w[0].float().t())       # whole numbers below 2^24: exact in any order


# tiles of eight wavefronts: a remainder of the k step, fewer steps than buffers, columns past a workgroup's
@pytest.mark.parametrize("N,K", [(1, 8), (257, 128), (515, 200), (64, 264), (768, 1024)])
@pytest.mark.parametrize("out_dtype,pad", [(torch.float32, 0), (torch.bfloat16, 8), (torch.float32, 1)])
def test_products_of_sorted_rows_in_tiles_of_128(N, K, out_dtype, pad):
    test_products_of_sorted_rows(128, N, K, out_dtype, pad)


@pytest.mark.parametrize("mean,experts,widths,rows", [(8, 32, (1536, 1536), 16), (16, 32, (1536, 1536), 32), (48, 32, (1536, 1536), 32), (64, 32, (1536, 1536), 128),
                                                      (128, 32, (1536, 1536), 64), (250, 32, (1536, 1536), 128), (32, 32, (2560, 3584), 64),
                                                      (64, 8, (4096, 1024), 32), (100, 8, (4096, 1024), 64), (16, 2, (12, 8), 16)])
def test_which_tiles_a_step_takes(mean, experts, widths, rows):
    from zedinfer_amd import ops
    assert ops.moe_tile_rows(torch.bfloat16, torch.bfloat16, widths, mean * experts, experts) == rows
    assert ops.moe_tile_rows(torch.float32, torch.bfloat16, widths, mean * experts, experts) == 16


@pytest.mark.parametrize("n,top,H", [(1, 1, 4), (3, 2, 260), (7, 4, 1536), (5, 5, 256), (33, 9, 132), (4, 3, 70), (2, 8, 1001)])
def test_pairs_results_combined(n, top, H):
    """Widths that are and are not whole pieces, a wavefront's columns not whole, one round of four pairs, a part of one and more."""
    from zedinfer_amd import ops
    g = torch.Generator().manual_seed(n * H)
    y, wt = torch.randn(n * top, H, generator=g), torch.rand(n, top, generator=g)
    place = torch.randperm(n * top, generator=g)
    out = torch.full((n + 1, H), 7.0, device="cuda")
    ops.moe_combine(y.cuda(), wt.cuda(), place.int().cuda(), out[:n])
    terms = wt.double()[..., None] * y.double()[place].view(n, top, H)
    # each of `top` multiply-adds rounds a sum that is at most the terms' sum of sizes
    assert bool(((out[:n].cpu().double() - terms.sum(1)).abs() <= (top + 1) * 2.0 ** -24 * terms.abs().sum(1)).all()) and bool((out[n:] == 7.0).all())
