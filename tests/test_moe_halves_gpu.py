"""Experts' products in tiles of 128 rows whose steps are two halves (``csrc/moe.hip``): the bits of the tiles of 64 rows, whose sums have
the same order, at the shortest k it takes, columns that end within a tile, experts of no, few and many rows, both results and the activation."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,K", [(256, 192), (515, 256), (1, 320), (260, 1536), (768, 1600)])
def test_the_bits_of_the_smaller_tiles(N, K, out_dtype):
    from zedinfer_amd import ops
    E, top, n = 5, 2, 401
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x = torch.randn((n, K + 8), generator=g, device="cuda").bfloat16()[:, :K]
    store = torch.full((E + 1, N, K), float("nan"), dtype=torch.bfloat16, device="cuda")
    store[:E] = 0.1 * torch.randn((E, N, K), generator=g, device="cuda").bfloat16()
    first = torch.where(torch.arange(n) < 130, 0, torch.where(torch.arange(n) < 131, 1, 2))
    idx = torch.stack([first, torch.full((n,), 4)], 1).int().cuda()          # (expert 3 has no rows, 1 has one, 4 has all)
    got = []
    for rows in (64, 128):
        for act in ("none", "gelu_erf"):
            tiles = ops.moe_max_tiles(n * top, E, rows)
            plan = torch.empty(1 + 3 * tiles, dtype=torch.int32, device="cuda")
            order, place = (torch.empty(n * top, dtype=torch.int32, device="cuda") for _ in range(2))
            ops.moe_group(idx, E, rows, plan, order, place)
            kw = {} if act == "none" else dict(activation=act)
            out = torch.full((n * top, N + 4), 7.0, device="cuda", dtype=out_dtype)
            ops.moe_linear(x, store[:E], plan, rows, tiles, out=out[:, :N], source=order, source_div=top, **kw)
            assert bool((out[:, N:] == 7.0).all())
            got.append(out[:, :N][place.long()])
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3]) and not torch.equal(got[0], got[1])
