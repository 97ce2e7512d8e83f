"""Experts' products (csrc/moe.hip): every number of steps of 64 columns around the turns through the buffers, in every size of tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [16, 32, 64, 128])
@pytest.mark.parametrize("K", [8, 64, 72, 128, 192, 256, 264, 320, 376, 384, 392, 448, 504, 512, 520, 576, 640, 704, 768, 776, 832, 896, 960, 1152, 1160, 1536, 1600])
def test_whole_numbers_come_out_exact(rows, K):
    """|sum| <= 1,600 * 9: exact in float32 in any order.  What lies behind the weights and beside the tokens is no number."""
    from zedinfer_amd import ops
    dev, E, N, top, n = "cuda", 3, 70, 2, 75
    g = torch.Generator().manual_seed(K + rows)
    x, w = (torch.randint(-3, 4, s, generator=g).bfloat16() for s in ((n, K), (E, N, K)))
    room = torch.full((n, K + 8), float("nan"), dtype=torch.bfloat16)
    room[:, :K] = x
    store = torch.full((E + 1, N, K), float("nan"), dtype=torch.bfloat16, device=dev)
    store[:E] = w.to(dev)
    idx = torch.stack([torch.zeros(n), 1 + torch.arange(n) % 2], 1).int()
    tiles = ops.moe_max_tiles(n * top, E, rows)
    plan = torch.empty(1 + 3 * tiles, dtype=torch.int32, device=dev)
    order, place = (torch.empty(n * top, dtype=torch.int32, device=dev) for _ in range(2))
    ops.moe_group(idx.to(dev), E, rows, plan, order, place)
    out = ops.moe_linear(room.to(dev)[:, :K], store[:E], plan, rows, tiles, out=torch.empty((n * top, N), device=dev), source=order, source_div=top)
    want = torch.einsum("tpnk,tk->tpn", w.double()[idx.long()], x.double()).reshape(n * top, N)
    assert torch.equal(out[place.long()].double().cpu(), want)
