"""Latent attention on the matrix cores (csrc/latent_cores.hip): ranks at and beside whole groups of 16 tiles of 16 dims, one block of keys and more."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rank,rot", [(8, 8), (120, 64), (136, 64), (256, 64), (264, 24), (504, 64), (512, 64), (320, 0)])
@pytest.mark.parametrize("past,count", [(0, 33), (31, 1), (70, 300)])
def test_against_64_bits(rank, rot, past, count):
    """Probabilities and results are rounded to bfloat16: 2 * 2^-9 of the largest value a result is a mean of."""
    from zedinfer_amd import ops
    dev, heads, ps, window, keys = "cuda", 16, 16, 64, past + count
    if not ops.latent_attention_cores_supported(torch.bfloat16, rank, rot):
        pytest.skip("sizes that the kernel does not take")
    g = torch.Generator().manual_seed(rank + count)
    qa, k = (torch.randn(s, generator=g).bfloat16() for s in ((count, heads, rank + rot), (keys, rank + rot)))
    pages = -(-keys // ps)
    order = torch.randperm(pages + 2, generator=g)[:pages]
    pool = torch.full((pages + 2, ps, rank + rot), float("nan"), dtype=torch.bfloat16)
    pool[order] = torch.cat([k, torch.full((pages * ps - keys, rank + rot), float("nan"))]).bfloat16().view(pages, ps, -1)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    scale = (rank + rot) ** -0.5
    s = torch.einsum("nhd,kd->nhk", qa.double(), k.double()) * scale
    at, pos = torch.arange(keys), past + torch.arange(count)[:, None, None]
    want = s.masked_fill((at > pos) | (at <= pos - window), float("-inf")).softmax(-1) @ k[:, :rank].double()
    for units in (1, 256):       # 64 rows a workgroup, and 16 with the keys cut into chunks
        waves, chunk, chunks = ops.latent_attention_cores_plan(count, 1, heads, window, units, keys)
        ws = torch.empty(max(1, ops.latent_attention_cores_workspace(count, heads, rank, chunks)), device=dev)
        out = ops.latent_attention_cores(qa.to(dev), pool[..., :rank].contiguous().to(dev), pool[..., rank:].contiguous().to(dev), i32([0]),
                                         i32([count]), i32([past]), order.int()[None].to(dev), scale, window,
                                         torch.empty((count, heads, rank), dtype=torch.bfloat16, device=dev), waves, chunk, chunks, ws)
        assert (out.double().cpu() - want).abs().max() <= 2.0 ** -8 * k.double().abs().max(), (waves, chunks)
