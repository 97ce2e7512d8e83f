"""A sublayer's last product as partial sums in a block's stack of terms: the parts, the stack a parallel block hands on, and the number of
sums, at both sides of 64 and 128 rows and of what a norm adds at once."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _mlp(hidden, inter, dtype=torch.bfloat16):
    from zedinfer_amd.config.forward_config import PartSpec
    from zedinfer_amd.parts.base import FEED_FORWARDS, Runtime
    g = torch.Generator().manual_seed(hidden + inter)
    w = {k: (torch.randn(s, generator=g) * 0.05).to(dtype).cuda() for k, s in
         (("gate", (inter, hidden)), ("up", (inter, hidden)), ("down", (hidden, inter)))}
    spec = PartSpec("gated_mlp", {"hidden_size": hidden, "intermediate_size": inter, "activation": "silu"}, {k: k for k in w})
    return FEED_FORWARDS.get("gated_mlp")(spec, w, Runtime("cuda", dtype))


@pytest.mark.parametrize("rows", [1, 17, 64, 65, 128, 129])
@pytest.mark.parametrize("hidden,inter", [(1536, 8960), (256, 2048), (64, 72)])
def test_a_feed_forwards_sums_are_its_result(rows, hidden, inter):
    from zedinfer_amd import ops
    part = _mlp(hidden, inter)
    x = torch.randn(rows, hidden, generator=torch.Generator().manual_seed(rows)).bfloat16().cuda()
    whole = part.forward(x, out=torch.empty(rows, hidden, device="cuda"))
    S = part.out_sums(rows)
    assert S == (1 if rows > 128 else ops.linear_splits(rows, hidden, inter))
    if S == 1:
        return
    sums = part.forward(x, out=torch.full((S, rows, hidden), float("nan"), device="cuda"))
    added = ops.reduce_sums(sums, out_dtype=torch.float32)
    if rows <= ops.FEW_ROWS:      # the launch that is saved adds these sums
        assert torch.equal(added, whole)
    else:                         # beyond, the whole result is the library's: bfloat16 products are exact, so float32 sums of `inter` terms
        assert float((added - whole).norm() / whole.norm()) <= 1e-5


def test_who_leaves_sums():
    assert _mlp(64, 2048, torch.float32).out_sums(8) == 1
    assert _mlp(256, 2048).out_sums(8) > 1 and _mlp(256, 2048).out_sums(0) == 1


def test_a_parallel_blocks_stack():
    """Terms of both sublayers one after the other, mixer first, and whole ones where there would be more than a norm adds at once."""
    from zedinfer_amd import ops
    from zedinfer_amd.parts.blocks import ParallelBlock
    from zedinfer_amd.parts.base import Runtime

    class Norm:
        def forward(self, resid):
            return resid.bfloat16()

    class Mixer:
        writes_into = True

        def __init__(self, part, sums):
            self.part, self.sums = part, sums

        def out_sums(self, rows):
            return self.sums

        def forward(self, x, batch, memory, out):
            return self.part.forward(x, out=out)

    mlp = _mlp(1536, 8960)
    mlp.reads_batch, resid = False, torch.randn(5, 1536, generator=torch.Generator().manual_seed(3)).cuda()
    S = mlp.out_sums(5)
    small = _mlp(1536, 1536)
    for part in (mlp, small):
        block = ParallelBlock({"input": Norm()}, Mixer(part, part.out_sums(5)), mlp, Runtime("cuda", torch.bfloat16))
        terms = block.forward(resid, None, None, None)
        most = part.out_sums(5) + S
        assert terms.shape[0] == (most if most <= 16 else 2)
        want = part.forward(resid.bfloat16(), out=torch.empty(5, 1536, device="cuda")) + mlp.forward(resid.bfloat16(), out=torch.empty(5, 1536, device="cuda"))
        assert float((terms.sum(0) - want).norm() / want.norm()) <= 1e-6
        k = part.out_sums(5) if most <= 16 else 1
        assert torch.equal(ops.reduce_sums(terms[k:].contiguous(), out_dtype=torch.float32), mlp.forward(resid.bfloat16(), out=torch.empty(5, 1536, device="cuda")))


@pytest.mark.parametrize("splits", [1, 2, 7, 15, 16, 17])
@pytest.mark.parametrize("rows,width,pad", [(1, 4, 0), (3, 70, 0), (5, 1000, 8), (33, 132, 2), (2, 260, 4)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sums_added_four_columns_at_a_time(splits, rows, width, pad, dtype):
    """Widths and strides that are and are not whole pieces, one sum and as many as there are kernels for and one more; with a bias and
    without: float32 additions in rising order."""
    from zedinfer_amd import ops
    g = torch.Generator().manual_seed(splits * width)
    sums, bias = torch.randn(splits, rows, width, generator=g).cuda(), torch.randn(width, generator=g).bfloat16().cuda()
    want = torch.zeros(rows, width, device="cuda")
    for s in sums:
        want = want + s
    for b in (None, bias):
        store = torch.full((rows, width + pad), 7.0, dtype=dtype, device="cuda")
        ops.reduce_sums(sums, b, out=store[:, :width])
        assert torch.equal(store[:, :width], (want + b.float() if b is not None else want).to(dtype)) and bool((store[:, width:] == 7.0).all())
