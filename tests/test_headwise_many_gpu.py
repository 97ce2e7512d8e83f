"""A product per head for 128 tokens and more (csrc/latent_cores.hip): edges of the tiles of 64 tokens, 128 outputs and 64 k."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [128, 191, 192, 321])
@pytest.mark.parametrize("vdim,rank", [(1, 8), (33, 64), (127, 72), (128, 128), (130, 136), (264, 200), (128, 512)])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
def test_whole_numbers_come_out_exact(n, vdim, rank, dtype, out_dtype):
    """|sum| <= 512 * 9: exact in float32 in any order; the gate: its float32 exponential and one rounding to bfloat16."""
    from zedinfer_amd import ops
    heads, dev = 3, "cuda"
    g = torch.Generator().manual_seed(n * vdim + rank)
    o = torch.randint(-3, 4, (n, heads, rank), generator=g).double()
    uv = torch.randint(-3, 4, (heads * vdim, rank), generator=g).double()
    want = torch.einsum("nhr,hvr->nhv", o, uv.view(heads, vdim, rank)).reshape(n, -1)
    args = o.to(dtype).to(dev), uv.bfloat16().to(dev), vdim
    for pad in (0, 1):        # rows from any address
        room = torch.full((n, heads * vdim + 8), 77.0, dtype=out_dtype, device=dev)
        out = ops.latent_value(*args, out=room[:, pad:pad + heads * vdim])
        assert torch.equal(out.cpu(), want.to(out_dtype)), pad
        assert (room[:, :pad] == 77).all() and (room[:, pad + heads * vdim:] == 77).all()
    gate = torch.randn((2, n, heads * vdim), generator=g)
    out = ops.latent_value(*args, out=torch.empty((n, heads * vdim), dtype=out_dtype, device=dev), gate=gate.to(dev))
    ref = want * torch.sigmoid(gate.double().sum(0))
    assert (out.double().cpu() - ref).abs().le(ref.abs() * (2.0 ** -8 if out_dtype == torch.bfloat16 else 1e-5)).all()


@pytest.mark.parametrize("n", [128, 195])
@pytest.mark.parametrize("vdim", [8, 16, 31, 32, 33, 48, 64, 65, 96, 130])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_tiles_of_32_and_64_outputs_with_either_gate(n, vdim, dtype):
    """As above, 32 outputs a tile up to that many, else 64; gates in bfloat16 and as one and five terms."""
    from zedinfer_amd import ops
    heads, rank, dev = 5, 72, "cuda"
    g = torch.Generator().manual_seed(n * vdim)
    o = torch.randint(-3, 4, (n, heads, rank), generator=g).double()
    uv = torch.randint(-3, 4, (heads * vdim, rank), generator=g).double()
    want = torch.einsum("nhr,hvr->nhv", o, uv.view(heads, vdim, rank)).reshape(n, -1)
    for gate in (torch.randn((n, heads * vdim), generator=g).bfloat16(), torch.randn((1, n, heads * vdim), generator=g),
                 torch.randn((5, n, heads * vdim), generator=g)):
        out = ops.latent_value(o.to(dtype).to(dev), uv.bfloat16().to(dev), vdim, torch.empty((n, heads * vdim), dtype=dtype, device=dev), gate=gate.to(dev))
        ref = want * torch.sigmoid(gate.double() if gate.dim() == 2 else gate.double().sum(0))
        # (the terms' sum: five roundings of at most 2^-24 of 16; the exponential and the division)
        assert (out.double().cpu() - ref).abs().le(ref.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 1e-5)).all()
