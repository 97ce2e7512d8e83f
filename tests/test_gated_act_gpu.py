"""The gated activation four columns a thread (csrc/elementwise.hip) against the kernel of one column a thread."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,inter", [(1, 4), (3, 1028), (257, 512)])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
def test_gated_activation_four_columns_a_thread(n, inter, dtype, out_dtype):
    """The same bits as column by column (rows that are not 16-byte aligned take that kernel)."""
    from zedinfer_amd import ops
    x = torch.randn(n, 2 * inter + 8, device="cuda").to(dtype)
    odd = torch.empty(n, 2 * inter + 9, device="cuda", dtype=dtype)[:, 1:]
    odd.copy_(x)
    out = torch.full((2, n, inter + 4), 7.0, device="cuda", dtype=out_dtype)
    for act in ("silu", "gelu_tanh", "gelu_erf"):
        for i, src in enumerate((x, odd)):
            ops.gated_act(src[:, :inter], src[:, inter + 8:], act, out=out[i, :, :inter])
        assert torch.equal(out[0], out[1]) and bool((out[0, :, inter:] == 7.0).all())
