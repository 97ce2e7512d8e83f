"""The workspace that a runtime keeps for float32 products of many rows: on the CPU, its size given instead of asked for."""
import torch

from zedinfer_amd import ops
from zedinfer_amd.parts.base import Runtime


def test_one_workspace_for_all_products_which_a_check_of_replays_sees(monkeypatch):
    """Products follow each other on one stream and share one allocation; the check that a replay writes all it reads makes every
    workspace of floating-point values NaN, and what holds parts and sums is one."""
    rt = Runtime("cpu", torch.float32)
    x, w = torch.zeros(450, 1536), torch.zeros(2048, 1536)
    need = 6144 * 29 * 24
    monkeypatch.setattr(ops, "linear_many_workspace", lambda x, w, gated=False: need * (2 if gated else 1))
    a, b = rt.product_workspace(x, w, gated=True), rt.product_workspace(x, w)
    assert a.numel() * a.element_size() == 2 * need and b.numel() * b.element_size() == need
    assert a.data_ptr() == b.data_ptr() and len(rt._buffers) == 1
    a.zero_()
    rt.poison()
    assert bool(a.isnan().all())
    monkeypatch.setattr(ops, "linear_many_workspace", lambda x, w, gated=False: 0)
    assert rt.product_workspace(x, w) is None
