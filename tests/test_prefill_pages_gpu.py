"""Prompt attention whose loads of keys and values lie in one page each (pages of 16 positions and more) against the kernel that stages them
through registers: the same bits wherever the last key falls in a block, a group of 16 keys and a page, with NaN in every slot that
holds no key and pages that a window has given back."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LENGTHS = [1, 7, 8, 9, 15, 16, 17, 31, 33, 64, 70, 127, 128, 129, 143, 161]


@pytest.mark.parametrize("ps", [8, 16, 32, 128])
@pytest.mark.parametrize("nh,nkv,d", [(4, 2, 128), (3, 1, 64)])
@pytest.mark.parametrize("past,window", [(0, 0), (115, 0), (130, 70)])
def test_the_bits_of_the_staged_kernel(ps, nh, nkv, d, past, window):
    from zedinfer_amd import ops
    g = torch.Generator().manual_seed(ps * d + past)
    totals = [past + n for n in LENGTHS]
    widths = [-(-t // ps) for t in totals]
    order = torch.randperm(sum(widths) + 3, generator=g)
    kc = torch.full((len(order), nkv, ps, d), float("nan"), dtype=torch.bfloat16)
    vc = torch.full((len(order), nkv, d, ps), float("nan"), dtype=torch.bfloat16)
    table = torch.full((len(totals), max(widths)), -1, dtype=torch.int32)
    at = 0
    for i, (t, w) in enumerate(zip(totals, widths)):
        for j in range(w):
            page, at = int(order[at]), at + 1
            if window and (j + 1) * ps <= past - window + 1:
                continue                     # no query of the portion sees this page any more: given back
            table[i, j] = page
            m = min(ps, t - j * ps)
            kc[page, :, :m] = torch.randn(nkv, m, d, generator=g).bfloat16()
            vc[page, :, :, :m] = torch.randn(nkv, d, m, generator=g).bfloat16()
    starts = [sum(LENGTHS[:i]) for i in range(len(LENGTHS))]
    q = torch.randn(sum(LENGTHS), nh * d, generator=g).bfloat16().cuda()
    kc, vc, table = kc.cuda(), vc.cuda(), table.cuda()
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731

    def attend(tile, alone=False):
        tiles = [(i, o) for i, n in enumerate(LENGTHS) for o in range(0, n, tile)]
        out = torch.full_like(q, 7.0)
        ops.attention_prefill(q, kc, vc, ints([t[0] for t in tiles]), ints([t[1] for t in tiles]), ints(starts), ints(LENGTHS),
                              ints([past] * len(LENGTHS)), table, nh, nkv, d, d ** -0.5, window, out=out, max_keys=max(totals), tile=tile,
                              alone=alone)
        return out

    got = attend(64)
    assert bool(torch.isfinite(got).all())
    before = ops.attention_prefill_variant(0)
    try:
        staged = attend(64)
    finally:
        ops.attention_prefill_variant(before)
    assert torch.equal(got, staged) and torch.equal(attend(128), got)
    # (workgroups of four wavefronts add a query's keys in another order)
    assert torch.equal(attend(64, True), attend(128, True)) and bool(((attend(64, True) - got).abs() <= 3e-2).all())
