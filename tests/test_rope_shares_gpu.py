"""Rotation and cache store of prompt tokens (csrc/rope_kv.hip): a tile in one workgroup and in four makes the same of it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,d,rot,ps", [(12, 2, 128, 128, 16), (5, 3, 80, 48, 8), (2, 1, 64, 0, 32)])
@pytest.mark.parametrize("scattered", [False, True])
@pytest.mark.parametrize("store", [True, False])
def test_a_tile_in_one_workgroup_and_in_four(nh, nkv, d, rot, ps, scattered, store):
    """4,107 tokens are more than two tiles a unit of 256; 4,096 and fewer are not."""
    from zedinfer_amd import ops
    n, pages = 4107, -(-4107 // ps) + 3
    g = torch.Generator(device="cuda").manual_seed(nh)
    qkv = torch.randn(n, (nh + 2 * nkv) * d, generator=g, device="cuda").bfloat16()
    slots = (torch.randperm(pages * ps, generator=torch.Generator().manual_seed(1))[:n] if scattered else torch.arange(n) + 8).to(torch.int32)
    slots[77] = -1
    slots = slots.cuda()
    table = torch.randn(n, rot // 2, 2, generator=g, device="cuda") if rot else None

    def run(step):
        x = qkv.clone()
        kc, vc = (torch.full(s, 3.0, dtype=torch.bfloat16, device="cuda") for s in ((pages, nkv, ps, d), (pages, nkv, d, ps)))
        for a in range(0, n, step):
            b = min(n, a + step)
            q, k, v = x[a:b, :nh * d], x[a:b, nh * d:(nh + nkv) * d], x[a:b, (nh + nkv) * d:]
            t = table[a:b] if rot else None
            if store:
                ops.rope_kv_store(q, k, v, t, slots[a:b], kc, vc, nh, nkv, d)
            else:
                ops.rope_kv_store(q, None, None, t, None, None, None, nh, 0, d)
        return x, kc, vc

    for one, four in zip(run(n), run(2053)):        # (2,053 and 2,054 tokens: the last tile is not whole)
        assert torch.equal(one, four)


@pytest.mark.parametrize("nh,d,rot", [(2, 64, 64), (16, 128, 64), (12, 128, 128), (33, 64, 64)])
def test_queries_alone_in_one_workgroup_and_in_four(nh, d, rot):
    """One, two, three and five pieces a thread and tile: shared never, up to a tile a unit, up to two; 8,200 tokens are more, 1,025 fewer
    than a tile a unit and 3,001 between one and two (of 256)."""
    from zedinfer_amd import ops
    n = 8200
    g = torch.Generator(device="cuda").manual_seed(nh)
    q, table = torch.randn(n, nh * d, generator=g, device="cuda").bfloat16(), torch.randn(n, rot // 2, 2, generator=g, device="cuda")

    def run(step):
        x = q.clone()
        for a in range(0, n, step):
            b = min(n, a + step)
            ops.rope_kv_store(x[a:b], None, None, table[a:b], None, None, None, nh, 0, d)
        return x

    one = run(n)
    assert torch.equal(one, run(1025)) and torch.equal(one, run(3001))
