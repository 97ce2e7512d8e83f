"""Float32 attention on the matrix cores (csrc/attention_f32.hip) against float64 softmax attention: head sizes, groups, pages,
windows, portions beside single tokens, sinks; the two ways a token can come give the same bits, in any company; what lies in
masked places does not matter."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def paged(lens, nkv, d, ps, g):
    """Keys and values of sequences in pages taken in a random order, with NaN wherever no position lies."""
    pages = [-(-n // ps) for n in lens]
    order = torch.randperm(sum(pages) + 2, generator=g)
    kc = torch.full((len(order), nkv, ps, d), float("nan"))
    vc = torch.full((len(order), nkv, d, ps), float("nan"))
    table = torch.full((len(lens), max(pages) + 1), -1, dtype=torch.int32)
    ks, vs, at = [], [], 0
    for i, n in enumerate(lens):
        k, v = torch.randn(n, nkv, d, generator=g), torch.randn(n, nkv, d, generator=g)
        for j in range(pages[i]):
            p = int(order[at])
            at += 1
            table[i, j] = p
            part = slice(j * ps, min((j + 1) * ps, n))
            m = part.stop - part.start
            kc[p, :, :m] = k[part].transpose(0, 1)
            vc[p, :, :, :m] = v[part].permute(1, 2, 0)
        ks.append(k.double())
        vs.append(v.double())
    return kc.cuda(), vc.cuda(), table.cuda(), ks, vs


def reference(q, ks, vs, seqs, poss, nh, nkv, d, scale, window, sinks):
    out = torch.empty(q.shape[0], nh, d, dtype=torch.float64)
    for t, (s, p) in enumerate(zip(seqs, poss)):
        lo = max(0, p - window + 1) if window else 0
        for h in range(nh):
            kv = h // (nh // nkv)
            sc = ks[s][lo:p + 1, kv] @ q[t, h * d:(h + 1) * d].double() * scale
            if sinks is not None:
                sc = torch.cat([sc, sinks[h:h + 1].double()])
            w = torch.softmax(sc, 0)
            out[t, h] = w[:p + 1 - lo] @ vs[s][lo:p + 1, kv]
    return out.view(q.shape[0], nh * d)


# heads, key/value heads, head size, page, tokens before and brought by each sequence, window
CASES = [(12, 2, 128, 16, [(0, 1)], 0), (4, 4, 16, 16, [(0, 17), (15, 1), (16, 2)], 0), (6, 2, 80, 32, [(130, 1), (0, 33), (200, 40)], 0),
         (16, 1, 64, 48, [(300, 5), (31, 1), (0, 16)], 40), (20, 1, 32, 16, [(127, 1), (128, 1), (129, 20)], 1), (2, 1, 112, 16, [(0, 300)], 100)]


@pytest.mark.parametrize("nh,nkv,d,ps,entries,window", CASES)
@pytest.mark.parametrize("with_sinks", [False, True])
def test_float32_attention(nh, nkv, d, ps, entries, window, with_sinks):
    from zedinfer_amd import ops
    g = torch.Generator().manual_seed(nh * d + len(entries))
    kc, vc, table, ks, vs = paged([a + b for a, b in entries], nkv, d, ps, g)
    seqs = [s for s, (a, b) in enumerate(entries) for _ in range(b)]
    poss = [a + j for a, b in entries for j in range(b)]
    n = len(seqs)
    q = torch.randn(n, nh * d, generator=g)
    sinks = torch.randn(nh, generator=g) if with_sinks else None
    scale = 1.0 / math.sqrt(d)
    args = (kc, vc, torch.tensor(seqs, dtype=torch.int32).cuda(), torch.tensor(poss, dtype=torch.int32).cuda(), table, nh, nkv, d, scale, window)
    kw = dict(sinks=sinks.cuda()) if with_sinks else {}
    got = ops.attention(q.cuda(), *args, **kw)
    ref = reference(q, ks, vs, seqs, poss, nh, nkv, d, scale, window, sinks)
    # the scores, about 5 at most here, carry d roundings of 2^-24 of a sum of |q k| (about 0.64 d, scaled); a probability is off
    # by as much, relatively, and an output of size up to about 4 by twice that; 4e-6 for 128 dims and 2e-6 for the rest
    assert float((got.cpu().double() - ref).abs().max()) <= 2e-5
    # a token a workgroup, and any subset of the tokens: the same bits
    assert torch.equal(ops.attention(q.cuda(), *args, decoded=True, **kw), got)
    some = torch.arange(n - 1, -1, -3, dtype=torch.int32).flip(0).cuda()
    part = torch.zeros_like(got)
    ops.attention(q.cuda(), *args, out=part, tok_index=some, **kw)
    assert torch.equal(part[some.long()], got[some.long()]) and int((part != 0).any(1).sum()) == some.numel()
    # a query row among wider ones
    wide = torch.zeros(n, nh * d + 8, device="cuda")
    wide[:, 4:-4] = q.cuda()
    assert torch.equal(ops.attention(wide[:, 4:-4], *args, **kw), got)


def test_float32_attention_sees_no_later_token():
    """A later token's infinities and NaN stay out of an earlier token's result, also in the block and the workgroup they share."""
    from zedinfer_amd import ops
    nh, nkv, d, ps, n = 6, 2, 64, 16, 45
    g = torch.Generator().manual_seed(3)
    kc, vc, table, ks, vs = paged([n, n], nkv, d, ps, g)
    q = torch.randn(2 * n, nh * d, generator=g).cuda()
    seq = torch.arange(2, dtype=torch.int32).repeat_interleave(n).cuda()
    pos = torch.arange(n, dtype=torch.int32).repeat(2).cuda()
    clean = ops.attention(q, kc, vc, seq, pos, table, nh, nkv, d, 0.1)
    assert bool(torch.isfinite(clean).all())
    at, page = 37, int(table[0, 37 // ps])
    vc[page, 1, 3, at % ps], kc[page, 0, at % ps, 5] = float("nan"), float("inf")
    got = ops.attention(q, kc, vc, seq, pos, table, nh, nkv, d, 0.1)
    assert torch.allclose(got[:at], clean[:at], rtol=1e-5, atol=1e-6) and torch.equal(got[n:], clean[n:])
    assert bool(torch.isnan(got[at:n].view(-1, nh, d)[:, 3:, 3]).all())


@pytest.mark.parametrize("n,window", [(17, 0), (33, 0), (150, 0), (40, 3)])
@pytest.mark.parametrize("with_sinks", [False, True])
def test_a_seen_key_of_minus_infinite_score_has_no_weight(n, window, with_sinks):
    """A key with an infinite component against the query's sign scores minus infinity: weight zero, also where it is all that a
    wavefront sees; a column that sees nothing else is NaN (without a sink), and so is one that sees a NaN."""
    from zedinfer_amd import ops
    nh, nkv, d, ps = 4, 2, 32, 16
    g = torch.Generator().manual_seed(n)
    kc, vc, table, ks, vs = paged([n], nkv, d, ps, g)
    q = torch.rand(n, nh * d, generator=g) + 0.1                # every query positive
    sinks = torch.randn(nh, generator=g) if with_sinks else None
    at = [n - 1, 0] + [j for j in range(n) if 16 <= j < 32]     # the 17th token alone in its block, then all of the block; the first
    for j in at:
        kc[table[0, j // ps].long(), 0, j % ps, 5] = float("-inf")
        ks[0][j, 0, 5] = float("-inf")
    seq, pos = torch.zeros(n, dtype=torch.int32), torch.arange(n, dtype=torch.int32)
    args = (kc, vc, seq.cuda(), pos.cuda(), table, nh, nkv, d, 0.2, window)
    kw = dict(sinks=sinks.cuda()) if with_sinks else {}
    ref = reference(q, ks, vs, seq.tolist(), pos.tolist(), nh, nkv, d, 0.2, window, sinks)
    assert with_sinks or bool(torch.isnan(ref[0, :d]).all())
    for decoded in (False, True):
        got = ops.attention(q.cuda(), *args, decoded=decoded, **kw).cpu().double()
        assert torch.equal(torch.isnan(got), torch.isnan(ref))
        assert float((got - ref)[~torch.isnan(ref)].abs().max()) <= 2e-5      # (as in test_float32_attention)
    kc[table[0, (n - 1) // ps].long(), 1, (n - 1) % ps, 0] = float("nan")
    got = ops.attention(q.cuda(), *args, **kw)
    assert bool(torch.isnan(got[n - 1, 2 * d:]).all()) and not bool(torch.isnan(got[:n - 1, 2 * d:]).any())


@pytest.mark.parametrize("d", [16, 80, 128])
def test_what_lies_in_cells_that_are_not_seen_changes_no_bit(d):
    """Cells past a sequence's end hold NaN, or what a sequence left that had the page before: the same bits as with zeros there;
    and the same for a token before one whose values are not finite, in its block and workgroup."""
    from zedinfer_amd import ops
    nh, nkv, ps, lens = 4, 2, 16, [37, 5, 70]
    g = torch.Generator().manual_seed(d)
    kc, vc, table, ks, vs = paged(lens, nkv, d, ps, g)
    q = torch.randn(sum(lens), nh * d, generator=g).cuda()
    seq = torch.repeat_interleave(torch.arange(3), torch.tensor(lens)).to(torch.int32).cuda()
    pos = torch.cat([torch.arange(n) for n in lens]).to(torch.int32).cuda()
    run = lambda k, v, decoded=False: ops.attention(q, k, v, seq, pos, table, nh, nkv, d, 0.1, decoded=decoded)  # noqa: E731
    want = run(kc.nan_to_num(0.0), vc.nan_to_num(0.0))
    assert bool(torch.isfinite(want).all())
    for k, v in ((kc, vc), (kc.nan_to_num(3.0), vc.nan_to_num(-5.0))):
        assert torch.equal(run(k, v), want) and torch.equal(run(k, v, True), want)
    vc[int(table[0, 2]), 1, 3, 35 % ps], vc[int(table[0, 2]), 1, 4, 36 % ps] = float("nan"), float("-inf")
    got = run(kc, vc)
    assert torch.equal(got[:35], want[:35]) and torch.equal(got[37:], want[37:])
    bad = got[35:37].view(2, nh, d)[:, 2:]
    assert bool(torch.isnan(bad[:, :, 3]).all()) and bool(torch.isinf(bad[1, :, 4]).all())
    rest = [i for i in range(d) if i not in (3, 4)]
    assert torch.equal(bad[:, :, rest], want[35:37].view(2, nh, d)[:, 2:][:, :, rest])


@pytest.mark.parametrize("nh,nkv,d", [(40, 1, 32), (34, 2, 48), (17, 1, 128)])
def test_groups_of_more_than_16_heads(nh, nkv, d):
    """Decoded tokens of such a group are several workgroups, each of up to 16 of its heads: the same bits as in tiles of tokens."""
    from zedinfer_amd import ops
    g = torch.Generator().manual_seed(nh)
    entries = [(30, 1), (0, 1), (64, 3), (5, 1), (15, 20)]
    kc, vc, table, ks, vs = paged([a + b for a, b in entries], nkv, d, 16, g)
    seqs = [s for s, (a, b) in enumerate(entries) for _ in range(b)]
    poss = [a + j for a, b in entries for j in range(b)]
    q = torch.randn(len(seqs), nh * d, generator=g)
    args = (kc, vc, torch.tensor(seqs, dtype=torch.int32).cuda(), torch.tensor(poss, dtype=torch.int32).cuda(), table, nh, nkv, d, 0.2)
    got = ops.attention(q.cuda(), *args, decoded=True)
    assert float((got.cpu().double() - reference(q, ks, vs, seqs, poss, nh, nkv, d, 0.2, 0, None)).abs().max()) <= 2e-5
    every = torch.arange(len(seqs), dtype=torch.int32).cuda()
    assert torch.equal(ops.attention(q.cuda(), *args, tok_index=every), got)


def test_which_tokens_are_taken_one_by_one():
    """Tokens of 16 and more a sequence in tiles, single tokens one by one, in between as measured."""
    from zedinfer_amd import ops
    for nh, nkv in ((12, 2), (16, 16), (40, 1), (1, 1)):
        for E in (1, 8, 64):
            assert ops.attention_f32_by_heads(E, E, nh, nkv) and not ops.attention_f32_by_heads(16 * E, E, nh, nkv)
    assert ops.attention_f32_by_heads(100, 20, 12, 2) and ops.attention_f32_by_heads(192, 64, 12, 2)
    assert ops.attention_f32_by_heads(128, 64, 16, 16) and not ops.attention_f32_by_heads(256, 64, 16, 16)


@pytest.mark.parametrize("nh,nkv,d,n", [(12, 2, 128, 32), (12, 2, 128, 33), (8, 8, 64, 8), (8, 8, 64, 9), (4, 4, 64, 65), (6, 2, 112, 3)])
def test_tokens_one_by_one_give_the_bits_of_tiles(nh, nkv, d, n):
    """A token by heads, its dims shared by four workgroups (few workgroups, head sizes 64 and 128) or not, and in a tile of 16 tokens."""
    from zedinfer_amd import ops
    g = torch.Generator().manual_seed(n + d)
    lens = [1 + 37 * i % 300 for i in range(n)]
    kc, vc, table, _, _ = paged(lens, nkv, d, 16, g)
    q = torch.randn(n, nh * d, generator=g).cuda()
    seqs, poss = torch.arange(n, dtype=torch.int32).cuda(), torch.tensor([m - 1 for m in lens], dtype=torch.int32).cuda()
    index = torch.arange(n, dtype=torch.int32).cuda()
    args = (q, kc, vc, seqs, poss, table, nh, nkv, d, d ** -0.5)
    one = ops.attention(*args, tok_index=index, decoded=True)
    assert torch.equal(one, ops.attention(*args, tok_index=index, decoded=False)) and bool(torch.isfinite(one).all())


@pytest.mark.parametrize("nh,nkv,d,ps", [(12, 2, 128, 16), (4, 4, 16, 32), (3, 1, 24, 16), (6, 2, 40, 8)])
@pytest.mark.parametrize("decoded", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_token_that_sees_no_key_has_zeros(nh, nkv, d, ps, decoded, dtype):
    """What stands behind a step's requests to fill it up: a sequence that holds no page, in the kernel of the matrix cores and in the plain one
    (head sizes of 24 and 40, bfloat16).  The tokens beside it keep their bits."""
    from zedinfer_amd import ops
    g = torch.Generator().manual_seed(nh * d)
    kc, vc, table, _, _ = paged([40, 7], nkv, d, ps, g)
    kc, vc = kc.to(dtype), vc.to(dtype)
    table = torch.cat([table, torch.full_like(table[:1], -1)])
    q = torch.randn(5, nh * d, generator=g).to(dtype).cuda()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    seq, pos = i32([0, 1, 2, 0, 2]), i32([39, 6, 0, 21, 0])
    got = ops.attention(q, kc, vc, seq, pos, table, nh, nkv, d, d ** -0.5, decoded=decoded)
    assert bool((got[[2, 4]] == 0).all()) and bool(torch.isfinite(got).all())
    real = [0, 1, 3]
    assert torch.equal(got[real], ops.attention(q[real].contiguous(), kc, vc, seq[real].contiguous(), pos[real].contiguous(), table, nh, nkv, d, d ** -0.5, decoded=decoded))


def test_a_latent_token_that_sees_no_key_has_zeros():
    from zedinfer_amd import ops
    g = torch.Generator(device="cuda").manual_seed(5)
    rank, rot, heads, ps = 40, 8, 3, 16
    c, kr = (torch.randn(3, ps, n, generator=g, device="cuda") for n in (rank, rot))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    qa = torch.randn(3, heads, rank + rot, generator=g, device="cuda")
    out = ops.latent_attention(qa, c, kr, i32([0, 1, 0]), i32([20, 0, 3]), i32([[2, 0], [-1, -1]]), 0.2, 0, torch.empty(3, heads, rank, device="cuda"))
    assert bool((out[1] == 0).all()) and bool(torch.isfinite(out).all()) and bool((out[[0, 2]] != 0).any())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_pooled_token_that_sees_no_key_has_zeros(dtype):
    """... and one whose every score is minus infinity has no number, as a softmax over them has none."""
    from zedinfer_amd import ops
    g = torch.Generator(device="cuda").manual_seed(6)
    nh, nkv, d, ps = 4, 2, 32, 16
    kc, vc = (torch.randn(3, ps, nkv, d, generator=g, device="cuda").to(dtype) for _ in range(2))
    q = torch.randn(3, nh * d, generator=g, device="cuda").to(dtype)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    run = lambda: ops.pooled_attention(q, kc, vc, None, None, i32([0, 1, 0]), i32([20, 0, 3]), i32([[2, 0], [-1, -1]]), None, nh, nkv, d, d, 0, 0,  # noqa: E731
                                       d ** -0.5, torch.empty_like(q)).clone()
    out = run()
    assert bool((out[1] == 0).all()) and bool(torch.isfinite(out).all()) and bool((out[[0, 2]] != 0).any())
    kc[2, :4], q[2] = float("-inf"), q[2].abs() + 1
    assert bool(torch.isnan(run()[2]).all())
