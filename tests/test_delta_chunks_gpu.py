"""The delta rule in chunks (csrc/delta_chunks.hip) against the rule token by token in float64: entries around the bound and the
chunk's edges beside short ones, head sizes, decays down to zero, keys alike, and values that are not finite."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(lens, heads, kvh, dim, vdim, seed, alike=0.0, decay=0.2):
    n, g = sum(lens), torch.Generator().manual_seed(seed)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)  # noqa: E731
    q = unit(torch.randn(n, kvh, dim, generator=g)) * dim ** -0.5
    k = unit(torch.randn(n, kvh, dim, generator=g) + alike * torch.randn(1, kvh, dim, generator=g))
    v, beta = torch.randn(n, heads, vdim, generator=g), torch.rand(n, heads, generator=g)
    gate = torch.exp(-decay * torch.rand(n, heads, generator=g) ** 4)
    state = torch.randn(len(lens) + 1, heads * dim * vdim + 12, generator=g) * 0.2
    return q, k, v, beta, gate, state


def _run(ops, lens, q, k, v, beta, gate, state, chunked):
    n, kvh, dim = q.shape
    heads, vdim, E = v.shape[1], v.shape[2], len(lens)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    qk, bg = torch.cat([q.reshape(n, -1), k.reshape(n, -1)], 1).cuda(), torch.stack([beta, gate], 1).cuda()
    need = ops.delta_rule_workspace(n, E, heads, dim, vdim)
    assert bool(need) == (n - (E - 1) >= 64) or dim % 16 or vdim % 16
    ws = torch.full((need,), float("nan"), device="cuda") if chunked and need else None
    out, st = torch.full((n, heads * vdim), 7.0, device="cuda"), state.cuda()
    ops.delta_rule(qk, v.reshape(n, -1).cuda(), bg, st, i32([sum(lens[:e]) for e in range(E)]), i32(lens), i32(list(range(E, 0, -1))),
                   heads, kvh, dim, vdim, out=out, workspace=ws)
    return out.cpu().view(n, heads, vdim), st.cpu()


def _plain(lens, q, k, v, beta, gate, state):
    n, kvh, dim = q.shape
    heads, vdim, at = v.shape[1], v.shape[2], 0
    out, left = torch.empty(n, heads, vdim, dtype=torch.float64), state.double().clone()
    q, k = (t.double().repeat_interleave(heads // kvh, 1) for t in (q, k))
    for e, ln in enumerate(lens):
        S = left[len(lens) - e, :heads * dim * vdim].view(heads, dim, vdim)      # (a view: updated in place)
        for t in range(at, at + ln):
            S *= gate[t].double()[:, None, None]
            u = beta[t].double()[:, None] * (v[t].double() - torch.einsum("hdv,hd->hv", S, k[t]))
            S += k[t][:, :, None] * u[:, None]
            out[t] = torch.einsum("hdv,hd->hv", S, q[t])
        at += ln
    return out, left


# entries, heads, key heads, dim, vdim, keys alike, decay
CASES = [([64], 1, 1, 16, 16, 0.0, 0.2), ([63, 1, 65], 2, 1, 32, 48, 0.0, 3.0), ([127, 3, 128, 1, 129], 3, 3, 112, 16, 0.0, 0.05),
         ([200, 70], 12, 6, 128, 128, 3.0, 0.02), ([256], 9, 3, 64, 144, 0.0, 300.0), ([1] * 70 + [100], 2, 2, 48, 32, 1.0, 0.5)]


@pytest.mark.parametrize("lens,heads,kvh,dim,vdim,alike,decay", CASES)
def test_delta_rule_in_chunks(lens, heads, kvh, dim, vdim, alike, decay):
    from zedinfer_amd import ops
    x = _inputs(lens, heads, kvh, dim, vdim, seed=dim + vdim, alike=alike, decay=decay)
    want, left = _plain(lens, *x)
    got, state = _run(ops, lens, *x, chunked=True)
    alone, alone_state = _run(ops, lens, *x, chunked=False)
    # token by token in float32 shows what rounding does to these inputs; another order of the same sums may be off by a few times
    # that (T's entries are bounded by one, so nothing grows in between)
    for a, b, ref in ((got, alone, want), (state, alone_state, left)):
        own = float((b.double() - ref).norm() / ref.norm())
        assert own < 2e-6 and float((a.double() - ref).norm() / ref.norm()) <= 3 * own + 2e-7
    assert torch.equal(state[0], x[5][0]) and torch.equal(state[:, heads * dim * vdim:], x[5][:, heads * dim * vdim:])      # others' memory


def test_a_decay_of_zero_and_values_that_are_not_finite():
    """A decay of zero forgets all at once; a NaN or an infinity reaches its own and later tokens of its head and no earlier ones."""
    from zedinfer_amd import ops
    lens = [150, 90]
    q, k, v, beta, gate, state = _inputs(lens, 4, 2, 32, 32, seed=3)
    gate[70], gate[100, 1] = 0.0, 0.0
    want, left = _plain(lens, q, k, v, beta, gate, state)
    got, st = _run(ops, lens, q, k, v, beta, gate, state, True)
    assert float((got.double() - want).norm() / want.norm()) < 1e-6 and float((st.double() - left).norm() / left.norm()) < 1e-6
    k[140, 0, 3], v[60, 3, 5] = float("nan"), float("inf")       # heads 0 and 1 read key head 0
    bad, _ = _run(ops, lens, q, k, v, beta, gate, state, True)
    plain, _ = _run(ops, lens, q, k, v, beta, gate, state, False)
    assert torch.equal(torch.isnan(bad), torch.isnan(plain)) and torch.equal(torch.isinf(bad), torch.isinf(plain))
    fine = torch.isfinite(plain)
    assert bool(fine[:60].all()) and bool(fine[:140, :3].all()) and not bool(fine[140:150, :2].any()) and bool(fine[150:].all())
    assert float((bad - got)[fine & torch.isfinite(bad)].abs().max()) < 1e-5


@pytest.mark.parametrize("heads,kvh,dim,vdim", [(1, 1, 16, 4), (4, 2, 40, 64), (3, 3, 128, 68), (6, 2, 130, 128), (2, 1, 256, 100)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_step_of_single_tokens(heads, kvh, dim, vdim, dtype):
    """Single tokens with the read-out's norm and gate in one launch against float64; entries of more tokens are left alone."""
    from zedinfer_amd import ops
    lens = [1] * 7
    q, k, v, beta, gate, state = _inputs(lens, heads, kvh, dim, vdim, seed=dim)
    want, left = _plain(lens, q, k, v, beta, gate, state)
    w, z = torch.randn(vdim) + 1, torch.randn(7, heads * vdim + 8)
    want = want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-5) * w.double()
    zz = z[:, 4:-4].double().view(7, heads, vdim)
    want = (want * zz / (1 + torch.exp(-zz))).reshape(7, -1)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    qk, bg = torch.cat([q.reshape(7, -1), k.reshape(7, -1)], 1).cuda(), torch.stack([beta, gate], 1).cuda()
    st, out = state.cuda(), torch.full((7, heads * vdim), 7.0, dtype=dtype, device="cuda")
    assert ops.delta_rule_steps(dim, vdim, st) and not ops.delta_rule_steps(dim, 132, st) and not ops.delta_rule_steps(dim, 6, st)
    lens_dev = i32([1, 1, 1, 0, 1, 1, 1])
    ops.delta_rule_step(qk, v.reshape(7, -1).cuda(), bg, st, i32(list(range(7))), lens_dev, i32(list(range(7, 0, -1))), heads, kvh, dim, vdim,
                        w.cuda(), z.cuda()[:, 4:-4], 1e-5, out=out)
    rows = [0, 1, 2, 4, 5, 6]
    # dot products of dim float32 terms, one after the other in 16 chains: a few 2^-24 of their sums; bfloat16 rounds once
    tol = 2e-5 if dtype == torch.float32 else 2.0 ** -8
    assert bool(((out.cpu().double() - want).abs()[rows] <= tol * want.abs()[rows] + 2e-5).all())
    assert bool((out[3] == 7.0).all()) and torch.equal(st[4].cpu(), state[4]) and torch.equal(st[0].cpu(), state[0])
    others = [1, 2, 3, 5, 6, 7]
    assert float((st.cpu().double() - left)[others].abs().max()) < 5e-6


@pytest.mark.parametrize("heads,kvh,dim,vdim", [(2, 1, 4, 6), (4, 2, 64, 20), (3, 3, 128, 128), (2, 1, 256, 258), (2, 2, 8, 1024)])
@pytest.mark.parametrize("lens", [[1], [3, 1, 2], [1] * 5 + [1018, 4, 7], [2050]])
def test_preparing_four_channels_a_thread(heads, kvh, dim, vdim, lens):
    """Convolution over the kept tail, SiLU and unit vectors against float64, with runs of tokens that cross entries; few
    tokens and enough for four a thread."""
    from zedinfer_amd import ops
    g = torch.Generator().manual_seed(dim + len(lens))
    n, E, C = sum(lens), len(lens), 2 * kvh * dim + heads * vdim
    width, off = C + heads * vdim + 2 * heads, heads * dim * vdim
    proj = torch.randn(n, width + (-width) % 4, generator=g)
    conv, a_log, dt = torch.randn(C, 4, generator=g), torch.randn(heads, generator=g), torch.randn(heads, generator=g)
    state = torch.randn(E + 1, ops.delta_state_floats(heads, dim, vdim, kvh, 4), generator=g)
    starts = [sum(lens[:e]) for e in range(E)]
    slots = list(range(E, 0, -1))
    x = torch.empty(n, C, dtype=torch.float64)
    for s, length, slot in zip(starts, lens, slots):
        rows = torch.cat([state[slot, off:off + 3 * C].view(3, C), proj[s:s + length, :C]]).double()
        y = sum(rows[j:j + length] * conv[:, j].double() for j in range(4))
        x[s:s + length] = y / (1 + torch.exp(-y))
    unit = x[:, :2 * kvh * dim].view(n, 2, kvh, dim)
    unit = unit / torch.sqrt((unit * unit).sum(-1, keepdim=True) + 1e-6)
    unit[:, 0] *= dim ** -0.5
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")  # noqa: E731
    qk, v, bg = (torch.full(s, 7.0, device="cuda") for s in ((n, 2 * kvh * dim), (n, heads * vdim), (n, 2, heads)))
    seq = i32([e for e, length in enumerate(lens) for _ in range(length)])
    ops.delta_prepare(proj.cuda()[:, :width], conv.cuda(), a_log.cuda(), dt.cuda(), state.cuda(), seq, i32(starts), i32(slots), heads, kvh,
                      dim, vdim, 4, qk, v, bg)
    # four products and their sum, an exponential and a quotient: some ten roundings of values of a few units; near-zero heads lose more
    assert float((v.cpu().double() - x[:, 2 * kvh * dim:]).abs().max()) < 1e-5
    assert float((qk.cpu().double().view_as(unit) - unit).abs().max()) < 1e-4
    b, a = proj[:, width - 2 * heads:width - heads].double(), proj[:, width - heads:width].double()
    assert float((bg[:, 0].cpu().double() - torch.sigmoid(b)).abs().max()) < 1e-6
    decay = torch.exp(-torch.exp(a_log.double()) * torch.nn.functional.softplus(a + dt.double()))
    assert float((bg[:, 1].cpu().double() - decay).abs().max()) < 1e-5


@pytest.mark.parametrize("heads,kvh,dim,vdim,lens", [(240, 4, 128, 128, [70, 1, 300, 64, 500, 3]), (600, 300, 128, 128, [200, 129]), (64, 2, 64, 16, [6000])])
def test_chunks_in_rounds(heads, kvh, dim, vdim, lens):
    """Heads and tokens whose chunks are more than one round's workspace: the rule token by token, and a value that is not finite in
    a later round or an earlier one."""
    from zedinfer_amd import ops
    x = _inputs(lens, heads, kvh, dim, vdim, seed=heads)
    n, E = sum(lens), len(lens)
    need = ops.delta_rule_workspace(n, E, heads, dim, vdim)
    cell = 64 * (3 * dim + vdim + 65)
    assert 0 < need <= (256 << 18) + heads * (n // 64 + E) and need < heads * cell * (n // 64)
    alone, alone_state = _run(ops, lens, *x, chunked=False)
    got, state = _run(ops, lens, *x, chunked=True)
    for a, b in ((got, alone), (state, alone_state)):       # (each within 2e-6 of float64, see above)
        assert float((a.double() - b.double()).norm() / b.double().norm()) < 4e-6
    for bad in (n - 5, 40):                                 # of the last and of the first long entry
        v = x[2].clone()
        v[bad, 3, 1] = float("inf")
        args = (*x[:2], v, *x[3:])
        odd, odd_state = _run(ops, lens, *args, chunked=True)
        plain, plain_state = _run(ops, lens, *args, chunked=False)
        assert torch.equal(torch.isfinite(odd), torch.isfinite(plain)) and torch.equal(torch.isfinite(odd_state), torch.isfinite(plain_state))
        at = torch.isfinite(plain)
        assert not bool(at.all()) and torch.equal(odd[:bad // 64 * 64 if E == 1 else 0], got[:bad // 64 * 64 if E == 1 else 0])
        assert float((odd - plain)[at].abs().max()) < 2e-5 * float(plain[at].abs().max())


def test_more_heads_than_a_round_holds():
    from zedinfer_amd import ops
    assert ops.delta_rule_workspace(200, 1, 1817, 128, 128) > 0 and ops.delta_rule_workspace(200, 1, 1818, 128, 128) == 0


def test_finite_values_whose_sums_are_not():
    """Two tokens whose values are near the largest float32 make an infinity between them: it reaches them and later tokens of their
    head and no earlier one of their chunk."""
    from zedinfer_amd import ops
    lens = [150]
    q, k, v, beta, gate, state = _inputs(lens, 2, 1, 32, 32, seed=5)
    k[101] = k[100]
    beta[100:102], gate[100:102] = 0.99, 1.0
    v[100, 1, 4], v[101, 1, 4] = 3e38, -3e38
    got, _ = _run(ops, lens, q, k, v, beta, gate, state, True)
    plain, _ = _run(ops, lens, q, k, v, beta, gate, state, False)
    assert bool(torch.isfinite(plain[:100]).all()) and not bool(torch.isfinite(plain[101:, 1, 4]).any())
    assert torch.equal(torch.isfinite(got), torch.isfinite(plain))
    at = torch.isfinite(plain) & (plain.abs() < 1e30)
    assert float((got - plain)[at].abs().max()) < 1e-5
    gate[60] = 1.5                                              # no decay: the rule token by token
    got, _ = _run(ops, lens, q, k, v.clamp(-3, 3), beta, gate, state, True)
    plain, _ = _run(ops, lens, q, k, v.clamp(-3, 3), beta, gate, state, False)
    assert torch.equal(got, plain)


def test_when_chunks_pay():
    """A long entry in chunks, many of 64 tokens with few heads token by token, steps without a long entry without the launches."""
    import numpy as np
    from zedinfer_amd import ops
    pay = lambda lens, *sizes: ops.delta_rule_chunks_pay(np.array(lens, dtype=np.int32), *sizes)  # noqa: E731
    for sizes in ((12, 128, 128), (2, 128, 128), (32, 128, 128), (6, 64, 64), (16, 32, 64)):
        assert pay([500], *sizes) and pay([1] * 31 + [500], *sizes) and pay([300] * 8, *sizes)
        assert not pay([63], *sizes) and not pay([2] * 64, *sizes) and not pay([1] * 200, *sizes)
    for sizes in ((2, 128, 128), (6, 64, 64), (16, 32, 64)):
        assert not pay([64] * 32, *sizes) and not pay([64] * 128, *sizes)
    assert pay([64] * 32, 12, 128, 128) and pay([100] * 20, 32, 128, 128) and not pay([64], 16, 32, 64)
    assert not pay([2000], 4, 256, 256) and not pay([2000], 6, 48, 40)       # (no multiples of 16, more than 128)
