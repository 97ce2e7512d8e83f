"""Products of many rows in tiles (``csrc/gemm_tiles.hip``) at the edges of every tile, against float64 products of the same bfloat16
operands.  Sums are float32, of K products each of which is exact: their error is below K 2^-24 of the sum of the products'
magnitudes (K a few hundred to thousands, errors of both signs: a fiftieth of that bound is allowed here), and bfloat16 results are
rounded once, by at most 2^-8 of their size (eight bits: half of 2^-7 of the power of two below)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16, F32, SWIGLU, GATED = 0, 1, 2, 3
# rows and weight rows of the tiles, in the kernel's order
TILES = [(64, 64), (128, 64), (128, 96), (128, 128), (128, 192), (192, 160), (192, 224), (128, 256), (192, 192), (256, 256)]


def rnd(*shape, seed=0, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).bfloat16().cuda()


def tiles(epi, x, w, N, bias=None, out=None, up_at=0, act=0, tile=-1):
    from zedinfer_amd.ops import _lib
    from zedinfer_amd.ops.functional import _p, _stream
    M, K = x.shape
    if out is None:
        out = torch.full((M, N), float("nan"), dtype=torch.float32 if epi == F32 else torch.bfloat16, device="cuda")
    _lib.call("zi_gemm_tiles", _p(out), epi, _p(x), _p(w), _p(bias), M, N, K, x.stride(0), w.stride(0),
              out.stride(0), up_at, act, tile, _stream())
    return out


def close(got, x, w, epi, bias=None, act=None, up=None):
    """``act``: what is made of gate and up; ``up``: the up rows."""
    X = x.double()
    ref, size = X @ w.double().t(), X.abs() @ w.double().abs().t()
    bound = size * (x.shape[1] * 2.0 ** -24 / 50) + 2.0 ** -23 * ref.abs()
    if bias is not None:
        ref = ref + bias.double()
        bound = bound + 2.0 ** -23 * ref.abs()
    if act is not None:
        u = X @ up.double().t()
        bound = 1.2 * bound * u.abs() + ref.abs() * (X.abs() @ up.double().abs().t()) * (x.shape[1] * 2.0 ** -24 / 50)      # (slopes of the activations: up to 1.13)
        ref = act(ref) * u
        bound = bound + 2.0 ** -20 * ref.abs()
    if epi != F32:
        bound = bound + 2.0 ** -8 * (ref.abs() + bound)
    assert not got.isnan().any()
    assert bool(((got.double() - ref).abs() <= bound + 1e-30).all()), float(((got.double() - ref).abs() / (bound + 1e-30)).max())


def gelu_tanh(z):
    return torch.nn.functional.gelu(z, approximate="tanh")


def test_the_kernels_tiles():
    from zedinfer_amd import ops
    assert ops.load().zi_gemm_tiles_count() == len(TILES)


@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("rows,cols,K", [(0, 0, 320), (1, 8, 384), (-1, -8, 704), (17, 24, 640)])
def test_every_tile_at_its_edges(tile, rows, cols, K):
    """One tile and a little more or less, and several of them, with and without a bias, into rows of a wider buffer."""
    bm, bn = TILES[tile]
    for many in (1, 3):
        M, N = many * bm + rows, max(8, many * bn + cols)
        x, w, bias = rnd(M, K, seed=tile), rnd(N, K, seed=tile + 50, scale=0.2), rnd(N, seed=tile + 90)
        close(tiles(BF16, x, w, N, bias, tile=tile), x, w, BF16, bias)
        close(tiles(F32, x, w, N, tile=tile), x, w, F32)
        wide = torch.zeros(M, N + 16, dtype=torch.bfloat16, device="cuda")
        tiles(BF16, x, w, N, out=wide[:, 8:N + 8], tile=tile)
        close(wide[:, 8:N + 8], x, w, BF16)
        assert float(wide[:, :8].abs().max()) == 0 and float(wide[:, N + 8:].abs().max()) == 0
        apart = rnd(M, K + 24, seed=tile)[:, 8:K + 8]
        close(tiles(BF16, apart, w, N, tile=tile), apart, w, BF16)


@pytest.mark.parametrize("tile", [t for t in range(len(TILES)) if TILES[t][1] // 32 % 2 == 0])
@pytest.mark.parametrize("rows,cols,K", [(0, 0, 320), (1, 8, 384), (-1, -8, 704)])
def test_gate_and_up(tile, rows, cols, K):
    """Gate and up rows in turn and one block after the other, up to rows that no column of the result belongs to."""
    bm, bn = TILES[tile]
    M, N = bm + rows, max(8, bn + cols)
    x, g, u = rnd(M, K, seed=tile), rnd(N, K, seed=tile + 50, scale=0.2), rnd(N, K, seed=tile + 90, scale=0.2)
    turns = torch.stack([g.view(N // 8, 8, K), u.view(N // 8, 8, K)], dim=1).reshape(2 * N, K).contiguous()
    close(tiles(SWIGLU, x, turns, N, tile=tile), x, g, SWIGLU, act=torch.nn.functional.silu, up=u)
    for act, fn in enumerate((torch.nn.functional.silu, gelu_tanh, torch.nn.functional.gelu)):
        up_at = N + 8 * act
        halves = torch.full((up_at + N, K), float("nan"), dtype=torch.bfloat16, device="cuda")
        halves[:N], halves[up_at:] = g, u
        close(tiles(GATED, x, halves, N, up_at=up_at, act=act, tile=tile), x, g, GATED, act=fn, up=u)


def test_large_and_infinite_gates():
    """up * silu(gate) where the exponential overflows or vanishes, and of what is no number, as the activation's own kernel has it."""
    from zedinfer_amd import ops
    K, N = 320, 64
    gates = torch.tensor([0.0, -0.0, 1e-30, -1e-30, 30.0, -30.0, 87.0, -87.0, 88.8, -88.8, 104.0, -104.0, 3e4, -3e4, 3e38, -3e38, float("inf"),
                          float("-inf"), float("nan")])
    x = torch.zeros(300, K, dtype=torch.bfloat16, device="cuda")
    x[:, 0] = 1.0
    x[:len(gates), 1] = gates.bfloat16().cuda()
    turns = torch.zeros(2 * N, K, dtype=torch.bfloat16, device="cuda")
    turns[torch.arange(2 * N, device="cuda") % 16 < 8, 1] = 1.0      # gates: x[:, 1]
    turns[torch.arange(2 * N, device="cuda") % 16 >= 8, 0] = 1.5     # ups
    got = tiles(SWIGLU, x, turns, N)
    both = torch.zeros(300, 2 * N, dtype=torch.bfloat16, device="cuda")
    both[:, torch.arange(2 * N, device="cuda") % 16 < 8] = x[:, 1:2]
    both[:, torch.arange(2 * N, device="cuda") % 16 >= 8] = 1.5
    # (zeros times what is no number are none either: those rows' ups)
    both[torch.isinf(x[:, 1]) | torch.isnan(x[:, 1])] = float("nan")
    want = ops.swiglu(both, interleave=8)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isinf(), want.isinf())
    good = want.isfinite()
    # (two roundings of nearly the same value; a quotient below 2^-126 is zero, times a gate of up to 89 and 1.5)
    assert bool(((got - want)[good].float().abs() <= 2.0 ** -7 * want[good].float().abs() + 140 * 2.0 ** -126).all())


def test_more_tiles_than_workgroups_and_replays():
    """Workgroups that take several tiles, of which the last are few; the same bits eagerly and from a replayed graph with other work between."""
    from zedinfer_amd import ops
    M, N, K = 1600, 4104, 576
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=0.2)
    for tile in (0, 3, 8, 9):
        out = tiles(BF16, x, w, N, tile=tile)
        close(out, x, w, BF16)
        again = torch.empty_like(out)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            tiles(BF16, x, w, N, out=again, tile=tile)
        for _ in range(3):
            again.zero_()
            g.replay()
            assert torch.equal(out, again)
            ops.linear(x[:64], w)
            torch.cuda.synchronize()


def test_which_products_take_the_tiles(monkeypatch):
    """``ops.linear`` of more than 256 rows by the sizes, and what the kernel cannot load by the library as before."""
    from zedinfer_amd import ops
    calls, real = [], ops._lib.call
    monkeypatch.setattr(ops._lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])

    def taken(M, N, K, bias=False, **kw):
        x, w = rnd(M, K, seed=3), rnd(N, K, seed=4, scale=0.1)
        b = rnd(N, seed=5) if bias else None
        calls.clear()
        out = ops.linear(x, w, b, **kw)
        ref = x.double() @ w.double().t() + (b.double() if bias else 0)
        assert float((out.double() - ref).norm() / ref.norm()) <= (1e-5 if out.dtype == torch.float32 else 3e-3)
        return calls == ["zi_gemm_tiles"]
    assert taken(257, 1536, 1536) and taken(2048, 2048, 1536, bias=True) and taken(640, 1536, 8960, out_dtype=torch.float32)
    assert not taken(256, 1536, 1536) and not taken(300, 1536, 1528) and not taken(300, 1532, 1536) and not taken(320, 512, 4608)
    x, w = rnd(300, 1544, seed=6)[:, 4:1540], rnd(1536, 1536, seed=7)      # rows that do not begin at 16 bytes
    calls.clear()
    ops.linear(x, w)
    assert "zi_gemm_tiles" not in calls
    assert ops.linear_tune(rnd(300, 1536), w) is None


def test_what_is_refused():
    from zedinfer_amd import ops
    x, w = rnd(300, 640), rnd(640, 640)
    for bad in (dict(N=644), dict(N=640, tile=len(TILES)), dict(N=320, epi=SWIGLU, tile=2),
                dict(N=320, epi=GATED, up_at=312), dict(N=320, epi=GATED, up_at=320, act=3)):
        with pytest.raises(ops.KernelLibraryError):
            tiles(bad.pop("epi", BF16), x, w, **bad)
    with pytest.raises(ops.KernelLibraryError):
        tiles(BF16, rnd(300, 256), rnd(640, 256), 640)


@pytest.mark.parametrize("kind,activation", [("swiglu", "silu"), ("gated_mlp", "silu"), ("gated_mlp", "gelu_tanh"), ("gated_mlp", "gelu_erf")])
@pytest.mark.parametrize("n,H,I", [(257, 640, 1000), (640, 1536, 2048)])
def test_feed_forwards_of_many_rows(kind, activation, n, H, I, monkeypatch):
    """Parts whose gate/up product ends in the activation: against float64, and nothing of it is timed or launched apart."""
    from zedinfer_amd.config.forward_config import PartSpec
    from zedinfer_amd.ops import _lib
    from zedinfer_amd.parts import FEED_FORWARDS
    from zedinfer_amd.parts.base import Runtime
    w = {"gate": rnd(I, H, seed=1, scale=0.05), "up": rnd(I, H, seed=2, scale=0.05), "down": rnd(H, I, seed=3, scale=0.05)}
    x, rt = rnd(n, H, seed=4), Runtime("cuda", torch.bfloat16)
    params = {"hidden_size": H, "intermediate_size": I, "activation": activation}
    part = FEED_FORWARDS.get(kind)(PartSpec(kind, params, {k: k for k in w}), w, rt)
    part.tune(n)
    assert not [k for k in rt.choices if k[0] == "gate_up_transposed" or k[2] > H]
    calls, real = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    got = part.forward(x).double()
    if got.dim() == 3:
        got = got.sum(0)
    assert calls[0] == "zi_gemm_tiles" and not {"zi_swiglu", "zi_swiglu_t", "zi_gated_act"} & set(calls)
    fn = {"silu": torch.nn.functional.silu, "gelu_tanh": gelu_tanh, "gelu_erf": torch.nn.functional.gelu}[activation]
    X = x.double()
    ref = (fn(X @ w["gate"].double().t()) * (X @ w["up"].double().t())) @ w["down"].double().t()
    # the activation and the result are rounded to bfloat16 once each, evenly: 2^-8 / sqrt(3) at most of every value, less of a sum
    assert float((got - ref).norm() / ref.norm()) <= 2 * 2.0 ** -8 / 3 ** 0.5


@pytest.mark.parametrize("kind", ["swiglu", "gated_mlp"])
def test_what_no_rule_tells_apart_is_measured_once(kind, monkeypatch):
    """``tune`` times the tiles against the library's products and records the faster, the forward pass follows the record, and a part that
    is given the record times nothing."""
    from zedinfer_amd import ops
    from zedinfer_amd.config.forward_config import PartSpec
    from zedinfer_amd.ops import _lib
    from zedinfer_amd.parts import FEED_FORWARDS
    from zedinfer_amd.parts.base import Runtime
    n, H, I = 1024, 2048, 5120
    w = {"gate": rnd(I, H, seed=1, scale=0.05), "up": rnd(I, H, seed=2, scale=0.05), "down": rnd(H, I, seed=3, scale=0.05)}
    x, params = rnd(n, H, seed=4), {"hidden_size": H, "intermediate_size": I, "activation": "silu"}
    parts = [FEED_FORWARDS.get(kind)(PartSpec(kind, params, {k: k for k in w}), w, Runtime("cuda", torch.bfloat16)) for _ in range(2)]
    assert 0 < ops.linear_tiles_gates_rule(x, parts[0].gate_up, I) < ops.TILES_SURELY
    calls, real = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    choices = parts[0].rt.choices
    parts[0].rt.buffer("norm_out", (n, H)).copy_(x)
    parts[0].tune(n)
    tiles = choices[("tiles_gates", n, 2 * I, H, False, False, "bfloat16")]
    assert isinstance(tiles, bool) and calls.count("zi_gemm_lt_tune") >= 1 and "zi_gemm_tiles" in calls
    if kind == "swiglu":         # (its down product is tuned too)
        assert isinstance(choices[("tiles_product", n, H, I, False, False, "bfloat16")], bool)
    parts[1].rt.choices.update(choices)
    outs = []
    for part in parts:
        calls.clear()
        part.tune(n)
        assert "zi_gemm_lt_tune" not in calls and "zi_gemm_tiles" not in calls and part.rt.choices == choices
        outs.append(part.forward(x).clone())
        made = [c for c in calls if c in ("zi_gemm_tiles", "zi_gemm_lt")]
        assert (made[0] == "zi_gemm_tiles") == tiles
        assert kind != "swiglu" or (made[1] == "zi_gemm_tiles") == choices[("tiles_product", n, H, I, False, False, "bfloat16")]
    assert torch.equal(outs[0], outs[1])
    # either record, the same result but for rounding
    for way in (False, True):
        parts[0].rt.choices[("tiles_gates", n, 2 * I, H, False, False, "bfloat16")] = way
        got = parts[0].forward(x).double()
        assert float((got - outs[1].double()).norm() / outs[1].double().norm()) <= 2 * 2.0 ** -8
