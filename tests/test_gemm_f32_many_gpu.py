"""float32 products of many rows whose x is split once, in a workspace (``csrc/gemm_f32_split.hip``): the bits of the kernels without
one, in every tile and cut, at the edges of rows, columns and k.  Those kernels are held against float64 in test_gemm_f32_split_gpu.py."""
import pytest
import torch

pytestmark = pytest.mark.gpu
CUTS = [(4, 8), (6, 8), (8, 8), (4, 4), (6, 4), (8, 4), (4, 2), (6, 2), (8, 2)]
# k: the last chunk of 64 with 4 columns; whole; seven runs of four chunks, the last of one; six runs of five and one of two
SIZES = [(33, 132, 1412), (64, 128, 1536), (97, 260, 1600), (130, 516, 2052), (257, 64, 1476), (48, 1028, 8960)]


def _operands(M, N, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N + seed)
    return tuple(torch.randn(s, generator=g, device="cuda") for s in ((M, K), (N, K), (N,)))


def _many(x, w, bias, mt, runs, gated=False, out=None, whole=0):
    from zedinfer_amd.ops import _lib
    from zedinfer_amd.ops.functional import _p, _stream
    M, K, N = x.shape[0], x.shape[1], w.shape[0] // (2 if gated else 1)
    need = _lib.load().zi_gemm_f32_many_workspace(M, N, K, x.stride(0), w.stride(0), int(gated), mt, runs, whole)
    assert need > 0
    ws = torch.full((need // 4,), float("nan"), device="cuda")
    out = torch.full((M, N), 7.0, device="cuda") if out is None else out
    _lib.call("zi_gemm_f32_many", _p(out), _p(x), _p(w), _p(bias), M, N, K, x.stride(0), w.stride(0), out.stride(0), int(gated), mt, runs,
              whole, _p(ws), need, _stream())
    return out


@pytest.mark.parametrize("mt,runs", CUTS)
def test_the_bits_without_a_workspace(mt, runs):
    from zedinfer_amd import ops
    for M, N, K in SIZES:
        x, w, b = _operands(M, N, K)
        assert torch.equal(_many(x, w, b, mt, runs), ops.linear(x, w, b)), (M, N, K)
        assert torch.equal(_many(x, w, None, mt, runs), ops.linear(x, w)), (M, N, K)


@pytest.mark.parametrize("mt,runs", CUTS)
def test_rows_apart_in_memory(mt, runs):
    from zedinfer_amd import ops
    M, N, K = 101, 140, 1540
    x, w, b = _operands(M, N, K + 12)
    x, w = x[:, 4:K + 4], w[:, 8:K + 8]
    out = torch.full((M, N + 5), 7.0, device="cuda")
    _many(x, w, b, mt, runs, out=out[:, 1:N + 1])
    assert torch.equal(out[:, 1:N + 1], ops.linear(x.contiguous(), w.contiguous(), b))
    assert bool((out[:, 0] == 7.0).all()) and bool((out[:, N + 1:] == 7.0).all())


@pytest.mark.parametrize("mt", [4, 6, 8])
@pytest.mark.parametrize("M,I,K,runs,whole", [(100, 3001, 1500, 8, 0), (129, 4097, 1412, 8, 0), (200, 1032, 2052, 8, 0), (100, 3004, 1500, 2, 0),
                                              (129, 4100, 1412, 4, 4032), (200, 1036, 2052, 2, 512)])
def test_gate_and_up_end_in_the_activation(M, I, K, runs, whole, mt):
    from zedinfer_amd import ops
    x, w, _ = _operands(M, 2 * I, K)
    two = ops.linear(x, w)
    assert torch.equal(_many(x, w, None, mt, runs, gated=True, whole=whole), ops.swiglu(two[:, :I], two[:, I:]))


@pytest.mark.parametrize("mt", [4, 6, 8])
@pytest.mark.parametrize("runs", [2, 4])
def test_columns_in_two_cuts(mt, runs):
    from zedinfer_amd import ops
    x, w, b = _operands(140, 1028, 1540)
    x[5, 7], w[1000, 3] = float("nan"), float("inf")
    for whole in (128, 900, 1024):
        assert torch.equal(_many(x, w, b, mt, runs, whole=whole).nan_to_num(3.0), ops.linear(x, w, b).nan_to_num(3.0)), whole


@pytest.mark.parametrize("mt,runs", CUTS)
def test_sums_that_are_not_finite(mt, runs):
    """Values past what can be split, infinities and NaNs in rows of x (the first, one of the second 64, the last) and of the weights."""
    from zedinfer_amd import ops
    M, N, K = 130, 260, 1500
    x, w, b = _operands(M, N, K)
    x[0] = torch.where(x[0] < 0, -3.4e38, 3.4e38)
    x[70, 5], x[M - 1, K - 1], x[3, 2] = float("nan"), float("nan"), float("inf")
    w *= 2.0 ** -110
    w[7, 9], w[N - 1, 0] = float("nan"), float("-inf")
    got, ref = _many(x, w, b, mt, runs), ops.linear(x, w, b)
    rest = [m for m in range(M) if m != 0]       # (row 0 is made again from the operands, whose sums have an order of their own)
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(got[rest].nan_to_num(3.0), ref[rest].nan_to_num(3.0))
    fine = torch.isfinite(ref[0])
    assert float((got[0][fine].double() - ref[0][fine].double()).norm() / ref[0][fine].double().norm()) < 2.0 ** -20      # (both within 2^-21: K / 64 additions a lane)


def test_rows_beyond_what_is_split_at_a_time():
    from zedinfer_amd import ops
    from zedinfer_amd.ops import _lib
    M, N, K = 1411, 96, 65536
    x, w, b = _operands(M, N, K)
    ref = ops.linear(x, w, b)
    for mt, runs in ((4, 8), (8, 2)):
        assert _lib.load().zi_gemm_f32_many_workspace(M, N, K, K, K, 0, mt, runs, 0) < (258 << 20) + 8 * M * N * 4
        assert torch.equal(_many(x, w, b, mt, runs), ref)


def test_where_it_pays_and_what_is_refused():
    from zedinfer_amd import ops
    x, w, b = _operands(450, 3584, 3584)
    need = ops.linear_many_workspace(x, w)
    assert need > 0 and ops.linear_many_workspace(x[:20], w) == 0 and ops.linear_many_workspace(x[:, :1408], w[:, :1408]) == 0
    assert ops.linear_many_workspace(x.bfloat16(), w.bfloat16()) == 0 and ops.linear_many_workspace(x[:, 1:], w[:, 1:]) == 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    ref = ops.linear(x, w, b)
    assert torch.equal(ops.linear(x, w, b, workspace=ws), ref)
    assert torch.equal(ops.linear(x[:20], w, b, workspace=ws), ref[:20])          # (made without it)
    with pytest.raises(ValueError):
        ops.linear(x, w, b, workspace=ws[:need - 16])
    x2, w2, _ = _operands(450, 17920, 1536)
    gated = ops.linear_many_workspace(x2, w2, gated=True)
    assert gated > 0 and ops.linear_many_workspace(x2[:20], w2, gated=True) == 0
    assert torch.equal(ops.linear_swiglu_halves(x2, w2, workspace=torch.empty(gated, dtype=torch.uint8, device="cuda")), ops.linear_swiglu_halves(x2, w2))
    s, out = torch.cuda.Stream(), torch.zeros_like(ref)
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s), torch.cuda.graph(graph, stream=s):
        ops.linear(x, w, b, out=out, workspace=ws)
    for i in range(3):
        x.mul_(2.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ops.linear(x, w, b)), i
