"""Which products of many rows ``ops.linear`` gives to the tiles' kernel, with the launches recorded instead of made: on the CPU."""
import pytest
import torch

from zedinfer_amd import ops
from zedinfer_amd.ops import functional, mixing


@pytest.fixture
def launches(monkeypatch):
    """Names of the library's launches, none of which is made."""
    calls = []
    for ops_of in (functional, mixing):
        monkeypatch.setattr(ops_of, "_gpu", lambda *a: None)
        monkeypatch.setattr(ops_of, "_stream", lambda: None)
    monkeypatch.setattr(functional._lib, "call", lambda name, *a: calls.append(name))
    return calls


def operands(M, N, K):
    return torch.zeros(M, K, dtype=torch.bfloat16), torch.zeros(N, K, dtype=torch.bfloat16)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float64, torch.int32, torch.int16, torch.int8, torch.uint8, torch.bool])
def test_a_result_of_another_type_is_refused(dtype, launches):
    """257 rows at sizes that the tiles take: a type that they do not store raises, as for fewer rows, and nothing is launched."""
    x, w = operands(257, 1536, 1536)
    ops.linear(x, w)
    ops.linear(x, w, out_dtype=torch.float32)
    assert launches == ["zi_gemm_tiles"] * 2
    launches.clear()
    for call in (lambda: ops.linear(x, w, out_dtype=dtype), lambda: ops.linear(x, w, out=torch.zeros(257, 1536, dtype=dtype)),
                 lambda: ops.linear(x[:256], w, out_dtype=dtype), lambda: ops.linear_tune(x, w, out_dtype=dtype)):
        with pytest.raises(TypeError):
            call()
    assert not launches


def test_gate_and_up_rows_that_are_no_whole_blocks_are_refused(launches):
    """8 gate rows, then 8 up rows, and so on: a weight with a row more has no place for it."""
    x, w = operands(2048, 2 * 8960 + 1, 1536)
    ops.linear_tiles_swiglu(x, w[:-1])
    assert launches == ["zi_gemm_tiles"]
    with pytest.raises(ValueError):
        ops.linear_tiles_swiglu(x, w)
    assert launches == ["zi_gemm_tiles"]


def pays(M, N, K, gates=False):
    return ops.load().zi_gemm_tiles_pays(M, N, K, int(gates))


def test_the_rule_is_bounded_to_where_it_tells_the_ways_apart():
    """0: not taken; 1: taken, the library faster; 2: the tiles faster; 3: surely (a gate/up product)."""
    assert [pays(M, 1536, 1536) for M in (256, 257)] == [0, 2] and pays(300, 512, 4608) == pays(300, 4608, 512) == pays(300, 1536, 1528) == 0
    assert pays(640, 2048, 1536, True) == pays(257, 1000, 640, True) == 3 and pays(2048, 8960, 1536, True) == 2
    # large products, among them those of a prompt of 16,384 tokens at 32B sizes: the library was a quarter faster at some
    assert pays(4096, 16384, 4096) == pays(2048, 3584, 18944) == 1
    assert [pays(16384, N, K) for N, K in ((7168, 5120), (5120, 5120), (5120, 27648))] == [1, 1, 1] and pays(16384, 27648, 5120, True) == 1


@pytest.fixture
def runtime(launches, monkeypatch):
    from zedinfer_amd.parts.base import Runtime
    for name in ("ZEDINFER_PRODUCT_TILES", "ZEDINFER_GATE_UP_TRANSPOSED"):
        monkeypatch.delenv(name, raising=False)
    return Runtime("cpu", torch.bfloat16)


def test_a_runtime_reads_the_variable(monkeypatch):
    from zedinfer_amd.parts.base import Runtime
    for given, tiles in (("0", False), ("1", True), ("", None), ("yes", None)):
        monkeypatch.setenv("ZEDINFER_PRODUCT_TILES", given)
        assert Runtime("cpu", torch.bfloat16).product_tiles is tiles


@pytest.mark.parametrize("M,N,K,rule", [(640, 1536, 2048, True), (2560, 4608, 5120, False)])
def test_products_are_made_as_recorded(M, N, K, rule, launches, runtime, monkeypatch):
    """Without a record by the rule; a variable before it; a record before that, also an earlier run's of the library's algorithm."""
    x, w = operands(M, N, K)

    def made():
        launches.clear()
        runtime.linear(x, w, out=torch.zeros(M, N, dtype=torch.bfloat16))
        assert len(launches) == 1
        return launches[0] == "zi_gemm_tiles"
    assert made() == rule
    for given in (False, True):
        monkeypatch.setattr(runtime, "product_tiles", given)
        assert made() == given
        for recorded in (True, False):
            runtime.choices[("tiles_product", M, N, K, False, False, "bfloat16")] = recorded
            assert made() == recorded
        runtime.choices.clear()
    runtime.choices[("library_product", M, N, K, False, False, "bfloat16")] = 3
    assert not made()
    runtime.choices[("tiles_product", M, N, K, False, False, "bfloat16")] = True
    assert made()
    few, _ = operands(256, N, K)
    runtime.linear(few, w, out=torch.zeros(256, N, dtype=torch.bfloat16))
    assert "zi_gemm_tiles" not in launches[1:]


@pytest.mark.parametrize("kind", ["swiglu", "gated_mlp"])
def test_gate_and_up_are_made_as_recorded(kind, launches, runtime, monkeypatch):
    from zedinfer_amd.config.forward_config import PartSpec
    from zedinfer_amd.parts import FEED_FORWARDS
    n, H, I = 640, 1536, 2048
    w = {"gate": torch.zeros(I, H, dtype=torch.bfloat16), "up": torch.zeros(I, H, dtype=torch.bfloat16), "down": torch.zeros(H, I, dtype=torch.bfloat16)}
    params = {"hidden_size": H, "intermediate_size": I, "activation": "silu"}
    part = FEED_FORWARDS.get(kind)(PartSpec(kind, params, {k: k for k in w}), w, runtime)
    x, choices = torch.zeros(n, H, dtype=torch.bfloat16), runtime.choices
    TILES, STRAIGHT, TURNED = ["zi_gemm_tiles"], ["zi_gemm_lt", "zi_swiglu" if kind == "swiglu" else "zi_gated_act"], ["zi_gemm_lt", "zi_swiglu_t"]
    tiles, library = ("tiles_gates", n, 2 * I, H, False, False, "bfloat16"), ("library_product", n, 2 * I, H, False, False, "bfloat16")

    def made():
        launches.clear()
        part.forward(x)
        return launches[:-1]         # (the last is the down product's)
    assert made() == TILES
    choices[tiles] = False
    assert made() == STRAIGHT
    choices.clear()
    choices[library] = 3
    assert made() == STRAIGHT
    choices[tiles] = True
    assert made() == TILES
    choices.clear()
    monkeypatch.setattr(runtime, "product_tiles", False)
    assert made() == STRAIGHT
    if kind == "swiglu":             # the library's way round: a variable and a record of it are the library's
        for given, way in (("0", STRAIGHT), ("1", TURNED)):
            monkeypatch.setattr(runtime, "product_tiles", True)
            monkeypatch.setenv("ZEDINFER_GATE_UP_TRANSPOSED", given)
            assert made() == way
            monkeypatch.delenv("ZEDINFER_GATE_UP_TRANSPOSED")
            choices[("gate_up_transposed", n, 2 * I, H)] = given == "1"
            assert made() == way
            choices[tiles] = True
            assert made() == TILES
            choices.clear()
