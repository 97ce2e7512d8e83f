"""Which products of many rows ``ops.linear`` gives to the tiles' kernel, with the launches recorded instead of made: on the CPU."""
import pytest
import torch

from zedinfer_amd import ops
from zedinfer_amd.ops import functional


@pytest.fixture
def launches(monkeypatch):
    """Names of the library's launches, none of which is made."""
    calls = []
    monkeypatch.setattr(functional, "_gpu", lambda *a: None)
    monkeypatch.setattr(functional, "_stream", lambda: None)
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
    assert [pays(M, 1536, 1536) for M in (256, 257)] == [0, 1] and pays(300, 512, 4608) == pays(300, 4608, 512) == pays(300, 1536, 1528) == 0
    assert pays(640, 2048, 1536, True) == pays(257, 1000, 640, True) == pays(2048, 8960, 1536, True) == 1
    # large products, among them those of a prompt of 16,384 tokens at 32B sizes: the library was a quarter faster at some
    assert pays(4096, 16384, 4096) == pays(2048, 3584, 18944) == 0
    assert [pays(16384, N, K) for N, K in ((7168, 5120), (5120, 5120), (5120, 27648))] == [0, 0, 0] and pays(16384, 27648, 5120, True) == 0
