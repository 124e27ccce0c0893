"""Which library calls FP8WeightAct.linear makes, with the calls themselves replaced (no GPU)."""
import pytest
import torch

from engine.quantization.fp8 import FP8WeightAct
from kernels import quant_ops as ops

K, N = 256, 48


@pytest.fixture
def calls(monkeypatch):
    made = []

    def linear(x, w, s):
        made.append(("linear", x))
        return torch.zeros(x.shape[0], N, dtype=torch.bfloat16)

    def gemm(xq, xs, w, s):
        made.append(("gemm", xq))
        return torch.zeros(xq.shape[0], N, dtype=torch.bfloat16)

    monkeypatch.setattr(ops, "fp8_linear", linear)
    monkeypatch.setattr(ops, "fp8_gemm", gemm)
    return made


WEIGHT = dict(qweight=torch.zeros(N, K, dtype=torch.float8_e4m3fn), scale=torch.ones(N))


class Halved(FP8WeightAct):
    @staticmethod
    def quantize_activation(x2d):
        return (x2d / 2).to(torch.float8_e4m3fn), torch.full((x2d.shape[0], 1), 2.0)


@pytest.mark.parametrize("on_object", [False, True])
def test_a_replaced_quantizer_is_called(calls, on_object):
    """quantize_activation of a subclass or set on the method object quantizes the activations."""
    m = FP8WeightAct(backend="native") if on_object else Halved(backend="native")
    if on_object:
        m.quantize_activation = Halved.quantize_activation
    x = torch.full((3, K), 8.0)
    assert m.linear(x, **WEIGHT).shape == (3, N)
    (name, xq), = calls
    assert name == "gemm" and (xq.float() == 4.0).all()


@pytest.mark.parametrize("shape", [(K,), (5, K), (2, 3, K)])
def test_one_call_for_the_rows_of_any_shape(calls, shape):
    """The library gets x as rows, and a strided x of three dimensions is copied once."""
    m = FP8WeightAct(backend="native")
    x = torch.randn(*shape)
    y = m.linear(x, **WEIGHT)
    assert y.shape == (*shape[:-1], N) and y.dtype == x.dtype
    (name, rows), = calls
    assert name == "linear" and torch.equal(rows, x.reshape(-1, K))
    if len(shape) == 3:
        m.linear(torch.randn(3, 2, K).transpose(0, 1), **WEIGHT)
        assert calls[1][1].dim() == 2 and calls[1][1].is_contiguous()
