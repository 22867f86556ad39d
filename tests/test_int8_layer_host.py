"""What an Int8Linear call reads and calls, on the CPU: the layer's attributes
however they were set, and whatever stands for its quantizer, its
forward_quantized and int8_matmul at the time of the call."""
import pytest
import torch

from lynnreal_omni_amd import int8, int8_gemm, kernels
from lynnreal_omni_amd.int8 import Int8Linear, quantize_activations


def _layer(gemm="hip", cls=Int8Linear):
    g = torch.Generator().manual_seed(5)
    w = torch.randint(-127, 128, (24, 32), dtype=torch.int8, generator=g)
    scale = torch.rand(24, 1, generator=g) * 4e-3 + 1e-3
    layer = cls.from_packed(w, scale, torch.randn(24, generator=g).bfloat16(), gemm=gemm)
    layer.fused_ops = True
    return layer


X = torch.randn(2, 3, 32, generator=torch.Generator().manual_seed(6)).bfloat16()


@pytest.fixture
def on_cpu(monkeypatch):
    """kernels.quantize_rows and int8_gemm.int8_matmul replaced, as a caller's
    wrappers would be, by torch forms that record their calls."""
    calls = []

    def quantize_rows(value):
        calls.append("quantize_rows")
        return quantize_activations(value)

    def int8_matmul(a, b, row_scale, column_scale, bias=None, **kw):
        calls.append("int8_matmul")
        return int8_gemm._torch_matmul(a, b, row_scale, column_scale, bias)

    monkeypatch.setattr(kernels, "quantize_rows", quantize_rows)
    monkeypatch.setattr(int8_gemm, "int8_matmul", int8_matmul)
    return calls


def test_wrappers_of_quantizer_and_gemm_are_called(on_cpu):
    layer = _layer()
    y = layer(X)
    assert on_cpu == ["quantize_rows", "int8_matmul"] and y.shape == (2, 3, 24)
    rows = X.reshape(-1, 32)
    want = layer.forward_quantized(*quantize_activations(rows), (2, 3))
    assert on_cpu[2:] == ["int8_matmul"] and torch.equal(y, want)


@pytest.mark.parametrize("name", ["quantize_rows", "int8_matmul"])
def test_one_wrapper_is_enough(on_cpu, monkeypatch, name):
    """With only one of the two replaced the layer still calls it (the other,
    this package's own, refuses CPU tensors)."""
    other = {"quantize_rows": (int8_gemm, "int8_matmul", int8._INT8_MATMUL),
             "int8_matmul": (kernels, "quantize_rows", int8._QUANTIZE_ROWS)}[name]
    monkeypatch.setattr(*other)
    with pytest.raises(ValueError, match="GPU"):
        _layer()(X)
    assert on_cpu == (["quantize_rows"] if name == "quantize_rows" else [])


@pytest.mark.parametrize("where", ["instance", "class", "subclass"])
def test_forward_quantized_is_called(monkeypatch, on_cpu, where):
    monkeypatch.setattr(int8_gemm, "int8_matmul", int8._INT8_MATMUL)   # so nothing but forward_quantized differs
    seen = []

    def replacement(*args, **kw):
        seen.append(args[-1])
        return "projected"

    layer = _layer()
    if where == "instance":
        layer.forward_quantized = replacement
    elif where == "class":
        monkeypatch.setattr(Int8Linear, "forward_quantized", replacement)
    else:
        layer = _layer(cls=type("Own", (Int8Linear,), {"forward_quantized": replacement}))
    assert layer(X) == "projected" and seen == [torch.Size([2, 3])]


@pytest.mark.parametrize("name", ["weight_int8", "weight_scale", "bias"])
@pytest.mark.parametrize("as_parameter", [False, True])
def test_tensors_set_as_plain_attributes(on_cpu, name, as_parameter):
    """A buffer deleted and set again as a plain tensor or a Parameter is read
    by the call, with and without wrappers on the two functions."""
    layer = _layer()
    want = layer(X)
    value = getattr(layer, name)
    delattr(layer, name)
    setattr(layer, name, torch.nn.Parameter(value, requires_grad=False) if as_parameter else value)
    assert torch.equal(layer(X), want)


@pytest.mark.parametrize("name", ["weight_int8", "weight_scale", "bias"])
def test_tensors_of_the_fused_call(monkeypatch, name):
    """The same for the call that fuses quantizer and GEMM."""
    got = []
    monkeypatch.setattr(int8_gemm, "linear_rows", lambda rows, *tensors: got.append(tensors) or rows[:, :24])
    layer = _layer()
    value = getattr(layer, name)
    delattr(layer, name)
    setattr(layer, name, value)
    layer(X)
    assert all(a is b for a, b in zip(got[0], (layer.weight_int8, layer.weight_scale, layer.bias)))


@pytest.mark.parametrize("where", ["instance", "subclass"])
@pytest.mark.parametrize("name", ["weight_int8", "weight_scale", "bias"])
def test_tensors_that_hide_a_buffer(monkeypatch, name, where):
    """An attribute that hides the buffer of its name is what the fused call reads."""
    got = []
    monkeypatch.setattr(int8_gemm, "linear_rows", lambda rows, *tensors: got.append(tensors) or rows[:, :24])
    layer = _layer()
    other = getattr(layer, name).clone()
    if where == "instance":
        layer.__dict__[name] = other
    else:      # as torch.nn.utils.parametrize does it
        layer.__class__ = type("Own", (Int8Linear,), {name: property(lambda self: other)})
    layer(X)
    assert got[0][("weight_int8", "weight_scale", "bias").index(name)] is not layer._buffers[name]
    assert all(a is b for a, b in zip(got[0], (layer.weight_int8, layer.weight_scale, layer.bias)))
