"""GPU check of linear_rows, the fused-ops call of an Int8Linear: equal bit for
bit to quantize_rows followed by int8_matmul over the row types, widths, weight
layouts, scale and bias forms that the layer accepts."""
import pytest
import torch

from lynnreal_omni_amd import int8_gemm, kernels
from lynnreal_omni_amd.int8 import Int8Linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
@pytest.mark.parametrize("m,n,k", [(1, 8, 16), (3, 130, 100), (32, 512, 4096), (257, 264, 1040), (40, 33, 7)])
def test_equals_the_two_calls(m, n, k, dtype):
    g = torch.Generator().manual_seed(m + n + k)
    x = (torch.randn(m, k, generator=g) * 3).to(dtype).cuda()
    w = torch.randint(-127, 128, (n, k), dtype=torch.int8, generator=g).cuda()
    cs = (torch.rand(1, n, generator=g) * 4e-3 + 1e-3).cuda()
    b = (0.02 * torch.randn(n, generator=g)).bfloat16().cuda()
    q, s = kernels.quantize_rows(x)
    for weight in (w.t(), w.t().contiguous()):
        for scale, bias in ((cs, b), (cs.reshape(-1), None), (cs.double(), b),
                            (torch.stack([cs, cs], -1)[..., 0], torch.stack([b, b], -1)[:, 0])):
            got = int8_gemm.linear_rows(x, weight, scale, bias)
            assert torch.equal(got, int8_gemm.int8_matmul(q, weight, s, scale, bias))


def test_layer_and_its_errors():
    g = torch.Generator().manual_seed(1)
    w = torch.randint(-127, 128, (64, 256), dtype=torch.int8, generator=g)
    layer = Int8Linear.from_packed(w.cuda(), torch.rand(64, 1).cuda(), None, gemm="hip")
    x = torch.randn(2, 5, 256, generator=g).bfloat16().cuda()
    plain = layer.forward_quantized(*kernels.quantize_rows(x.reshape(-1, 256)), x.shape[:-1])
    layer.fused_ops = True
    assert torch.equal(layer(x), plain) and layer(x).shape == (2, 5, 64)
    assert layer(x[:, :0]).shape == (2, 0, 64)
    # Rows that are a view of a larger tensor are copied in order first.
    wide = torch.randn(2, 5, 512, generator=g).bfloat16().cuda()
    assert torch.equal(layer(wide[..., ::2]), layer(wide[..., ::2].contiguous()))
    with pytest.raises(RuntimeError, match="not supported"):
        layer(x.double())
    with pytest.raises(ValueError, match="GPU"):
        layer(x.cpu())
    with pytest.raises(ValueError, match="is on cpu"):
        int8_gemm.linear_rows(x[0], w.t(), layer.weight_scale, None)


@pytest.mark.parametrize("rows", [1, 512, 513])
@pytest.mark.parametrize("width", [2048, 2056, 4088, 4096, 4104, 6144, 6152, 8192, 8200, 12296])
def test_quantizer_at_the_edges_of_its_kernels(rows, width):
    """A wave and a block per row, at the widths and counts where one takes over
    from the other and at their chunk counts, against the torch restatement."""
    from oracle import torch_path as tp
    g = torch.Generator().manual_seed(rows + width)
    x = (torch.randn(rows, width, generator=g) * 5).bfloat16()
    x[0] = 0
    q, s = kernels.quantize_rows(x.cuda())
    want_q, want_s = tp.quantize(x)
    assert torch.equal(q.cpu(), want_q) and torch.equal(s.cpu().reshape(-1), want_s.reshape(-1))
