"""Operands that are not contiguous: the wrappers copy them, and every copy lives until the call
has been made.  Against the same call on contiguous tensors, bit for bit."""
import pytest
import torch

from iconnx_amd import ops

pytestmark = pytest.mark.gpu


def same(a, b):
    assert torch.equal(a.contiguous().view(torch.int32), b.contiguous().view(torch.int32))


@pytest.mark.parametrize("B,S,H", [(2, 40, 3), (1, 129, 2)])
def test_attention_over_slices_of_one_packed_tensor(B, S, H):
    g = torch.Generator(device="cuda").manual_seed(S)
    qkv = torch.randn((B, S, 3 * H * 64), generator=g, device="cuda")
    q, k, v = qkv.split(H * 64, dim=-1)
    assert not q.is_contiguous()
    same(ops.gpu_attention(q, k, v, H, 8.0), ops.gpu_attention(q.clone(memory_format=torch.contiguous_format),
                                                               k.contiguous(), v.contiguous(), H, 8.0))


def test_attention_over_transposed_tensors():
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn((50, 2, 128), generator=g, device="cuda").transpose(0, 1) for _ in range(3))
    same(ops.gpu_attention(q, k, v, 2, 8.0),
         ops.gpu_attention(*(t.contiguous() for t in (q, k, v)), 2, 8.0))


@pytest.mark.parametrize("cols", [768, 384, 37])
def test_layer_norm_strided_scale_and_bias(cols):
    g = torch.Generator(device="cuda").manual_seed(cols)
    x, r = (torch.randn((cols, 60), generator=g, device="cuda").t() for _ in range(2))
    scale, bias = (torch.randn((2 * cols,), generator=g, device="cuda")[::2] for _ in range(2))
    same(ops.gpu_layer_norm(x, scale, bias, 1e-5, r),
         ops.gpu_layer_norm(x.contiguous(), scale.contiguous(), bias.contiguous(), 1e-5, r.contiguous()))


def test_pow_strided_exponent():
    base = torch.rand((30, 50), device="cuda") + 0.5
    e = (torch.rand((50, 30), device="cuda") + 0.5).t()
    same(ops.gpu_pow(base.t().contiguous().t(), e), ops.gpu_pow(base, e.contiguous()))
