"""Pointers that are aligned to their own type only: a bias inside a packed
parameter vector, a gradient that starts anywhere in a bf16 buffer. The same
bits as from allocations of their own."""
import pytest
import torch

from tests.test_unet_kernels import _lib, _p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ci,co", [(16, 16), (16, 32), (32, 64)])
def test_bias_at_any_float(ci, co):
    L = _lib()
    torch.manual_seed(ci + co)
    dims = (1, 4, 6, 40)
    x = torch.randn(dims + (ci,), device="cuda").bfloat16()
    w = torch.randn(27, co, ci, device="cuda").bfloat16()
    packed = torch.randn(co + 8, device="cuda")
    outs = []
    for at in range(4):
        bias = packed[at:at + co]
        own = bias.clone()
        ya, yb = (torch.empty(dims + (co,), dtype=torch.bfloat16, device="cuda") for _ in "ab")
        for b, y in ((bias, ya), (own, yb)):
            assert L.agdu_conv3(_p(x), _p(w), _p(b), None, _p(y), *dims, ci, co, 3, None) == 0
        torch.cuda.synchronize()
        assert torch.equal(ya, yb)
        outs.append(ya)
    assert not torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("at", [1, 3, 8])
def test_loss_gradient_at_any_bf16(at):
    L = _lib()
    torch.manual_seed(at)
    nvox, c = 1000, 16
    y = torch.randn(nvox, c, device="cuda").bfloat16()
    t = torch.randn(nvox, device="cuda")
    part = torch.empty(int(L.agdu_loss_parts(nvox)), device="cuda")
    own = torch.empty(nvox * c, dtype=torch.bfloat16, device="cuda")
    buf = torch.full((nvox * c + 16,), 7.0, dtype=torch.bfloat16, device="cuda")
    inside = buf[at:at + nvox * c]
    for dy in (own, inside):
        assert L.agdu_l2_loss(_p(y), _p(t), _p(dy), _p(part), nvox, c, 0.5, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(own, inside)
    assert bool((buf[:at] == 7).all()) and bool((buf[at + nvox * c:] == 7).all())
