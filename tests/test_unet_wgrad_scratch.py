"""The weight gradient's scratch: agdu_wgrad_part_len floats, all of them
written and none beyond (one or many row chunks, one or many tile pairs)."""
import pytest
import torch

from tests.test_unet_kernels import _lib, _p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ci,co,shape", [(16, 16, (1, 1, 1, 1)), (48, 16, (2, 9, 33, 70)),
                                         (32, 64, (3, 20, 31, 65)), (96, 32, (1, 16, 16, 128))])
def test_scratch_is_what_is_asked_for(ci, co, shape):
    L = _lib()
    n, guard, mark = L.agdu_wgrad_part_len(*shape, ci, co), 4096, 12345.678
    x = torch.randn(shape + (ci,), device="cuda").bfloat16()
    dy = torch.randn(shape + (co,), device="cuda").bfloat16()
    part = torch.full((n + guard,), mark, device="cuda")
    dw = torch.empty((27, co, ci), device="cuda")
    db = torch.empty(co, device="cuda")
    assert L.agdu_conv3_wgrad(_p(x), _p(dy), _p(part), _p(dw), _p(db), *shape, ci, co, None) == 0
    torch.cuda.synchronize()
    unwritten = part == part.new_tensor(mark)
    assert bool(unwritten[n:].all())
    assert not bool(unwritten[:n].any())
