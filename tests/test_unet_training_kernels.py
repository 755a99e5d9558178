"""The training pass's fused resampling kernels against the separate ones,
bit for bit, and the weight gradient at the edges of its row chunks (64
voxels of w in halves of 32, runs of rows over h, d and n) against the FP64
restatement, to the bound of test_unet_kernels (FP32 sums: 1e-4)."""
import numpy as np
import pytest
import torch

from tests import unet_ref as R
from tests.test_unet_kernels import _bf, _close, _lib, _p

pytestmark = pytest.mark.gpu


def _rand(rng, *shape):
    return _bf(R.bf16_round(rng.standard_normal(shape)))


@pytest.mark.parametrize("ci,co,shape", [
    (16, 16, (1, 1, 1, 1)), (16, 16, (1, 1, 2, 65)), (16, 16, (2, 2, 1, 66)),
    (16, 32, (3, 16, 17, 31)), (48, 16, (5, 7, 23, 33)), (32, 64, (2, 9, 16, 64))])
def test_weight_gradient_at_row_chunk_edges(ci, co, shape):
    rng = np.random.default_rng(7 * ci + co + shape[-1])
    x = R.bf16_round(rng.standard_normal(shape + (ci,)))
    dy = R.bf16_round(rng.standard_normal(shape + (co,)))
    L = _lib()
    part = torch.empty(L.agdu_wgrad_part_len(*shape, ci, co), dtype=torch.float32, device="cuda")
    dw = torch.empty((27, co, ci), dtype=torch.float32, device="cuda")
    db = torch.empty(co, dtype=torch.float32, device="cuda")
    x_d, dy_d = _bf(x), _bf(dy)
    assert L.agdu_conv3_wgrad(_p(x_d), _p(dy_d), _p(part), _p(dw), _p(db), *shape, ci, co,
                              None) == 0
    torch.cuda.synchronize()
    _close(dw.cpu().numpy().astype(np.float64), R.conv3_weight_grad(x, dy), 1e-4)
    _close(db.cpu().numpy().astype(np.float64), dy.sum(axis=(0, 1, 2, 3)), 1e-4)


@pytest.mark.parametrize("cu,cs,shape", [(32, 16, (2, 4, 6, 20)), (64, 32, (1, 2, 2, 300)),
                                         (8, 8, (3, 2, 4, 2))])
def test_concat_up_is_upsample_and_copy(cu, cs, shape):
    rng = np.random.default_rng(cu + shape[-1])
    n, d, h, w = shape
    xu, xs = _rand(rng, n, d // 2, h // 2, w // 2, cu), _rand(rng, *shape, cs)
    a, b = (torch.zeros(shape + (cu + cs,), dtype=torch.bfloat16, device="cuda") for _ in "ab")
    L = _lib()
    assert L.agdu_concat_up(_p(xu), _p(xs), _p(a), *shape, cu, cs, None) == 0
    assert L.agdu_upsample(_p(xu), _p(b), n, d // 2, h // 2, w // 2, cu, cu + cs, 0, None) == 0
    assert L.agdu_copy_channels(_p(xs), _p(b), n * d * h * w, cs, 0, cu + cs, cu, cs, 0, None,
                                None) == 0
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    assert L.agdu_concat_up(_p(xu), _p(xs), _p(a), n, d, h, w - 1, cu, cs, None) == 1


@pytest.mark.parametrize("c,ca,c0,shape", [(16, 48, 32, (2, 4, 6, 20)), (32, 96, 64, (1, 2, 2, 130))])
def test_maxpool_bwd_add_is_gradient_plus_copy(c, ca, c0, shape):
    rng = np.random.default_rng(c + shape[-1])
    n, d, h, w = shape
    x, add = _rand(rng, *shape, c), _rand(rng, *shape, ca)
    y = torch.empty((n, d // 2, h // 2, w // 2, c), dtype=torch.bfloat16, device="cuda")
    arg = torch.empty(y.shape, dtype=torch.uint8, device="cuda")
    dy = _rand(rng, *y.shape)
    a, b = torch.empty_like(x), torch.empty_like(x)
    L = _lib()
    assert L.agdu_maxpool(_p(x), _p(y), _p(arg), *shape, c, None) == 0
    assert L.agdu_maxpool_bwd_add(_p(dy), _p(arg), _p(add), ca, c0, _p(a), *shape, c, None) == 0
    assert L.agdu_maxpool_bwd(_p(dy), _p(arg), _p(b), *shape, c, None) == 0
    assert L.agdu_copy_channels(_p(add), _p(b), n * d * h * w, ca, c0, c, 0, c, 1, None, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    assert L.agdu_maxpool_bwd_add(_p(dy), _p(arg), _p(add), ca, ca - 8, _p(a), *shape, c, None) == 1
