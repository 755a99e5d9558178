"""The resampling kernels on very many and on very few rows. One block per
row of a volume of 2 x (2^25 + 2) rows would be more threads than a
launch may have (2^32), and on eight rows of 100000 voxels it would leave the
chip idle (ninety times the time of as many voxels in a cube). Bit for bit against torch (whole-voxel copies, one
winner of a pooling window, the maximum itself; the upsampling's gradient of
eight equal powers of two, exact in bf16)."""
import pytest
import torch

from tests.test_unet_kernels import _lib, _p

pytestmark = pytest.mark.gpu

N, D, H, W, C = 1, 2, (1 << 25) + 2, 2, 8  # 2^26 + 4 rows


def _values(*shape):
    """positive finite bf16 values of random bits"""
    v = torch.randint(0x3c00, 0x4400, shape, dtype=torch.int16, device="cuda")
    return v.view(torch.bfloat16)


def test_pooling_and_its_gradient():
    L = _lib()
    torch.manual_seed(1)
    x = _values(N, D, H, W, C)
    y = torch.empty(N, D // 2, H // 2, W // 2, C, dtype=torch.bfloat16, device="cuda")
    arg = torch.empty(y.shape, dtype=torch.uint8, device="cuda")
    assert L.agdu_maxpool(_p(x), _p(y), _p(arg), N, D, H, W, C, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(y, x.view(N, 1, 2, H // 2, 2, W // 2, 2, C).amax(dim=(2, 4, 6)))
    dx = torch.empty_like(x)
    assert L.agdu_maxpool_bwd(_p(y), _p(arg), _p(dx), N, D, H, W, C, None) == 0
    torch.cuda.synchronize()
    cells = dx.view(N, 1, 2, H // 2, 2, W // 2, 2, C)
    for o in range(8):
        assert torch.equal(cells[:, :, o >> 2, :, (o >> 1) & 1, :, o & 1],
                           torch.where(arg == o, y, torch.zeros_like(y)))


def test_pooling_of_as_many_output_rows():
    L = _lib()
    torch.manual_seed(2)
    x = _values(N, 2 * D, 2 * H, 2, C)
    y = torch.empty(N, D, H, 1, C, dtype=torch.bfloat16, device="cuda")
    arg = torch.empty(y.shape, dtype=torch.uint8, device="cuda")
    assert L.agdu_maxpool(_p(x), _p(y), _p(arg), N, 2 * D, 2 * H, 2, C, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(y, x.view(N, D, 2, H, 2, 1, 2, C).amax(dim=(2, 4, 6)))


def test_concatenation_and_upsampling_gradient():
    L = _lib()
    torch.manual_seed(3)
    xu, xs = _values(N, D // 2, H // 2, W // 2, 8), _values(N, D, H, W, 8)
    y = torch.empty(N, D, H, W, 16, dtype=torch.bfloat16, device="cuda")
    assert L.agdu_concat_up(_p(xu), _p(xs), _p(y), N, D, H, W, 8, 8, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(y[..., 8:], xs)
    cells = y[..., :8].view(N, 1, 2, H // 2, 2, W // 2, 2, 8)
    for o in range(8):
        assert torch.equal(cells[:, :, o >> 2, :, (o >> 1) & 1, :, o & 1], xu)
    # dx of D x H rows from dy = the upsampling of 2^k
    dx = torch.empty(N, D, H, 1, 8, dtype=torch.bfloat16, device="cuda")
    g = torch.exp2(torch.randint(-9, 9, dx.shape, device="cuda", dtype=torch.int8).float()).bfloat16()
    dy = g.view(N, D, 1, H, 1, 1, 1, 8).expand(N, D, 2, H, 2, 1, 2, 8).reshape(N, 2 * D, 2 * H, 2, 8)
    dy = dy.contiguous()
    assert L.agdu_upsample_bwd(_p(dy), _p(dx), N, D, H, 1, 8, 8, 0, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(dx, g * 8)


def _us(call):
    call()
    best = 1e9
    for _ in range(5):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in "ab")
        a.record()
        for _ in range(10):
            assert call() == 0
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 100)
    return best


def test_few_long_rows_take_no_longer():
    L = _lib()
    times = []
    for d, h, w in ((2, 2, 100000), (20, 20, 1000)):
        x = _values(2, d, h, w, 32)
        y = torch.empty(2, d // 2, h // 2, w // 2, 32, dtype=torch.bfloat16, device="cuda")
        arg = torch.empty(y.shape, dtype=torch.uint8, device="cuda")
        cat = torch.empty(2, d, h, w, 64, dtype=torch.bfloat16, device="cuda")
        st = torch.cuda.current_stream().cuda_stream
        times.append([
            _us(lambda: L.agdu_maxpool(_p(x), _p(y), _p(arg), 2, d, h, w, 32, st)),
            _us(lambda: L.agdu_maxpool_bwd(_p(y), _p(arg), _p(x), 2, d, h, w, 32, st)),
            _us(lambda: L.agdu_concat_up(_p(y), _p(x), _p(cat), 2, d, h, w, 32, 32, st)),
            _us(lambda: L.agdu_upsample_bwd(_p(x), _p(y), 2, d // 2, h // 2, w // 2, 32, 32, 0, st))])
    print("us of eight rows", times[0], "of a cube", times[1], flush=True)
    assert all(a < 3 * b + 5 for a, b in zip(*times))
