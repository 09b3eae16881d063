"""The blur's windows: radii of every remainder by the window's four, screens that end
inside a lane's outputs, and the largest staged radius along y and along x with one
more, against the post-processing oracle (1e-6 of the largest value, the bound of the
other bloom tests: the taps are summed in its order)."""
import numpy as np
import pytest

from oracle import postp
from test_gpu_postp import _field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('W,H,radius', [(2, 2, 1), (517, 66, 2), (1031, 131, 3), (130, 70, 4), (515, 67, 5), (90, 640, 6),
                                         (60, 50, 284), (60, 50, 285), (40, 20, 4992), (40, 20, 4993)])
def test_bloom_windows(gpu, W, H, radius):
    import torch
    import taichi_three_amd as tina
    print(f'case: bloom {W}x{H} radius {radius}', flush=True)
    rng = np.random.default_rng(radius)
    img = (rng.random((H, W, 3)) ** 3 * 4).astype(np.float32)
    img[H // 3:H // 2, W // 4:W // 2] = 6.0
    bl = tina.Blooming((W, H))
    bl.radius = radius
    bl.init_gwei()
    f = _field(img)
    bl.apply(f)
    torch.cuda.synchronize()
    want = postp.bloom(img, gwei=bl.gwei.cpu().numpy(), radius=radius)
    assert np.abs(f.storage.cpu().numpy() - want).max() <= 1e-6 * max(1.0, float(np.abs(want).max()))
