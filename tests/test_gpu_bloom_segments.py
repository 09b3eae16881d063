"""The blur along x writes its 256-pixel segments out of LDS in memory order: rows that
end on, before and after a segment's last pixel, at small radii, against the
post-processing oracle (1e-6 of the largest value, the bound of the other bloom tests:
the taps are summed in its order), with the half-size buffer's neighbours untouched."""
import numpy as np
import pytest

from oracle import postp
from test_gpu_postp import _field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('W', [510, 512, 514, 1030])
@pytest.mark.parametrize('radius', [1, 8])
def test_bloom_segments(gpu, W, radius):
    import torch
    import taichi_three_amd as tina
    H = 10
    print(f'case: bloom {W}x{H} radius {radius}', flush=True)
    rng = np.random.default_rng(W + radius)
    img = (rng.random((H, W, 3)) ** 3 * 4).astype(np.float32)
    bl = tina.Blooming((W, H))
    bl.radius = radius
    bl.init_gwei()
    wide = torch.full((H // 2 + 2, W // 2, 3), -7.0, dtype=torch.float32, device='cuda')
    bl.tmp = wide[1:-1]
    f = _field(img)
    bl.apply(f)
    torch.cuda.synchronize()
    assert (wide[0] == -7.0).all() and (wide[-1] == -7.0).all()
    want = postp.bloom(img, gwei=bl.gwei.cpu().numpy(), radius=radius)
    assert np.abs(f.storage.cpu().numpy() - want).max() <= 1e-6 * max(1.0, float(np.abs(want).max()))
