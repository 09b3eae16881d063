"""The sliced prefilter bake at the edges of its tiling: texel counts around the
workgroup's texels and below, sample counts around a chunk of 512, maps whose
level takes 1 to 64 texels a workgroup."""
import numpy as np
import pytest

from oracle import orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('ow,oh,nsamples,roughness', [
    (2, 2, 1, 0.5),          # four texels: one a workgroup, one sample
    (3, 5, 511, -1.0),       # odd map, one short chunk
    (31, 15, 512, 0.08),     # 465 texels (two a workgroup), exactly one chunk
    (37, 19, 513, 1.0),      # a chunk and one sample
    (84, 42, 1025, -1.0),    # 3,528 texels (sixteen), two chunks and one sample
    (150, 76, 40, 0.18),     # 11,400 texels, the last workgroup part-full
    (259, 129, 7, 0.03),     # 33,411 texels (64), fewer samples than slices
])
def test_bake_tiling(gpu, ow, oh, nsamples, roughness):
    """Both sides are binary64 and differ by the order of the sum and libm rounding
    (about 1e-13 relative), far below one rounding of the float32 store (6e-8)."""
    import torch
    from taichi_three_amd.skybox import procedural_sky, bake_level
    print(f'case: {ow}x{oh} n={nsamples} r={roughness}', flush=True)
    env = procedural_sky(97, 51)
    out = torch.full((ow * oh + 64, 3), -7.0, dtype=torch.float32, device='cuda')
    bake_level(torch.from_numpy(env).cuda(), 97, 51, out, ow, oh, roughness, nsamples)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert (got[ow * oh:] == -7.0).all()
    ref = orc.bake_lambert(env, ow, oh, nsamples) if roughness < 0 else \
        orc.bake_ggx(env, ow, oh, np.float32(roughness), nsamples)
    assert np.allclose(got[:ow * oh].reshape(ow, oh, 3), ref, rtol=2e-7, atol=1e-9)
