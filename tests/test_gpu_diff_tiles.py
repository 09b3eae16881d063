"""The tiled adjoint at the edges of its tables: screens that are no multiple of a
tile, a mesh so fine that a tile sees more vertices than its LDS table holds (the
rest goes straight to memory), more tiles than persistent workgroups."""
import numpy as np
import pytest

from test_gpu_diff import NAMES, _gpu_grads, _setup, _torch_reference_grads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('res,freq,crowded', [
    (16, 3, False),      # one tile
    (37, 60, False),     # every pixel its own face, tiles part-full
    (48, 120, True),     # a full tile of such pixels: 768 vertices
    (61, 20, False),     # ragged tiles, two or three pixels a face
    (791, 12, False),    # 2,500 tiles, large faces
])
def test_adjoint_tiles(gpu, res, freq, crowded):
    """Against plain PyTorch in float64 on the same ids, to the bound that the
    adjoint's other test holds (the binary32 weights of small faces lose digits)."""
    import torch
    print(f'case: dshade adjoint {res}x{res} icosphere({freq})', flush=True)
    d, ids, case, p, tp = _setup(res=res, freq=freq)
    tgt = np.random.default_rng(4).uniform(0, 1, (res, res, 3))
    g = _gpu_grads(d, tp, torch.from_numpy(tgt.astype(np.float32)).cuda())
    if crowded:
        tile = ids[16:32, 16:32]
        assert len(np.unique(case[5][tile[tile >= 0]])) > 512
    ref = _torch_reference_grads(case, ids, p, tgt)
    for name in NAMES:
        scale = np.abs(ref[name]).max()
        err = float(np.abs(g[name] - ref[name]).max())
        assert err <= 1e-3 * scale, (name, err, scale)
