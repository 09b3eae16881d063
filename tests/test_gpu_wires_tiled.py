"""Wire calls by tile (65,536 wires and more, twice that on small screens), depth and ids bit for bit against the
oracle: just below and at the count, long and short wires mixed so that a call takes
both ways, screens that are no multiple of a tile, more wires than the scratch holds
at a time, entries that do not fit (those groups are drawn), wires with no length,
of 10^7 pixels and in front of the near plane among them, and a second call into the
keys of the first."""
import numpy as np
import pytest

from oracle import orc
from test_gpu_wires import _camera, _oracle, _wires

pytestmark = pytest.mark.gpu


def _draw(W, H, wires, clip=False):
    import torch
    import taichi_three_amd as tina
    scene = tina.Scene(W, H, maxfaces=1, maxwires=len(wires), clipping=clip)
    mesh = tina.SimpleMesh(len(wires), npolygon=2)
    mesh.set_face_verts(wires)
    scene.add_object(mesh)
    scene.set_camera(*_camera(W, H))
    scene.render()
    torch.cuda.synchronize()
    return scene, scene.engine.ids.to_numpy().T, scene.engine.depth.to_numpy().T


@pytest.mark.parametrize('W,H,n,reach,clip', [
    (1001, 667, 65531, 0.3, False),    # 65,536 with the five extremes: ragged tiles, long wires
    (1001, 667, 65530, 0.3, False),    # one fewer: drawn into memory
    (1200, 450, 70000, 0.004, True),   # about a pixel each: every group draws
    (97, 61, 262300, 1.2, False),      # more than the 262,144 that go at a time
    (16384, 3, 131067, 1.2, False),    # the small screen's count; 512 tiles in a row: more entries than there is room for
])
def test_tiled_wires_bit_exact(gpu, W, H, n, reach, clip):
    print(f'case: {n} wires {W}x{H} reach {reach} clip={clip}', flush=True)
    rng = np.random.default_rng(8)
    wires = _wires(n, 3, W, H)
    if reach < 1.2:
        wires[:n, 1] = wires[:n, 0] + rng.uniform(-reach, reach, (n, 3)).astype(np.float32)
        wires[:n:7, 1] = rng.uniform(-1.2, 1.2, wires[:n:7, 1].shape) if reach > 0.1 else wires[:n:7, 1]
    scene, ids, depth = _draw(W, H, wires, clip)
    odepth, oid = _oracle(scene, wires, 2 if clip else 0)[:2]
    assert np.array_equal(ids, oid), f'{(ids != oid).sum()} ids differ'
    assert np.array_equal(depth, odepth)


def test_two_tiled_calls_share_the_keys(gpu):
    """Two wire objects of 66,000 and 70,000: half their groups short, half long."""
    import torch
    import taichi_three_amd as tina
    W, H = 1000, 700
    print('case: two tiled wire objects 1000x700', flush=True)
    rng = np.random.default_rng(9)
    sets = []
    for k, n in enumerate((66000, 70000)):
        w = _wires(n, 20 + k, W, H, extreme=False)
        w[:n // 2, 1] = w[:n // 2, 0] + rng.uniform(-0.02, 0.02, (n // 2, 3)).astype(np.float32)
        sets.append(w)
    scene = tina.Scene(W, H, maxfaces=1)
    for w in sets:
        mesh = tina.SimpleMesh(len(w), npolygon=2)
        mesh.set_face_verts(w)
        scene.add_object(mesh)
    scene.set_camera(*_camera(W, H))
    for _ in range(2):
        scene.render()
    torch.cuda.synchronize()
    d, o = _oracle(scene, sets[0], 0)[:2]
    d, o = _oracle(scene, sets[1], 0, id_base=66000, depth=d, occ=o)[:2]
    assert np.array_equal(scene.engine.ids.to_numpy().T, o)
    assert np.array_equal(scene.engine.depth.to_numpy().T, d)
