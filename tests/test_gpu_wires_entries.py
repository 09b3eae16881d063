"""Wire calls by tile with more entries than there is room for: groups that find none
left are drawn, the others listed; and a screen of 3840 x 2160, whose wires have room
for twice as many entries as those of 1920 x 1080.  Depth and ids bit for bit against
the oracle."""
import numpy as np
import pytest

from test_gpu_wires import _camera, _oracle

pytestmark = pytest.mark.gpu


def _across(W, H, n, seed):
    """Wires from the left edge of the screen to the right one."""
    from taichi_three_amd.util.matrix import camera_matrices
    rng = np.random.default_rng(seed)
    ndc = np.ones((n, 2, 4))
    ndc[:, 0, 0], ndc[:, 1, 0] = -0.99, 0.99
    ndc[:, :, 1] = rng.uniform(-0.99, 0.99, (n, 2))
    ndc[:, :, 2] = rng.uniform(0.3, 0.99, (n, 2))
    h = ndc @ np.float64(camera_matrices(*_camera(W, H))[1]).T
    return (h[..., :3] / h[..., 3:]).astype(np.float32)


@pytest.mark.parametrize('W,H,n,fits', [(1200, 800, 200000, False), (3840, 2160, 66000, True)])
def test_entries_and_their_room(gpu, W, H, n, fits):
    import torch
    import taichi_three_amd as tina
    print(f'case: {n} wires across {W}x{H}', flush=True)
    wires = _across(W, H, n, 7)
    # a wire crosses every tile column, and a row whenever it changes it; 262,144 wires
    # have room for a quarter of the tile columns and rows each, 24 at least
    tx, ty = -(-W // 32), -(-H // 32)
    rows = np.abs(np.diff(np.clip(_rows(W, H, wires) // 32, 0, ty - 1), axis=1))
    entries, room = n * tx + int(rows.sum()), 262144 * max(24, (tx + ty) // 4)
    assert (1.02 * entries < room) if fits else (0.9 * entries > room)
    scene = tina.Scene(W, H, maxfaces=1, maxwires=n)
    mesh = tina.SimpleMesh(n, npolygon=2)
    mesh.set_face_verts(wires)
    scene.add_object(mesh)
    scene.set_camera(*_camera(W, H))
    for _ in range(2):
        scene.render()
    torch.cuda.synchronize()
    depth, oid = _oracle(scene, wires, 0)[:2]
    assert np.array_equal(scene.engine.ids.to_numpy().T, oid)
    assert np.array_equal(scene.engine.depth.to_numpy().T, depth)


def _rows(W, H, wires):
    from taichi_three_amd.util.matrix import camera_matrices
    h = np.concatenate([wires, np.ones_like(wires[..., :1])], -1) @ np.float64(camera_matrices(*_camera(W, H))[0]).T
    return ((h[..., 1] / h[..., 3]) * 0.5 + 0.5) * H
