"""How a wire call of 65,536 and more chooses between drawing and listing by tile: frames
of one scene that list, draw and list again (what a call leaves for the next), groups
unlike the sample by which the others decide, and a count that leaves no lanes for the
sample; depth and ids bit for bit against the oracle."""
import numpy as np
import pytest

from test_gpu_wires import _camera, _oracle, _wires

pytestmark = pytest.mark.gpu


def _scene(W, H, n):
    import taichi_three_amd as tina
    scene = tina.Scene(W, H, maxfaces=1, maxwires=n)
    mesh = tina.SimpleMesh(n, npolygon=2)
    scene.set_camera(*_camera(W, H))
    return scene, mesh


def _check(scene, wires, what):
    import torch
    torch.cuda.synchronize()
    depth, oid = _oracle(scene, wires, 0)[:2]
    ids = scene.engine.ids.to_numpy().T
    assert np.array_equal(ids, oid), (what, int((ids != oid).sum()))
    assert np.array_equal(scene.engine.depth.to_numpy().T, depth), what


def test_long_and_short_frames_in_turn(gpu):
    W, H, n = 1100, 520, 70000
    print(f'case: {n} wires {W}x{H}, long, short, long, short, long', flush=True)
    scene, mesh = _scene(W, H, n)
    long = _wires(n, 31, W, H, extreme=False)
    short = _wires(n, 32, W, H, extreme=False)
    short[:, 1] = short[:, 0] + np.random.default_rng(1).uniform(-0.01, 0.01, (n, 3)).astype(np.float32)
    added = False
    for k, wires in enumerate((long, short, long, short, long)):
        mesh.set_face_verts(wires)
        if not added:
            scene.add_object(mesh)
            added = True
        scene.render()
        _check(scene, wires, k)


@pytest.mark.parametrize('n', [66000, 131072, 250000])
@pytest.mark.parametrize('part', [0.1, 0.5])
def test_groups_unlike_the_sample(gpu, n, part):
    """Runs of long wires among short ones, at the front and at the end of the call."""
    W, H = 1000, 560
    print(f'case: {n} wires {W}x{H}, {part} of them long', flush=True)
    scene, mesh = _scene(W, H, n)
    rng = np.random.default_rng(n)
    wires = _wires(n, 33, W, H, extreme=False)
    k = int(n * part / 2)
    wires[k:n - k, 1] = wires[k:n - k, 0] + rng.uniform(-0.004, 0.004, (n - 2 * k, 3)).astype(np.float32)
    mesh.set_face_verts(wires)
    scene.add_object(mesh)
    scene.render()
    _check(scene, wires, part)
