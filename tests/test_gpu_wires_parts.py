"""Wire calls drawn into memory: several waves share 64 wires and walk a part of their
steps each.  One wire, a whole and a broken last 64, every number of waves to a share
(64 down to four), wires of no length and of 10^7 pixels among them; depth and ids bit
for bit against the oracle."""
import numpy as np
import pytest

from test_gpu_wires import _camera, _oracle, _wires

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('W,H,n', [(640, 360, 1), (640, 360, 59), (333, 217, 60), (640, 360, 4092), (641, 359, 5000),
                                   (500, 300, 12000), (500, 300, 40000), (320, 200, 130000)])
def test_shared_wires_bit_exact(gpu, W, H, n):
    import torch
    import taichi_three_amd as tina
    print(f'case: {n} + 5 wires {W}x{H}', flush=True)
    wires = _wires(n, n, W, H)
    scene = tina.Scene(W, H, maxfaces=1, maxwires=len(wires))
    mesh = tina.SimpleMesh(len(wires), npolygon=2)
    mesh.set_face_verts(wires)
    scene.add_object(mesh)
    scene.set_camera(*_camera(W, H))
    scene.render()
    torch.cuda.synchronize()
    depth, oid = _oracle(scene, wires, 0)[:2]
    assert np.array_equal(scene.engine.ids.to_numpy().T, oid)
    assert np.array_equal(scene.engine.depth.to_numpy().T, depth)
