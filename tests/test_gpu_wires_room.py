"""One wire launch of more groups than units (300,000 wires), a scratch that grows when
a raster for more wires joins the engine, and a call of more wires than were reserved,
depth and ids bit for bit against the oracle."""
import numpy as np
import pytest

from test_gpu_wires import _camera, _oracle, _wires

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('reserved', [(300005,), (70000, 300005), (70000,)])
def test_many_groups_and_a_growing_scratch(gpu, reserved):
    import torch
    import taichi_three_amd as tina
    from taichi_three_amd.wireframe import WireframeRaster
    W, H, n = 800, 700, 300000
    print(f'case: {n} + 5 wires {W}x{H}, scratch for {reserved}', flush=True)
    wires = _wires(n, 12, W, H)
    wires[:n:2, 1] = wires[:n:2, 0] + np.float32(0.01)
    scene = tina.Scene(W, H, maxfaces=1)
    for k in reserved[:-1]:
        WireframeRaster(scene.engine, maxwires=k)
    raster = WireframeRaster(scene.engine, maxwires=n + 5)
    if reserved == (70000,):               # the scratch of another raster, made for fewer
        scene = tina.Scene(W, H, maxfaces=1)
        scene.engine.reserve_wires(70000)
        scene.engine.reserve_wires, keep = (lambda k: None), scene.engine.reserve_wires
        raster = WireframeRaster(scene.engine, maxwires=n + 5)
        scene.engine.reserve_wires = keep
    mesh = tina.SimpleMesh(n + 5, npolygon=2)
    mesh.set_face_verts(wires)
    scene.add_object(mesh, raster=raster)
    scene.set_camera(*_camera(W, H))
    for _ in range(2):
        scene.render()
    torch.cuda.synchronize()
    depth, oid = _oracle(scene, wires, 0)[:2]
    assert np.array_equal(scene.engine.ids.to_numpy().T, oid)
    assert np.array_equal(scene.engine.depth.to_numpy().T, depth)
