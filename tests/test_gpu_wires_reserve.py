"""Wire calls by tile from the first frame on, where that frame is a captured one: the
scratch is there once the object is added, no frame allocates device memory, and the
graph's replays equal the oracle with eager frames between them."""
import numpy as np
import pytest

from test_gpu_wires import _camera, _oracle, _wires

pytestmark = pytest.mark.gpu


def test_first_frame_captured(gpu):
    import torch
    import taichi_three_amd as tina
    W, H, n = 1200, 800, 70000
    print(f'case: captured first frame, {n} wires {W}x{H}', flush=True)
    wires = _wires(n, 6, W, H, extreme=False)
    mesh = tina.SimpleMesh(n, npolygon=2)
    mesh.set_face_verts(wires)

    def make():
        s = tina.Scene(W, H, maxfaces=1, maxwires=n)
        s.set_camera(*_camera(W, H))
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        s.add_object(mesh)
        assert before - torch.cuda.mem_get_info()[0] > 30e6  # 262,144 wires' records and lists
        return s
    make().render()                        # the kernels are loaded
    scene = make()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        scene.render()
    depth, oid = _oracle(scene, wires, 0)[:2]
    keys = scene.engine.keys()
    for k in range(3):
        keys.fill_(k)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(scene.engine.ids.to_numpy().T, oid), k
        assert np.array_equal(scene.engine.depth.to_numpy().T, depth), k
        keys.fill_(k)
        scene.render()
        torch.cuda.synchronize()
        assert np.array_equal(scene.engine.ids.to_numpy().T, oid), k
