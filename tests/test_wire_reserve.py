"""The wire raster asks for the scratch of its largest call when it is made and never
in a frame (no GPU: the engine is a recorder)."""
import numpy as np
import pytest


class _Engine:
    def __init__(self):
        self.res, self._id_cursor, self.reserved = np.array([640, 360]), 0, []

    def reserve_wires(self, n):
        self.reserved.append(n)


class _Wires:
    def __init__(self, n):
        import torch
        self.fb = dict(nfaces=n, verts=torch.zeros((n, 2, 3)))

    def get_npolygon(self):
        return 2

    def face_buffers(self):
        return self.fb


@pytest.mark.parametrize('maxwires,counts', [(70000, (10, 70000, 65536)), (100, (100, 1))])
def test_scratch_is_asked_for_once_and_outside_the_frame(maxwires, counts):
    from taichi_three_amd.wireframe import WireframeRaster
    eng = _Engine()
    raster = WireframeRaster(eng, maxwires=maxwires)
    assert eng.reserved == [maxwires]
    for n in counts:                       # what Scene.render does with an object each frame
        raster.set_object(_Wires(n))
        assert raster.nfaces == n
    assert eng.reserved == [maxwires]
