"""SSR over every size of block in the coarse depth table (16, 32 and 64 pixels) and with
a single sample, which every fixed program traces in one slice, against the oracle."""
import numpy as np
import pytest

from oracle import orc

pytestmark = pytest.mark.gpu

MOST_BLOCKS = 2048                         # words of the table a workgroup keeps


@pytest.mark.parametrize('W,H,block,material,nsamples,nsteps', [
    (640, 360, 16, 'pbr', 4, 12),
    (1279, 721, 32, 'pbr', 4, 12),
    (1920, 1080, 32, 'diffuse', 2, 10),
    (2600, 820, 64, 'classic', 4, 12),
    (131, 75, 16, 'pbr', 1, 12),
    (131, 75, 16, 'diffuse', 1, 12),
    (131, 75, 16, 'classic', 1, 13),
    (131, 75, 16, 'blinn', 1, 12),
])
def test_ssr_tables(gpu, W, H, block, material, nsamples, nsteps):
    """Both sides trace the same binary32 rays; only their binary64 cosines, sines and
    powers may differ in the last place, which moves one binary32 value in some 10^8.
    At most one pixel in ten thousand of those that meet a surface may differ."""
    import torch
    import taichi_three_amd as tina
    from taichi_three_amd.matr import lower_material
    from test_ssr_oracle import _grid
    print(f'case: ssr tables {W}x{H} {material} ns={nsamples} steps={nsteps}', flush=True)
    size = 16
    while -(-W // size) * -(-H // size) > MOST_BLOCKS:
        size *= 2
    assert size == block
    scene = tina.Scene(W, H, ssr=True, tonemap=False, maxfaces=4000)
    scene.engine.set_camera(tina.lookat([0, -0.2, 0], [0.2, 1.0, 3.0]), tina.perspective(50, W / H, 0.1, 30))
    # a floor in front of a wall, with posts of several depths standing on it
    floor_v = _grid((-4, -0.7, 2), (8, 0, 0), (0, 0, -5), 16)
    wall_v = np.concatenate([_grid((-4, -0.7, -1.5), (8, 0, 0), (0, 2.2, 0), 12)] +
                            [_grid((-2.2 + 0.55 * k, -0.7, -1.2 + 0.3 * (k % 4)), (0.12, 0, 0), (0, 0.9, 0), 2)
                             for k in range(9)])
    mat = {'pbr': lambda: tina.PBR(basecolor=(0.6, 0.6, 0.7), metallic=0.7, roughness=0.3),
           'diffuse': lambda: tina.Diffuse(color=(0.8, 0.3, 0.2)),
           'classic': lambda: tina.Classic(color=(0.8, 0.3, 0.2), shineness=40),
           'blinn': lambda: tina.Blinn(color=(0.2, 0.3, 0.9), shineness=40, specular=0.7)}[material]()
    wall = tina.Lamp(color=(0.9, 0.6, 0.3))
    sets = ((floor_v, mat), (wall_v, wall))
    for v, m in sets:
        mesh = tina.SimpleMesh()
        mesh.set_face_verts(v)
        scene.add_object(mesh, m)
    ssr = scene.ssr
    ssr.nsamples, ssr.nsteps = nsamples, nsteps
    got, apply = {}, ssr.apply

    def wrapped(image):
        got['pre'], got['buf'] = image.storage.cpu().numpy().copy(), ssr.img.cpu().numpy().copy()
        apply(image)
    ssr.apply = wrapped
    scene.render()
    torch.cuda.synchronize()
    ids, depth = scene.engine.ids.to_numpy().T.copy(), scene.engine.depth.to_numpy().T.copy()
    norm = scene.norm_buffer.storage.cpu().numpy()
    cam = orc.camera(scene.engine.W2V, scene.engine.V2W)
    out, base = np.zeros((H, W, 4), np.float32), 0
    for v, m in sets:
        hm = orc.HostMesh(v)
        hm.struct.id_base, hm.struct.nfaces = base, len(v)
        orc.ssr(W, H, cam, hm, lower_material(m, dict(attrs={})).struct, depth, ids, norm, got['pre'],
                nsamples=nsamples, nsteps=nsteps, blur=ssr.blurring, out=out)
        base += len(v)
    hits = int((out[..., 3] > 0).sum())
    d = np.abs(got['buf'] - out).max(axis=2)
    print(f'{hits} pixels with hits, max diff {d.max():.2e}, {int((d > 1e-5).sum())} above 1e-5', flush=True)
    assert hits > 0.02 * W * H
    assert (d > 1e-5).sum() <= 1e-4 * hits
