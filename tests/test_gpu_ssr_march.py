"""The sliced, coarse-table SSR march at the edges of its tiling, for every fixed
material program and a walked one: screens that are no multiple of 8 or 16 pixels,
sample counts that four slices do not divide (fewer than four among them), odd step
counts, box sizes that are no power of two, a screen wide enough for 32-pixel
blocks in the coarse table."""
import numpy as np
import pytest

from oracle import orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('W,H,material,nsamples,nsteps,blur', [
    (97, 61, 'pbr', 5, 7, 4),
    (97, 61, 'diffuse', 1, 1, 3),
    (64, 48, 'classic', 32, 32, 4),
    (129, 95, 'blinn', 3, 33, 5),
    (121, 80, 'walked', 6, 12, 4),
    (2600, 820, 'pbr', 4, 8, 4),
])
def test_ssr_programs_and_edges(gpu, W, H, material, nsamples, nsteps, blur):
    """Up to one pixel in a thousand may land on the other side of a depth test
    (binary64 cos and sin differ between the host's and this library's series in
    the last bit before rounding); the others' sums differ by binary32 rounding."""
    import torch
    import taichi_three_amd as tina
    from taichi_three_amd.matr import lower_material
    from test_ssr_oracle import _grid
    print(f'case: ssr {W}x{H} {material} ns={nsamples} steps={nsteps} blur={blur}', flush=True)
    rng = np.random.default_rng(5)
    scene = tina.Scene(W, H, ssr=True, tonemap=False, maxfaces=4000)
    scene.engine.set_camera(tina.lookat([0, -0.2, 0], [0.2, 1.0, 3.0]), tina.perspective(50, W / H, 0.1, 30))
    fl, wa = tina.SimpleMesh(), tina.SimpleMesh()
    floor_v, wall_v = _grid((-3, -0.7, 2), (6, 0, 0), (0, 0, -5), 16), _grid((-3, -0.7, -1.5), (6, 0, 0), (0, 1.5, 0), 12)
    rough = rng.uniform(0.1, 0.9, len(floor_v)).astype(np.float32)
    fl.set_face_verts(floor_v)
    fl.set_face_attr('rough', rough)
    wa.set_face_verts(wall_v)
    mat = {'pbr': lambda: tina.PBR(basecolor=(0.6, 0.6, 0.7), metallic=0.7, roughness=tina.FaceAttr('rough')),
           'diffuse': lambda: tina.Diffuse(color=(0.8, 0.3, 0.2)),
           'classic': lambda: tina.Classic(color=(0.8, 0.3, 0.2), shineness=12),
           'blinn': lambda: tina.Blinn(color=(0.2, 0.3, 0.9), shineness=20, specular=0.7),
           'walked': lambda: tina.Diffuse(color=(0.8, 0.3, 0.2)) + tina.Phong(shineness=9)}[material]()
    wall = tina.Lamp(color=(0.9, 0.6, 0.3))
    scene.add_object(fl, mat)
    scene.add_object(wa, wall)
    ssr = scene.ssr
    ssr.nsamples, ssr.nsteps, ssr.blurring = nsamples, nsteps, blur
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
    for v, m, attrs in ((floor_v, mat, {'rough': rough}), (wall_v, wall, {})):
        hm = orc.HostMesh(v)
        hm.struct.id_base, hm.struct.nfaces = base, len(v)
        orc.ssr(W, H, cam, hm, lower_material(m, dict(attrs=attrs)).struct, depth, ids, norm, got['pre'],
                nsamples=nsamples, nsteps=nsteps, blur=blur, out=out)
        base += len(v)
    assert ((ids >= 0) & (ids < len(floor_v))).sum() > 0.1 * W * H
    if nsteps > 1:
        assert (out[..., 3] > 0).sum() > 50
    d = np.abs(got['buf'] - out).max(axis=2)
    print(f'max diff {d.max():.2e}, {int((d > 1e-5).sum())} pixels above 1e-5', flush=True)
    assert (d > 1e-5).sum() <= 1e-3 * W * H
