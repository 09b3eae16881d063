"""Particle sets under each material program that has a kernel of its own, and under
a composed one, with lights and with a sky: coverage, ids and the tone-mapped colour
against the binary32 oracle (1e-5, the bound of the other particle tests), an odd
screen whose last chunk of pixels is partial."""
import numpy as np
import pytest

from oracle import orc
from test_gpu_particles import _camera, _check_colour, _cloud, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('name,sky', [('diffuse', False), ('classic', False), ('blinn', False), ('pbr', False),
                                      ('composed', False), ('diffuse', True), ('pbr', True), ('composed', True)])
def test_particle_programs(gpu, name, sky):
    import taichi_three_amd as tina
    from taichi_three_amd import _abi
    from taichi_three_amd.matr import lower_material
    W, H, n = 333, 217, 4000
    print(f'case: particles {W}x{H} n={n} {name} sky={sky}', flush=True)
    material = {'diffuse': tina.Diffuse, 'classic': tina.Classic, 'blinn': tina.Blinn,
                'pbr': lambda: tina.PBR(roughness=0.35, metallic=0.2),
                'composed': lambda: tina.ScaleMaterial(tina.PBR(roughness=0.5, metallic=0.7), 0.75)}[name]()
    opts = dict(ibl=True, skybox=tina.Skybox.procedural(128, 64), ibl_precision=2) if sky else {}
    pos, rad, col = _cloud(n, 5)
    scene = tina.Scene(W, H, maxpars=n, **opts)
    pars = tina.SimpleParticles(n)
    pars.set_particles(pos)
    pars.set_particle_radii(rad)
    pars.set_particle_colors(col)
    scene.add_object(pars, material)
    scene.set_camera(*_camera(W, H))
    scene.lighting.clear_lights()
    scene.lighting.add_light(dir=(0.3, 0.5, 0.8), color=(1.5, 1.2, 1.0))
    scene.lighting.add_light(pos=(1.0, -2.0, 2.0), color=(2.0, 3.0, 2.5))
    ids, depth, img = _run(scene)
    eng = scene.engine
    cam = orc.camera(eng.W2V, eng.V2W, eng.bias)
    od, oi = orc.raster_particles(W, H, cam, pos, rad, flags=_abi.CLIP)
    assert np.array_equal(ids, oi) and np.array_equal(depth, od)
    ibl, keep = scene.lighting.ibltab.host_copy() if sky else (None, None)
    flags = _abi.PARTICLES | _abi.VCOLOR | _abi.BG | _abi.TONEMAP | (_abi.IBL if sky else 0)
    o32 = orc.shade(W, H, cam, orc.particle_mesh(pos, rad, col), lower_material(material, dict(attrs={})).struct,
                    scene.lighting.to_struct(), oi, flags, ibl=ibl)
    assert (oi >= 0).sum() > 0.2 * W * H
    _check_colour(img, o32)
