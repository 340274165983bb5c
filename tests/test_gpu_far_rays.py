"""Rays that start far outside the scene and graze turned solids, of one prim and of several,
where the single-precision quadric test reports hits on rays that pass the exact surface by
far more than from inside: the ray query and the propagation of photons from there give the
hits of the oracle's unculled loop in every tree and bound form, bit for bit."""
import numpy as np
import pytest

from oxr import abi, gensteps as G
from oxr.csg import Foundry, box3, cylinder, rotate_z_to, scale, sphere, translate

from test_gpu_parity import bits
from test_gpu_placed_boxes import SOLIDS

pytestmark = pytest.mark.gpu

# several prims to a solid, so that the solid's own tree is walked in its frame
GROUPS = {'pair': [lambda: sphere(50.0), lambda: box3(30.0).moved(translate(0.0, 0.0, 120.0))],
          'row': [lambda k=k: sphere(20.0 + k).moved(scale(1.0, 1.5, 0.7)).moved(translate(90.0 * k, 0.0, 0.0)) for k in range(5)] +
                 [lambda: cylinder(15.0, -200.0, 200.0).moved(translate(0.0, 150.0, 0.0))]}
FORMS = [dict(bvh_mode=b, bvh_radial=r) for b in (0, 1) for r in (0, 1)]


def scene(name, rng, turned=True):
    """24 copies of one solid within 2.5 m of the origin and nothing around them."""
    makes, r = (GROUPS[name], 50.0) if name in GROUPS else ([SOLIDS[name][0]], SOLIDS[name][1])
    f = Foundry()
    f.add_material('Air', 1.0)
    f.add_material('Glass', 1.5)
    f.begin_solid('r0')
    for make in makes:
        f.add_prim(make(), f.boundary('Air', None, None, 'Glass'))
    f.end_solid()
    centres = rng.uniform(-2500.0, 2500.0, size=(24, 3))
    for c in centres:
        f.add_instance((rotate_z_to(rng.normal(size=3)) if turned else np.eye(4)) @ translate(*c), 0)
    return f.arrays(), f.physics(), centres, r


def grazing(rng, n, centres, r, away):
    """Origins at the given distances from the solids, directions that pass their axes at up
    to a few times what the quadric test's rounding reaches from there."""
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    side = np.cross(d, rng.normal(size=(n, 3)))
    side /= np.linalg.norm(side, axis=1)[:, None]
    dist = away * rng.uniform(0.5, 1.0, size=n)
    off = np.sqrt(np.maximum(r * r + rng.uniform(-0.05, 1.0, size=n) * 4e-7 * dist * dist, 0.0))
    return (centres[rng.integers(0, len(centres), size=n)] + off[:, None] * side - dist[:, None] * d), d


@pytest.mark.parametrize('away', [3e4, 2e5, 1e6])
@pytest.mark.parametrize('name', sorted(SOLIDS) + ['pair', 'row', 'pair unturned'])
def test_far_rays(engine_mod, oracle_lib, name, away):
    rng = np.random.default_rng(len(name) + int(away))
    g, p, centres, r = scene(name.split()[0], rng, turned='unturned' not in name)
    n = 40_000
    rays = np.zeros((n, 2, 4), dtype=np.float32)
    rays[:, 0, :3], rays[:, 1, :3] = grazing(rng, n, centres, r, away)
    rays[:, 0, 3], rays[:, 1, 3] = 0.05, 1e9
    cfg = abi.default_config()
    print('far rays', name, away, flush=True)
    want = oracle_lib.Oracle(g, p, cfg).trace(rays)
    assert (bits(want)[:, 1, 2] != 0xffffffff).mean() > 0.005
    with engine_mod.Engine(g, p, cfg) as e:
        for form in FORMS:
            e.set_tuning(**form)
            got = e.trace(rays)
            bad = (bits(got) != bits(want)).any(axis=(1, 2))
            assert not bad.any(), (name, away, form, int(bad.sum()))


@pytest.mark.parametrize('name', ['ball', 'bulb', 'rod', 'pair', 'row'])
def test_far_photons(engine_mod, oracle_lib, name):
    rng = np.random.default_rng(len(name))
    g, p, centres, r = scene(name, rng)
    n = 20_000
    photons = np.zeros((n, 4, 4), dtype=np.float32)
    photons[:, 0, :3], d = grazing(rng, n, centres, r, 2e5)
    photons[:, 1, :3] = d
    pol = np.cross(d, rng.normal(size=(n, 3)))
    photons[:, 2, :3] = pol / np.linalg.norm(pol, axis=1)[:, None]
    photons[:, 2, 3] = 440.0
    cfg = abi.default_config(max_bounce=4, tmax=1e9)
    gs = G.input_photon(n)
    print('far photons', name, flush=True)
    want = oracle_lib.Oracle(g, p, cfg).simulate(gs, input_photons=photons, seq=False)['photon']
    with engine_mod.Engine(g, p, cfg) as e:
        e.set_input_photons(photons)
        e.set_gensteps(gs)
        for form in FORMS:
            e.set_tuning(**form)
            for kind in (abi.OXR_FORM_PLAIN, abi.OXR_FORM_PERSISTENT):
                e.launch(kind)
                got = e.photons()
                bad = (got.view(np.uint32) != want.view(np.uint32)).reshape(n, -1).any(axis=1)
                assert not bad.any(), (name, form, kind, int(bad.sum()))
