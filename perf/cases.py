"""The calls that users of the engine make, as timed cases: each through the public entry
points of ``oxr`` (``Engine.simulate``, ``launch`` with its gathers, the serving loop, the
geometry queries), over the sizes, forms, precisions and outputs in use.

A program builds one engine for its detector and keeps it; what changes from event to event
is the gensteps (or input photons, rays), which is what ``prepare`` makes from the seed. So
the engines (geometry, tuning, serving loop) are made once per configuration and shared by
the states of a case.

Hits come back in a buffer that the program keeps for them, with their number; rows that no
hit of the event fills stay zero.

Photon, hit and history arrays mix floats with packed integers word by word, and every bit
of them is fixed by the inputs; they are returned as their 32-bit words. Ray queries return
their distances and normals as floats.
"""
import ctypes
import json
import math
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, 'eic-opticks_amd')
if PKG not in sys.path:
    sys.path.insert(0, PKG)

from oxr import abi, gdml, gensteps as G, scenes  # noqa: E402
from oxr.engine import Engine, Server, lib  # noqa: E402

PERSISTENT, PLAIN = 'persistent', 'plain'


def listed():
    return [
        # a photon text file's ten photons through the C++ example's path: pure latency
        dict(name='photon_file_10', kind='photon_file', photons=10),
        # the quick-start geometry with the engine's defaults (plain form, default tuning)
        dict(name='boxes_100k', kind='photons', scene='nested_boxes', photons=100_000, form=PLAIN, tuned=False),
        # a whole shower in the crystal calorimeter: scintillation and Cerenkov gensteps, few
        # hits, long diffuse-reflection histories; the production setting
        dict(name='calorimeter_2m', kind='hits', scene='csi_calorimeter', photons=2_075_000, form=PERSISTENT, tuned=True),
        # a small shower in the same detector before anything is tuned
        dict(name='calorimeter_60k', kind='hits', scene='csi_calorimeter', photons=62_250, form=PLAIN, tuned=False),
        # the benchmark's event: 10M photons among 20,000 instanced CSG solids
        dict(name='instanced_10m', kind='hits', scene='instanced_csg', photons=10_000_000, form=PERSISTENT, tuned=True),
        # one event of median serving size, its hits merged per sensor and nanosecond
        dict(name='instanced_merged_200k', kind='merged', scene='instanced_csg', photons=200_003, form=PERSISTENT, tuned=True),
        # concentric thin shells, every photon's end point gathered
        dict(name='shells_500k', kind='photons', scene='thin_shells', photons=500_000, form=PERSISTENT, tuned=True),
        # the same with double-precision roots, as precision studies run it
        dict(name='shells_fp64_150k', kind='photons', scene='thin_shells', photons=150_001, form=PERSISTENT, tuned=True, fp64=True),
        # an imported detector: polyhedra, cones and boolean solids, default tuning
        dict(name='pfrich_300k', kind='photons', scene='pfrich', photons=300_000, form=PERSISTENT, tuned=False),
        # histories for debugging: end points, step sequences and records of a re-emitting
        # scintillator
        dict(name='history_40k', kind='history', scene='scintillator_sphere', photons=40_000, form=PLAIN, tuned=False),
        # the serving loop with events of mixed size submitted at once
        dict(name='serving_24', kind='serving', scene='instanced_csg', events=24, tuned=True),
        # a closest-hit query for a batch of rays
        dict(name='rays_250k', kind='rays', scene='scintillator_sphere', rays=250_000, tuned=False),
    ]


# photons a drawn event may have: (fewest, most)
DRAWN = {'nested_boxes': (1_000, 500_000), 'csi_calorimeter': (2_000, 2_000_000), 'instanced_csg': (1_000, 8_000_000),
         'thin_shells': (1_000, 500_000), 'pfrich': (1_000, 500_000)}


def log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['hits', 'hits', 'hits', 'photons', 'photons', 'merged', 'photon_file', 'history', 'serving', 'rays'])
    if kind == 'photon_file':
        return dict(kind=kind, photons=log_size(rng, 1, 5_000))
    if kind == 'history':
        return dict(kind=kind, scene='scintillator_sphere', photons=log_size(rng, 500, 50_000),
                    form=rng.choice([PLAIN, PERSISTENT]), tuned=False)
    if kind == 'serving':
        return dict(kind=kind, scene='instanced_csg', events=rng.randint(3, 24), tuned=True)
    if kind == 'rays':
        return dict(kind=kind, scene='scintillator_sphere', rays=log_size(rng, 1_000, 500_000), tuned=False)
    scene = rng.choice({'hits': ['csi_calorimeter', 'instanced_csg'], 'photons': ['nested_boxes', 'thin_shells', 'pfrich'],
                        'merged': ['instanced_csg', 'csi_calorimeter']}[kind])
    case = dict(kind=kind, scene=scene, photons=log_size(rng, *DRAWN[scene]), form=rng.choice([PLAIN, PERSISTENT, PERSISTENT]),
                tuned=scene != 'pfrich' and rng.random() < 0.7)
    if scene == 'thin_shells':
        case['fp64'] = rng.random() < 0.3
        if case['fp64']:
            case['photons'] = case['photons'] * 3 // 10 + 1
    return case


# ---------------------------------------------------------------------------
_scenes, _engines, _servers = {}, {}, {}


def scene_of(name):
    if name not in _scenes:
        if name == 'pfrich':
            _scenes[name] = gdml.load_gdml(os.path.join(ROOT, 'tests', 'golden', 'geom', 'pfrich_min_FINAL.gdml'))
        elif name == 'scintillator_sphere':
            _scenes[name] = scenes.scintillator_sphere()
        else:
            _scenes[name] = scenes.SCENES[name]()
    return _scenes[name]


def tuning_of(name):
    """The package's measured launch settings for a detector, as a program loads them."""
    with open(os.path.join(PKG, 'oxr', 'tuning_gfx950.json')) as f:
        return json.load(f)[name]


def engine_of(case):
    name = case.get('scene', 'raindrop')
    history = case['kind'] == 'history'
    fp64 = bool(case.get('fp64', False))
    tuned = bool(case.get('tuned', False))
    key = (name, history, fp64, tuned, case['kind'] == 'serving')
    if key not in _engines:
        s = scene_of(name)
        cfg = dict(max_bounce=32) if name == 'pfrich' else dict(s.config)
        if fp64:
            cfg['fp64_roots'] = 1
        if history:
            cfg.update(seq_enabled=1, max_record=10)
        e = Engine(s.geometry, s.physics, abi.default_config(**cfg))
        if tuned:
            e.set_tuning(**tuning_of(name))
        _engines[key] = e
    return _engines[key]


def gensteps_of(name, photons, seed):
    """An event of the scene's own source with exactly this many photons (the calorimeter's
    shower has Poisson counts about it)."""
    rng = np.random.default_rng(seed)
    s = scene_of(name)
    if name == 'csi_calorimeter':
        return s.gensteps(seed=seed, scale_photons=photons / 2_075_000)
    if name == 'pfrich':
        n = max(1, min(16, photons // 1000))
        return exactly(G.torch(np.full(n, photons // n), pos=rng.uniform(-60.0, 60.0, size=(n, 3)), wavelength=400.0,
                               type=G.T_POINT_ISOTROPIC), photons)
    if name == 'instanced_csg':
        return exactly(s.gensteps(seed=seed, scale_photons=photons / 10_000_000), photons)
    if name == 'thin_shells':   # one source at the centre: an event differs by its random streams
        return G.torch(photons, pos=(0.0, 0.0, 0.0), wavelength=400.0, type=G.T_POINT_ISOTROPIC)
    n = max(1, min(32, photons // 500))
    r, wavelength = {'nested_boxes': (45.0, 420.0), 'scintillator_sphere': (300.0, 350.0)}[name]
    return exactly(G.torch(np.full(n, photons // n), pos=rng.uniform(-r, r, size=(n, 3)), wavelength=wavelength,
                           type=G.T_POINT_ISOTROPIC), photons)


def exactly(gs, photons):
    """gs with its photons spread over the gensteps so that they add up to the number."""
    n = gs.view(np.uint32)[:, 0, 3]
    n[:] = photons // len(gs)
    n[:photons - int(n.sum())] += 1
    return gs


def form_of(case):
    return abi.OXR_FORM_PLAIN if case.get('form') == PLAIN else abi.OXR_FORM_PERSISTENT


# hits a program leaves room for, per photon of the event
ROOM = {'instanced_csg': 0.4, 'csi_calorimeter': 0.05}


def room_for(name, photons):
    return np.zeros((int(photons * ROOM[name]) + 64, 4, 4), dtype=np.float32)


def serving_events(n, seed):
    """Events of the serving stream: the photon numbers of its log-normal (median 200,000,
    at most a million), the same for every seed, from origins of the seed's."""
    rng = np.random.default_rng(seed)
    _, counts, _ = scenes.serving_stream(np.random.default_rng(n), n_events=n, hi=1_000_000)
    evs = []
    for c in counts.tolist():
        k = max(1, min(64, c // 20_000))
        evs.append(exactly(G.torch(np.full(k, c // k), pos=rng.uniform(-9_000.0, 9_000.0, size=(k, 3)), wavelength=430.0,
                                   type=G.T_POINT_ISOTROPIC), c))
    return evs


def rays_of(n, seed):
    """Start points through the 1200 mm world sphere of scintillator_sphere, isotropic directions."""
    rng = np.random.default_rng(seed)
    rays = np.zeros((n, 2, 4), dtype=np.float32)
    v = rng.normal(size=(n, 3))
    rays[:, 0, :3] = v / np.linalg.norm(v, axis=1)[:, None] * (1190.0 * rng.uniform(size=n) ** (1.0 / 3.0))[:, None]
    rays[:, 0, 3] = 0.05
    d = rng.normal(size=(n, 3))
    rays[:, 1, :3] = d / np.linalg.norm(d, axis=1)[:, None]
    rays[:, 1, 3] = 1e6
    return rays


def prepare(case, seed):
    e = engine_of(case)
    kind = case['kind']
    st = dict(kind=kind, engine=e, form=form_of(case), event=seed % 1000)
    if kind == 'photon_file':
        n = case['photons']
        rng = np.random.default_rng(seed)
        p = np.resize(scenes.raindrop_input_photons(), (n, 4, 4)).copy()
        p[:, 0, :3] += rng.uniform(-5.0, 5.0, size=(n, 3)).astype(np.float32)
        st.update(photons=p, gs=G.input_photon(n), out=np.zeros((n, 4, 4), dtype=np.float32))
    elif kind == 'serving':
        if e not in _servers:
            _servers[e] = Server(e, max_step_photons=4 << 20)
        evs = serving_events(case['events'], seed)
        st.update(server=_servers[e], events=evs, out=[room_for(case['scene'], G.num_photons(gs)) for gs in evs])
    elif kind == 'rays':
        st['rays'] = rays_of(case['rays'], seed)
    else:
        st['gs'] = gensteps_of(case['scene'], case['photons'], seed)
        if kind in ('hits', 'merged'):
            st['out'] = room_for(case['scene'], case['photons'])
    return st


def words(a):
    return a.view(np.int32)


def run(state):
    e, kind, out = state['engine'], state['kind'], state.get('out')
    if kind in ('hits', 'photon_file'):
        if kind == 'photon_file':
            e.set_input_photons(state['photons'])
        hits, _ = e.simulate(state['gs'], event_index=state['event'], form=state['form'], hit_capacity=len(out), out=out)
        return dict(number=len(hits), hits=words(out))
    if kind == 'serving':
        srv = state['server']
        for k, gs in enumerate(state['events']):
            srv.submit(k, gs, state['event'] + k)
        number = [0] * len(out)
        for _ in state['events']:
            r = srv.wait()
            k = r['request_id']
            number[k] = len(srv.take_hits(k, r['num_hit'], out=out[k]))
        return dict(number=np.array(number), hits=[words(h) for h in out])
    if kind == 'rays':
        prd = e.trace(state['rays'])
        return dict(normal=prd[:, 0, :3], distance=prd[:, 0, 3], identity=words(prd[:, 1, 2:]))
    e.set_gensteps(state['gs'], event_index=state['event'])
    e.launch(state['form'])
    if kind == 'merged':   # the C entry point, as a C++ host calls it
        n = ctypes.c_int64()
        rc = lib().oxr_event_get_merged(e.h, abi.OXR_GET_HIT, ctypes.c_float(1.0), abi.ptr(out), len(out), ctypes.byref(n))
        if rc != 0:
            raise RuntimeError(lib().oxr_last_error().decode())
        return dict(number=n.value, hits=words(out))
    if kind == 'history':
        return dict(photons=words(e.photons()), seq=e.seq().view(np.int64), record=words(e.get(abi.OXR_GET_RECORD)))
    return words(e.photons())


# bounce steps per photon and the share of photons that end as hits, measured per scene
STEPS = {'nested_boxes': 3.4, 'csi_calorimeter': 15.0, 'instanced_csg': 1.5, 'thin_shells': 50.0, 'pfrich': 5.0,
         'scintillator_sphere': 4.0, 'raindrop': 2.0}
HITS = {'csi_calorimeter': 0.006, 'instanced_csg': 0.2, 'raindrop': 1.0}
# floating-point operations of one bounce step that no traversal avoids: one surface
# intersection with its normal, two distances from logarithms, three table rows, and
# Fresnel or surface physics
STEP_FLOPS = 400


def work(case):
    kind, name = case['kind'], case.get('scene', 'raindrop')
    if kind == 'rays':
        return dict(bytes=case['rays'] * 64, flops=case['rays'] * 100)
    n = case['events'] * 280_000 if kind == 'serving' else case['photons']
    out = n * 64 * (1.0 if kind in ('photons', 'history') else HITS.get(name, 0.0))
    if kind == 'history':
        out += n * (32 + 10 * 64)
    if kind == 'photon_file':
        out += n * 64
    return dict(bytes=96 * max(1, n // 1000) + out, flops=n * STEPS[name] * STEP_FLOPS)


def exact(case, seed):
    """The ray query in 64 bits: the nearest of the three concentric spheres beyond tmin. A
    propagated photon has no such value: its history branches on single-precision draws, so
    another precision follows another history (its words are compared bit for bit)."""
    if case['kind'] != 'rays':
        return None
    rays = rays_of(case['rays'], seed).astype(np.float64)
    o, d, tmin = rays[:, 0, :3], rays[:, 1, :3], rays[:, 0, 3]
    a, b = (d * d).sum(1), (o * d).sum(1)
    best, radius = np.full(len(o), np.inf), np.zeros(len(o))
    for r in (1200.0, 1000.0, 600.0):
        disc = b * b - a * ((o * o).sum(1) - r * r)
        root = np.sqrt(np.maximum(disc, 0.0))
        t1, t2 = (-b - root) / a, (-b + root) / a
        t = np.where(disc > 0.0, np.where(t1 > tmin, t1, t2), -1.0)
        closer = (t > tmin) & (t < best)
        best, radius = np.where(closer, t, best), np.where(closer, r, radius)
    return dict(normal=(o + best[:, None] * d) / radius[:, None], distance=best, identity=None)
