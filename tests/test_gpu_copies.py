"""Staged copies at the edges of how they are cut up (1 MB in one piece, 2 MB without helpers,
four slots of 2 MB, longer ones reusing them): every row arrives, up and down, compared with
the same rows in copies of one piece; and from several engines, and several callers of one
server, at once."""
import threading

import numpy as np
import pytest

from oxr import abi, gensteps as G, scenes

from test_gpu_parity import bits

pytestmark = pytest.mark.gpu

SCENE = scenes.scintillator_sphere()


def rays_of(rng, n):
    rays = np.zeros((n, 2, 4), dtype=np.float32)
    rays[:, 0, :3] = rng.uniform(-600.0, 600.0, size=(n, 3))
    rays[:, 0, 3] = 0.05
    d = rng.normal(size=(n, 3))
    rays[:, 1, :3] = d / np.linalg.norm(d, axis=1)[:, None]
    rays[:, 1, 3] = 1e6
    return rays


def in_pieces(e, rays):
    return np.concatenate([e.trace(rays[k:k + 20_000]) for k in range(0, len(rays), 20_000)])


def test_rays_up_and_down(engine_mod):
    rays = rays_of(np.random.default_rng(1), 700_000)
    with engine_mod.Engine(SCENE.geometry, SCENE.physics, abi.default_config()) as e:
        want = in_pieces(e, rays)
        assert len(np.unique(bits(want)[:, 0, 3])) > 100_000        # rows can be told apart
        MB = (1 << 20) // 32
        for n in (1, MB - 1, MB, MB + 1, 2 * MB - 1, 2 * MB, 2 * MB + 1, 8 * MB - 1, 8 * MB, 8 * MB + 1, 16 * MB + 7, 700_000, 33):
            print('rays', n, flush=True)
            first = (n * 37) % (len(rays) - n + 1)
            assert np.array_equal(bits(e.trace(rays[first:first + n])), bits(want[first:first + n])), n


def test_photons_up_and_down(engine_mod):
    rng = np.random.default_rng(2)
    n = 300_000
    photons = rng.normal(size=(n, 4, 4)).astype(np.float32)
    photons[:, 1, :3] /= np.linalg.norm(photons[:, 1, :3], axis=1)[:, None]
    photons[:, 2, 3] = rng.uniform(300.0, 600.0, size=n)
    photons[:, 3, :] = 0.0
    cfg = abi.default_config(max_bounce=0, hitmask=1 << 2)   # every photon is a hit
    MB = (1 << 20) // 64
    with engine_mod.Engine(SCENE.geometry, SCENE.physics, cfg) as e:
        for m in (5, MB - 1, MB, MB + 1, 2 * MB, 2 * MB + 1, 8 * MB, 8 * MB + 1, n, MB):
            print('photons', m, flush=True)
            part = photons[n - m:]
            e.set_input_photons(part)
            e.set_gensteps(G.input_photon(m))
            st = e.launch(abi.OXR_FORM_PERSISTENT)
            got, hit = e.photons(), e.hits()
            for words in (np.s_[:, 0, :], np.s_[:, 1, :3], np.s_[:, 2, :]):
                assert np.array_equal(bits(got[words]), bits(part[words])), m
            assert st['num_hit'] == m and np.array_equal(bits(hit), bits(got)), m


def run_together(jobs):
    failed = []

    def guarded(job):
        try:
            job()
        except BaseException as x:   # reported by the test's own thread
            failed.append(x)
    th = [threading.Thread(target=guarded, args=(j,)) for j in jobs]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not failed, failed


def test_engines_at_once(engine_mod):
    engines = [engine_mod.Engine(SCENE.geometry, SCENE.physics, abi.default_config()) for _ in range(3)]
    rays = [rays_of(np.random.default_rng(10 + k), 200_000 + 40_001 * k) for k in range(3)]
    want = [in_pieces(e, r) for e, r in zip(engines, rays)]

    def job(k):
        def work():
            for n in (len(rays[k]), 70_000, 33_000, len(rays[k])):
                assert np.array_equal(bits(engines[k].trace(rays[k][:n])), bits(want[k][:n])), (k, n)
        return work
    print('three engines at once', flush=True)
    run_together([job(k) for k in range(3)])
    for e in engines:
        e.close()


def test_hits_taken_at_once(engine_mod):
    s = scenes.nested_boxes()
    cfg = abi.default_config(**dict(s.config, hitmask=1 << 2))
    sizes = [200_000, 90_001, 16_385, 150_007, 1000]
    gs = [G.torch(np.array([n]), pos=np.array([[1.0 + k, 2.0, 3.0]]), wavelength=430.0, type=G.T_POINT_ISOTROPIC)
          for k, n in enumerate(sizes)]
    with engine_mod.Engine(s.geometry, s.physics, cfg) as e:
        want = [e.simulate(g, event_index=k, form=abi.OXR_FORM_PERSISTENT, hit_capacity=n)[0]
                for k, (g, n) in enumerate(zip(gs, sizes))]
        srv = engine_mod.Server(e, max_step_photons=1 << 20)
        for turn in range(3):
            print('hits taken at once', turn, flush=True)
            for k, g in enumerate(gs):
                srv.submit(k, g, k)
            done = [srv.wait() for _ in gs]

            def job(r):
                def work():
                    got = srv.take_hits(r['request_id'], r['num_hit'])
                    assert np.array_equal(bits(got), bits(want[r['request_id']])), r['request_id']
                return work
            run_together([job(r) for r in done])
        srv.close()
