"""The hits of a launch are its photons with the mask's bits, in photon order, at the edges of
what the selection and the copies work in: 4096 photons a workgroup, 1024 hits written straight
to the host, 1 MB (16384 photons) a copy in one piece, 2 MB without helpers, four slots of
2 MB. One engine takes all sizes in turn, so each launch follows one that left other counts
behind."""
import numpy as np
import pytest

from oxr import abi, gensteps as G, scenes

pytestmark = pytest.mark.gpu

TORCH, REFLECT = 4, 1 << 10


@pytest.mark.parametrize('form', [abi.OXR_FORM_PLAIN, abi.OXR_FORM_PERSISTENT])
@pytest.mark.parametrize('mask', [TORCH, TORCH | REFLECT])
def test_selection_at_the_edges(engine_mod, oracle_lib, mask, form):
    s = scenes.raindrop()
    cfg = abi.default_config(**dict(s.config, hitmask=mask))
    o = oracle_lib.Oracle(s.geometry, s.physics, cfg)
    with engine_mod.Engine(s.geometry, s.physics, cfg) as e:
        for n in (1, 1023, 1024, 1025, 4095, 4096, 4097, 16384, 16385, 32767, 32768, 32769, 131073, 63):
            gs = G.torch(np.array([n]), pos=np.array([[1.0, 2.0, 3.0]]), wavelength=440.0, type=G.T_POINT_ISOTROPIC)
            print('selection', mask, form, n, flush=True)
            e.set_gensteps(gs, event_index=n % 7)
            for _ in range(2):
                st = e.launch(form)
                ph, hit = e.photons(), e.hits()
                flagmask = ph.view(np.uint32).reshape(n, 16)[:, 15]
                want = ph[(flagmask & mask) == mask]
                assert st['num_photon'] == n and st['num_hit'] == len(want) == len(hit), n
                assert np.array_equal(hit.view(np.uint32), want.view(np.uint32)), n
            if n <= 4097:
                ref = o.simulate(gs, event_index=n % 7, seq=False)['photon']
                assert np.array_equal(ph.view(np.uint32), ref.view(np.uint32)), n
            if mask == TORCH:
                assert len(hit) == n
