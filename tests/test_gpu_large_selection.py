"""Hit selection of launches of more than 16.8 million photons, where the counts of 256 blocks
are summed first: the hits are the photons with the mask's bits, in photon order, on both sides
of that size and at the edges of a block and of a group. With the second mask, hits are those
of the photons that a surface has reflected, so blocks hold different numbers of them."""
import numpy as np
import pytest

from oxr import abi, gensteps as G, scenes

pytestmark = pytest.mark.gpu

EDGE = 4096 * 4096
TORCH, REFLECT = 1 << 2, 1 << 10


@pytest.mark.parametrize('mask', [TORCH, TORCH | REFLECT])
def test_large_launches(engine_mod, mask):
    s = scenes.nested_boxes()
    cfg = abi.default_config(**dict(s.config, hitmask=mask, max_photon=20_000_000))
    with engine_mod.Engine(s.geometry, s.physics, cfg) as e:
        for n in (EDGE, EDGE + 1, EDGE + 256 * 4096 + 4095, EDGE - 1):
            gs = G.torch(np.array([n - 7, 7]), pos=np.array([[1.0, 2.0, 3.0], [0.0, 0.0, 0.0]]), wavelength=440.0,
                         type=G.T_POINT_ISOTROPIC)
            print('large selection', mask, n, flush=True)
            e.set_gensteps(gs, event_index=n % 5)
            st = e.launch(abi.OXR_FORM_PERSISTENT)
            ph = e.photons().view(np.uint32).reshape(n, 16)
            want = (ph[:, 15] & mask) == mask
            number = int(want.sum())
            assert st['num_photon'] == n and st['num_hit'] == number
            if mask == TORCH:
                assert number == n
            else:
                assert 1000 < number < n - 1000
            hit = e.hits().view(np.uint32).reshape(-1, 16)
            assert len(hit) == number
            for at in range(0, n, 1 << 22):   # a few chunks, so that no copy of all of them is made
                sel = ph[at:at + (1 << 22)][want[at:at + (1 << 22)]]
                k = int(want[:at].sum())
                assert np.array_equal(hit[k:k + len(sel)], sel), (n, at)
