"""Compiler options by unit: the float rules hold in every unit, the option that is for the
traversal loop in the units that hold one and in no other."""
import pytest

from oxr import build


@pytest.mark.parametrize('src', build.SOURCES)
def test_flags(src):
    f = build.flags(src)
    assert '-ffp-contract=off' in f and '-packed-fp32-ops' in f and '-fhip-fp32-correctly-rounded-divide-sqrt' in f
    assert ('-disable-machine-licm' in f) == (src == 'oxr_kernels.hip' or src.startswith('oxr_sim_'))
