"""A lane's sum of bounce steps (eic-opticks_amd/csrc/oxr_steps.h), on the CPU: 32 bits of it
are kept, and what has been handed over plus what is left is the 64-bit sum, for photons of up
to the largest max_bounce and for many more of them than 32 bits hold."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, 'eic-opticks_amd', 'csrc')

PROGRAM = r'''
#include "oxr_steps.h"
#include <cstdlib>
int main(int, char** a) {
    const long long photons = std::atoll(a[1]);
    const int bounces = std::atoi(a[2]);
    unsigned long long handed = 0, want = 0;
    uint32_t steps = 0;
    for (long long k = 0; k < photons; k++) {
        const int b = k % 3 ? bounces : int(k % 1000);
        oxd::add_steps(steps, b, [&](uint32_t n) { handed += n; });
        want += (unsigned long long)b;
    }
    return handed + steps == want ? 0 : 1;
}
'''


@pytest.fixture(scope='module')
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp('steps')
    (d / 'steps.cpp').write_text(PROGRAM)
    subprocess.check_call(['g++', '-O2', '-std=c++17', '-I', CSRC, str(d / 'steps.cpp'), '-o', str(d / 'steps')])
    return str(d / 'steps')


@pytest.mark.parametrize('photons,bounces', [(1, 31), (1000, 31), (100_000, 43_000), (7, 2**31 - 1), (5000, 2**31 - 1),
                                             (20_000_000, 1000)])
def test_sum(program, photons, bounces):
    subprocess.check_call([program, str(photons), str(bounces)])
