"""The photon loop's sine and cosine (sincos_bounded in eic-opticks_amd/csrc/oxr_device.h),
compiled for the host: equal to the library's double-precision functions rounded once, for
every angle that a Philox uniform gives and for arguments up to 8e5 in magnitude."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, 'eic-opticks_amd', 'csrc', 'oxr_device.h')

PROGRAM = r'''
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#define OXD static inline
%s
static long bad = 0, n = 0;
static void check(float x) {
    float s, c;
    sincos_bounded(x, s, c);
    const float ws = float(std::sin(double(x))), wc = float(std::cos(double(x)));
    n++;
    if (std::memcmp(&s, &ws, 4) != 0 || std::memcmp(&c, &wc, 4) != 0) {
        if (bad++ < 5) std::printf("%%.9g: %%.9g %%.9g for %%.9g %%.9g\n", x, s, c, ws, wc);
    }
}
int main(int, char** a) {
    const float PIf = 3.14159265358979323846f;
    if (!std::strcmp(a[1], "uniforms")) {
        for (uint32_t k = 0; k < (1u << 24); k++) {
            const float u = float(k + 1u) * (1.0f / 16777216.0f);
            check(2.f * PIf * u);
        }
    } else {   // the floats up to 8e5, every 127th, both signs
        uint32_t top;
        const float limit = 8e5f;
        std::memcpy(&top, &limit, 4);
        for (uint32_t w = 1; w <= top; w += 127) {
            float x;
            std::memcpy(&x, &w, 4);
            check(x);
            check(-x);
        }
    }
    std::printf("%%ld of %%ld\n", bad, n);
    return bad ? 1 : 0;
}
'''


@pytest.fixture(scope='module')
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp('sincos')
    body = re.search(r'OXD void sincos_bounded\(.*?\n}\n', open(HEADER).read(), re.S).group(0)
    (d / 'sincos.cpp').write_text(PROGRAM % body)
    subprocess.check_call(['g++', '-O2', '-std=c++17', '-ffp-contract=off', str(d / 'sincos.cpp'), '-o', str(d / 'sincos')])
    return str(d / 'sincos')


@pytest.mark.parametrize('which', ['uniforms', 'floats'])
def test_rounded_once(program, which):
    subprocess.run([program, which], check=True, timeout=120)
