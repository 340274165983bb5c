"""The device buffers that an engine keeps between calls (eic-opticks_amd/csrc/oxr_dbuf.h), on
the CPU with a device of a few GB made of counters: what is kept stays bounded, a call that
fails keeps nothing, and what is kept gives way to an allocation that finds no memory."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, 'eic-opticks_amd', 'csrc')

PROGRAM = r'''
#include "oxr_dbuf.h"
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
static std::map<void*, size_t> blocks;
static size_t free_bytes;
static bool error_left = false;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
    static char* next = reinterpret_cast<char*>(size_t(1) << 40);
    *p = nullptr;
    if (n > free_bytes) { error_left = true; return hipErrorOutOfMemory; }
    free_bytes -= n;
    *p = next;
    next += n + 256;
    blocks[*p] = n;
    return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
    if (!blocks.count(p)) { std::puts("freed what was not allocated"); std::exit(2); }
    free_bytes += blocks[p];
    blocks.erase(p);
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError() {
    const bool e = error_left;
    error_left = false;
    return e ? hipErrorOutOfMemory : hipSuccess;
}
using namespace oxl;
static const size_t MB = size_t(1) << 20;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

static bool call(Workspace& w, std::initializer_list<size_t> want, bool ok = true) {
    WorkCall c(w);
    int k = 0;
    for (size_t n : want) if (w.get(k++, n) != hipSuccess) return false;
    if (ok) c.keep();
    return true;
}

int main(int, char** a) {
    const size_t ALL = 4096 * MB;
    free_bytes = ALL;
    Workspace w;
    if (!std::strcmp(a[1], "bounded")) {
        CHECK(call(w, {100 * MB, 200 * MB}) && free_bytes == ALL - 300 * MB);
        CHECK(call(w, {10 * MB, 210 * MB}) && free_bytes == ALL - 310 * MB);   // grown, not added
        CHECK(call(w, {1, 1, 202 * MB}) && free_bytes == ALL - 512 * MB);      // at the bound
        CHECK(call(w, {1, 1, 1, 1}) && free_bytes == ALL);                     // beyond it
        CHECK(call(w, {2000 * MB, 2000 * MB}) && free_bytes == ALL);
    } else if (!std::strcmp(a[1], "failed")) {
        CHECK(!call(w, {3000 * MB, 3000 * MB}) && free_bytes == ALL && w.bytes() == 0);
        CHECK(call(w, {1 * MB}) && free_bytes == ALL - MB);
        CHECK(call(w, {2 * MB, 3 * MB}, false) && free_bytes == ALL);          // failed after its allocations
        CHECK(!call(w, {1 * MB, 5000 * MB}) && free_bytes == ALL);
    } else if (!std::strcmp(a[1], "gives_way")) {
        CHECK(call(w, {100 * MB, 300 * MB, 50 * MB}));
        oxh::DBuf<double> event;
        (void)hipGetLastError();
        CHECK(w.reserve(event, 500 * MB) == hipSuccess && event.n == 500 * MB);   // 4000 MB
        CHECK(free_bytes == 96 * MB && w.bytes() == 0);
        CHECK(hipGetLastError() == hipSuccess);      // the first try's error is not left for the next launch
        event.release();
        CHECK(call(w, {100 * MB, 300 * MB, 50 * MB}));
        CHECK(call(w, {3900 * MB}) && free_bytes == ALL);   // a call's own slot, the others given up
        CHECK(w.reserve(event, 513 * MB) == hipErrorOutOfMemory && free_bytes == ALL);
        {
            WorkCall c(w);                          // slots of the call under way are not given up
            CHECK(w.get(3, 200 * MB) == hipSuccess && w.reserve(event, 500 * MB) == hipErrorOutOfMemory);
            CHECK(w.slot[3].p && w.slot[3].n == 200 * MB);
        }
        CHECK(free_bytes == ALL && blocks.empty());
    }
    return 0;
}
'''


@pytest.fixture(scope='module')
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp('kept')
    (d / 'kept.cpp').write_text(PROGRAM)
    rocm = os.environ.get('ROCM_PATH', '/opt/rocm')
    subprocess.check_call(['g++', '-O1', '-std=c++17', '-D__HIP_PLATFORM_AMD__', '-I', os.path.join(rocm, 'include'), '-I', CSRC,
                           str(d / 'kept.cpp'), '-o', str(d / 'kept')])
    return str(d / 'kept')


@pytest.mark.parametrize('what', ['bounded', 'failed', 'gives_way'])
def test_kept(program, what):
    subprocess.run([program, what], check=True, timeout=60)
