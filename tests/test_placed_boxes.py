"""World boxes of placed prims (eic-opticks_amd/csrc/oxr_boxes.cpp), on the CPU: points of the
leaves' surfaces lie in them, also those that a single-precision test reports from a ray's
length away; they stay within the prim's turned object box; a prim with any other leaf keeps
that box; and making them for every placed prim takes less time than the tree over them."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, 'eic-opticks_amd', 'csrc')

PROGRAM = r'''
#include "oxr_boxes.h"
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
using namespace oxh;
typedef std::mt19937_64 Rng;
static double uni(Rng& r, double a, double b) { return std::uniform_real_distribution<double>(a, b)(r); }
static float bitf(uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }

// a rotation about a random axis times a scale along the axes, row convention, with translation
static void transform(Rng& r, double smin, double smax, double shift, double M[4][4], double I[4][4]) {
    double a[3], n = 0.0;
    for (double& x : a) { x = uni(r, -1, 1); n += x * x; }
    for (double& x : a) x /= std::sqrt(n);
    const double t = uni(r, 0, 6.28), c = std::cos(t), s = std::sin(t);
    double R[3][3] = {{c + a[0] * a[0] * (1 - c), a[0] * a[1] * (1 - c) + a[2] * s, a[0] * a[2] * (1 - c) - a[1] * s},
                      {a[0] * a[1] * (1 - c) - a[2] * s, c + a[1] * a[1] * (1 - c), a[1] * a[2] * (1 - c) + a[0] * s},
                      {a[0] * a[2] * (1 - c) + a[1] * s, a[1] * a[2] * (1 - c) - a[0] * s, c + a[2] * a[2] * (1 - c)}};
    double T[3];
    for (int i = 0; i < 4; i++) for (int k = 0; k < 4; k++) M[i][k] = I[i][k] = i == k;
    for (int k = 0; k < 3; k++) T[k] = uni(r, -shift, shift);
    for (int i = 0; i < 3; i++) {
        const double sc = uni(r, smin, smax);
        for (int k = 0; k < 3; k++) { M[i][k] = sc * R[i][k]; I[k][i] = R[i][k] / sc; }
    }
    for (int k = 0; k < 3; k++) {
        M[3][k] = T[k];
        I[3][k] = -(T[0] * I[0][k] + T[1] * I[1][k] + T[2] * I[2][k]);
    }
}
static void apply(const double M[4][4], const double* p, double* w) {
    for (int k = 0; k < 3; k++) w[k] = p[0] * M[0][k] + p[1] * M[1][k] + p[2] * M[2][k] + M[3][k];
}

struct Geo {
    std::vector<float> node, itra, prim;
    std::vector<double> M;     // 16 per leaf: leaf to object
    oxr_geometry g() const {
        oxr_geometry x;
        std::memset(&x, 0, sizeof(x));
        x.node = node.data(); x.itra = itra.data(); x.prim = prim.data();
        x.num_node = int64_t(node.size() / 16); x.num_itra = int64_t(itra.size() / 16); x.num_prim = int64_t(prim.size() / 16);
        return x;
    }
    void op(uint32_t subs) { float q[16] = {0}; q[0] = bitf(subs); q[14] = bitf(1); node.insert(node.end(), q, q + 16); }
    void leaf(Rng& r, uint32_t type, bool turned) {
        float q[16] = {0};
        if (type == 110) { for (int k = 0; k < 3; k++) q[k] = float(uni(r, 5, 100)); }
        else { q[3] = float(uni(r, 5, 100)); q[4] = float(-uni(r, 1, 80)); q[5] = float(uni(r, 1, 80)); }
        if (type == 103) { q[4] = float(uni(r, -0.9, 0.0) * q[3]); q[5] = float(uni(r, 0.0, 0.9) * q[3]); }
        if (type == 101 || type == 103) for (int k = 0; k < 3; k++) q[k] = float(uni(r, -20, 20));
        q[14] = bitf(type);
        double A[4][4], I[4][4];
        for (int i = 0; i < 4; i++) for (int k = 0; k < 4; k++) A[i][k] = i == k;
        if (turned) {
            transform(r, 0.5, 1.8, 60, A, I);
            for (int i = 0; i < 16; i++) itra.push_back(float(I[i / 4][i % 4]));
            q[15] = bitf(uint32_t(itra.size() / 16) | (r() % 2 ? 0x80000000u : 0u));
        }
        for (int i = 0; i < 16; i++) M.push_back(A[i / 4][i % 4]);
        node.insert(node.end(), q, q + 16);
    }
    void one_prim() {
        float p[16] = {0};
        const int32_t n = int32_t(node.size() / 16), at = 0;
        std::memcpy(p, &n, 4); std::memcpy(p + 1, &at, 4);
        prim.assign(p, p + 16);
    }
};
static const uint32_t TYPES[4] = {101, 103, 105, 110};

// a point that the leaf's test may report: on its surface, quadrics' radius grown by reach
static void surface(Rng& r, const float* q, uint32_t type, double grow, double* p) {
    const double z = uni(r, -1, 1), a = uni(r, 0, 6.2831853);
    if (type == 110) {
        for (int k = 0; k < 3; k++) p[k] = uni(r, -0.5, 0.5) * q[k];
        const int k = int(r() % 3);
        p[k] = (r() % 2 ? 0.5 : -0.5) * q[k];
        return;
    }
    const double R = std::sqrt(double(q[3]) * q[3] + grow);
    if (type == 105) {
        const bool cap = r() % 3 == 0;
        const double rr = cap ? R * std::sqrt(uni(r, 0, 1)) : R;
        p[0] = rr * std::cos(a); p[1] = rr * std::sin(a);
        p[2] = cap ? (r() % 2 ? q[4] : q[5]) : uni(r, q[4], q[5]);
        return;
    }
    double h = z * R;
    if (type == 103) h = std::min(std::max(h, double(q[4])), double(q[5]));
    const double s = std::sqrt(std::max(0.0, R * R - h * h)) * (type == 103 && (h == q[4] || h == q[5]) ? std::sqrt(uni(r, 0, 1)) : 1.0);
    p[0] = q[0] + s * std::cos(a); p[1] = q[1] + s * std::sin(a); p[2] = q[2] + h;
}

static int contain(unsigned seed, bool other) {
    Rng r(seed);
    for (int turn = 0; turn < 300; turn++) {
        Geo geo;
        const bool tree = turn % 2;
        if (tree) { geo.op(7); geo.op(0); geo.op(0); geo.M.resize(48); }
        for (int i = 0; i < (tree ? 4 : 1); i++) geo.leaf(r, other && i == 0 ? 108 : TYPES[r() % 4], r() % 3 != 0);
        geo.one_prim();
        const double reach = std::pow(10.0, uni(r, 3, 5));
        double A[4][4], I[4][4], inv[4][3];
        transform(r, turn % 5 ? 1.0 : 0.7, turn % 5 ? 1.0 : 1.5, 1000, A, I);
        float inst[16];
        for (int i = 0; i < 16; i++) inst[i] = float(A[i / 4][i % 4]);
        invert_instance(inst, inv);
        for (int i = 0; i < 4; i++) for (int k = 0; k < 3; k++) A[i][k] = inst[4 * i + k];
        Box ob;
        for (int k = 0; k < 3; k++) { ob.lo[k] = -600; ob.hi[k] = 600; }
        Box turned = Box::empty();
        for (int c = 0; c < 8; c++) {
            double p[3] = {c & 1 ? 600. : -600., c & 2 ? 600. : -600., c & 4 ? 600. : -600.}, w[3];
            apply(A, p, w);
            turned.grow_point(w);
        }
        LeafBoxes boxes(new oxr_geometry(geo.g()), reach);
        const Box b = boxes.placed(0, ob, inst, inv);
        for (int k = 0; k < 3; k++) {
            if (b.lo[k] < turned.lo[k] - 1e-6 || b.hi[k] > turned.hi[k] + 1e-6) return 1;
            if (other && (b.lo[k] > turned.lo[k] + 1e-6 || b.hi[k] < turned.hi[k] - 1e-6)) return 2;
        }
        if (other) continue;
        for (size_t n = tree ? 3 : 0; n < geo.node.size() / 16; n++) {
            const float* q = &geo.node[16 * n];
            uint32_t type;
            std::memcpy(&type, q + 14, 4);
            double M[4][4];
            for (int i = 0; i < 16; i++) M[i / 4][i % 4] = geo.M[16 * n + size_t(i)];
            for (int s = 0; s < 200; s++) {
                double p[3], o[3], w[3];
                surface(r, q, type, 1e-6 * reach * reach / 4, p);   // a leaf scaled up to 1.8 and placed up to 1.5 shrinks the reach at most 2.7 times
                apply(M, p, o);
                if (s % 2 || type == 110) surface(r, q, type, 0, p), apply(M, p, o);
                apply(A, o, w);
                for (int k = 0; k < 3; k++) if (w[k] < b.lo[k] - 1e-3 || w[k] > b.hi[k] + 1e-3) {
                    if (w[k] < turned.lo[k] || w[k] > turned.hi[k]) continue;   // cut by the object box
                    std::printf("seed %u turn %d type %u out by %g\n", seed, turn, type, std::max(b.lo[k] - w[k], w[k] - b.hi[k]));
                    return 4;
                }
            }
        }
    }
    return 0;
}

static int timing() {
    Rng r(5);
    Geo geo;
    geo.op(15);
    for (int i = 1; i < 7; i++) geo.op(0);
    geo.M.resize(7 * 16);
    for (int i = 0; i < 5; i++) geo.leaf(r, TYPES[i % 4], i != 0);
    for (int i = 0; i < 3; i++) { float q[16] = {0}; geo.node.insert(geo.node.end(), q, q + 16); }
    geo.one_prim();
    const oxr_geometry g = geo.g();
    const int n = 200000;
    std::vector<float> inst(size_t(n) * 16);
    std::vector<double> inv(size_t(n) * 12);
    for (int i = 0; i < n; i++) {
        double A[4][4], I[4][4];
        transform(r, 1.0, 1.0, 10000, A, I);
        for (int k = 0; k < 16; k++) inst[size_t(16 * i + k)] = float(A[k / 4][k % 4]);
        invert_instance(&inst[size_t(16 * i)], reinterpret_cast<double(*)[3]>(&inv[size_t(12 * i)]));
    }
    Box ob;
    for (int k = 0; k < 3; k++) { ob.lo[k] = -300; ob.hi[k] = 300; }
    double best[2] = {1e9, 1e9};
    for (int rep = 0; rep < 3; rep++) {
        std::vector<Box> out(static_cast<size_t>(n));
        const auto t0 = std::chrono::steady_clock::now();
        LeafBoxes boxes(&g, 35000.0);
        for (int i = 0; i < n; i++)
            out[size_t(i)] = boxes.placed(0, ob, &inst[size_t(16 * i)], reinterpret_cast<const double(*)[3]>(&inv[size_t(12 * i)]));
        const auto t1 = std::chrono::steady_clock::now();
        build_bvh(out, 0, 0.0);
        const auto t2 = std::chrono::steady_clock::now();
        best[0] = std::min(best[0], std::chrono::duration<double>(t1 - t0).count());
        best[1] = std::min(best[1], std::chrono::duration<double>(t2 - t1).count());
    }
    std::printf("%.3f us a placed prim of five leaves, %.3f us of its tree\n", best[0] * 1e6 / n, best[1] * 1e6 / n);
    return best[0] < best[1] ? 0 : 1;
}

int main(int, char** a) {
    if (!std::strcmp(a[1], "time")) return timing();
    return contain(unsigned(std::atoi(a[2])), !std::strcmp(a[1], "other"));
}
'''


@pytest.fixture(scope='module')
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp('boxes')
    (d / 'boxes.cpp').write_text(PROGRAM)
    subprocess.check_call(['g++', '-O2', '-std=c++17', '-I', CSRC, str(d / 'boxes.cpp'), os.path.join(CSRC, 'oxr_boxes.cpp'),
                           os.path.join(CSRC, 'oxr_bvh.cpp'), '-o', str(d / 'boxes')])
    return str(d / 'boxes')


@pytest.mark.parametrize('seed', range(4))
@pytest.mark.parametrize('kind', ['simple', 'other'])
def test_boxes(program, kind, seed):
    subprocess.run([program, kind, str(seed)], check=True, timeout=120)


def test_less_time_than_the_tree(program):
    subprocess.run([program, 'time'], check=True, timeout=120)
