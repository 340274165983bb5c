// oxr_boxes.cpp -- the world boxes of oxr_boxes.h.
#include "oxr_boxes.h"
#include <algorithm>
#include <cmath>
#include <cstring>

namespace oxh {

static uint32_t word(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }

void invert_instance(const float* q, double W[4][3]) {
    double a[3][3], t[3];
    for (int r = 0; r < 3; r++) for (int k = 0; k < 3; k++) a[r][k] = q[4 * r + k];
    for (int k = 0; k < 3; k++) t[k] = q[12 + k];
    double det = a[0][0] * (a[1][1] * a[2][2] - a[1][2] * a[2][1]) - a[0][1] * (a[1][0] * a[2][2] - a[1][2] * a[2][0]) +
                 a[0][2] * (a[1][0] * a[2][1] - a[1][1] * a[2][0]);
    double inv[3][3];
    inv[0][0] = (a[1][1] * a[2][2] - a[1][2] * a[2][1]) / det;
    inv[0][1] = (a[0][2] * a[2][1] - a[0][1] * a[2][2]) / det;
    inv[0][2] = (a[0][1] * a[1][2] - a[0][2] * a[1][1]) / det;
    inv[1][0] = (a[1][2] * a[2][0] - a[1][0] * a[2][2]) / det;
    inv[1][1] = (a[0][0] * a[2][2] - a[0][2] * a[2][0]) / det;
    inv[1][2] = (a[0][2] * a[1][0] - a[0][0] * a[1][2]) / det;
    inv[2][0] = (a[1][0] * a[2][1] - a[1][1] * a[2][0]) / det;
    inv[2][1] = (a[0][1] * a[2][0] - a[0][0] * a[2][1]) / det;
    inv[2][2] = (a[0][0] * a[1][1] - a[0][1] * a[1][0]) / det;
    for (int i = 0; i < 3; i++) for (int k = 0; k < 3; k++) W[i][k] = inv[i][k];
    for (int k = 0; k < 3; k++) W[3][k] = -(t[0] * inv[0][k] + t[1] * inv[1][k] + t[2] * inv[2][k]);
}

double stretch_of(const float* q, const double inv[4][3]) {
    double a = 0.0, b = 0.0;
    for (int r = 0; r < 3; r++) for (int k = 0; k < 3; k++) { a += double(q[4 * r + k]) * q[4 * r + k]; b += inv[r][k] * inv[r][k]; }
    return std::sqrt(a * b);
}

LeafBoxes::LeafBoxes(const oxr_geometry* g, double reach) : reach_(reach) {
    first_.push_back(0);
    for (int64_t p = 0; p < g->num_prim; p++) {
        int32_t at;
        std::memcpy(&at, g->prim + 16 * p + 1, 4);
        const float* root = g->node + 16 * int64_t(at);
        const uint32_t rtc = word(root[14]);
        const bool tree = rtc >= 1u && rtc <= 3u;
        const int64_t n = tree ? word(root[0]) : 1;
        const size_t begin = leaves_.size();
        for (int64_t i = 0; i < n; i++) {
            const float* q = root + 16 * i;
            const uint32_t tc = word(q[14]), gt = word(q[15]) & 0x7fffffffu;
            if (tc <= 3u) continue;   // an operator, or nothing
            if (tc != 101u && tc != 103u && tc != 105u && tc != 110u) { leaves_.resize(begin); break; }
            Leaf l{};
            l.type = tc;
            l.turned = gt > 0u;
            if (l.turned) {
                const float* t = g->itra + 16 * (int64_t(gt) - 1);
                invert_instance(t, l.to_object);
                for (int r = 0; r < 3; r++) for (int k = 0; k < 3; k++) l.to_leaf[r][k] = t[4 * r + k];
            }
            l.x = q[0]; l.y = q[1]; l.z = q[2]; l.r = q[3]; l.z1 = q[4]; l.z2 = q[5];
            leaves_.push_back(l);
        }
        first_.push_back(int64_t(leaves_.size()));
    }
}

bool LeafBoxes::leaf_box(const Leaf& l, const double A[4][3], const double inv[4][3], Box& out) const {
    double T[4][3];   // leaf to world, row convention
    double norm2 = 0.0;
    if (l.turned) {
        for (int r = 0; r < 4; r++) for (int k = 0; k < 3; k++)
            T[r][k] = l.to_object[r][0] * A[0][k] + l.to_object[r][1] * A[1][k] + l.to_object[r][2] * A[2][k] + (r == 3 ? A[3][k] : 0.0);
        for (int r = 0; r < 3; r++) for (int k = 0; k < 3; k++) {
            const double x = inv[r][0] * l.to_leaf[0][k] + inv[r][1] * l.to_leaf[1][k] + inv[r][2] * l.to_leaf[2][k];
            norm2 += x * x;
        }
    } else {
        for (int r = 0; r < 3; r++) for (int k = 0; k < 3; k++) norm2 += inv[r][k] * inv[r][k];
    }
    const double (*M)[3] = l.turned ? T : A;
    const double far = reach_ * std::sqrt(norm2);   // the reach in the leaf's frame
    double all = far;                               // not finite if any term is not
    for (int r = 0; r < 4; r++) for (int k = 0; k < 3; k++) all += std::fabs(M[r][k]);
    if (!std::isfinite(all)) return false;
    double col[3];                                  // length of M's columns: how far a unit sphere reaches
    for (int k = 0; k < 3; k++) col[k] = std::sqrt(M[0][k] * M[0][k] + M[1][k] * M[1][k] + M[2][k] * M[2][k]);
    const double flat = 16.0 * 6e-8 * far;          // planes: a few ulps of the distance
    auto map = [&](double x, double y, double z, double* w) {
        for (int k = 0; k < 3; k++) w[k] = x * M[0][k] + y * M[1][k] + z * M[2][k] + M[3][k];
    };
    auto around = [&](const double* c, double hx, double hy, double hz, Box& b) {   // the box of a leaf-frame box
        for (int k = 0; k < 3; k++) {
            const double h = std::fabs(M[0][k]) * hx + std::fabs(M[1][k]) * hy + std::fabs(M[2][k]) * hz;
            b.lo[k] = c[k] - h; b.hi[k] = c[k] + h;
        }
    };
    double c[3];
    if (l.type == 110u) {
        map(0.0, 0.0, 0.0, c);
        around(c, 0.5 * std::fabs(l.x) + flat, 0.5 * std::fabs(l.y) + flat, 0.5 * std::fabs(l.z) + flat, out);
        return true;
    }
    const double R = std::sqrt(l.r * l.r + 2e-6 * far * far);
    const double zc = 0.5 * (l.z1 + l.z2), hz = 0.5 * std::fabs(l.z2 - l.z1) + flat;
    if (l.type == 105u) {
        map(0.0, 0.0, zc, c);
        for (int k = 0; k < 3; k++) {
            const double h = R * std::sqrt(M[0][k] * M[0][k] + M[1][k] * M[1][k]) + hz * std::fabs(M[2][k]);
            out.lo[k] = c[k] - h; out.hi[k] = c[k] + h;
        }
        return true;
    }
    map(l.x, l.y, l.z, c);
    for (int k = 0; k < 3; k++) { out.lo[k] = c[k] - R * col[k]; out.hi[k] = c[k] + R * col[k]; }
    if (l.type == 103u) {   // and the slab between its planes
        Box slab;
        map(l.x, l.y, l.z + zc, c);
        around(c, R, R, hz, slab);
        for (int k = 0; k < 3; k++) { out.lo[k] = std::max(out.lo[k], slab.lo[k]); out.hi[k] = std::min(out.hi[k], slab.hi[k]); }
    }
    return true;
}

Box LeafBoxes::placed(int64_t prim, const Box& ob, const float* inst, const double inv[4][3]) const {
    double A[4][3];
    for (int r = 0; r < 4; r++) for (int k = 0; k < 3; k++) A[r][k] = inst[4 * r + k];
    Box b;   // the object box's, turned
    for (int k = 0; k < 3; k++) {
        double c = A[3][k], h = 0.0;
        for (int r = 0; r < 3; r++) {
            c += 0.5 * (ob.lo[r] + ob.hi[r]) * A[r][k];
            h += 0.5 * (ob.hi[r] - ob.lo[r]) * std::fabs(A[r][k]);
        }
        b.lo[k] = c - h; b.hi[k] = c + h;
    }
    Box all = Box::empty();
    for (int64_t i = first_[size_t(prim)]; i < first_[size_t(prim) + 1]; i++) {
        Box lb;
        if (!leaf_box(leaves_[size_t(i)], A, inv, lb)) return b;
        all.grow(lb);
    }
    if (first_[size_t(prim)] == first_[size_t(prim) + 1]) return b;
    Box cut = b;
    for (int k = 0; k < 3; k++) {
        cut.lo[k] = std::max(b.lo[k], all.lo[k]);
        cut.hi[k] = std::min(b.hi[k], all.hi[k]);
        if (!(cut.lo[k] <= cut.hi[k])) return b;   // box and shape disagree: the box stands
    }
    return cut;
}

} // namespace oxh
