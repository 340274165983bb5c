// oxr_boxes.h -- world boxes of placed prims, on the host.
#pragma once
#include <cstdint>
#include <vector>
#include "oxr_bvh.h"
#include "../../include/oxr.h"

namespace oxh {

// Inverse of the 4x4 transform q in double (row convention, last column taken as identity).
void invert_instance(const float* q, double W[4][3]);
// How much longer a distance in front of q may become behind its inverse and back: the
// product of both norms, 3 for a rotation.
double stretch_of(const float* q, const double inv[4][3]);

// The world box of one placed prim from its leaves' own shapes, when they are all spheres,
// zspheres, cylinders or boxes: the union of the leaves' boxes, complemented ones too, so
// every surface point a test can report lies in it. The corners of the prim's object box
// turned into the world reach up to 1.7 times as far (a photomultiplier's bulb and neck, turned
// 45 degrees: 2.2 times the area), and each such box costs node visits and prim tests along
// its rays. reach is the longest distance from a ray's origin to anything in the scene: a
// quadric's discriminant in single precision is off by at most 16 ulps of its square, so a ray
// may be reported to hit a sphere or cylinder up to sqrt(r^2 + 2e-6 reach^2) from its axis
// (twice that bound), and the boxes take that radius. A ray from further away than the scene
// is wide widens the boxes as it meets them (far_pad, oxr_trace.h).
// Instanced CSG, 10M photons: 7.7 -> 6.1 ms; 200k photons 540 -> 466 us; the served stream of 24
// events 9.5 -> 7.9 ms.
//
// The leaves and their transforms are read and inverted once per prim, when this is made.
class LeafBoxes {
public:
    LeafBoxes(const oxr_geometry* g, double reach);
    // Prim's object box ob placed by inst (object to world; inv its inverse), cut to its leaves'
    // boxes where their shapes are known.
    Box placed(int64_t prim, const Box& ob, const float* inst, const double inv[4][3]) const;
private:
    struct Leaf {
        uint32_t type;
        bool turned;             // has a transform of its own
        double to_object[4][3];
        double to_leaf[3][3];    // its inverse, without the translation
        double x, y, z, r;       // centre and radius, or full sides in x, y, z
        double z1, z2;
    };
    bool leaf_box(const Leaf& l, const double A[4][3], const double inv[4][3], Box& out) const;
    double reach_;
    std::vector<Leaf> leaves_;
    std::vector<int64_t> first_;   // of each prim in leaves_, and the end; none: shapes not known
};

} // namespace oxh
