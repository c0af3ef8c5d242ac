// The part of the device scene that the one-ray traversal reads.
#pragma once
#include "gk_math.hpp"

namespace gk {
struct InstDev { float inv[16]; uint32_t root; };
struct DScene {
    const Bvh4Node* blas;
    const TriRec* tris;
    const Bvh4Node* tlas;
    const uint32_t* tlas_prims;
    const InstDev* inst;
    uint32_t blas_root;
};
struct SHit { float t, u, v; uint32_t prim, inst; };
}  // namespace gk
