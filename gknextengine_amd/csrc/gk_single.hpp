// gk_single.hpp - one ray per thread, traversed inside the kernel that shades it (the
// differentiable renderer, whose paths live in registers from camera to end).
//
// Same triangle test, box test (the entry and exit distances of k_trace's slab4_ordered, bit
// for bit) and (t, instance, primitive) tie-break as k_trace, so it returns the same hit for
// the same ray. What it takes over from k_trace for speed: leaf children are ordered near to
// far with the internal ones, and in single-level scenes a lane keeps the leaf it reaches and
// goes on with nodes, and the wave tests leaves together once half of its live lanes hold one
// (leaves tested as they are met run the triangle code for a few lanes at a time). The stack's
// first kSingleLds entries are a column per thread in LDS, deeper ones private memory; a ray
// that needs more of them ends, and says so.
#pragma once
#include "gk_scene.hpp"

namespace gk {

constexpr uint32_t kSingleLds = 24;    // stack entries per thread in LDS
// Further entries in private memory. Geometry in nested clusters makes a radix tree of 63-bit
// codes a chain; its wide nodes take three binary levels each and leave three waiting entries
// on each of about 30 levels, in both levels of the scene, with a mark between them. (Leaves
// wait as entries; tested as they are met they took none, and 96 held such a scene.)
constexpr uint32_t kSingleDeep = 168;
constexpr uint32_t kSingleNone = 0xfffffffeu;

struct SingleStack {
    // This thread's column of the LDS part, entry k at [k * blockDim.x]. A pointer of the LDS
    // address space: with a generic one the compiler turns a pop, which reads LDS or private
    // memory, into one flat load of a chosen address.
    typedef __attribute__((address_space(3))) uint32_t* Column;
    Column lds;
    uint32_t* overflow;  // set to 1 when a ray ended because its stack was full
};

// The scenes a traversal is compiled for. In a single-level one of up to kSingleNear nodes a
// node is 32 bits of offset from the array (one register per plane loaded); 2^25 nodes are
// 4 GiB, and beyond, as in two-level scenes, whose nodes lie in two arrays, it is an address
// of 64 bits: 512 x 512, 4 spp, primal and adjoint 1.00 and 1.23 ms against 0.98 and 1.21.
enum class SingleScene { near, far, two };
constexpr uint64_t kSingleNear = uint64_t(1) << 25;

template <bool ANY, SingleScene SCENE>
__device__ inline bool trace_single(const DScene& s, const f3 wO, const f3 wD, const float tmin, const float tmax,
                                    SHit& best, SingleStack stack) {
    constexpr bool TWO = SCENE == SingleScene::two;
    uint32_t deep[kSingleDeep];
    uint32_t sp = 0;
    const uint32_t stride = blockDim.x;
    // An entry past the last one is counted but not kept, and the ray ends with the step that
    // pushed it. (The return mark of an instance always fits: it takes the place of the
    // instance's entry, popped just before.)
    constexpr uint32_t kFull = kSingleLds + kSingleDeep;
    auto push = [&](uint32_t e) {
        if (sp < kSingleLds) stack.lds[sp * stride] = e;
        else if (sp < kFull) deep[sp - kSingleLds] = e;
        ++sp;
    };
    auto pop = [&]() {
        --sp;
        uint32_t e;
        if (sp < kSingleLds) e = stack.lds[sp * stride];
        else e = deep[sp - kSingleLds];
        return e;
    };
    auto is_leaf = [](uint32_t e) { return (e & 0xc0000000u) == kBlasLeaf; };
    f3 O = wO, D = wD;
    f3 rD = f3{safercp(D.x), safercp(D.y), safercp(D.z)};
    // byte offset of each axis's near plane within a node's lo/hi pair
    uint32_t sx, sy, sz;
    auto orient = [&]() {
        sx = (__float_as_uint(rD.x) >> 27) & 16u;
        sy = (__float_as_uint(rD.y) >> 27) & 16u;
        sz = (__float_as_uint(rD.z) >> 27) & 16u;
    };
    orient();
    uint32_t level = TWO ? 0u : 1u, inst = 0u;
    uint32_t node = TWO ? 0u : s.blas_root, leaf = kSingleNone;
    bool found = false, active = true;
    best.t = tmax;
    best.u = best.v = 0.f;
    best.prim = best.inst = 0xffffffffu;
    auto test_leaf = [&](uint32_t e) {
        const uint32_t first = e & kLeafFirstMask, cnt = (e >> 27) & 7u;
        for (uint32_t k = 0; k < cnt; ++k) {
            const TriRec tr = s.tris[first + k];
            const f3 v0 = ld3(tr.v0), e1 = ld3(tr.e1), e2 = ld3(tr.e2);
            const f3 h = cross(D, e2);
            const float a = dot(e1, h);
            if (fabsf(a) < 0.0000001f) continue;
            const float f = 1 / a;
            const f3 sv = O - v0;
            const float u = f * dot(sv, h);
            if (u < 0 || u > 1) continue;
            const f3 q = cross(sv, e1);
            const float v = f * dot(D, q);
            if (v < 0 || u + v > 1) continue;
            const float t = f * dot(e2, q);
            if (!(t > tmin && t < tmax)) continue;
            if (ANY) { found = true; active = false; return; }
            const uint32_t prim = __float_as_uint(tr.v0.w);
            if (!found || t < best.t || (t == best.t && (inst < best.inst || (inst == best.inst && prim < best.prim)))) {
                best.t = t; best.u = u; best.v = v; best.prim = prim; best.inst = inst;
                found = true;
            }
        }
    };
    // One loop trip per wave step, with a single way back to its head: with early ways back
    // (continue) lanes went round apart from the others, a ballot saw only a part of the wave,
    // and its rays were given up as finished.
    bool more = true;
    while (more) {
        bool step = false;  // this lane tests a node
        if (!TWO) {
            if (active) {
                if (leaf == kSingleNone && node != kSingleNone && is_leaf(node)) { leaf = node; node = kSingleNone; }
                if (leaf == kSingleNone && node == kSingleNone && sp == 0u) active = false;
            }
            const bool nodeable = active && (node != kSingleNone ? !is_leaf(node) : sp != 0u);
            const uint64_t live = __ballot(active), bn = __ballot(nodeable);
            const uint64_t bl = __ballot(active && leaf != kSingleNone);
            more = live != 0ull;
            if (bn == 0ull || 2 * __popcll(bl) >= __popcll(live)) {
                if (active && leaf != kSingleNone) {
                    test_leaf(leaf);
                    leaf = kSingleNone;
                }
            } else if (nodeable) {
                step = true;
                if (node == kSingleNone) {
                    const uint32_t e = pop();
                    if (is_leaf(e) && leaf == kSingleNone) leaf = e;
                    else node = e;  // a second leaf waits for the leaf phase
                    step = node != kSingleNone && !is_leaf(e);
                }
            }
        } else {
            more = __ballot(active) != 0ull;
            if (active) {
                step = true;
                if (node == kSingleNone) {
                    step = false;
                    if (sp == 0u) {
                        active = false;
                    } else {
                        const uint32_t e = pop();
                        if (e == kStackMark) {
                            O = wO; D = wD;
                            rD = f3{safercp(D.x), safercp(D.y), safercp(D.z)};
                            orient();
                            level = 0u;
                        } else if (e & kInstFlag) {
                            inst = e & ~kInstFlag;
                            const InstDev& I = s.inst[inst];
                            const float* M = I.inv;
                            const f3 r = f3{M[0] * wO.x + M[1] * wO.y + M[2] * wO.z + M[3],
                                            M[4] * wO.x + M[5] * wO.y + M[6] * wO.z + M[7],
                                            M[8] * wO.x + M[9] * wO.y + M[10] * wO.z + M[11]};
                            const float w = M[12] * wO.x + M[13] * wO.y + M[14] * wO.z + M[15];
                            O = w == 1.0f ? r : r * (1.f / w);
                            D = f3{M[0] * wD.x + M[1] * wD.y + M[2] * wD.z, M[4] * wD.x + M[5] * wD.y + M[6] * wD.z,
                                   M[8] * wD.x + M[9] * wD.y + M[10] * wD.z};
                            rD = f3{safercp(D.x), safercp(D.y), safercp(D.z)};
                            orient();
                            push(kStackMark);
                            level = 1u;
                            node = I.root;
                        } else {
                            node = e;
                            step = !(level != 0u && is_leaf(e));
                        }
                    }
                } else if (level != 0u && is_leaf(node)) {
                    test_leaf(node);
                    node = kSingleNone;
                    step = false;
                }
            }
        }
        if (step) {
            // one node: four boxes, children near to far
            const bool top = TWO && level == 0u;
            constexpr bool NEAR = SCENE == SingleScene::near;
            const char* nb = reinterpret_cast<const char*>((top ? s.tlas : s.blas) + (NEAR ? 0u : node));
            const uint32_t base = NEAR ? node * uint32_t(sizeof(Bvh4Node)) : 0u;
            auto ld = [&](uint32_t off) { return *reinterpret_cast<const float4*>(nb + off); };
            const float4 nx = ld(base | sx), fx = ld((base | sx) ^ 16u);
            const float4 ny = ld((base | sy) + 32u), fy = ld(((base | sy) ^ 16u) + 32u);
            const float4 nz = ld((base | sz) + 64u), fz = ld(((base | sz) ^ 16u) + 64u);
            const uint4 ch = *reinterpret_cast<const uint4*>(nb + base + 96u);
            const float nxs[4] = {nx.x, nx.y, nx.z, nx.w}, fxs[4] = {fx.x, fx.y, fx.z, fx.w};
            const float nys[4] = {ny.x, ny.y, ny.z, ny.w}, fys[4] = {fy.x, fy.y, fy.z, fy.w};
            const float nzs[4] = {nz.x, nz.y, nz.z, nz.w}, fzs[4] = {fz.x, fz.y, fz.z, fz.w};
            float kt[4];
            uint32_t kc[4] = {ch.x, ch.y, ch.z, ch.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float lo = fmaxf(fmaxf((nxs[i] - O.x) * rD.x, (nys[i] - O.y) * rD.y), (nzs[i] - O.z) * rD.z);
                float hi = fminf(fminf((fxs[i] - O.x) * rD.x, (fys[i] - O.y) * rD.y), (fzs[i] - O.z) * rD.z);
                lo = __builtin_fmaf(-__builtin_fabsf(lo), 0x1p-16f, lo);
                hi = __builtin_fmaf(__builtin_fabsf(hi), 0x1p-16f, hi);
                kt[i] = (hi >= lo && hi >= tmin && lo <= best.t) ? lo : __builtin_inff();
            }
            node = kSingleNone;
            if (top) {
                const uint4 me = *reinterpret_cast<const uint4*>(nb + 112u);
                const uint32_t m4[4] = {me.x, me.y, me.z, me.w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (m4[i] == 0u || !(kt[i] < __builtin_inff())) continue;
                    if (m4[i] == 1u) {  // a one-instance leaf is ordered with the other children
                        kc[i] = kInstFlag | s.tlas_prims[kc[i]];
                    } else {
                        for (uint32_t k = 0; k < m4[i]; ++k) push(kInstFlag | s.tlas_prims[kc[i] + k]);
                        kt[i] = __builtin_inff();
                    }
                }
            }
            auto cx = [&](int a, int b) {
                const bool sw = kt[b] < kt[a];
                const float ta = kt[a], tb = kt[b];
                const uint32_t ca = kc[a], cb = kc[b];
                kt[a] = sw ? tb : ta; kt[b] = sw ? ta : tb;
                kc[a] = sw ? cb : ca; kc[b] = sw ? ca : cb;
            };
            cx(0, 1); cx(2, 3); cx(0, 2); cx(1, 3); cx(1, 2);
#pragma unroll
            for (int k = 3; k >= 1; --k)
                if (kt[k] < __builtin_inff()) push(kc[k]);
            if (kt[0] < __builtin_inff()) {
                if (TWO && (kc[0] & kInstFlag)) push(kc[0]);  // instances are entered by the pop path
                else node = kc[0];
            }
            if (sp > kFull) active = false;
        }
    }
    if (sp > kFull) atomicOr(stack.overflow, 1u);
    return found;
}

}  // namespace gk
