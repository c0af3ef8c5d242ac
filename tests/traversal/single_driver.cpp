// The traversal of one ray per thread (csrc/gk_single.hpp) on the CPU: hits against a test of
// every triangle, and trees whose waiting children fill its stack.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>
#include <vector>

#include <sys/mman.h>

#include "gk_single.hpp"

using namespace gk;

namespace {

using Box = std::pair<f3, f3>;
constexpr float kBig = 1e9f;

Bvh4Node empty_node() {
    Bvh4Node n{};
    n.lox = n.loy = n.loz = make_float4(1e30f, 1e30f, 1e30f, 1e30f);
    n.hix = n.hiy = n.hiz = make_float4(1e30f, 1e30f, 1e30f, 1e30f);
    return n;
}
void set_child(Bvh4Node& n, int k, const Box& b, uint32_t child, uint32_t meta) {
    (&n.lox.x)[k] = b.first.x; (&n.hix.x)[k] = b.second.x;
    (&n.loy.x)[k] = b.first.y; (&n.hiy.x)[k] = b.second.y;
    (&n.loz.x)[k] = b.first.z; (&n.hiz.x)[k] = b.second.z;
    (&n.child.x)[k] = child;
    (&n.meta.x)[k] = meta;
}
uint32_t tri_leaf(uint32_t first, uint32_t count) { return kBlasLeaf | (count << 27) | first; }
TriRec triangle(f3 a, f3 e1, f3 e2, uint32_t prim) {
    return TriRec{make_float4(a.x, a.y, a.z, __uint_as_float(prim)), make_float4(e1.x, e1.y, e1.z, 0.f),
                  make_float4(e2.x, e2.y, e2.z, 0.f)};
}
// an instance moved by d
InstDev moved(f3 d, uint32_t root) {
    return InstDev{{1, 0, 0, -d.x, 0, 1, 0, -d.y, 0, 0, 1, -d.z, 0, 0, 0, 1}, root};
}

struct Run {
    bool found;
    SHit hit;
    uint32_t overflow;
};
template <bool ANY, SingleScene SCENE>
Run trace(const DScene& s, f3 O, f3 D) {
    std::vector<uint32_t> lds(kSingleLds);  // exactly the entries a thread has
    Run r{};
    r.found = trace_single<ANY, SCENE>(s, O, D, 0.f, 1e30f, r.hit, SingleStack{lds.data(), &r.overflow});
    return r;
}

struct Mesh {
    std::vector<TriRec> tris;
    std::vector<Box> boxes;
    std::vector<Bvh4Node> nodes;
    uint32_t build(int a, int b) {
        const uint32_t id = uint32_t(nodes.size());
        nodes.push_back(empty_node());
        Bvh4Node n = empty_node();
        for (int k = 0; k < 4; ++k) {
            const int s = a + (b - a) * k / 4, e = a + (b - a) * (k + 1) / 4;
            if (s == e) continue;
            Box x = boxes[s];
            for (int i = s; i < e; ++i) x = {fmin3(x.first, boxes[i].first), fmax3(x.second, boxes[i].second)};
            if (e - s <= 4) set_child(n, k, x, tri_leaf(uint32_t(s), uint32_t(e - s)), uint32_t(e - s));
            else set_child(n, k, x, build(s, e), 0u);
        }
        nodes[id] = n;
        return id;
    }
};

int random_scenes() {
    std::mt19937 g(1);
    std::uniform_real_distribution<float> U(-1.f, 1.f);
    Mesh m;
    for (uint32_t i = 0; i < 200; ++i) {
        const f3 a{U(g), U(g), U(g)}, e1{U(g) * .4f, U(g) * .4f, U(g) * .4f}, e2{U(g) * .4f, U(g) * .4f, U(g) * .4f};
        m.tris.push_back(triangle(a, e1, e2, i));
        m.boxes.push_back({fmin3(a, fmin3(a + e1, a + e2)), fmax3(a, fmax3(a + e1, a + e2))});
    }
    m.build(0, 200);
    Box all = m.boxes[0];
    for (const Box& b : m.boxes) all = {fmin3(all.first, b.first), fmax3(all.second, b.second)};
    const f3 at[2] = {f3{0.f, 0.f, 0.f}, f3{1.5f, 0.25f, 0.f}};
    std::vector<InstDev> inst = {moved(at[0], 0), moved(at[1], 0)};
    const uint32_t prims[2] = {1, 0};
    Bvh4Node top = empty_node();
    for (int k = 0; k < 2; ++k) set_child(top, k, {all.first + at[prims[k]], all.second + at[prims[k]]}, uint32_t(k), 1u);
    const DScene s{m.nodes.data(), m.tris.data(), &top, prims, inst.data(), 0u};
    int bad = 0, hits = 0;
    for (int r = 0; r < 20000; ++r) {
        const f3 O{U(g), U(g), U(g)}, D{U(g), U(g), U(g)};
        float bt[2] = {1e30f, 1e30f};
        uint32_t bp[2] = {~0u, ~0u}, bi[2] = {~0u, ~0u};
        for (int two = 0; two < 2; ++two)
            for (uint32_t ii = 0; ii < (two ? 2u : 1u); ++ii)
                for (const TriRec& t : m.tris) {
                    const f3 o = O + f3{-at[ii].x, -at[ii].y, -at[ii].z};
                    const f3 e1 = ld3(t.e1), e2 = ld3(t.e2), h = cross(D, e2);
                    const float a = dot(e1, h);
                    if (std::fabs(a) < 1e-7f) continue;
                    const float f = 1 / a;
                    const f3 sv = o - ld3(t.v0);
                    const float u = f * dot(sv, h);
                    if (u < 0 || u > 1) continue;
                    const f3 q = cross(sv, e1);
                    const float v = f * dot(D, q);
                    if (v < 0 || u + v > 1) continue;
                    const float d = f * dot(e2, q);
                    if (d > 0 && d < bt[two]) { bt[two] = d; bp[two] = __float_as_uint(t.v0.w); bi[two] = ii; }
                }
        const Run one = trace<false, SingleScene::near>(s, O, D), two = trace<false, SingleScene::two>(s, O, D);
        const Run any = trace<true, SingleScene::near>(s, O, D), any2 = trace<true, SingleScene::two>(s, O, D);
        hits += one.found + two.found;
        bad += one.hit.prim != bp[0] || two.hit.prim != bp[1] || two.hit.inst != bi[1];
        bad += (one.found && one.hit.t != bt[0]) || (two.found && two.hit.t != bt[1]);
        bad += any.found != one.found || any2.found != two.found;
        const Run far = trace<false, SingleScene::far>(s, O, D);
        bad += far.found != one.found || far.hit.t != one.hit.t || far.hit.prim != one.hit.prim;
        bad += one.overflow | two.overflow | any.overflow | any2.overflow;
    }
    printf("random: %d bad of %d hits\n", bad, hits);
    return bad || hits < 1000;
}

// A ray along +x through a chain of `levels` wide nodes: child 0 is the next node and the
// nearest, the other three wait on the stack. In the BLAS they are leaves; of mesh 0, child 3 of
// the last node, the last to be pushed, holds the triangle at x = 20 that the ray hits.
std::vector<Bvh4Node> blas_chain(uint32_t levels) {
    std::vector<Bvh4Node> n(levels + 1u, empty_node());  // the last one: mesh 1, a node without children
    for (uint32_t l = 0; l < levels; ++l)
        for (int k = 0; k < 4; ++k) {
            const Box b{f3{k == 0 ? 1.f : 10.f + float(3 - k), -kBig, -kBig}, f3{kBig, kBig, kBig}};
            const bool last = l + 1 == levels;
            if (k == 0 && !last) set_child(n[l], 0, b, l + 1, 0u);
            else set_child(n[l], k, b, tri_leaf(last && k == 3 ? 0u : 1u, 1u), 1u);
        }
    return n;
}
std::vector<TriRec> chain_tris() {
    return {triangle(f3{20.f, -1.f, -1.f}, f3{0.f, 4.f, 0.f}, f3{0.f, 0.f, 4.f}, 7u),
            triangle(f3{20.f, 50.f, 50.f}, f3{0.f, 1.f, 0.f}, f3{0.f, 0.f, 1.f}, 8u)};
}
// The same in the TLAS, where the waiting children are nodes of one instance leaf each. The
// last node's nearest holds mesh 0, entered while all others wait, and they mesh 1.
std::vector<Bvh4Node> tlas_chain(uint32_t levels) {
    std::vector<Bvh4Node> n(levels, empty_node());
    for (uint32_t l = 0; l < levels; ++l)
        for (int k = 0; k < 4; ++k) {
            const Box b{f3{k == 0 ? 1.f : 10.f + float(3 - k), -kBig, -kBig}, f3{kBig, kBig, kBig}};
            const bool last = l + 1 == levels;
            if (k == 0 && !last) { set_child(n[l], 0, b, l + 1, 0u); continue; }
            const uint32_t id = uint32_t(n.size());
            n.push_back(empty_node());
            set_child(n[id], 0, b, k == 0 ? 0u : 1u, 1u);
            set_child(n[l], k, b, id, 0u);
        }
    return n;
}

int chains(uint32_t top_levels, uint32_t levels, bool want_overflow) {
    const std::vector<Bvh4Node> blas = blas_chain(levels), tlas = tlas_chain(top_levels);
    const std::vector<TriRec> tris = chain_tris();
    const uint32_t prims[2] = {0, 1};
    const InstDev inst[2] = {moved(f3{0.f, 0.f, 0.f}, 0u), moved(f3{0.f, 0.f, 0.f}, levels)};
    const DScene s{blas.data(), tris.data(), tlas.data(), prims, inst, 0u};
    const f3 O{0.f, 0.f, 0.f}, D{1.f, 0.f, 0.f};
    int bad = 0;
    auto check = [&](const char* what, const Run& r, bool closest) {
        const bool ok = want_overflow ? r.overflow == 1u
                                      : r.overflow == 0u && r.found && (!closest || (r.hit.t == 20.f && r.hit.prim == 7u));
        printf("%s, %u over %u levels: found %d overflow %u %s\n", what, top_levels, levels, int(r.found), r.overflow,
               ok ? "ok" : "WRONG");
        bad += !ok;
    };
    if (top_levels == 0) {
        check("closest, one level", trace<false, SingleScene::near>(s, O, D), true);
        check("closest, one level, far", trace<false, SingleScene::far>(s, O, D), true);
        check("any, one level", trace<true, SingleScene::near>(s, O, D), false);
    } else {
        check("closest, two levels", trace<false, SingleScene::two>(s, O, D), true);
        check("any, two levels", trace<true, SingleScene::two>(s, O, D), false);
    }
    return bad;
}

// A root at node `at` of an array that is reserved but not filled, with two leaves: the hit
// lies in a node whose offset passes 32 bits when `at` is 2^25 - 1 or more.
template <SingleScene SCENE>
int far_node(uint32_t at) {
    const size_t bytes = (size_t(at) + 2u) * sizeof(Bvh4Node);
    void* mem = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (mem == MAP_FAILED) return 1;
    Bvh4Node* nodes = static_cast<Bvh4Node*>(mem);
    const Box all{f3{1.f, -kBig, -kBig}, f3{kBig, kBig, kBig}};
    nodes[at] = nodes[at + 1u] = empty_node();
    set_child(nodes[at], 0, all, at + 1u, 0u);
    set_child(nodes[at + 1u], 2, all, tri_leaf(0u, 2u), 2u);
    const std::vector<TriRec> tris = chain_tris();
    const uint32_t prims[1] = {0};
    const InstDev inst[1] = {moved(f3{0.f, 0.f, 0.f}, at)};
    Bvh4Node top = empty_node();
    set_child(top, 0, all, 0u, 1u);
    const DScene s{nodes, tris.data(), &top, prims, inst, at};
    const Run r = trace<false, SCENE>(s, f3{0.f, 0.f, 0.f}, f3{1.f, 0.f, 0.f});
    const bool ok = r.found && r.hit.t == 20.f && r.hit.prim == 7u;
    printf("node %u: found %d %s\n", at, int(r.found), ok ? "ok" : "WRONG");
    munmap(mem, bytes);
    return !ok;
}

}  // namespace

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "random") return random_scenes();
    if (what == "chain" && argc == 5)
        return chains(uint32_t(atoi(argv[2])), uint32_t(atoi(argv[3])), atoi(argv[4]) != 0);
    if (what == "far" && argc == 3) {
        const uint32_t at = uint32_t(atoll(argv[2]));
        int bad = far_node<SingleScene::far>(at) + far_node<SingleScene::two>(at);
        if (uint64_t(at) + 2u <= kSingleNear) bad += far_node<SingleScene::near>(at);
        return bad;
    }
    return 2;
}
