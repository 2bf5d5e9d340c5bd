// Walks of four- and eight-wide trees collapsed from many binary ones hold no
// more stack entries than walkStackEntries says, and reach every leaf once.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "scene_build.h"

using namespace wpt;

namespace {

std::mt19937 rng(7);

float uniform(float lo, float hi) { return std::uniform_real_distribution<float>(lo, hi)(rng); }

// A binary tree of `leaves` leaves in preorder; `lean`: the share of leaves
// that goes left (0 and 1: a chain).
uint32_t grow(HostBvh& t, uint32_t leaves, float lean, uint32_t& depth) {
    if (leaves == 1) {
        depth = 0;
        t.order.push_back(t.primCount());
        return kLeafBit | (t.primCount() - 1u);
    }
    uint32_t self = static_cast<uint32_t>(t.nodes.size());
    t.nodes.push_back(BvhNode{});
    float share = lean < 0.0f ? uniform(0.0f, 1.0f) : lean;
    uint32_t left = std::min(leaves - 1u, std::max(1u, static_cast<uint32_t>(share * leaves)));
    uint32_t dl, dr;
    uint32_t l = grow(t, left, lean, dl), r = grow(t, leaves - left, lean, dr);
    BvhNode& n = t.nodes[self];
    n.lmaxx = uniform(0, 1), n.lmaxy = uniform(0, 1), n.lmaxz = uniform(0, 1);
    n.rmaxx = uniform(0, 1), n.rmaxy = uniform(0, 1), n.rmaxz = uniform(0, 1);
    n.left = l;
    n.right = r;
    depth = 1 + std::max(dl, dr);
    return self;
}

struct Need {
    uint32_t entries, leaves;
};

// The most entries a walk below `child` holds: every other child of a node
// waits on the stack while the deepest is walked (`all`: and that one too
// before it is popped, as the eight-wide walk does).
template <class Children>
Need need(uint32_t child, bool all, const Children& children) {
    if (child & kLeafBit) return {0, 1};
    Need r{0, 0};
    uint32_t deepest = 0, count = 0;
    children(child, [&](uint32_t c) {
        if (c == kInvalid) return;
        Need n = need(c, all, children);
        deepest = std::max(deepest, n.entries);
        r.leaves += n.leaves;
        ++count;
    });
    r.entries = std::max(count - 1u + deepest, all ? count : 0u);
    return r;
}

Need quadNeed(const HostBvh& t) {
    return need(t.primCount() > 1 ? 0u : kLeafBit, false, [&](uint32_t i, auto&& visit) {
        const QuadNode q = quadNode(t.nodes.data(), i);
        for (uint32_t c : q.child) visit(c);
    });
}

int failures = 0;
uint32_t fullest = 0;  // entries that a walk of an accepted depth needed

void expect(bool ok, const char* what, const HostBvh& t, uint32_t a, uint32_t b) {
    if (ok) return;
    std::printf("%s: %u leaves, depth %u: %u against %u\n", what, t.primCount(), t.depth, a, b);
    ++failures;
}

void check(const HostBvh& t, const HostBvh& below) {
    HostSceneData s;
    Need q = quadNeed(t);
    s.flat = t;
    expect(q.entries <= walkStackEntries(s), "flat", t, q.entries, walkStackEntries(s));
    expect(q.leaves == t.primCount(), "leaves", t, q.leaves, t.primCount());
    uint32_t stack = 0;
    s.flatWide = collapseWide(t, &stack);
    s.flatWideStack = stack;
    if (!s.flatWide.empty()) {
        Need w = need(0u, true, [&](uint32_t i, auto&& visit) {
            for (uint32_t c : s.flatWide[i].child) visit(c);
        });
        expect(w.entries <= walkStackEntries(s), "wide", t, w.entries, walkStackEntries(s));
        expect(w.leaves == t.primCount(), "wide leaves", t, w.leaves, t.primCount());
    }
    HostSceneData two;
    two.tlas = t;
    two.maxBlasDepth = below.depth;
    uint32_t both = q.entries + quadNeed(below).entries;
    expect(both <= walkStackEntries(two), "two levels", t, both, walkStackEntries(two));
    if (t.depth + below.depth <= 62) {
        fullest = std::max(fullest, both);
        expect(both <= 96, "limit", t, both, 96);
    }
}

}  // namespace

int main() {
    std::vector<HostBvh> trees;
    for (uint32_t leaves : {1u, 2u, 3u, 4u, 5u, 6u, 7u, 8u, 9u, 17u, 32u, 33u, 63u})
        for (float lean : {0.0f, 1.0f, 0.5f, 0.34f, 0.9f, -1.0f, -1.0f, -1.0f}) {
            HostBvh t;
            uint32_t depth = 0;
            t.root = grow(t, leaves, lean, depth);
            t.depth = depth;
            trees.push_back(std::move(t));
        }
    for (uint32_t n : {1u, 2u, 3u, 5u, 40u, 3000u})
        for (bool median : {false, true}) {
            std::vector<Aabb> boxes(n);
            for (uint32_t i = 0; i < n; ++i)
                for (int k = 0; k < 3; ++k) {
                    // Half of them at sizes and distances that halve: deep trees.
                    float at = i % 2 ? uniform(-1, 1) : std::ldexp(1.0f, -static_cast<int>(i % 60)), size = 0.1f * std::fabs(at);
                    boxes[i].mn[k] = at - size;
                    boxes[i].mx[k] = at + size;
                }
            trees.push_back(buildBvh2(boxes, 1, median));
        }
    std::vector<TriShade> slivers(300);
    for (TriShade& t : slivers) {
        t.v0 = Vec3(uniform(-1, 1), uniform(-1, 1), uniform(-1, 1));
        t.v1 = t.v0 + Vec3(uniform(-4, 4), uniform(-4, 4), uniform(-4, 4));
        t.v2 = t.v1 + Vec3(0.01f, 0.0f, 0.01f);
    }
    trees.push_back(buildSpatialSplitBvh2(slivers));
    for (size_t i = 0; i < trees.size(); ++i)
        for (size_t k : {i, (i * 7 + 3) % trees.size(), trees.size() - 1 - i}) check(trees[i], trees[k]);
    std::printf("%zu trees, fullest walk of an accepted depth %u entries, %d failures\n", trees.size(), fullest, failures);
    return failures ? 1 : 0;
}
