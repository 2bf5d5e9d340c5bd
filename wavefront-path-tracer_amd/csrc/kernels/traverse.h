// Closest-hit and shadow any-hit traversal over the device scene.
//
// Reference: include/renderer/device_traversal.cuh:24-91 (sphere/triangle
// tests), :182-222 (slab test), :239-313 (BLAS BVH2), :789-878 (sphere leaf,
// mesh instance, TLAS), :1035-1184 (isOccluded, traceRay).
//
// The node layout differs from the reference (128 B nodes holding the boxes of
// four children, or 256 B eight-wide nodes for flat triangles, see
// device_scene.h), and one loop serves closest-hit and any-hit queries.  The primitive tests
// are the reference's, in the same FP32 operation order, so each candidate's
// distance and barycentrics are bit-identical to the reference's.  The
// nearest hit is the candidate first in (distance, category, instance,
// primitive) order.  That is the reference's result whenever the nearest
// distance is held by one primitive, and across categories on exact ties;
// on an exact tie inside one tree (a ray through a shared edge) the
// reference keeps whichever triangle its tree visits first, while this
// order keeps the lower index, whatever the tree.
#pragma once

#include "../common/vec.h"
#include "../scene/device_scene.h"
#include "material.h"

namespace wpt {

constexpr float kNoHit = 1e30f;

// Winning primitive of a closest-hit query.
struct HitRecord {
    float t;
    float u, v;
    uint32_t kind;      // WPT_HIT_* values
    uint32_t instance;  // instance index for instance triangles
    uint32_t prim;      // sphere / triangle index in the caller's order
    uint32_t material;  // resolved (override applied)
    uint32_t rank;      // tie order of the hit's category (kRank*)
};

// Hits at exactly the same distance are ordered by category -- spheres,
// direct-instance triangles, static triangles, TLAS-instance triangles,
// flat triangles -- then by instance, then by primitive.  Across categories
// this is the reference's outcome (traceRay visits the categories in that
// order and a sphere displaces an equally distant triangle,
// device_traversal.cuh:789-800,1115-1184).  Within a BVH the reference keeps
// whichever tie its tree visits first; fixing the order instead makes the
// nearest hit independent of tree shape and visit order, so that any BVH
// (binary or wide, host- or device-built) gives the same hits.
constexpr uint32_t kRankSphere = 0, kRankDirectInstance = 1, kRankStatic = 2, kRankTlasInstance = 3, kRankFlat = 4;

// Boxes are culled only beyond tieReach(closestT): a box holding a hit at
// exactly closestT can have a computed entry distance a few ulps above it,
// and must still be opened for that hit to take part in the tie order.
WPT_HD float tieReach(float closestT) { return closestT * 1.00000095f; }

WPT_HD bool nearer(float t, uint32_t rank, uint32_t instance, uint32_t prim, const HitRecord& best) {
    if (t != best.t) return t < best.t;
    if (rank != best.rank) return rank < best.rank;
    if (instance != best.instance) return instance < best.instance;
    return prim < best.prim;
}

// Alpha mask of a candidate triangle hit (reference intersectTriangleHit,
// device_traversal.cuh:146-151): masked materials below their cutoff are
// passed through; textured ones test opacity x albedo alpha at the hit.
WPT_HD bool textureCutAway(const DevScene& s, uint32_t material, const TriShade& tri, float u, float v) {
    const Material& m = s.materials[material];
    return materialOpacity(s, m, triangleUv(tri, u, v), triangleUv1(s, tri, u, v)) < m.alphaCutoff;
}

// `Full` kernels serve every scene; the others only scenes without
// environment maps, punctual lights or texture bindings, and leave that code
// out (it costs registers on every path).
template <bool Full>
WPT_HD bool cutAway(const DevScene& s, uint32_t material, const TriShade* tris, uint32_t prim, float u, float v) {
    uint8_t policy = s.materialCutout[material];
    if (policy == kCutNever) return false;
    return policy == kCutAlways || (Full && textureCutAway(s, material, tris[prim], u, v));
}

constexpr uint32_t kHitNone = 0, kHitSphere = 1, kHitStatic = 2, kHitInstance = 3, kHitFlat = 4;

WPT_HD HitRecord emptyHit() {
    HitRecord h;
    h.t = kNoHit;
    h.u = h.v = 0.0f;
    h.kind = kHitNone;
    h.instance = kInvalid;
    h.prim = kInvalid;
    h.material = kInvalid;
    h.rank = kInvalid;
    return h;
}

// Quadratic with unnormalized b; nearest root beyond the cutoff.
WPT_HD bool intersectSphere(const Ray& ray, const Vec3& center, float radius, float& t) {
    Vec3 oc = ray.origin - center;
    float a = dot(ray.direction, ray.direction);
    float b = 2.0f * dot(oc, ray.direction);
    float c = dot(oc, oc) - radius * radius;
    float discriminant = b * b - 4.0f * a * c;
    if (discriminant < 0.0f) return false;
    float sqrtD = sqrtf(discriminant);
    float t0 = (-b - sqrtD) / (2.0f * a);
    float t1 = (-b + sqrtD) / (2.0f * a);
    if (t0 > kRayMinDistance) {
        t = t0;
        return true;
    }
    if (t1 > kRayMinDistance) {
        t = t1;
        return true;
    }
    return false;
}

// Moller-Trumbore with the determinant guard relative to its own products.
WPT_HD bool intersectEdges(const Ray& ray, const Vec3& v0, const Vec3& edge1, const Vec3& edge2, float& t, float& u,
    float& v) {
    Vec3 p = cross(ray.direction, edge2);
    float determinant = dot(edge1, p);
    const Vec3& d = ray.direction;
    float scale = fabsf(edge1.x) * (fabsf(d.y * edge2.z) + fabsf(d.z * edge2.y)) +
        fabsf(edge1.y) * (fabsf(d.z * edge2.x) + fabsf(d.x * edge2.z)) +
        fabsf(edge1.z) * (fabsf(d.x * edge2.y) + fabsf(d.y * edge2.x));
    if (!isFinite(determinant) || fabsf(determinant) <= 8.0f * kFltEpsilon * scale) return false;
    float inverseDeterminant = 1.0f / determinant;
    Vec3 originToVertex = ray.origin - v0;
    u = dot(originToVertex, p) * inverseDeterminant;
    if (u < 0.0f || u > 1.0f) return false;
    Vec3 q = cross(originToVertex, edge1);
    v = dot(ray.direction, q) * inverseDeterminant;
    if (v < 0.0f || u + v > 1.0f) return false;
    t = dot(edge2, q) * inverseDeterminant;
    return t > kRayMinDistance;
}

WPT_HD bool intersectTriangle(const Ray& ray, const Vec3& v0, const Vec3& v1, const Vec3& v2, float& t, float& u,
    float& v) {
    return intersectEdges(ray, v0, v1 - v0, v2 - v0, t, u, v);
}

struct RayInv {
    Ray ray;
    Vec3 inv;
};

WPT_HD RayInv makeRayInv(const Ray& r) {
    RayInv ri;
    ri.ray = r;
    ri.inv = Vec3(1.0f / r.direction.x, 1.0f / r.direction.y, 1.0f / r.direction.z);
    return ri;
}

WPT_HD bool slab(const RayInv& r, float mnx, float mny, float mnz, float mxx, float mxy, float mxz, float closestT,
    float& nearT) {
    float tx0 = (mnx - r.ray.origin.x) * r.inv.x;
    float tx1 = (mxx - r.ray.origin.x) * r.inv.x;
    float ty0 = (mny - r.ray.origin.y) * r.inv.y;
    float ty1 = (mxy - r.ray.origin.y) * r.inv.y;
    float tz0 = (mnz - r.ray.origin.z) * r.inv.z;
    float tz1 = (mxz - r.ray.origin.z) * r.inv.z;
    float tmin = fmaxf(fminf(tx0, tx1), fmaxf(fminf(ty0, ty1), fminf(tz0, tz1)));
    float tmax = fminf(fmaxf(tx0, tx1), fminf(fmaxf(ty0, ty1), fmaxf(tz0, tz1)));
    nearT = tmin;
    return tmax >= fmaxf(tmin, kRayMinDistance) && tmin <= tieReach(closestT);
}

// A ray prepared for the boxes of QuadNodes: per axis the inverse direction
// and the biases that make a plane's entry distance fma(plane, inv, nearBias)
// and its exit distance fma(plane, inv, farBias), half the operations of
// slab().
//
// This box test passes every box that slab() passes: fma(plane, inv, -origin *
// inv) is off by at most 2 u |origin * inv| (u = 2^-24: the product's and the
// bias's rounding) and u of its value, slab's distance by 3 u of its value;
// the biases move entries down and exits up by 8 u |origin * inv|, and the
// interval may be empty by 32 u (boxReach), against the 16 u of tieReach.  It
// passes some boxes more, so a candidate found in a leaf counts only if slab()
// passes the leaf's own box (leafOpen; slotOpen for TLAS leaves and for the
// clipped triangles of spatial splits): slab's distances grow with the box, so
// that this one test stands for the boxes around it, and hits are those of a
// binary walk that tests every box with slab() in the same order (visitQuad;
// the biases can put two entries in another order when origin * inv is a
// million times their distances: 1 of 150 million rays aimed at edges; clipped
// boxes reach out of those around them by rounding, where a binary walk misses a
// few hits at their seams that this one finds: 1 in 100,000 such rays).
// Rays with a component outside 2^-60 .. 2^60 in size (a zero component of the
// direction has an infinite inverse), which would overflow, take slab() at
// every node: their nearBias.x is NaN.
struct BoxRay {
    Ray ray;
    Vec3 inv, nearBias, farBias;
    WPT_HD RayInv exact() const { return RayInv{ray, inv}; }
    WPT_HD bool regular() const { return nearBias.x == nearBias.x; }
};

WPT_HD bool boxAxis(float origin, float inv, float& nearBias, float& farBias) {
    constexpr float kLarge = 1.1529215e18f, kSmall = 8.6736174e-19f;  // 2^60, 2^-60
    float oi = origin * inv;
    float slack = fabsf(oi) * 4.76837158e-7f;  // 2^-21
    nearBias = -oi - slack;
    farBias = slack - oi;
    return fabsf(inv) <= kLarge && fabsf(inv) >= kSmall && fabsf(origin) <= kLarge;
}

WPT_HD BoxRay makeBoxRay(const Ray& ray, const Vec3& inv) {
    BoxRay b;
    b.ray = ray;
    b.inv = inv;
    bool x = boxAxis(ray.origin.x, inv.x, b.nearBias.x, b.farBias.x);
    bool y = boxAxis(ray.origin.y, inv.y, b.nearBias.y, b.farBias.y);
    bool z = boxAxis(ray.origin.z, inv.z, b.nearBias.z, b.farBias.z);
    if (!(x && y && z)) b.nearBias.x = __builtin_nanf("");
    return b;
}

// The leaf box of a triangle in a tree over whole triangles.
WPT_HD bool leafOpen(const RayInv& r, const Vec3& a, const Vec3& b, const Vec3& c, float closestT) {
    float nearT;
    return slab(r, fminf(a.x, fminf(b.x, c.x)), fminf(a.y, fminf(b.y, c.y)), fminf(a.z, fminf(b.z, c.z)),
        fmaxf(a.x, fmaxf(b.x, c.x)), fmaxf(a.y, fmaxf(b.y, c.y)), fmaxf(a.z, fmaxf(b.z, c.z)), closestT, nearT);
}

// The leaf box of a slot, from a list of them: TLAS leaves, clipped triangles.
WPT_HD bool slotOpen(const float4* boxes, const RayInv& r, uint32_t slot, float closestT) {
    const float4 mn = boxes[2 * slot], mx = boxes[2 * slot + 1];
    float nearT;
    return slab(r, mn.x, mn.y, mn.z, mx.x, mx.y, mx.z, closestT, nearT);
}

constexpr float kBoxMissed = __builtin_inff();

// Distances up to boxReach(t) count as within t for the boxes of QuadNodes
// and for the stack entries they push.
WPT_HD float boxReach(float t) { return t * 1.00000191f; }  // 1 + 2^-19

WPT_HD Vec3 xyz(const float4& f) { return Vec3(f.x, f.y, f.z); }
WPT_HD uint32_t wbits(const float4& f) { return bitsOf(f.w); }

// Traversal stacks hold (node pointer, entry distance) pairs and expose
// `size`, push, pop and clear.  This private-array stack serves host-side
// builds of the traversal code; the kernels use an LDS-resident stack with
// the same interface.  The scene build rejects trees whose combined
// TLAS+BLAS depth (of the binary trees, plus two) exceeds kMaxTreeDepth.  A
// four-wide level spans at least two binary levels on the way to any interior
// child and leaves at most three entries behind, so a walk of a TLAS d deep
// over a BLAS e deep (d + e <= 62) holds at most 3 (ceil(d/2) + ceil(e/2))
// <= 96 entries.
constexpr uint32_t kMaxTreeDepth = 64;
constexpr uint32_t kMaxStackDepth = 96;
struct PrivateStack {
    static constexpr uint32_t kCapacity = kMaxStackDepth;
    uint32_t node[kCapacity];
    float tmin[kCapacity];
    uint32_t size = 0;
    WPT_HD void push(uint32_t n, float t) {
        node[size] = n;
        tmin[size] = t;
        ++size;
    }
    WPT_HD void pop(uint32_t& n, float& t) {
        --size;
        n = node[size];
        t = tmin[size];
    }
    WPT_HD void clear() { size = 0; }
    // Entry k below the top (k < 8).
    WPT_HD uint2 peek(uint32_t k) const { return make_uint2(node[size - 1 - k], bitsOf(tmin[size - 1 - k])); }
    WPT_HD void poke(uint32_t k, uint2 e) {
        node[size - 1 - k] = e.x;
        tmin[size - 1 - k] = fromBits32(e.y);
    }
};

// Pops until an entry within `reach`, the reach of the box test that pushed
// the entries: boxReach(closestT), or tieReach(closestT) for slab() alone;
// false when the traversal level (entries above `base`) is exhausted.
template <class Stack>
WPT_HD bool popLive(Stack& stack, uint32_t base, float reach, uint32_t& cur) {
    while (stack.size > base) {
        float t;
        stack.pop(cur, t);
        if (t <= reach) return true;
    }
    return false;
}

// As a binary walk: the right one first unless the left one is nearer.
WPT_HD void orderPair(float& ta, uint32_t& a, float& tb, uint32_t& b) {
    bool swap = tb <= ta;
    float t = swap ? tb : ta;
    uint32_t c = swap ? b : a;
    tb = swap ? ta : tb;
    b = swap ? a : b;
    ta = t;
    a = c;
}

// visitQuad for the rays that are not regular(): the children's entry distances
// and those of the two pairs' unions.
WPT_HD void exactBoxes(const QuadNode& n, const RayInv& r, float closestT, float t[kQuadChildren], float pair[2]) {
    for (uint32_t k = 0; k < kQuadChildren; ++k) {
        float tmin;
        bool hit = n.child[k] != kInvalid &&
            slab(r, n.mn[0][k], n.mn[1][k], n.mn[2][k], n.mx[0][k], n.mx[1][k], n.mx[2][k], closestT, tmin);
        t[k] = hit ? tmin : kBoxMissed;
    }
    for (uint32_t k = 0; k < 2; ++k) {
        float mn[3], mx[3];
        for (int c = 0; c < 3; ++c) {
            mn[c] = fminf(n.mn[c][2 * k], n.mn[c][2 * k + 1]);
            mx[c] = fmaxf(n.mx[c][2 * k], n.mx[c][2 * k + 1]);
        }
        (void)slab(r, mn[0], mn[1], mn[2], mx[0], mx[1], mx[2], closestT, pair[k]);
    }
}

// One interior node: the first child whose box the ray reaches becomes `cur`,
// the others are pushed, the last first; false when there is none.
// A walk is bound by VALU issue where the chip is full and by the latency of
// its chain of node fetches where it is not.  Four boxes a visit halve the
// chain, for the 128 B line that is fetched either way, and take about 110
// vector instructions where two binary visits with ordered planes took 150:
// sphere field 1920x1080, 64 spp, closest-hit passes 58.4 -> 39.9 ms; terrain,
// 16 spp, 66 -> 49 ms and event rays 62 -> 45 ms; 2M camera rays 529 -> 338 us.
// Which plane of an axis a ray enters through depends on the sign of its
// direction alone, so a lane loads each node's entry and exit planes as such
// (minima at byte 0, 16, 32, maxima 48 further) instead of ordering them.
// The order is that of a binary walk: the pair whose union is entered first,
// its nearer child first, distances behind the origin included.  Which of two
// triangles counts depends on it where one is hit a little before the ray
// enters its box (rounding at an edge) and the other's distance lies between:
// with all four children ordered by their own clamped distances up to 10 of
// 400,000 rays aimed at edges under a median tree hit another triangle than in a
// binary walk, so none.  That order took 2 to 5% less time (a child of a child
// could fill a slot left free, and fewer registers were live; with the entries
// of all four children computed first, 3 to 5 spills less but terrain 139.9 ->
// 146.2 ms; with one slack for the three axes instead of biases, flat trees 350
// -> 785 us, as rays almost parallel to an axis pass nearly every box).
template <class Stack>
WPT_HD bool visitQuad(const QuadNode* nodes, const BoxRay& r, float closestT, uint32_t& cur, Stack& stack) {
    const char* p = reinterpret_cast<const char*>(nodes + cur);
    const uint32_t ox = (bitsOf(r.inv.x) >> 31) * 48u, oy = (bitsOf(r.inv.y) >> 31) * 48u,
                   oz = (bitsOf(r.inv.z) >> 31) * 48u;
    const float4 nx = *reinterpret_cast<const float4*>(p + ox), fx = *reinterpret_cast<const float4*>(p + (ox ^ 48u)),
                 ny = *reinterpret_cast<const float4*>(p + oy + 16), fy = *reinterpret_cast<const float4*>(p + (oy ^ 48u) + 16),
                 nz = *reinterpret_cast<const float4*>(p + oz + 32), fz = *reinterpret_cast<const float4*>(p + (oz ^ 48u) + 32);
    const uint4 child = *reinterpret_cast<const uint4*>(p + 96);
    auto enter = [&](float nx, float ny, float nz) {
        return Vec3(fmaf(nx, r.inv.x, r.nearBias.x), fmaf(ny, r.inv.y, r.nearBias.y), fmaf(nz, r.inv.z, r.nearBias.z));
    };
    auto box = [&](const Vec3& e, float fx, float fy, float fz) {
        float tmin = fmaxf(fmaxf(e.x, e.y), e.z);
        float tmax = fminf(fminf(fminf(fmaf(fx, r.inv.x, r.farBias.x), fmaf(fy, r.inv.y, r.farBias.y)),
                               fmaf(fz, r.inv.z, r.farBias.z)), closestT);
        return fmaxf(tmin, kRayMinDistance) <= boxReach(tmax) ? tmin : kBoxMissed;
    };
    auto both = [](const Vec3& a, const Vec3& b) {
        return fmaxf(fmaxf(fminf(a.x, b.x), fminf(a.y, b.y)), fminf(a.z, b.z));
    };
    const Vec3 e0 = enter(nx.x, ny.x, nz.x), e1 = enter(nx.y, ny.y, nz.y);
    float t0 = box(e0, fx.x, fy.x, fz.x), t1 = box(e1, fx.y, fy.y, fz.y), left = both(e0, e1);
    const Vec3 e2 = enter(nx.z, ny.z, nz.z), e3 = enter(nx.w, ny.w, nz.w);
    float t2 = box(e2, fx.z, fy.z, fz.z), t3 = box(e3, fx.w, fy.w, fz.w), right = both(e2, e3);
    if (!r.regular()) {
        float t[kQuadChildren], pair[2];
        exactBoxes(nodes[cur], r.exact(), closestT, t, pair);
        t0 = t[0];
        t1 = t[1];
        t2 = t[2];
        t3 = t[3];
        left = pair[0];
        right = pair[1];
    }
    uint32_t c0 = child.x, c1 = child.y, c2 = child.z, c3 = child.w;
    orderPair(t0, c0, t1, c1);
    orderPair(t2, c2, t3, c3);
    if (t2 < kBoxMissed && (t0 == kBoxMissed || right <= left)) {
        float t = t0;
        t0 = t2;
        t2 = t;
        t = t1;
        t1 = t3;
        t3 = t;
        uint32_t c = c0;
        c0 = c2;
        c2 = c;
        c = c1;
        c1 = c3;
        c3 = c;
    }
    if (t3 < kBoxMissed) stack.push(c3, t3);
    if (t2 < kBoxMissed) stack.push(c2, t2);
    if (t1 < kBoxMissed) stack.push(c1, t1);
    cur = c0;
    return t0 < kBoxMissed;
}

// Query kinds.  A closest-hit query keeps the nearest hit in the tie order
// above; an any-hit query (shadow rays) stops at the first blocker closer
// than its distance limit.  kEither picks one of the two per lane at run
// time, so that lanes of one wave running different kinds of query step
// through the same traversal loop together.
enum class Query { kClosest, kAny, kEither };

// Offers a candidate at distance t to the query.  Any-hit queries accept
// anything strictly closer than their limit (held in best.t); closest-hit
// queries apply the tie order.
WPT_HD bool wanted(bool any, float t, uint32_t rank, uint32_t instance, uint32_t prim, const HitRecord& best) {
    return any ? t < best.t : nearer(t, rank, instance, prim, best);
}

WPT_HD void record(HitRecord& best, float t, float u, float v, uint32_t kind, uint32_t instance, uint32_t prim,
    uint32_t material, uint32_t rank) {
    best.t = t;
    best.u = u;
    best.v = v;
    best.kind = kind;
    best.instance = instance;
    best.prim = prim;
    best.material = material;
    best.rank = rank;
}

// Triangles of one BVH (the flat-triangle BVH, world space).  Returns true
// when an any-hit query found its blocker.
template <bool Full, class Stack>
WPT_HD bool queryBvh(const DevScene& s, const RayInv& r, const Bvh& bvh, const float4* geometry, const TriShade* tris,
    uint32_t materialOverride, uint32_t kind, uint32_t rank, uint32_t instance, bool any, HitRecord& best,
    Stack& stack) {
    float nearT;
    if (!slab(r, bvh.rootMin[0], bvh.rootMin[1], bvh.rootMin[2], bvh.rootMax[0], bvh.rootMax[1], bvh.rootMax[2],
            best.t, nearT))
        return false;
    const BoxRay b = makeBoxRay(r.ray, r.inv);
    uint32_t base = stack.size;
    uint32_t cur = bvh.root;
    while (true) {
        if (cur & kLeafBit) {
            uint32_t slot = cur & ~kLeafBit;
            // A clipped leaf's box first: fetched after the triangle's test it
            // costs kTrace five spills (terrain 1080p, 16 spp: 136.4 -> 139.0 ms).
            if (!s.flatClipped || slotOpen(geometry + 3 * bvh.primCount, r, slot, best.t)) {
                float4 a = geometry[3 * slot + 0];
                float4 e = geometry[3 * slot + 1];
                float4 c = geometry[3 * slot + 2];
                float t, u, v;
                if (intersectTriangle(r.ray, xyz(a), xyz(e), xyz(c), t, u, v) &&
                    wanted(any, t, rank, instance, wbits(a), best) &&
                    (s.flatClipped || leafOpen(r, xyz(a), xyz(e), xyz(c), best.t))) {
                    uint32_t material = materialOverride == kInvalid ? wbits(e) : materialOverride;
                    if (!cutAway<Full>(s, material, tris, wbits(a), u, v)) {
                        record(best, t, u, v, kind, instance, wbits(a), material, rank);
                        if (any) {
                            stack.clear();
                            return true;
                        }
                    }
                }
            }
        } else {
            if (visitQuad(bvh.nodes, b, best.t, cur, stack)) continue;
        }
        if (!popLive(stack, base, boxReach(best.t), cur)) return false;
    }
}

// Triangles under eight-wide nodes (the flat-triangle accelerator
// WPT_FLAT_WIDE8).  A node's children that the ray reaches are pushed so that
// the nearest ends on top (insertion from the top of the stack, at most
// eight entries, all in the stack's LDS part), then the walk pops as for
// binary nodes.  Returns true when an any-hit query found its blocker.
template <bool Full, class Stack>
WPT_HD bool queryWide(const DevScene& s, const RayInv& r, const Bvh& bvh, const WideNode* nodes, const float4* geometry,
    const TriShade* tris, uint32_t kind, uint32_t rank, bool any, HitRecord& best, Stack& stack) {
    float nearT;
    if (!slab(r, bvh.rootMin[0], bvh.rootMin[1], bvh.rootMin[2], bvh.rootMax[0], bvh.rootMax[1], bvh.rootMax[2],
            best.t, nearT))
        return false;
    uint32_t base = stack.size;
    uint32_t cur = bvh.primCount > 1 ? 0u : (kLeafBit | 0u);
    while (true) {
        if (cur & kLeafBit) {
            uint32_t slot = cur & ~kLeafBit;
            float4 a = geometry[3 * slot + 0];
            float4 b = geometry[3 * slot + 1];
            float4 c = geometry[3 * slot + 2];
            float t, u, v;
            if (intersectTriangle(r.ray, xyz(a), xyz(b), xyz(c), t, u, v) &&
                wanted(any, t, rank, kInvalid, wbits(a), best)) {
                uint32_t material = wbits(b);
                if (!cutAway<Full>(s, material, tris, wbits(a), u, v)) {
                    record(best, t, u, v, kind, kInvalid, wbits(a), material, rank);
                    if (any) {
                        stack.clear();
                        return true;
                    }
                }
            }
        } else {
            const WideNode& n = nodes[cur];
            uint32_t pushed = 0;
            for (uint32_t k = 0; k < kWideChildren; ++k) {
                uint32_t child = n.child[k];
                if (child == kInvalid) break;
                float t;
                if (!slab(r, n.minX[k], n.minY[k], n.minZ[k], n.maxX[k], n.maxY[k], n.maxZ[k], best.t, t)) continue;
                stack.push(child, t);
                // Keep the pushed entries ordered, nearest on top.
                for (uint32_t j = 0; j < pushed; ++j) {
                    uint2 top = stack.peek(j), below = stack.peek(j + 1);
                    if (!(fromBits32(top.y) > fromBits32(below.y))) break;
                    stack.poke(j, below);
                    stack.poke(j + 1, top);
                }
                ++pushed;
            }
        }
        if (!popLive(stack, base, tieReach(best.t), cur)) return false;
    }
}

// Brute force over original-order triangles (direct instances, static
// triangles, flat triangles without a BVH): `edges` holds 9 floats per
// triangle, v0, v1 - v0 and v2 - v0.  Every lane reads the same triangle, so
// the floats come through the scalar cache into scalar registers; as vector
// loads of whole TriShade records the loop waited for the L1 in every
// iteration (72 triangles, forward and adjoint of 512x512, 16 samples: 18.6 ->
// 17.1 ms; Cornell box, 12 triangles, 256x256, 16 samples: 861 -> 835 us).
// Returns true when an any-hit query found its blocker.
#if defined(__HIP_DEVICE_COMPILE__)
using UniformFloats = const __attribute__((address_space(4))) float*;
#else
using UniformFloats = const float*;
#endif
template <bool Full>
WPT_HD bool queryBrute(const DevScene& s, const Ray& ray, const float* edges, const TriShade* tris, uint32_t count,
    uint32_t materialOverride, uint32_t kind, uint32_t rank, uint32_t instance, bool any, HitRecord& best) {
    UniformFloats e = (UniformFloats)edges;
    for (uint32_t i = 0; i < count; ++i, e += 9) {
        float t, u, v;
        if (!intersectEdges(ray, Vec3(e[0], e[1], e[2]), Vec3(e[3], e[4], e[5]), Vec3(e[6], e[7], e[8]), t, u, v) ||
            !wanted(any, t, rank, instance, i, best))
            continue;
        uint32_t material = materialOverride == kInvalid ? tris[i].material : materialOverride;
        if (cutAway<Full>(s, material, tris, i, u, v)) continue;
        record(best, t, u, v, kind, instance, i, material, rank);
        if (any) return true;
    }
    return false;
}

WPT_HD Ray toLocal(const InstanceTransform& tr, const Ray& ray) {
    Ray local;
    local.origin = inverseTransformVector(tr, ray.origin - tr.translation);
    local.direction = inverseTransformVector(tr, ray.direction);
    return local;
}

// Sphere candidate: nearer root wins; on an exact tie the lower sphere index
// wins (reference device_traversal.cuh:789-800).  Returns true when an
// any-hit query found its blocker.
WPT_HD bool querySphere(const DevScene& s, const Ray& ray, uint32_t index, bool any, HitRecord& best) {
    float4 sp = s.spheres[index];
    float t;
    if (!intersectSphere(ray, xyz(sp), sp.w, t) || !wanted(any, t, kRankSphere, kInvalid, index, best)) return false;
    record(best, t, 0.0f, 0.0f, kHitSphere, kInvalid, index, s.sphereMaterial[index], kRankSphere);
    return any;
}

// querySphere for the sphere in TLAS slot `slot`, under BoxRay's rule: its
// box is tested only once the sphere is found to be hit.
WPT_HD bool queryTlasSphere(const DevScene& s, const BoxRay& r, uint32_t slot, uint32_t index, bool any,
    HitRecord& best) {
    float4 sp = s.spheres[index];
    float t;
    if (!intersectSphere(r.ray, xyz(sp), sp.w, t) || !wanted(any, t, kRankSphere, kInvalid, index, best) ||
        !slotOpen(s.tlasBounds, r.exact(), slot, best.t))
        return false;
    record(best, t, 0.0f, 0.0f, kHitSphere, kInvalid, index, s.sphereMaterial[index], kRankSphere);
    return any;
}

// One query in the reference's category order: direct spheres, direct
// instances, static triangles, TLAS, flat triangles (traceRay /
// isOccluded, device_traversal.cuh:1035-1184).  `maxDistance` bounds
// any-hit queries.  The result's kind is kHitNone when nothing was found;
// for an any-hit query any other kind means the ray is blocked.
//
// The TLAS and the BLASes of its instance leaves are walked by one loop: on
// an instance leaf whose BLAS root box is hit, the loop switches its node
// array, ray and stack floor to the BLAS; when the BLAS level is exhausted
// it switches back and resumes popping the TLAS.  The visit order is that of
// the nested walk (each BLAS finishes before the TLAS resumes), but lanes at
// different levels -- and, for kEither, lanes running different kinds of
// query -- run the same node-visit code in the same iteration.
//
// TlasWalk is the same query as a resumable walk: start() runs the
// categories before the TLAS and enters its root, visitNode() and visitLeaf()
// each make one iteration of traceQuery's loop, finish() runs the categories
// after the TLAS.  A kernel can thus interleave the walks of several rays in
// one lane, and choose for a whole wave which kind of visit runs next; each
// ray's visits, and so its result, are those of traceQuery.  traceQuery keeps
// its own loop: as start/visit/finish its code is slower (the sphere field's
// closest-hit pass: 69 -> 80 ms per 64-sample frame).
enum class Walk { kTlas, kAfter, kDone };  // walking the TLAS; categories after it left; complete

template <bool Full, Query Q>
struct TlasWalk {
    Ray ray;
    BoxRay r;
    Vec3 worldInv;  // 1 / ray.direction
    HitRecord best;
    const QuadNode* nodes;
    const float4* geometry;
    uint32_t cur, instance, materialOverride, base, blasBase;
    bool anyHit;

    WPT_HD bool any() const { return Q == Query::kAny || (Q == Query::kEither && anyHit); }

    template <class Stack>
    WPT_HD Walk start(const DevScene& s, const Ray& query, float maxDistance, bool shadow, Stack& stack) {
        ray = query;
        anyHit = shadow;
        best = emptyHit();
        if (any()) best.t = maxDistance;
        for (uint32_t i = 0; i < s.directSphereCount; ++i)
            if (querySphere(s, ray, s.directSpheres[i], any(), best)) return Walk::kDone;
        for (uint32_t i = 0; i < s.directInstanceCount; ++i) {
            uint32_t index = s.directInstances[i];
            const Instance& inst = s.instances[index];
            const Blas& blas = s.blases[inst.mesh];
            if (queryBrute<Full>(s, toLocal(inst.transform, ray), blas.edges, blas.triangles, blas.triangleCount,
                    inst.materialOverride, kHitInstance, kRankDirectInstance, index, any(), best))
                return Walk::kDone;
        }
        if (queryBrute<Full>(s, ray, s.staticEdges, s.staticTriangles, s.staticCount, kInvalid, kHitStatic, kRankStatic, kInvalid,
                any(), best))
            return Walk::kDone;
        if (s.tlas.primCount == 0) return Walk::kAfter;
        RayInv world = makeRayInv(ray);
        float nearT;
        if (!slab(world, s.tlas.rootMin[0], s.tlas.rootMin[1], s.tlas.rootMin[2], s.tlas.rootMax[0], s.tlas.rootMax[1],
                s.tlas.rootMax[2], best.t, nearT))
            return Walk::kAfter;
        worldInv = world.inv;
        r = makeBoxRay(ray, worldInv);
        base = stack.size;
        blasBase = base;
        cur = s.tlas.root;
        nodes = s.tlas.nodes;
        geometry = nullptr;
        instance = kInvalid;  // kInvalid while in the TLAS
        materialOverride = kInvalid;
        return Walk::kTlas;
    }

    // The next live entry of the level being walked; when a BLAS is
    // exhausted, of the TLAS around it.
    template <class Stack>
    WPT_HD Walk next(const DevScene& s, Stack& stack) {
        if (instance != kInvalid) {
            if (popLive(stack, blasBase, boxReach(best.t), cur)) return Walk::kTlas;
            instance = kInvalid;
            nodes = s.tlas.nodes;
            r = makeBoxRay(ray, worldInv);
        }
        return popLive(stack, base, boxReach(best.t), cur) ? Walk::kTlas : Walk::kAfter;
    }

    WPT_HD bool atLeaf() const { return (cur & kLeafBit) != 0u; }

    // One interior node (atLeaf() is false).
    template <class Stack>
    WPT_HD Walk visitNode(const DevScene& s, Stack& stack) {
        if (visitQuad(nodes, r, best.t, cur, stack)) return Walk::kTlas;
        return next(s, stack);
    }

    // One leaf (atLeaf() is true): a BLAS triangle, or a TLAS sphere or
    // instance, whose BLAS the walk enters.
    template <class Stack>
    WPT_HD Walk visitLeaf(const DevScene& s, Stack& stack) {
        uint32_t slot = cur & ~kLeafBit;
        if (instance != kInvalid) {
            float4 a = geometry[3 * slot + 0];
            float4 b = geometry[3 * slot + 1];
            float4 c = geometry[3 * slot + 2];
            float t, u, v;
            if (intersectTriangle(r.ray, xyz(a), xyz(b), xyz(c), t, u, v) &&
                wanted(any(), t, kRankTlasInstance, instance, wbits(a), best) &&
                leafOpen(r.exact(), xyz(a), xyz(b), xyz(c), best.t)) {
                uint32_t material = materialOverride == kInvalid ? wbits(b) : materialOverride;
                if (s.materialCutout[material] == kCutNever ||
                    !cutAway<Full>(s, material, s.blases[s.instances[instance].mesh].triangles, wbits(a), u, v)) {
                    record(best, t, u, v, kHitInstance, instance, wbits(a), material, kRankTlasInstance);
                    if (any()) {
                        stack.clear();
                        return Walk::kDone;
                    }
                }
            }
            return next(s, stack);
        }
        uint32_t leaf = s.tlasLeaves[slot];
        if (leaf & kTlasSphereBit) {
            if (queryTlasSphere(s, r, slot, leaf & ~kTlasSphereBit, any(), best)) {
                stack.clear();
                return Walk::kDone;
            }
            return next(s, stack);
        }
        if (!slotOpen(s.tlasBounds, r.exact(), slot, best.t)) return next(s, stack);
        const Instance& inst = s.instances[leaf];
        const Blas& blas = s.blases[inst.mesh];
        Ray local = toLocal(inst.transform, ray);
        if (blas.bvh.primCount != 0) {
            RayInv rl = makeRayInv(local);
            float nearT;
            if (slab(rl, blas.bvh.rootMin[0], blas.bvh.rootMin[1], blas.bvh.rootMin[2], blas.bvh.rootMax[0],
                    blas.bvh.rootMax[1], blas.bvh.rootMax[2], best.t, nearT)) {
                r = makeBoxRay(local, rl.inv);
                instance = leaf;
                nodes = blas.bvh.nodes;
                geometry = blas.geometry;
                materialOverride = inst.materialOverride;
                blasBase = stack.size;
                cur = blas.bvh.root;
                return Walk::kTlas;
            }
        } else if (queryBrute<Full>(s, local, blas.edges, blas.triangles, blas.triangleCount, inst.materialOverride, kHitInstance,
                       kRankTlasInstance, leaf, any(), best)) {
            stack.clear();
            return Walk::kDone;
        }
        return next(s, stack);
    }

    template <class Stack>
    WPT_HD void finish(const DevScene& s, Stack& stack) {
        if (s.flatCount == 0) return;
        if (s.flatWide) {
            RayInv rf = makeRayInv(ray);
            queryWide<Full>(s, rf, s.flat, s.flatWide, s.flatGeometry, s.flatTriangles, kHitFlat, kRankFlat, any(), best,
                stack);
        } else if (s.flat.primCount != 0) {
            RayInv rf = makeRayInv(ray);
            queryBvh<Full>(s, rf, s.flat, s.flatGeometry, s.flatTriangles, kInvalid, kHitFlat, kRankFlat, kInvalid,
                any(), best, stack);
        } else {
            queryBrute<Full>(s, ray, s.flatEdges, s.flatTriangles, s.flatCount, kInvalid, kHitFlat, kRankFlat, kInvalid, any(),
                best);
        }
    }
};

template <bool Full, Query Q, class Stack>
WPT_HD HitRecord traceQuery(const DevScene& s, const Ray& ray, float maxDistance, bool anyHit, Stack& stack) {
    const bool any = Q == Query::kAny || (Q == Query::kEither && anyHit);
    HitRecord best = emptyHit();
    if (any) best.t = maxDistance;
    for (uint32_t i = 0; i < s.directSphereCount; ++i)
        if (querySphere(s, ray, s.directSpheres[i], any, best)) return best;
    for (uint32_t i = 0; i < s.directInstanceCount; ++i) {
        uint32_t index = s.directInstances[i];
        const Instance& inst = s.instances[index];
        const Blas& blas = s.blases[inst.mesh];
        if (queryBrute<Full>(s, toLocal(inst.transform, ray), blas.edges, blas.triangles, blas.triangleCount, inst.materialOverride,
                kHitInstance, kRankDirectInstance, index, any, best))
            return best;
    }
    if (queryBrute<Full>(s, ray, s.staticEdges, s.staticTriangles, s.staticCount, kInvalid, kHitStatic, kRankStatic, kInvalid, any,
            best))
        return best;
    if (s.tlas.primCount != 0) {
        RayInv world = makeRayInv(ray);
        float nearT;
        if (slab(world, s.tlas.rootMin[0], s.tlas.rootMin[1], s.tlas.rootMin[2], s.tlas.rootMax[0], s.tlas.rootMax[1],
                s.tlas.rootMax[2], best.t, nearT)) {
            const Vec3 worldInv = world.inv;
            BoxRay r = makeBoxRay(ray, worldInv);
            const uint32_t base = stack.size;
            uint32_t blasBase = base;
            uint32_t cur = s.tlas.root;
            const QuadNode* nodes = s.tlas.nodes;
            const float4* geometry = nullptr;
            uint32_t instance = kInvalid;  // kInvalid while in the TLAS
            uint32_t materialOverride = kInvalid;
            while (true) {
                if (cur & kLeafBit) {
                    uint32_t slot = cur & ~kLeafBit;
                    if (instance != kInvalid) {
                        float4 a = geometry[3 * slot + 0];
                        float4 b = geometry[3 * slot + 1];
                        float4 c = geometry[3 * slot + 2];
                        float t, u, v;
                        if (intersectTriangle(r.ray, xyz(a), xyz(b), xyz(c), t, u, v) &&
                            wanted(any, t, kRankTlasInstance, instance, wbits(a), best) &&
                            leafOpen(r.exact(), xyz(a), xyz(b), xyz(c), best.t)) {
                            uint32_t material = materialOverride == kInvalid ? wbits(b) : materialOverride;
                            if (s.materialCutout[material] == kCutNever ||
                                !cutAway<Full>(s, material, s.blases[s.instances[instance].mesh].triangles, wbits(a), u, v)) {
                                record(best, t, u, v, kHitInstance, instance, wbits(a), material, kRankTlasInstance);
                                if (any) {
                                    stack.clear();
                                    return best;
                                }
                            }
                        }
                    } else {
                        uint32_t leaf = s.tlasLeaves[slot];
                        if (leaf & kTlasSphereBit) {
                            if (queryTlasSphere(s, r, slot, leaf & ~kTlasSphereBit, any, best)) {
                                stack.clear();
                                return best;
                            }
                        } else if (slotOpen(s.tlasBounds, r.exact(), slot, best.t)) {
                            const Instance& inst = s.instances[leaf];
                            const Blas& blas = s.blases[inst.mesh];
                            Ray local = toLocal(inst.transform, ray);
                            if (blas.bvh.primCount != 0) {
                                RayInv rl = makeRayInv(local);
                                if (slab(rl, blas.bvh.rootMin[0], blas.bvh.rootMin[1], blas.bvh.rootMin[2],
                                        blas.bvh.rootMax[0], blas.bvh.rootMax[1], blas.bvh.rootMax[2], best.t, nearT)) {
                                    r = makeBoxRay(local, rl.inv);
                                    instance = leaf;
                                    nodes = blas.bvh.nodes;
                                    geometry = blas.geometry;
                                    materialOverride = inst.materialOverride;
                                    blasBase = stack.size;
                                    cur = blas.bvh.root;
                                    continue;
                                }
                            } else if (queryBrute<Full>(s, local, blas.edges, blas.triangles, blas.triangleCount,
                                           inst.materialOverride, kHitInstance, kRankTlasInstance, leaf, any, best)) {
                                stack.clear();
                                return best;
                            }
                        }
                    }
                } else {
                    if (visitQuad(nodes, r, best.t, cur, stack)) continue;
                }
                if (instance != kInvalid) {
                    if (popLive(stack, blasBase, boxReach(best.t), cur)) continue;
                    instance = kInvalid;
                    nodes = s.tlas.nodes;
                    r = makeBoxRay(ray, worldInv);
                }
                if (!popLive(stack, base, boxReach(best.t), cur)) break;
            }
        }
    }
    if (s.flatCount != 0) {
        if (s.flatWide) {
            RayInv r = makeRayInv(ray);
            queryWide<Full>(s, r, s.flat, s.flatWide, s.flatGeometry, s.flatTriangles, kHitFlat, kRankFlat, any, best,
                stack);
        } else if (s.flat.primCount != 0) {
            RayInv r = makeRayInv(ray);
            queryBvh<Full>(s, r, s.flat, s.flatGeometry, s.flatTriangles, kInvalid, kHitFlat, kRankFlat, kInvalid, any,
                best, stack);
        } else {
            queryBrute<Full>(s, ray, s.flatEdges, s.flatTriangles, s.flatCount, kInvalid, kHitFlat, kRankFlat, kInvalid, any, best);
        }
    }
    return best;
}

template <bool Full = true, class Stack>
WPT_HD HitRecord traceClosest(const DevScene& s, const Ray& ray, Stack& stack) {
    return traceQuery<Full, Query::kClosest>(s, ray, kNoHit, false, stack);
}

// Shadow query: any blocker with t < maxDistance.
template <bool Full = true, class Stack>
WPT_HD bool traceOccluded(const DevScene& s, const Ray& ray, float maxDistance, Stack& stack) {
    return traceQuery<Full, Query::kAny>(s, ray, maxDistance, true, stack).kind != kHitNone;
}

}  // namespace wpt
