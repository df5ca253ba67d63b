// Scene raycasts on the device: Scene::raycastClosest (src/Physecs.cpp:571-621) for a batch
// of rays, each in one world. A ray walks the LBVH of its world's dynamic colliders (built
// from the current bounds for the query) and then its world's non-dynamic colliders. The
// reference walks its dynamic AABB tree; a leaf is reached when the ray enters the leaf's
// own bounds within maxDistance, and every ancestor's box holds those bounds, so pruning
// with the same ray-box test on the LBVH's boxes accepts the same hits. Of the accepted
// hits the closest is kept; equal distances go to the lower collider index (the
// reference settles them by its tree's shape). The filter rejects one entity per ray.
#include <cstring>
#include <limits>
#include "pgx_internal.h"
#include "shape_bounds.h"

using namespace pgx;

namespace {

__device__ __forceinline__ float comp(f3 v, int i) { return i == 0 ? v.x : (i == 1 ? v.y : v.z); }

// 1 / d per axis, for ray_aabb: a walk divides once
__device__ __forceinline__ f3 ray_inverse(f3 d) { return mk3(1.f / d.x, 1.f / d.y, 1.f / d.z); }

// intersectRayAABB (src/Raycast.cpp:5-30); inv: ray_inverse(d)
__device__ __forceinline__ bool ray_aabb(f3 o, f3 d, f3 inv, f3 mn, f3 mx, float& t) {
    float tMin = 0.f;
    float tMax = 3.402823466e+38f;   // std::numeric_limits<float>::max()
    for (int i = 0; i < 3; ++i) {
        const float oi = comp(o, i), di = comp(d, i), lo = comp(mn, i), hi = comp(mx, i);
        if (gabs(di) < 0.001f) {
            if (oi < lo || oi > hi) return false;   // parallel to the slab, outside it
        } else {
            const float ood = comp(inv, i);
            float t1 = (lo - oi) * ood;
            float t2 = (hi - oi) * ood;
            if (t1 > t2) { float x = t1; t1 = t2; t2 = x; }
            if (t1 > tMin) tMin = t1;
            if (t2 < tMax) tMax = t2;
            if (tMin > tMax) return false;
        }
    }
    t = tMin;
    return true;
}

// intersectRaySphere (src/Raycast.cpp:32-46)
__device__ bool ray_sphere(f3 o, f3 d, f3 pos, float radius, float& t) {
    f3 m = sub(o, pos);
    float b = dot(m, d);
    float c = dot(m, m) - radius * radius;
    if (c > 0.f && b > 0.f) return false;
    float discr = b * b - c;
    if (discr < 0.f) return false;
    t = -b - sqrtf(discr);
    if (t < 0.f) t = 0.f;
    return true;
}

// intersectRayCapsule (src/Raycast.cpp:48-103): top hemisphere, cylinder, bottom hemisphere
__device__ bool ray_capsule(f3 o, f3 d0, f3 pos, qf ori, float hh, float radius, float& t) {
    qf inv = qinverse(ori);
    f3 p = qrot(inv, sub(o, pos));
    f3 d = qrot(inv, d0);
    float pd = dot(p, d);
    float hdy = hh * d.y;
    float thpy = 2.f * hh * p.y;
    float phr = dot(p, p) + hh * hh - radius * radius;
    float tMin = 3.402823466e+38f;
    bool hit = false;
    float b = pd - hdy, c = phr - thpy, discr = b * b - c;
    if (discr >= 0.f) {
        t = -b - sqrtf(discr);
        if (t < 0.f) t = 0.f;
        if (add(p, mul(t, d)).y >= hh) { hit = true; tMin = t; }
    }
    float a = d.x * d.x + d.z * d.z;
    b = p.x * d.x + p.z * d.z;
    c = p.x * p.x + p.z * p.z - radius * radius;
    discr = b * b - a * c;
    if (discr >= 0.f) {
        t = (-b - sqrtf(discr)) / a;
        if (t < 0.f) t = 0.f;
        float y = add(p, mul(t, d)).y;
        if (-hh <= y && y < hh && t < tMin) { hit = true; tMin = t; }
    }
    b = pd + hdy;
    c = phr + thpy;
    discr = b * b - c;
    if (discr >= 0.f) {
        t = -b - sqrtf(discr);
        if (t < 0.f) t = 0.f;
        if (add(p, mul(t, d)).y < -hh && t < tMin) { hit = true; tMin = t; }
    }
    t = tMin;
    return hit;
}

// intersectRayBox (src/Raycast.cpp:105-110)
__device__ bool ray_box(f3 o, f3 d, f3 pos, qf ori, f3 he, float& t) {
    const qf inv = qinverse(ori);
    const f3 dl = qrot(inv, d);
    return ray_aabb(qrot(inv, sub(o, pos)), dl, ray_inverse(dl), neg(he), he, t);
}

// intersectRayConvexMesh (src/Raycast.cpp:112-139): the faces' half-spaces, in face order
// convex meshes: per mesh {first vertex, vertex count, first face, face count}; per face
// outward normal and centroid
struct ConvexFaces { const int4* mesh; const float4 *faceN, *faceC; };

__device__ bool ray_convex(f3 o, f3 d, f3 pos, qf ori, const ConvexFaces& cv, int mesh, f3 scale, float& t) {
    const int4 mi = cv.mesh[mesh];
    float tMin = 0.f;
    float tMax = 3.402823466e+38f;
    for (int f = 0; f < mi.w; ++f) {
        f3 planeOrig = add(pos, qrot(ori, mulv(scale, xyz(cv.faceC[mi.z + f]))));
        f3 planeNormal = qrot(ori, mulv(divv(s3(1.f), scale), xyz(cv.faceN[mi.z + f])));
        float denom = dot(d, planeNormal);
        float dist = dot(sub(planeOrig, o), planeNormal);
        if (denom == 0.f) {
            if (dist > 0.f) return false;
        } else {
            t = dist / denom;
            if (denom < 0.f) { if (t > tMin) tMin = t; }
            else { if (t < tMax) tMax = t; }
            if (tMin > tMax) return false;
        }
    }
    t = tMin;
    return true;
}

// What the colliders of a tree allow its walks: whether only the tree's own order will do,
// what is not skipped however far (RaySkip::near), whether nothing may be skipped.
struct RayRules {
    int32_t inOrder;
    float near;
    int32_t noSkip;
};

struct RayScene {
    int W, nLeaves;
    const int32_t *worldRoot, *worldStop, *worldStaticStart, *staticCols, *mvals;
    const RayRules* rules;
    const float4 *rayNode, *rayLeaf;   // k_ray_records
    const float4 *leafA, *nodeA, *nodeB;
    const float4 *cbmin, *cbmax, *cparams, *clpos, *clquat, *bpos, *bquat;
    const int32_t *cbody, *ctype;
    const uint32_t* centity;
    ConvexFaces cv;
    const float4* cvVerts;
    const float* cvSlender;
};

__device__ __forceinline__ bool ray_shape(int type, const float4& prm, f3 pos, qf q, const ConvexFaces& cv, f3 o, f3 d,
                                          float& t) {
    switch (type) {
        case PGX_SPHERE: return ray_sphere(o, d, pos, prm.x, t);
        case PGX_CAPSULE: return ray_capsule(o, d, pos, q, prm.x, prm.y, t);
        case PGX_BOX: return ray_box(o, d, pos, q, xyz(prm), t);
        case PGX_CONVEX_MESH: return ray_convex(o, d, pos, q, cv, (int)prm.w, xyz(prm), t);
        default: return false;   // triangle meshes are never hit (src/Raycast.cpp:148)
    }
}

// one collider: the reference's leaf test (its bounds, then its geometry, both within
// maxDistance, and the filter), kept when closer than the best so far
__device__ __forceinline__ void test_collider(const RayScene& S, int c, f3 o, f3 d, f3 inv, float maxDist, uint32_t ignore,
                                              float& bestT, int& best) {
    if (S.centity[c] == ignore) return;
    float t;
    if (!ray_aabb(o, d, inv, xyz(S.cbmin[c]), xyz(S.cbmax[c]), t) || t > maxDist) return;
    const int b = S.cbody[c];
    const qf bq = q4(S.bquat[b]);
    const f3 pos = add(xyz(S.bpos[b]), qrot(bq, xyz(S.clpos[c])));
    const qf q = qmul(bq, q4(S.clquat[c]));
    const bool hit = ray_shape(S.ctype[c], S.cparams[c], pos, q, S.cv, o, d, t);
    if (!hit || t > maxDist) return;
    if (best < 0 || t < bestT || (t == bestT && c < best)) { best = c; bestT = t; }
}

// What a walk may skip once it has a hit: the boxes that the ray enters beyond it. A shape's
// hit distance comes from its own formula and can lie before the float entry distance of its
// box, so a box is skipped by the entry into itself widened by a margin. The computed hit
// point is within the margin of the shape, and so of every box around it (k_ray_records sees
// to it that they are: poses may be written without the bounds): with m the distance to the
// shape the formulas' error is that of a difference of squares (sqrt(8 eps m^2), and
// sqrt(2e-6 m^2) for a direction that is a unit vector to 2e-6: under 2e-3 m, in a sphere's,
// capsule's or plane's direction), and a direction component under 0.001 counts as parallel
// (intersectRayAABB, a drift of up to 0.001 t per axis). m and t are at most the distance to
// the far corner of the tree's box. Far from the world's origin the boxes' corners and the
// entry are rounded at the size of the coordinates (2^-24 of them each), the shapes' distances
// are not: the margin grows with the coordinates too.
//
// A capsule is the exception (src/Raycast.cpp:65-100): where the ray's line leaves its cylinder
// behind the origin, carried on beyond the caps, the hit counts as one at 0 if the origin lies
// between the caps' planes, however far ahead the ray enters the capsule's box. How far that is:
// with H the distance from the capsule's centre to the farthest corner of its box, half its
// half height, the ray moves away from the axis from its origin on and is at most H from it
// where it enters the box, so its origin is at most H from the axis and half <= H from the
// centre along it, sqrt(2) H from the centre, and the entry at most (1 + sqrt(2)) H from the
// origin. Boxes that the ray enters within 2.5 H of the tree's largest capsule are not skipped
// (the rest is for rounding and drift, which are under a hundredth of such a distance).
struct RaySkip {
    f3 inv;          // 1 / d, 0 on a parallel axis
    float margin;    // negative: nothing is skipped
    float near;      // what is entered up to here is not skipped
    bool numbers;    // false: a hit distance could be a NaN, walk in the tree's order
};
// The formulas take directions as unit vectors, of which the margin holds, and their squares
// stay finite up to 1e9. Directions of other lengths give numbers too, up to 1e6.
__device__ __forceinline__ RaySkip ray_skip(f3 o, f3 d, f3 inv, f3 mn, f3 mx, float near, bool skips) {
    RaySkip r;
    r.near = near;
    r.inv = mk3(fabsf(d.x) < 0.001f ? 0.f : inv.x, fabsf(d.y) < 0.001f ? 0.f : inv.y, fabsf(d.z) < 0.001f ? 0.f : inv.z);
    const f3 far = mk3(fmaxf(fabsf(mn.x - o.x), fabsf(mx.x - o.x)), fmaxf(fabsf(mn.y - o.y), fabsf(mx.y - o.y)),
                       fmaxf(fabsf(mn.z - o.z), fabsf(mx.z - o.z)));
    const float reach = far.x + far.y + far.z;
    const float size = fmaxf(fabsf(mn.x), fabsf(mx.x)) + fmaxf(fabsf(mn.y), fabsf(mx.y)) +
                       fmaxf(fabsf(mn.z), fabsf(mx.z)) + fabsf(o.x) + fabsf(o.y) + fabsf(o.z);
    const float dd = dot(d, d);
    r.numbers = dd < 1e12f && reach < 1e9f && dot(o, o) < 1e18f;
    r.margin = skips && fabsf(dd - 1.f) < 2e-6f ? 4e-3f * reach + 4e-6f * size : -1.f;
    return r;
}
// a lower bound of the distance at which the ray enters the widened box
__device__ __forceinline__ float widened_entry(const RaySkip& r, f3 o, f3 mn, f3 mx) {
    float t = 0.f;
    t = fmaxf(t, fminf((mn.x - r.margin - o.x) * r.inv.x, (mx.x + r.margin - o.x) * r.inv.x));
    t = fmaxf(t, fminf((mn.y - r.margin - o.y) * r.inv.y, (mx.y + r.margin - o.y) * r.inv.y));
    t = fmaxf(t, fminf((mn.z - r.margin - o.z) * r.inv.z, (mx.z + r.margin - o.z) * r.inv.z));
    return t * (1.f - 1e-5f);
}

// leaf i's record; what it asks of RaySkip::near
__device__ __forceinline__ float ray_leaf(int i, const RayScene& S, const float4* __restrict__ clquat,
                                          float4* __restrict__ rayLeaf, RayRules* __restrict__ rules) {
    const int c = S.mvals[i], b = S.cbody[c];
    const float4 mn = S.cbmin[c], mx = S.cbmax[c], l = clquat[c], q = S.bquat[b];
    const bool bounded = mn.x > -1e9f && mn.y > -1e9f && mn.z > -1e9f && mx.x < 1e9f && mx.y < 1e9f && mx.z < 1e9f;
    const float ll = l.x * l.x + l.y * l.y + l.z * l.z + l.w * l.w, qq = q.x * q.x + q.y * q.y + q.z * q.z + q.w * q.w;
    const qf lq = qmul(q4(q), q4(l));
    const f3 pos = add(xyz(S.bpos[b]), qrot(q4(q), xyz(S.clpos[c])));
    const int type = S.ctype[c];
    const float4 prm = S.cparams[c];
    bool numbers = bounded && ll > 0.25f && ll < 4.f && qq > 0.25f && qq < 4.f;
    bool skips = fabsf(ll - 1.f) < 1e-5f && fabsf(qq - 1.f) < 1e-5f;
    if (type != PGX_TRIANGLE_MESH) {   // the bounds hold the shape as it is now (rays never hit a mesh)
        f3 lo, hi;
        shape_bounds(type, prm, pos, lq, S.cvVerts, S.cv.mesh, nullptr, nullptr, lo, hi);
        numbers = numbers && lo.x > -1e9f && lo.y > -1e9f && lo.z > -1e9f && hi.x < 1e9f && hi.y < 1e9f && hi.z < 1e9f;
        skips = skips && mn.x <= lo.x && mn.y <= lo.y && mn.z <= lo.z && lo.x <= hi.x && lo.y <= hi.y && lo.z <= hi.z &&
                hi.x <= mx.x && hi.y <= mx.y && hi.z <= mx.z;
        if (type == PGX_CAPSULE) skips = skips && prm.y >= 0.f;   // a radius below 0 narrows the bounds alone
    }
    if (type == PGX_CONVEX_MESH) {   // its half-spaces end at its vertices
        const float x = fabsf(prm.x), y = fabsf(prm.y), z = fabsf(prm.z);
        const float least = fminf(x, fminf(y, z)), most = fmaxf(x, fmaxf(y, z)), slender = S.cvSlender[(int)prm.w];
        numbers = numbers && least >= 1e-6f && most <= 1e6f && slender == slender;
        skips = skips && slender * most <= 32.f * least;
    }
    if (!numbers) rules->inOrder = 1;
    if (!skips) rules->noSkip = 1;
    rayLeaf[4 * (size_t)i] = f4(pos, __int_as_float(type));
    rayLeaf[4 * (size_t)i + 1] = f4(mk3(lq.x, lq.y, lq.z), lq.w);
    rayLeaf[4 * (size_t)i + 2] = prm;
    rayLeaf[4 * (size_t)i + 3] = make_float4(__int_as_float(c), __uint_as_float(S.centity[c]), 0.f, 0.f);
    if (type != PGX_CAPSULE) return 0.f;
    const f3 far = mk3(fmaxf(pos.x - mn.x, mx.x - pos.x), fmaxf(pos.y - mn.y, mx.y - pos.y), fmaxf(pos.z - mn.z, mx.z - pos.z));
    return 2.5f * length(far);
}

// The walk's records, 64 bytes each so that a visit takes one line: per inner node
// {left box min, left}, {left max, right}, {right min}, {right max}; per leaf
// {position, type}, {orientation}, {params}, {collider, entity}.
// And the rules, 0 before: nothing is skipped if the margin does not hold for a dynamic
// collider (its bounds do not hold the shape, its orientation is not a unit quaternion, or it
// is a hull whose half-spaces go on beyond its vertices: k_hull_slenderness; up to 32 the planes'
// rounding, some 1e-6 of the distance and 2^-23 of the coordinates, stays within the margin);
// and the tree's order is kept if a hit distance could be a NaN, which makes the result depend
// on the order of the tests (bounds, orientations or scales that are not finite or are far
// from 1).
__global__ __launch_bounds__(256) void k_ray_records(int n, const int32_t* __restrict__ child, RayScene S,
                                                     const float4* __restrict__ leafB, const float4* __restrict__ clquat,
                                                     float4* __restrict__ rayNode, float4* __restrict__ rayLeaf,
                                                     RayRules* __restrict__ rules) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    float reach = 0.f;
    if (i < n - 1) {
        const int l = child[2 * i], r = child[2 * i + 1], ll = l & ~LEAF_BIT, rl = r & ~LEAF_BIT;
        rayNode[4 * (size_t)i] = f4(xyz(l & LEAF_BIT ? S.leafA[ll] : S.nodeA[ll]), __int_as_float(l));
        rayNode[4 * (size_t)i + 1] = f4(xyz(l & LEAF_BIT ? leafB[ll] : S.nodeB[ll]), __int_as_float(r));
        rayNode[4 * (size_t)i + 2] = f4(xyz(r & LEAF_BIT ? S.leafA[rl] : S.nodeA[rl]), 0.f);
        rayNode[4 * (size_t)i + 3] = f4(xyz(r & LEAF_BIT ? leafB[rl] : S.nodeB[rl]), 0.f);
    }
    if (i < n) reach = ray_leaf(i, S, clquat, rayLeaf, rules);
    // one atomic a wave at most: the floats are not negative, so their bits order like them
    for (int o = WAVE / 2; o >= 1; o >>= 1) reach = fmaxf(reach, __shfl_xor(reach, o));
    if ((threadIdx.x & (WAVE - 1)) == 0 && reach > rules->near) atomicMax((unsigned int*)&rules->near, __float_as_uint(reach));
}

// How far a convex mesh's half-spaces, which are what a ray is tested against, reach beyond its
// vertices when their planes are moved out: by at most this factor (and one) times the move. It
// is the diameter over the inner radius about the vertices' mean, if the faces close the mesh:
// their planes hold every vertex, every edge is met as often in one direction as in the other
// (the sum of the directed edges' hashes is 0), and the volume that the faces enclose is at
// least a ball's of that radius (which a surface folded onto itself does not enclose). Meshes
// come with faces, normals and centroids as given, so they may not; infinite then, and for
// meshes too large to look at here, and a NaN if the planes are not numbers below 1e9. A wave
// per mesh, a face per lane: 34 us for 8,192 hulls of 24 points (on the host 140 ms).
__device__ __forceinline__ double wave_sum(double x) {
    for (int o = WAVE / 2; o >= 1; o >>= 1) x += __shfl_xor(x, o);
    return x;
}
__device__ __forceinline__ float wave_least(float x) {
    for (int o = WAVE / 2; o >= 1; o >>= 1) x = fminf(x, __shfl_xor(x, o));
    return x;
}
__device__ __forceinline__ uint64_t edge_hash(int a, int b) {   // of either direction, with its sign
    uint64_t x = ((uint64_t)(uint32_t)min(a, b) << 32) | (uint32_t)max(a, b);
    x = (x ^ (x >> 31)) * 0x9e3779b97f4a7c15ull;
    x = (x ^ (x >> 29)) * 0xbf58476d1ce4e5b9ull;
    x ^= x >> 32;
    return a < b ? x : 0 - x;
}
__global__ __launch_bounds__(WAVE) void k_hull_slenderness(const int4* __restrict__ mesh, const float4* __restrict__ verts,
                                                           const int2* __restrict__ face, const int32_t* __restrict__ faceIdx,
                                                           const float4* __restrict__ faceN, const float4* __restrict__ faceC,
                                                           float* __restrict__ slender) {
    const int4 m = mesh[blockIdx.x];
    const int nv = m.y, nf = m.w, lane = threadIdx.x;
    const float4* v = verts + m.x;
    bool planes = true;
    for (int f = lane; f < nf; f += WAVE) {
        const float4 n = faceN[m.z + f], c = faceC[m.z + f];
        planes = planes && fabsf(n.x) < 1e9f && fabsf(n.y) < 1e9f && fabsf(n.z) < 1e9f && fabsf(c.x) < 1e9f &&
                 fabsf(c.y) < 1e9f && fabsf(c.z) < 1e9f;
    }
    if (__ballot(!planes)) {
        if (lane == 0) slender[blockIdx.x] = __builtin_nanf("");
        return;
    }
    if (nv < 4 || nf < 4 || (long long)nv * nf > 1 << 24) {
        if (lane == 0) slender[blockIdx.x] = INFINITY;
        return;
    }
    double mx = 0.0, my = 0.0, mz = 0.0;
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {INFINITY, INFINITY, INFINITY};   // hi: of the negatives
    for (int i = lane; i < nv; i += WAVE) {
        const float p[3] = {v[i].x, v[i].y, v[i].z};
        mx += p[0]; my += p[1]; mz += p[2];
        for (int k = 0; k < 3; ++k) { lo[k] = fminf(lo[k], p[k]); hi[k] = fminf(hi[k], -p[k]); }
    }
    mx = wave_sum(mx) / nv; my = wave_sum(my) / nv; mz = wave_sum(mz) / nv;
    double diameter = 0.0;
    for (int k = 0; k < 3; ++k) {
        const double e = (double)-wave_least(hi[k]) - wave_least(lo[k]);
        diameter += e * e;
    }
    diameter = sqrt(diameter);
    const double tol = 1e-5 * diameter;
    bool closed = true;
    float inner = INFINITY;
    double volume = 0.0;
    uint64_t edges = 0;
    for (int f = lane; f < nf; f += WAVE) {
        const float4 n4 = faceN[m.z + f], c = faceC[m.z + f];
        const double length = sqrt((double)n4.x * n4.x + (double)n4.y * n4.y + (double)n4.z * n4.z);
        const double nx = n4.x / length, ny = n4.y / length, nz = n4.z / length;
        auto over = [&](const float4& p) { return (p.x - (double)c.x) * nx + (p.y - (double)c.y) * ny + (p.z - (double)c.z) * nz; };
        const double depth = (c.x - mx) * nx + (c.y - my) * ny + (c.z - mz) * nz;
        closed = closed && depth > 0.0;   // no NaN either
        inner = fminf(inner, (float)depth);
        for (int i = 0; i < nv; ++i) closed = closed && over(v[i]) <= tol;
        const int2 F = face[m.z + f];
        closed = closed && F.y >= 3;
        for (int k = 0; k < F.y; ++k) {
            const int a = faceIdx[F.x + k], b = faceIdx[F.x + (k + 1 < F.y ? k + 1 : 0)];
            if (a < 0 || a >= nv || b < 0 || b >= nv) { closed = false; break; }
            closed = closed && over(v[a]) >= -tol;
            edges += edge_hash(a, b);
            const double ax = v[a].x - mx, ay = v[a].y - my, az = v[a].z - mz;
            const double bx = v[b].x - mx, by = v[b].y - my, bz = v[b].z - mz;
            volume += ((c.x - mx) * (ay * bz - az * by) + (c.y - my) * (az * bx - ax * bz) + (c.z - mz) * (ax * by - ay * bx)) / 6.0;
        }
    }
    for (int o = WAVE / 2; o >= 1; o >>= 1) edges += (uint64_t)__shfl_xor((unsigned long long)edges, o);
    volume = wave_sum(volume);
    const double ball = wave_least(inner);
    const bool ok = !__ballot(!closed) && edges == 0 && fabs(volume) >= 4.0 * ball * ball * ball;
    if (lane == 0) slender[blockIdx.x] = ok ? (float)(diameter / ball) : INFINITY;
}

// Ray i: origin, direction and maxDistance as the caller holds them (3, 3 and 1 floats), the
// world it is cast in and the entity it ignores (null: world 0, none).
//
// The walk is a chain of dependent, scattered node loads, so its length and the lines it
// touches are the cost: on the 32k scene a ray's line meets the boxes of some thirty colliders
// deep in a pile that it ends in after one or two. Children are visited nearest first (the
// other one waits in an LDS stack with its entry distance) and boxes beyond the best hit are
// skipped; the lanes of a wave descend together, then test their leaves together; a visit
// reads one 64-byte record. Which order the colliders are tested in does not reach the result
// (least distance, then least index) while every distance is a number, so a ray that may not
// skip takes the same walk, entering every box; a subtree that finds the stack full, and a ray
// whose result could depend on the order, are walked along the escape links, which need no
// stack. 262,144 rays into 32k bodies: 1,616 us along the links, 560 us nearest first with
// skipping (nine loads of three arrays a visit), 390 us with the records, 407 us with the boxes
// near the origin kept; the records take 12 us to write. 1,048,576 rays of directions that are
// not unit vectors: 6.4 ms with the tree in a kernel that only follows the links, 8.6 ms where
// they did that here, 6.9 ms in this walk, 5.8 ms with a stack of 12 instead of 20 (six blocks
// of 24 KB a CU, not four; ten measure the same); half of them unit vectors, which wait for the
// others of their wave: 6.3, 8.0, 5.8 and 4.8 ms.
constexpr int RAY_THREADS = 256, RAY_STACK = 12;
__global__ __launch_bounds__(RAY_THREADS) void k_raycast(int n, const float* __restrict__ ro, const float* __restrict__ rd,
                                                 const float* __restrict__ rmax, const int32_t* __restrict__ rworld,
                                                 const uint32_t* __restrict__ ignore, RayScene S,
                                                 int32_t* __restrict__ hitCol, float* __restrict__ hitT) {
    __shared__ int32_t waiting[RAY_STACK][RAY_THREADS];
    __shared__ float entry[RAY_STACK][RAY_THREADS];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const f3 o = mk3(ro[3 * (size_t)i], ro[3 * (size_t)i + 1], ro[3 * (size_t)i + 2]);
    const f3 d = mk3(rd[3 * (size_t)i], rd[3 * (size_t)i + 1], rd[3 * (size_t)i + 2]);
    const f3 inv = ray_inverse(d);
    const float maxDist = rmax[i];
    const int wd = rworld ? rworld[i] : 0;
    const uint32_t ig = ignore ? ignore[i] : 0xffffffffu;
    float bestT = 0.f;
    int best = -1;
    const int root = S.worldRoot[wd];
    RaySkip skip{s3(0.f), -1.f, 0.f, false};
    if (root != -1 && !(root & LEAF_BIT) && !S.rules->inOrder)
        skip = ray_skip(o, d, inv, xyz(S.nodeA[root]), xyz(S.nodeB[root]), S.rules->near, !S.rules->noSkip);
    auto statics = [&]() {
        for (int st = S.worldStaticStart[wd]; st < S.worldStaticStart[wd + 1]; ++st)
            test_collider(S, S.staticCols[st], o, d, inv, maxDist, ig, bestT, best);
    };
    // enter: the box is met within maxDistance, and not beyond the best hit; t: where it may be met
    auto enter = [&](const float4& mn, const float4& mx, float& t) {
        if (!ray_aabb(o, d, inv, xyz(mn), xyz(mx), t) || !(t <= maxDist)) return false;
        if (skip.margin < 0.f) { t = 0.f; return true; }
        t = widened_entry(skip, o, xyz(mn), xyz(mx));
        return best < 0 || !(t > fmaxf(bestT, skip.near));
    };
    int visits = 0;   // a walk visits at most 2n - 1 nodes
    float t;
    auto leaf = [&](int node) { test_collider(S, S.mvals[node & ~LEAF_BIT], o, d, inv, maxDist, ig, bestT, best); };
    auto follow = [&](int node, int stop) {   // the subtree's nodes along the escape links
        while (node != stop && node != -1 && ++visits <= 2 * S.nLeaves) {
            if (node & LEAF_BIT) {
                leaf(node);
                node = __float_as_int(S.leafA[node & ~LEAF_BIT].w);
            } else {
                const float4 na = S.nodeA[node], nb = S.nodeB[node];
                node = enter(na, nb, t) ? __float_as_int(na.w) : __float_as_int(nb.w);
            }
        }
    };
    int sp = 0;
    auto pop = [&]() {   // the next waiting subtree that is not beyond the best hit by now
        while (sp > 0) {
            --sp;
            if (best < 0 || !(entry[sp][threadIdx.x] > fmaxf(bestT, skip.near))) return waiting[sp][threadIdx.x];
        }
        return -1;
    };
    auto shape = [&](int node) {   // a leaf whose box is entered: the rest of test_collider
        const float4* L = S.rayLeaf + 4 * (size_t)(node & ~LEAF_BIT);
        const float4 p = L[0], q = L[1], prm = L[2], id = L[3];
        const int c = __float_as_int(id.x);
        if (__float_as_uint(id.y) == ig) return;
        if (!ray_shape(__float_as_int(p.w), prm, xyz(p), q4(q), S.cv, o, d, t) || t > maxDist) return;
        if (best < 0 || t < bestT || (t == bestT && c < best)) { best = c; bestT = t; }
    };
    if (skip.numbers) statics();   // a wall behind the ray's pile ends its walk early
    // NaN: a static's, kept as the first hit; the order decides then
    if (!skip.numbers || bestT != bestT) {
        skip.margin = -1.f;
        best = -1; bestT = 0.f;
        if (root != -1) follow(root, S.worldStop[wd]);
        statics();
    } else {
        // the wave's lanes all descend to a leaf (or to the end), then all test theirs
        int node = root;
        if (!enter(S.nodeA[node], S.nodeB[node], t)) node = -1;
        while (node != -1) {
            while (!(node & LEAF_BIT)) {
                if (++visits > 2 * S.nLeaves) { node = -1; break; }
                const float4* N = S.rayNode + 4 * (size_t)node;
                const float4 n0 = N[0], n1 = N[1], n2 = N[2], n3 = N[3];
                const int l = __float_as_int(n0.w), r = __float_as_int(n1.w);
                float tl = 0.f, tr = 0.f;
                const bool hl = enter(n0, n1, tl), hr = enter(n2, n3, tr);
                if (hl && hr) {
                    const bool lf = !(tr < tl);
                    const int far = lf ? r : l;
                    if (sp < RAY_STACK) {
                        waiting[sp][threadIdx.x] = far;
                        entry[sp++][threadIdx.x] = lf ? tr : tl;
                    } else if (far & LEAF_BIT) {
                        shape(far);
                    } else {
                        follow(far, __float_as_int(S.nodeB[far].w));
                    }
                    node = lf ? l : r;
                } else {
                    node = hl ? l : hr ? r : pop();
                }
            }
            if (node == -1) break;   // (-1 has LEAF_BIT)
            shape(node);
            node = pop();
        }
    }
    hitCol[i] = best;
    hitT[i] = best >= 0 ? bestT : 0.f;
}

}  // namespace

namespace pgx {

void qr_raycast(World& w, int n, const float* origins, const float* dirs, const float* maxDist,
                const int32_t* rayWorld, const uint32_t* ignoreEntity, int32_t* hitCollider, float* hitDistance,
                double* deviceUs) {
    hipStream_t s = w.stream;
    const size_t n3 = 3 * (size_t)n, f = sizeof(float);
    w.qRays.alloc(7 * (size_t)n); w.qRayWorld.alloc(n); w.qIgnore.alloc(n); w.qHit.alloc(n); w.qT.alloc(n);
    PGX_HIP(hipMemcpyAsync(w.qRays.p, origins, f * n3, hipMemcpyHostToDevice, s));
    PGX_HIP(hipMemcpyAsync(w.qRays.p + n3, dirs, f * n3, hipMemcpyHostToDevice, s));
    PGX_HIP(hipMemcpyAsync(w.qRays.p + 2 * n3, maxDist, f * n, hipMemcpyHostToDevice, s));
    if (rayWorld) PGX_HIP(hipMemcpyAsync(w.qRayWorld.p, rayWorld, sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
    if (ignoreEntity)
        PGX_HIP(hipMemcpyAsync(w.qIgnore.p, ignoreEntity, sizeof(uint32_t) * n, hipMemcpyHostToDevice, s));
    if (!w.qEv[0])
        for (auto& e : w.qEv) PGX_HIP(hipEventCreate(&e));
    PGX_HIP(hipEventRecord(w.qEv[0], s));
    fill_i32(s, w.counters.p + 7, 0, 4);   // the refit's work counter and the walks' rules
    RayRules* const rules = (RayRules*)(w.counters.p + 8);
    bp_build(w);
    RayScene S;
    S.W = w.W;
    S.nLeaves = w.nDynCol;
    S.worldRoot = w.worldRoot.p; S.worldStop = w.worldStop.p;
    S.worldStaticStart = w.worldStaticStart.p; S.staticCols = w.staticCols.p; S.mvals = w.mvals.p;
    w.qRayNode.alloc(4 * (size_t)std::max(w.nDynCol, 1)); w.qRayLeaf.alloc(4 * (size_t)std::max(w.nDynCol, 1));
    S.rules = rules; S.rayNode = w.qRayNode.p; S.rayLeaf = w.qRayLeaf.p;
    S.leafA = w.leafA.p; S.nodeA = w.nodeA.p; S.nodeB = w.nodeB.p;
    S.cbmin = w.cbmin.p; S.cbmax = w.cbmax.p; S.cparams = w.cparams.p; S.clpos = w.clpos.p; S.clquat = w.clquat.p;
    S.bpos = w.bpos.p; S.bquat = w.bquat.p; S.cbody = w.cbody.p; S.ctype = w.ctype.p; S.centity = w.centity.p;
    S.cv = ConvexFaces{w.cvMesh.p, w.cvFaceN.p, w.cvFaceC.p};
    S.cvVerts = w.cvVerts.p; S.cvSlender = w.cvSlender.p;
    if (w.nDynCol == 0) {
        fill_i32(s, w.worldRoot.p, -1, w.W);   // no tree: static lists only
    } else {
        hipLaunchKernelGGL(k_ray_records, dim3(div_up(w.nDynCol, 256)), dim3(256), 0, s, w.nDynCol, w.nodeChild.p, S,
                           w.leafB.p, w.clquat.p, w.qRayNode.p, w.qRayLeaf.p, rules);
        PGX_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_raycast, dim3(div_up(n, RAY_THREADS)), dim3(RAY_THREADS), 0, s, n, w.qRays.p, w.qRays.p + n3,
                       w.qRays.p + 2 * n3, rayWorld ? w.qRayWorld.p : nullptr, ignoreEntity ? w.qIgnore.p : nullptr, S,
                       w.qHit.p, w.qT.p);
    PGX_LAUNCH_CHECK();
    PGX_HIP(hipEventRecord(w.qEv[1], s));
    PGX_HIP(hipMemcpyAsync(hitCollider, w.qHit.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost, s));
    PGX_HIP(hipMemcpyAsync(hitDistance, w.qT.p, sizeof(float) * n, hipMemcpyDeviceToHost, s));
    PGX_HIP(hipStreamSynchronize(s));
    if (deviceUs) {
        float ms = 0.f;
        PGX_HIP(hipEventElapsedTime(&ms, w.qEv[0], w.qEv[1]));
        *deviceUs = 1000.0 * ms;
    }
}

// query shapes to the device: params, position (.w = world id bits), orientation; types
static void upload_query_shapes(World& w, int n, const int32_t* types, const float* params, const float* positions,
                                const float* orientations, const int32_t* queryWorld) {
    std::vector<float4> hs(3 * (size_t)n);
    for (int i = 0; i < n; ++i) {
        int32_t wd = queryWorld ? queryWorld[i] : 0;
        float wbits;
        std::memcpy(&wbits, &wd, sizeof wbits);
        hs[i] = make_float4(params[4 * i], params[4 * i + 1], params[4 * i + 2], params[4 * i + 3]);
        hs[n + i] = make_float4(positions[3 * i], positions[3 * i + 1], positions[3 * i + 2], wbits);
        hs[2 * (size_t)n + i] = make_float4(orientations[4 * i], orientations[4 * i + 1], orientations[4 * i + 2],
                                            orientations[4 * i + 3]);
    }
    w.qShape.alloc(3 * (size_t)n); w.qType.alloc(n);
    PGX_HIP(hipMemcpyAsync(w.qShape.p, hs.data(), sizeof(float4) * 3 * (size_t)n, hipMemcpyHostToDevice, w.stream));
    PGX_HIP(hipMemcpyAsync(w.qType.p, types, sizeof(int32_t) * n, hipMemcpyHostToDevice, w.stream));
    PGX_HIP(hipStreamSynchronize(w.stream));   // hs is released on return
}

// Candidate triangles of one pass over the queries: 72 bytes each, and 144 more in a world with
// hulls, so at most 1.2 or 3.6 GB. A call with more of them is made of several passes.
constexpr int MTD_MAX_CANDS = 1 << 24;

// One pass: PGX_OK or PGX_ERR_CAPACITY, or, with *candidates set, MTD_TOO_MANY.
constexpr int MTD_TOO_MANY = 1;
static int overlap_mtd_pass(World& w, int n, const int32_t* types, const float* params, const float* positions,
                            const float* orientations, const int32_t* queryWorld, int capacity, int32_t* offsets,
                            int32_t* colliders, float* normalMtd, int32_t* total, double* deviceUs, int* candidates) {
    constexpr int MBITS = 8;   // manifold index within a pair (the kernels' MTD_MBITS)
    constexpr int MTD_COUNTS = 6;
    hipStream_t s = w.stream;
    int cbits = 1;
    while ((1L << cbits) < (long)w.C) ++cbits;
    int qbits = 1;
    while ((1L << qbits) < (long)n) ++qbits;
    if (qbits + cbits + MBITS > 64) throw PgxError{PGX_ERR_UNSUPPORTED, "too many queries and colliders for one call"};
    upload_query_shapes(w, n, types, params, positions, orientations, queryWorld);
    w.qMtdN.alloc(MTD_COUNTS);
    w.qKeys.alloc(std::max(capacity, 1)); w.qVals.alloc(std::max(capacity, 1)); w.qRes.alloc(std::max(capacity, 1));
    if (!w.qEv[0])
        for (auto& e : w.qEv) PGX_HIP(hipEventCreate(&e));
    MtdArgs A;
    A.n = n; A.nLeaves = w.nDynCol; A.cap = capacity; A.cbits = cbits;
    A.qPrm = w.qShape.p; A.qPos = w.qShape.p + n; A.qQuat = w.qShape.p + 2 * (size_t)n; A.qType = w.qType.p;
    A.worldRoot = w.worldRoot.p; A.worldStop = w.worldStop.p;
    A.worldStaticStart = w.worldStaticStart.p; A.staticCols = w.staticCols.p; A.mvals = w.mvals.p;
    A.leafA = w.leafA.p; A.nodeA = w.nodeA.p; A.nodeB = w.nodeB.p;
    A.cbmin = w.cbmin.p; A.cbmax = w.cbmax.p; A.cparams = w.cparams.p; A.clpos = w.clpos.p; A.clquat = w.clquat.p;
    A.bpos = w.bpos.p; A.bquat = w.bquat.p; A.cbody = w.cbody.p; A.ctype = w.ctype.p;
    A.counts = w.qMtdN.p; A.keys = w.qKeys.p; A.vals = w.qVals.p; A.res = w.qRes.p;
    int cnt[MTD_COUNTS] = {};
    int listCap = (int)std::max<size_t>(std::max<size_t>(w.qCvxPairs.n, 4096), 4 * (size_t)n);
    size_t cands = std::max<size_t>({(size_t)w.qMesh.candCap, (size_t)1 << 18,
                                     std::min<size_t>(2 * (size_t)n, MTD_MAX_CANDS)});
    float ms0 = 0.f;
    // the second attempt with pair lists, the third with candidate lists as long as was needed
    for (int attempt = 0; attempt < 3; ++attempt) {
        w.qCvxPairs.alloc(listCap); w.qMeshPairs.alloc(listCap);
        if (w.nTriMesh > 0) np_mesh_buffers(w, w.qMesh, listCap, cands);
        A.listCap = listCap; A.convexPairs = w.qCvxPairs.p; A.meshPairs = w.qMeshPairs.p;
        PGX_HIP(hipEventRecord(w.qEv[0], s));
        fill_i32(s, w.qMtdN.p, 0, MTD_COUNTS);
        fill_i32(s, w.counters.p + 7, 0, 1);   // the refit's work counter
        bp_build(w);
        if (w.nDynCol == 0) fill_i32(s, w.worldRoot.p, -1, w.W);   // no tree: static lists only
        np_mtd_launch(w, A);
        PGX_HIP(hipEventRecord(w.qEv[1], s));
        PGX_HIP(hipMemcpyAsync(cnt, w.qMtdN.p, sizeof cnt, hipMemcpyDeviceToHost, s));
        PGX_HIP(hipStreamSynchronize(s));
        PGX_HIP(hipEventElapsedTime(&ms0, w.qEv[0], w.qEv[1]));
        const bool pairs = std::max(cnt[1], cnt[2]) <= listCap;
        if (pairs && (w.nTriMesh == 0 || cnt[4] <= w.qMesh.candCap)) break;
        if (w.nTriMesh > 0 && cnt[4] > std::max(w.qMesh.candCap, MTD_MAX_CANDS) && n > 1) {
            *candidates = cnt[4];
            return MTD_TOO_MANY;
        }
        if (attempt == 2) throw PgxError{PGX_ERR_HIP, "MTD query: pair or candidate lists overflowed again"};
        if (!pairs) listCap = std::max(cnt[1], cnt[2]);
        else cands = (size_t)cnt[4];
    }
    if (cnt[3]) throw PgxError{PGX_ERR_CAPACITY, "MTD query: EPA or triangle-candidate workspace overflow in " +
                                                     std::to_string(cnt[3]) + " pairs"};
    *total = cnt[0];
    if (deviceUs) *deviceUs = 1000.0 * ms0;
    if (cnt[0] > capacity) return PGX_ERR_CAPACITY;
    const int m = cnt[0];
    float ms1 = 0.f;
    if (m > 1) {
        PGX_HIP(hipEventRecord(w.qEv[2], s));
        radix_sort_u64(s, w.qKeys.p, w.qVals.p, m, qbits + cbits + MBITS, w.sortT);
        PGX_HIP(hipEventRecord(w.qEv[3], s));
    }
    std::vector<uint64_t> keys((size_t)m);
    std::vector<int32_t> vals((size_t)m);
    std::vector<float4> res((size_t)m);
    if (m) {
        PGX_HIP(hipMemcpyAsync(keys.data(), w.qKeys.p, 8 * (size_t)m, hipMemcpyDeviceToHost, s));
        PGX_HIP(hipMemcpyAsync(vals.data(), w.qVals.p, 4 * (size_t)m, hipMemcpyDeviceToHost, s));
        PGX_HIP(hipMemcpyAsync(res.data(), w.qRes.p, 16 * (size_t)m, hipMemcpyDeviceToHost, s));
    }
    PGX_HIP(hipStreamSynchronize(s));
    if (m > 1 && deviceUs) {
        PGX_HIP(hipEventElapsedTime(&ms1, w.qEv[2], w.qEv[3]));
        *deviceUs = 1000.0 * (ms0 + ms1);
    }
    const uint64_t cmask = (1ull << cbits) - 1;
    int k = 0;
    for (int i = 0; i < n; ++i) {
        offsets[i] = k;
        while (k < m && (int)(keys[k] >> (cbits + MBITS)) == i) {
            colliders[k] = (int32_t)((keys[k] >> MBITS) & cmask);
            const float4 r = res[vals[k]];
            normalMtd[4 * k] = r.x; normalMtd[4 * k + 1] = r.y; normalMtd[4 * k + 2] = r.z; normalMtd[4 * k + 3] = r.w;
            ++k;
        }
    }
    offsets[n] = k;
    if (k != m) throw PgxError{PGX_ERR_HIP, "MTD query: result keys out of order"};
    return PGX_OK;
}

void qr_hull_slenderness(World& w) {
    w.cvSlender.alloc(w.nConvex);
    hipLaunchKernelGGL(k_hull_slenderness, dim3(w.nConvex), dim3(WAVE), 0, w.stream, w.cvMesh.p, w.cvVerts.p, w.cvFace.p,
                       w.cvFaceIdx.p, w.cvFaceN.p, w.cvFaceC.p, w.cvSlender.p);
    PGX_LAUNCH_CHECK();
}

int qr_overlap_mtd(World& w, int n, const int32_t* types, const float* params, const float* positions,
                   const float* orientations, const int32_t* queryWorld, int capacity, int32_t* offsets,
                   int32_t* colliders, float* normalMtd, int32_t* total, double* deviceUs) {
    int candidates = 0;
    const int rc = overlap_mtd_pass(w, n, types, params, positions, orientations, queryWorld, capacity, offsets,
                                    colliders, normalMtd, total, deviceUs, &candidates);
    if (rc != MTD_TOO_MANY) return rc;
    // parts of the queries with about half of what a pass may have each, and their results one
    // after the other; the caller's arrays are written only when all of them fit
    const int part = (int)std::max<long long>(1, (long long)n * (MTD_MAX_CANDS / 2) / candidates);
    std::vector<int32_t> off((size_t)n + 1), cols((size_t)capacity);
    std::vector<float> nm(4 * (size_t)capacity);
    long long found = 0;
    double us = 0.0;
    for (int lo = 0; lo < n; lo += part) {
        const int m = std::min(part, n - lo);
        const int room = (int)std::max<long long>(0, capacity - found);
        int32_t t = 0;
        double partUs = 0.0;
        const size_t at = (size_t)(capacity - room);
        const int r = qr_overlap_mtd(w, m, types + lo, params + 4 * (size_t)lo, positions + 3 * (size_t)lo,
                                     orientations + 4 * (size_t)lo, queryWorld ? queryWorld + lo : nullptr, room,
                                     off.data() + lo, cols.data() + at, nm.data() + 4 * at, &t, &partUs);
        if (r != PGX_OK && r != PGX_ERR_CAPACITY) return r;
        if (r == PGX_OK)
            for (int i = 0; i <= m; ++i) off[lo + i] += (int32_t)found;
        found += t;
        us += partUs;
    }
    if (found > std::numeric_limits<int32_t>::max())
        throw PgxError{PGX_ERR_CAPACITY, "MTD query: " + std::to_string(found) + " hits are more than a call can return"};
    *total = (int32_t)found;
    if (deviceUs) *deviceUs = us;
    if (found > capacity) return PGX_ERR_CAPACITY;
    std::copy(off.begin(), off.end(), offsets);
    std::copy(cols.begin(), cols.begin() + found, colliders);
    std::copy(nm.begin(), nm.begin() + 4 * found, normalMtd);
    return PGX_OK;
}

// CharacterController::move (src/CharacterController.cpp:5-45) for every character: the
// rounds of MTD queries run on the device for all characters still moving, and each
// character's hits are applied on the host in order, as the reference's loop does.
void qr_character_move(World& w, int n, pgx_character* chars, const float* translations, uint8_t* flags) {
    std::vector<f3> pos((size_t)n), up((size_t)n);
    int rounds = 0;
    for (int i = 0; i < n; ++i) {
        const pgx_character& c = chars[i];
        const qf q{c.orientation[0], c.orientation[1], c.orientation[2], c.orientation[3]};
        up[i] = qrot(q, mk3(0.f, 1.f, 0.f));
        pos[i] = add(mk3(c.position[0], c.position[1], c.position[2]),
                     mk3(translations[3 * i], translations[3 * i + 1], translations[3 * i + 2]));
        flags[i] = 0;
        rounds = std::max(rounds, (int)c.num_iterations);
    }
    std::vector<int32_t> idx, types, qworld, off, cols;
    std::vector<float> prm, qpos, qori, nm;
    int cap = 8 * n + 1024;
    for (int r = 0; r < rounds; ++r) {
        idx.clear(); types.clear(); qworld.clear(); prm.clear(); qpos.clear(); qori.clear();
        for (int i = 0; i < n; ++i) {
            const pgx_character& c = chars[i];
            if (r >= c.num_iterations) continue;
            idx.push_back(i);
            types.push_back(PGX_CAPSULE);
            qworld.push_back(c.world);
            prm.insert(prm.end(), {c.height * 0.5f, c.radius, 0.f, 0.f});
            const f3 centre = add(pos[i], mul(up[i], c.height * 0.5f + c.radius));
            qpos.insert(qpos.end(), {centre.x, centre.y, centre.z});
            qori.insert(qori.end(), {c.orientation[0], c.orientation[1], c.orientation[2], c.orientation[3]});
        }
        const int m = (int)idx.size();
        if (m == 0) continue;
        off.assign((size_t)m + 1, 0);
        int32_t total = 0;
        while (true) {
            cols.resize((size_t)cap);
            nm.resize(4 * (size_t)cap);
            if (qr_overlap_mtd(w, m, types.data(), prm.data(), qpos.data(), qori.data(), qworld.data(), cap,
                               off.data(), cols.data(), nm.data(), &total, nullptr) == PGX_OK)
                break;
            cap = total;   // PGX_ERR_CAPACITY: room for every hit
        }
        for (int j = 0; j < m; ++j) {
            const int i = idx[j];
            const float slope = chars[i].slope_limit;
            for (int k = off[j]; k < off[j + 1]; ++k) {
                const f3 nk = mk3(nm[4 * (size_t)k], nm[4 * (size_t)k + 1], nm[4 * (size_t)k + 2]);
                const float mtd = nm[4 * (size_t)k + 3];
                const float d = dot(nk, up[i]);
                if (d > 0.001f) flags[i] |= 1;          // DOWN
                else if (d < -0.001f) flags[i] |= 4;    // UP
                else flags[i] |= 2;                     // SIDES
                pos[i] = d > slope ? add(pos[i], divs(mul(up[i], mtd), d)) : add(pos[i], mul(nk, mtd));
            }
        }
    }
    for (int i = 0; i < n; ++i) {
        chars[i].position[0] = pos[i].x; chars[i].position[1] = pos[i].y; chars[i].position[2] = pos[i].z;
    }
}

int qr_overlap(World& w, int n, const int32_t* types, const float* params, const float* positions,
               const float* orientations, const int32_t* queryWorld, const int32_t* filters, int capacity,
               int32_t* offsets, int32_t* colliders, int32_t* total, double* deviceUs) {
    hipStream_t s = w.stream;
    int cbits = 1;
    while ((1L << cbits) < (long)w.C) ++cbits;
    int qbits = 1;
    while ((1L << qbits) < (long)n) ++qbits;
    std::vector<float4> hs(3 * (size_t)n);
    for (int i = 0; i < n; ++i) {
        int32_t wd = queryWorld ? queryWorld[i] : 0;
        float wbits;
        std::memcpy(&wbits, &wd, sizeof wbits);
        hs[i] = make_float4(params[4 * i], params[4 * i + 1], params[4 * i + 2], params[4 * i + 3]);
        hs[n + i] = make_float4(positions[3 * i], positions[3 * i + 1], positions[3 * i + 2], wbits);
        hs[2 * (size_t)n + i] = make_float4(orientations[4 * i], orientations[4 * i + 1], orientations[4 * i + 2],
                                            orientations[4 * i + 3]);
    }
    std::vector<int32_t> hf(filters ? filters : nullptr, filters ? filters + n : nullptr);
    if (!filters) hf.assign((size_t)n, 0);
    w.qShape.alloc(3 * (size_t)n); w.qType.alloc(n); w.qFilter.alloc(n); w.qCount.alloc((size_t)n + 2);
    w.qKeys.alloc(std::max(capacity, 1)); w.qVals.alloc(std::max(capacity, 1));
    PGX_HIP(hipMemcpyAsync(w.qShape.p, hs.data(), sizeof(float4) * 3 * (size_t)n, hipMemcpyHostToDevice, s));
    PGX_HIP(hipMemcpyAsync(w.qType.p, types, sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
    PGX_HIP(hipMemcpyAsync(w.qFilter.p, hf.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
    if (!w.qEv[0])
        for (auto& e : w.qEv) PGX_HIP(hipEventCreate(&e));
    OverlapArgs A;
    A.n = n; A.nLeaves = w.nDynCol; A.cap = capacity; A.cbits = cbits;
    A.qPrm = w.qShape.p; A.qPos = w.qShape.p + n; A.qQuat = w.qShape.p + 2 * (size_t)n;
    A.qType = w.qType.p; A.qFilter = w.qFilter.p;
    A.worldRoot = w.worldRoot.p; A.worldStop = w.worldStop.p;
    A.worldStaticStart = w.worldStaticStart.p; A.staticCols = w.staticCols.p; A.mvals = w.mvals.p;
    A.leafA = w.leafA.p; A.nodeA = w.nodeA.p; A.nodeB = w.nodeB.p;
    A.cbmin = w.cbmin.p; A.cbmax = w.cbmax.p; A.cparams = w.cparams.p; A.clpos = w.clpos.p; A.clquat = w.clquat.p;
    A.bpos = w.bpos.p; A.bquat = w.bquat.p; A.cbody = w.cbody.p; A.ctype = w.ctype.p; A.cdata = w.cdata.p;
    A.cv = ConvexView{w.cvVerts.p, w.cvMesh.p, w.cvFace.p, w.cvFaceIdx.p, w.cvFaceN.p, w.cvFaceC.p};
    A.count = w.qCount.p; A.total = w.qCount.p + n; A.keys = w.qKeys.p; A.nCvx = w.qCount.p + n + 1;
    std::vector<int32_t> cnt((size_t)n + 2);
    int listCap = (int)std::max<size_t>(std::max<size_t>(w.qCvxPairs.n, 4096), (size_t)n);
    float ms0 = 0.f;
    for (int attempt = 0; attempt < 2; ++attempt) {   // the second with a convex-pair list as long as needed
        w.qCvxPairs.alloc(listCap);
        A.cvxPairs = w.qCvxPairs.p; A.listCap = listCap;
        PGX_HIP(hipEventRecord(w.qEv[0], s));
        fill_i32(s, w.counters.p + 7, 0, 1);   // the refit's work counter
        fill_i32(s, w.qCount.p + n, 0, 2);     // the hit and convex-pair counters
        bp_build(w);
        if (w.nDynCol == 0) fill_i32(s, w.worldRoot.p, -1, w.W);   // no tree: static lists only
        np_overlap_launch(s, A, w.nConvex > 0);
        PGX_HIP(hipEventRecord(w.qEv[1], s));
        PGX_HIP(hipMemcpyAsync(cnt.data(), w.qCount.p, sizeof(int32_t) * ((size_t)n + 2), hipMemcpyDeviceToHost, s));
        PGX_HIP(hipStreamSynchronize(s));
        PGX_HIP(hipEventElapsedTime(&ms0, w.qEv[0], w.qEv[1]));
        if (cnt[n + 1] <= listCap) break;
        if (attempt == 1) throw PgxError{PGX_ERR_HIP, "overlap: the convex-pair list overflowed twice"};
        listCap = cnt[n + 1];
    }
    long sum = 0;
    for (int i = 0; i < n; ++i) {
        offsets[i] = (int32_t)sum;
        sum += cnt[i];
    }
    offsets[n] = (int32_t)sum;
    *total = (int32_t)sum;
    if (sum != cnt[n]) throw PgxError{PGX_ERR_HIP, "overlap: the per-query hit counts disagree with the total"};
    if (deviceUs) *deviceUs = 1000.0 * ms0;
    if (sum > capacity) return PGX_ERR_CAPACITY;
    if (sum == 0) return PGX_OK;
    // the hits of each query ascending by collider: sort the keys (query, collider)
    PGX_HIP(hipEventRecord(w.qEv[2], s));
    radix_sort_u64(s, w.qKeys.p, w.qVals.p, (int)sum, qbits + cbits, w.sortT);
    PGX_HIP(hipEventRecord(w.qEv[3], s));
    std::vector<uint64_t> keys((size_t)sum);
    PGX_HIP(hipMemcpyAsync(keys.data(), w.qKeys.p, sizeof(uint64_t) * sum, hipMemcpyDeviceToHost, s));
    PGX_HIP(hipStreamSynchronize(s));
    const uint64_t cmask = (1ull << cbits) - 1;
    for (long k = 0; k < sum; ++k) colliders[k] = (int32_t)(keys[k] & cmask);
    if (deviceUs) {
        float ms1 = 0.f;
        PGX_HIP(hipEventElapsedTime(&ms1, w.qEv[2], w.qEv[3]));
        *deviceUs = 1000.0 * (ms0 + ms1);
    }
    return PGX_OK;
}

}  // namespace pgx
