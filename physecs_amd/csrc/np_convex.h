// Convex-mesh narrowphase on the device: GJK (src/GJK.h:131-292); with np_wave.h, EPA
// (src/EPA.h:9-186) and the convex contact generators (src/Collision.cpp:352-426,488-499,694-887,
// src/ContactsUtil.cpp:109-204), operation for operation with the reference, including
// its mixed precision: simplex and polytope vertices are doubles, every support query
// narrows its direction to float, and the float helpers the reference feeds with double
// vectors (isZero, sqrDistPointToLine, distPointToPlane, the barycentric edges) narrow
// them the same way.
//
// Pairs with a convex mesh on either side are taken out of the one-pair-per-lane
// primitive kernel into a list and solved a wave per pair (np_wave.h). The single-lane GJK
// here serves the yes/no overlap tests.
// Included by narrowphase.hip (shares its clipping and box-face routines).
#pragma once

namespace pgx {

constexpr int CVX_MAXPOLY = 40;   // a clipped face polygon (faces have at most 16 vertices)


// ------------------------------------------------------------------ support maps
struct SupSphere {                                  // src/GJK.h:13-20
    f3 pos; float r;
    __device__ f3 operator()(f3 d) const { return add(pos, mul(d, r)); }
};
struct SupCapsule {                                 // src/GJK.h:22-31
    f3 pos, axis; float hh, r;
    __device__ f3 operator()(f3 d) const {
        return add(add(pos, mul(mul(axis, gsign(dot(d, axis))), hh)), mul(d, r));
    }
};
struct SupBox {                                     // src/GJK.h:33-45
    f3 pos; m3 l2w; f3 he;
    __device__ f3 operator()(f3 d) const {
        f3 s = pos;
        for (int i = 0; i < 3; ++i) {
            f3 c = col(l2w, i);
            s = add(s, mul(mul(gsign(dot(d, c)), c), at(he, i)));
        }
        return s;
    }
};
// src/GJK.h:47-107: four interleaved running maxima (vertex i -> lane i % 4, strict '>'),
// then the lanes compared in order with strict '>'
struct SupConvex {
    f3 pos; m3 l2w; f3 scale; const float4* v; int count;
    __device__ f3 operator()(f3 dir) const {
        dir = mulv(scale, mk3(dot(dir, l2w.c0), dot(dir, l2w.c1), dot(dir, l2w.c2)));
        float mv[4];
        int mi[4] = {0, 1, 2, 3};
        for (int k = 0; k < 4; ++k) mv[k] = -3.402823466e+38f;
        for (int i = 0; i < count; i += 4) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float4 p = v[i + k];
                float d = (p.x * dir.x + p.y * dir.y) + p.z * dir.z;
                if (d > mv[k]) mi[k] = i + k;
                mv[k] = d > mv[k] ? d : mv[k];
            }
        }
        int best = mi[0];
        float bv = mv[0];
        for (int k = 1; k < 4; ++k)
            if (mv[k] > bv) { bv = mv[k]; best = mi[k]; }
        return add(pos, mulmv(l2w, mulv(scale, xyz(v[best]))));
    }
};

// ------------------------------------------------------------------ GJK
struct GjkV { d3 pos, sp0, sp1; };

template <class S0, class S1>
__device__ __forceinline__ GjkV mdiff(const S0& s0, const S1& s1, f3 dir) {      // src/GJK.h:192-196
    f3 a = s0(dir);
    f3 b = s1(neg(dir));
    GjkV r;
    r.pos = wide(sub(a, b)); r.sp0 = wide(a); r.sp1 = wide(b);
    return r;
}
__device__ __forceinline__ float sqr_dist_point_line(f3 p, f3 a, f3 b) {          // src/GJK.h:142-148
    f3 r = sub(p, a), d = sub(b, a);
    f3 q = add(a, mul(dot(r, d) / dot(d, d), d));
    f3 pq = sub(p, q);
    return dot(pq, pq);
}
__device__ __forceinline__ float dist_point_plane(f3 p, f3 o, f3 n) { return gabs(dot(sub(p, o), n)); }
__device__ __forceinline__ bool is_zero(f3 v) { return (double)dot(v, v) < 1e-6; }

template <class S0, class S1>
__device__ bool check_direction(const S0& s0, const S1& s1, d3 dir, GjkV& v) {    // src/GJK.h:162-167
    dir = dnormalize(dir);
    v = mdiff(s0, s1, narrow(dir));
    return ddot(v.pos, dir) >= 0;
}
__device__ __forceinline__ bool check_face(d3 v0, d3 v1, d3 v2, d3 opp, d3& n) {  // src/GJK.h:169-173
    n = dcross(dsub(v1, v0), dsub(v2, v0));
    n = dmul(dsign(ddot(dsub(v0, opp), n)), n);
    return ddot(n, dneg(v0)) > (double)0.00001f;
}
template <class S0, class S1>
__device__ void complete_from_line(const S0& s0, const S1& s1, GjkV* s) {         // src/GJK.h:233-243
    d3 dir = dcross(dsub(s[0].pos, s[1].pos), mkd(0, 1, 0));
    if (is_zero(narrow(dir))) dir = dcross(dsub(s[0].pos, s[1].pos), mkd(0, 0, 1));
    s[2] = mdiff(s0, s1, narrow(dnormalize(dir)));
    if (sqr_dist_point_line(narrow(s[2].pos), narrow(s[0].pos), narrow(s[1].pos)) < 0.00001f)
        s[2] = mdiff(s0, s1, narrow(dneg(dir)));
    dir = dnormalize(dcross(dsub(s[1].pos, s[0].pos), dsub(s[2].pos, s[0].pos)));
    s[3] = mdiff(s0, s1, narrow(dir));
    if (dist_point_plane(narrow(s[3].pos), narrow(s[0].pos), narrow(dir)) < 0.0001f)
        s[3] = mdiff(s0, s1, narrow(dneg(dir)));
}
template <class S0, class S1>
__device__ bool gjk(const S0& s0, const S1& s1, f3 startDir, GjkV* s) {          // src/GJK.h:226-292
    d3 dir = wide(normalize(startDir));
    s[0] = mdiff(s0, s1, narrow(dir));
    if (is_zero(narrow(s[0].pos))) {
        dir = dneg(dir);
        s[1] = mdiff(s0, s1, narrow(dir));
        complete_from_line(s0, s1, s);
        return true;
    }
    dir = dneg(s[0].pos);
    if (!check_direction(s0, s1, dir, s[1])) return false;
    dir = dcross(dcross(dsub(s[0].pos, s[1].pos), dneg(s[1].pos)), dsub(s[0].pos, s[1].pos));
    if (is_zero(narrow(dir))) {
        complete_from_line(s0, s1, s);
        return true;
    }
    if (!check_direction(s0, s1, dir, s[2])) return false;
    dir = dcross(dsub(s[1].pos, s[0].pos), dsub(s[2].pos, s[0].pos));
    double sg = dsign(ddot(dneg(s[0].pos), dir));
    if (!sg) {
        dir = dnormalize(dir);
        s[3] = mdiff(s0, s1, narrow(dir));
        if (dist_point_plane(narrow(s[3].pos), narrow(s[0].pos), narrow(dir)) < 0.0001f)
            s[3] = mdiff(s0, s1, narrow(dneg(dir)));
        return true;
    }
    dir = dmul(sg, dir);
    if (!check_direction(s0, s1, dir, s[3])) return false;
    for (int i = 0; i < 100; ++i) {
        // simplexContainsOrigin (src/GJK.h:175-181)
        int fi = 2;
        bool outside = check_face(s[3].pos, s[0].pos, s[1].pos, s[2].pos, dir);
        if (!outside) { fi = 1; outside = check_face(s[3].pos, s[2].pos, s[0].pos, s[1].pos, dir); }
        if (!outside) { fi = 0; outside = check_face(s[3].pos, s[1].pos, s[2].pos, s[0].pos, dir); }
        if (!outside) return true;
        if (!check_direction(s0, s1, dir, s[fi])) return false;
        GjkV t = s[fi];
        s[fi] = s[3];
        s[3] = t;
    }
    return false;
}

// ------------------------------------------------------------------ contact generation
__device__ bool clip_line_n(f2& p0, f2& p1, const f2* clip, int nclip) {        // src/Clipping.cpp:55-71
    for (int i = 0; i < nclip; ++i) {
        int j = (i + 1) % nclip;
        bool in0 = inside(p0, clip[i], clip[j]), in1 = inside(p1, clip[i], clip[j]);
        if (in0 && in1) continue;
        if (in0) p1 = intersect2(p0, p1, clip[i], clip[j]);
        else if (in1) p0 = intersect2(p0, p1, clip[i], clip[j]);
        else return false;
    }
    return true;
}

__device__ __forceinline__ f3 world_face_normal(qf q, f3 n, f3 scale) { return normalize(qrot(q, divv(n, scale))); }

struct MeshRef {
    const ConvexView* cv; int4 info;
    __device__ int nfaces() const { return info.w; }
    __device__ int2 face(int f) const { return cv->face[info.z + f]; }
    __device__ f3 fnormal(int f) const { return xyz(cv->faceN[info.z + f]); }
    __device__ f3 fcentroid(int f) const { return xyz(cv->faceC[info.z + f]); }
    __device__ f3 vert(int i) const { return xyz(cv->verts[info.x + i]); }
    __device__ f3 face_vert(int2 fc, int k) const { return vert(cv->faceIdx[fc.x + k]); }
};

}  // namespace pgx
