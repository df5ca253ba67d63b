// Convex-mesh narrowphase on the device: GJK (src/GJK.h:131-292), EPA (src/EPA.h:9-186)
// and the convex contact generators (src/Collision.cpp:352-426,488-499,694-887,
// src/ContactsUtil.cpp:109-204), operation for operation with the reference, including
// its mixed precision: simplex and polytope vertices are doubles, every support query
// narrows its direction to float, and the float helpers the reference feeds with double
// vectors (isZero, sqrDistPointToLine, distPointToPlane, the barycentric edges) narrow
// them the same way.
//
// Pairs with a convex mesh on either side are taken out of the one-pair-per-lane
// primitive kernel into a list and solved a wave per pair (np_wave.h). The single-lane forms
// here serve the yes/no overlap tests and, with a polytope workspace laid out
// lane-interleaved (element e of lane l at e * lanes + l), the triangle-mesh MTD queries.
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

// ------------------------------------------------------------------ EPA
// one lane's polytope in the lane-interleaved workspace
struct EpaWs {
    double* vd;       // 9 doubles per vertex: pos, sp0, sp1
    int* fi;          // 3 ints per face
    double* fn;       // 3 doubles per face (unit normal)
    int* ed;          // 2 ints per loose edge
    size_t L;         // lanes
    int nv, nf;
    bool overflow;
    __device__ double& V(int v, int c) { return vd[(size_t)(v * 9 + c) * L]; }
    __device__ int& FI(int f, int k) { return fi[(size_t)(f * 3 + k) * L]; }
    __device__ double& FN(int f, int c) { return fn[(size_t)(f * 3 + c) * L]; }
    __device__ int& E(int e, int k) { return ed[(size_t)(e * 2 + k) * L]; }
    __device__ d3 pos(int v) { return mkd(V(v, 0), V(v, 1), V(v, 2)); }
    __device__ d3 normal(int f) { return mkd(FN(f, 0), FN(f, 1), FN(f, 2)); }
    __device__ void putV(int v, const GjkV& g) {
        V(v, 0) = g.pos.x; V(v, 1) = g.pos.y; V(v, 2) = g.pos.z;
        V(v, 3) = g.sp0.x; V(v, 4) = g.sp0.y; V(v, 5) = g.sp0.z;
        V(v, 6) = g.sp1.x; V(v, 7) = g.sp1.y; V(v, 8) = g.sp1.z;
    }
    __device__ GjkV getV(int v) {
        GjkV g;
        g.pos = mkd(V(v, 0), V(v, 1), V(v, 2));
        g.sp0 = mkd(V(v, 3), V(v, 4), V(v, 5));
        g.sp1 = mkd(V(v, 6), V(v, 7), V(v, 8));
        return g;
    }
    __device__ void create_face(int i0, int i1, int i2) {              // src/EPA.h:24-34
        if (nf >= EPA_MAXF) { overflow = true; return; }
        d3 n = dcross(dsub(pos(i0), pos(i1)), dsub(pos(i2), pos(i1)));
        double len = dlength(n);
        if (len) n = ddivs(n, len);
        FI(nf, 0) = i0; FI(nf, 1) = i1; FI(nf, 2) = i2;
        FN(nf, 0) = n.x; FN(nf, 1) = n.y; FN(nf, 2) = n.z;
        ++nf;
    }
    __device__ void copy_face(int dst, int src) {
        for (int k = 0; k < 3; ++k) { FI(dst, k) = FI(src, k); FN(dst, k) = FN(src, k); }
    }
    __device__ double face_distance(int f) { return ddot(pos(FI(f, 0)), normal(f)); }   // src/EPA.h:41-43
};

template <class S0, class S1>
__device__ f3 epa(const S0& s0, const S1& s1, GjkV* s, EpaWs& P, f3& cp0, f3& cp1) {   // src/EPA.h:171-186
    P.nv = 4; P.nf = 0; P.overflow = false;
    for (int i = 0; i < 4; ++i) P.putV(i, s[i]);
    {   // EpaPolytope(GjkSimplex&), src/EPA.h:50-66
        d3 n = dcross(dsub(s[0].pos, s[1].pos), dsub(s[2].pos, s[1].pos));
        if (ddot(dsub(s[3].pos, s[0].pos), n) < 0) {
            P.create_face(0, 1, 2); P.create_face(3, 1, 0); P.create_face(3, 2, 1); P.create_face(3, 0, 2);
        } else {
            P.create_face(0, 2, 1); P.create_face(3, 2, 0); P.create_face(3, 1, 2); P.create_face(3, 0, 1);
        }
    }
    float minDist = 0.f;
    d3 normal = mkd(0, 0, 0);
    int faceIndex = 0;
    for (int it = 0; it < 100 && !P.overflow; ++it) {
        // findClosestFace: a float running minimum compared against double distances (:68-79)
        minDist = __builtin_inff();
        for (int f = 0; f < P.nf; ++f) {
            double d = P.face_distance(f);
            if (d < (double)minDist) { minDist = (float)d; normal = P.normal(f); faceIndex = f; }
        }
        GjkV v = mdiff(s0, s1, narrow(normal));
        if (ddot(v.pos, normal) - (double)minDist < (double)0.00001f) break;
        // insertVertex (:81-120)
        if (P.nv >= EPA_MAXV) { P.overflow = true; break; }
        int ne = 0;
        for (int f = P.nf - 1; f >= 0; --f) {
            if (ddot(P.normal(f), dsub(v.pos, P.pos(P.FI(f, 0)))) > 0) {
                int e[3][2] = {{P.FI(f, 0), P.FI(f, 1)}, {P.FI(f, 1), P.FI(f, 2)}, {P.FI(f, 2), P.FI(f, 0)}};
                bool found[3] = {false, false, false};
                for (int j = 0; j < 3; ++j)
                    for (int k = ne - 1; k >= 0; --k)
                        if (P.E(k, 0) == e[j][1] && P.E(k, 1) == e[j][0]) {
                            found[j] = true;
                            P.E(k, 0) = P.E(ne - 1, 0);
                            P.E(k, 1) = P.E(ne - 1, 1);
                            --ne;
                            break;
                        }
                for (int j = 0; j < 3; ++j)
                    if (!found[j]) {
                        if (ne >= EPA_MAXE) { P.overflow = true; break; }
                        P.E(ne, 0) = e[j][0];
                        P.E(ne, 1) = e[j][1];
                        ++ne;
                    }
                P.copy_face(f, P.nf - 1);
                --P.nf;
            }
        }
        int vi = P.nv++;
        P.putV(vi, v);
        for (int k = 0; k < ne; ++k) P.create_face(vi, P.E(k, 0), P.E(k, 1));
    }
    // getClosestPoints (:122-168), including proj = normal + distance (:133)
    int fa = P.FI(faceIndex, 0), fb = P.FI(faceIndex, 1), fc = P.FI(faceIndex, 2);
    GjkV a = P.getV(fa), b = P.getV(fb), c = P.getV(fc);
    d3 proj = dadds(P.normal(faceIndex), P.face_distance(faceIndex));
    f3 v0 = narrow(dsub(b.pos, a.pos)), v1 = narrow(dsub(c.pos, a.pos)), v2 = narrow(dsub(proj, a.pos));
    double d00 = dot(v0, v0), d01 = dot(v0, v1), d11 = dot(v1, v1), d20 = dot(v2, v0), d21 = dot(v2, v1);
    double denom = d00 * d11 - d01 * d01;
    double u, vv, w;
    if (denom) {
        vv = (d20 * d11 - d21 * d01) / denom;
        w = (d00 * d21 - d01 * d20) / denom;
        u = 1.0 - vv - w;
    } else {
        w = 0;
        if (d00) { vv = d20 / d00; u = 1.0 - vv; }
        else { vv = 0; u = 1.0; }
    }
    cp0 = narrow(dadd(dadd(dmul(u, a.sp0), dmul(vv, b.sp0)), dmul(w, c.sp0)));
    cp1 = narrow(dadd(dadd(dmul(u, a.sp1), dmul(vv, b.sp1)), dmul(w, c.sp1)));
    return narrow(normal);
}

// ------------------------------------------------------------------ contact generation
template <int CAP>
__device__ void clip_polygon_n(f2* poly, int& n, const f2* clip, int nclip) {   // src/Clipping.cpp:21-53
    f2 out[CAP];
    for (int e = 0; e < nclip; ++e) {
        f2 a = clip[e], b = clip[(e + 1) % nclip];
        int m = 0;
        for (int i = 0; i < n; ++i) {
            int j = (i + 1) == n ? 0 : i + 1;
            bool ii = inside(poly[i], a, b), ji = inside(poly[j], a, b);
            if (ii && ji) { if (m < CAP) out[m++] = poly[j]; }
            else if (ii) { if (m < CAP) out[m++] = intersect2(poly[i], poly[j], a, b); }
            else if (ji) {
                if (m < CAP) out[m++] = intersect2(poly[i], poly[j], a, b);
                if (m < CAP) out[m++] = poly[j];
            }
        }
        n = m;
        for (int i = 0; i < m; ++i) poly[i] = out[i];
    }
}
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

// src/ContactsUtil.cpp:109-204
__device__ void polygon_polygon_face_contacts(f3 refPos, const m3& refToWorld, f3 refOrig, f3 refNormal,
                                              f3 incOrig, f3 incNormal, const f2* poly, int n, int cx, int cy,
                                              CPt* cps, int& numPoints) {
    f3 pen[CVX_MAXPOLY];
    int np = 0;
    float distRef = dot(refOrig, refNormal);
    f3 dir = mk3(0.f, 1.f, 0.f);
    for (int i = 0; i < n; ++i) {
        f3 p3 = mk3(poly[i].y, 0.f, poly[i].x);
        float distance = dot(sub(incOrig, p3), incNormal) / dot(dir, incNormal);
        if (distance < distRef + 1e-4f) {
            p3.y = distance;
            pen[np++] = p3;
        }
    }
    auto emit = [&](int slot, int idx) {
        f3 on = pen[idx];
        on.y = distRef;
        cps[slot].p0 = add(refPos, mulmv(refToWorld, on));
        cps[slot].p1 = add(refPos, mulmv(refToWorld, pen[idx]));
    };
    if (np > 4) {
        emit(0, 0);
        float maxD = 0.f;
        int maxDi = 0;
        for (int i = 0; i < np; ++i) {
            f3 d = sub(pen[i], pen[0]);
            float dd = dot(d, d);
            if (dd > maxD) { maxD = dd; maxDi = i; }
        }
        emit(1, maxDi);
        float maxA = 0.f, minA = 0.f;
        int maxAi = 0, minAi = 0;
        for (int i = 0; i < np; ++i) {
            f3 ca = sub(pen[0], pen[i]), cb = sub(pen[maxDi], pen[i]);
            float area = det2(mk2(at(ca, cx), at(ca, cy)), mk2(at(cb, cx), at(cb, cy)));
            if (area > maxA) { maxA = area; maxAi = i; }
        }
        emit(2, maxAi);
        for (int i = 0; i < np; ++i) {
            f3 da = sub(pen[0], pen[i]), db = sub(pen[maxDi], pen[i]);
            float area = det2(mk2(at(da, cx), at(da, cy)), mk2(at(db, cx), at(db, cy)));
            if (area < minA) { minA = area; minAi = i; }
        }
        emit(3, minAi);
        numPoints = 4;
    } else {
        for (int i = 0; i < np; ++i) emit(i, i);
        numPoints = np;
    }
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
