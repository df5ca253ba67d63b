// Narrowphase: one candidate pair per lane, writing a manifold slot (SoA) per pair.
//
// The pair routines follow the reference's src/Collision.cpp (dispatcher :895-1016,
// sphere/capsule/box closed forms :109-133,428-486, box-box SAT + face clipping
// :54-107,135-350, capsule-box :501-692), src/GeomUtil.cpp (segment distances and the
// segment-AABB regions :7-59,129-467), src/Clipping.cpp (:10-71) and
// src/ContactsUtil.cpp (:9-107), operation for operation, so the manifold is bit-identical
// to the reference's for the same poses. Face contacts of boxes, hulls and triangles are
// clipped by several lanes a pair, the polygons in LDS (k_box_faces, np_wave.h).
#include "pgx_internal.h"
#include "radix_block.h"
#include "shape_bounds.h"
#include <iterator>
#include <type_traits>

namespace pgx {

struct CPt { f3 p0, p1; };
struct Mf {
    int numPoints;
    CPt pts[4];
    f3 normal;
};

// ------------------------------------------------------------------ GeomUtil
__device__ f3 closest_point_on_segment(f3 point, f3 o, f3 d, float mn, float mx) {
    f3 r = sub(o, point);
    float t = -dot(r, d);
    t = gclamp(t, mn, mx);
    return add(o, mul(t, d));
}

__device__ void closest_points_segments(f3 o0, f3 d0, float mn0, float mx0, f3 o1, f3 d1, float mn1, float mx1,
                                        f3& p0, f3& p1) {
    float v1v2 = dot(d0, d1);
    f3 r = sub(o1, o0);
    float rv1 = dot(r, d0);
    float rv2 = dot(r, d1);
    float t1 = gabs(v1v2) > 1.f - 0.0001f ? 0.f : (rv1 * v1v2 - rv2) / (1.f - v1v2 * v1v2);
    float t0 = rv1 + t1 * v1v2;
    if (t0 < mn0 || t0 > mx0) {
        t0 = t0 < mn0 ? mn0 : mx0;
        p0 = add(o0, mul(t0, d0));
        t1 = -dot(sub(o1, p0), d1);
    } else {
        p0 = add(o0, mul(t0, d0));
    }
    if (t1 < mn1 || t1 > mx1) {
        t1 = t1 < mn1 ? mn1 : mx1;
        p1 = add(o1, mul(t1, d1));
        t0 = -dot(sub(o0, p1), d0);
        t0 = gclamp(t0, mn0, mx0);
        p0 = add(o0, mul(t0, d0));
    } else {
        p1 = add(o1, mul(t1, d1));
    }
}

__device__ float case_two_zeros(f3 p, int axis, f3 he, float& t, f3& q) {
    float sq = 0.f;
    t = at(he, axis) - at(p, axis);
    set(q, axis, at(p, axis) + t);
    for (int k = 1; k <= 2; ++k) {
        int a = (axis + k) % 3;
        float pa = at(p, a), ha = at(he, a);
        if (pa > ha) { float d = pa - ha; sq += d * d; set(q, a, ha); }
        else if (pa < -ha) { float d = pa + ha; sq += d * d; set(q, a, -ha); }
        else set(q, a, pa);
    }
    return sq;
}

__device__ float case_one_zero(f3 p, int z0, f3 dir, f3 he, float& t, f3& q) {
    float sq = 0.f;
    set(q, z0, at(p, z0));
    f3 pme = sub(p, he);
    int x = (z0 + 1) % 3, y = (z0 + 2) % 3;
    float prod0 = at(dir, y) * at(pme, x);
    float prod1 = at(dir, x) * at(pme, y);
    if (prod0 >= prod1) {
        set(q, x, at(he, x));
        float eY = at(p, y) + at(he, y);
        float delta = prod0 - at(dir, x) * eY;
        if (delta >= 0) {
            sq += delta * delta;
            set(q, y, -at(he, y));
            t = -(at(pme, x) * at(dir, x) + eY * at(dir, y));
        } else {
            set(q, y, at(p, y) - prod0 / at(dir, x));
            t = -at(pme, x) / at(dir, x);
        }
    } else {
        set(q, y, at(he, y));
        float eX = at(p, x) + at(he, x);
        float delta = prod1 - at(dir, y) * eX;
        if (delta >= 0) {
            sq += delta * delta;
            set(q, x, -at(he, x));
            t = -(eX * at(dir, x) + at(pme, y) * at(dir, y));
        } else {
            set(q, x, at(p, x) - prod1 / at(dir, y));
            t = -at(pme, y) / at(dir, y);
        }
    }
    float pz = at(p, z0), hz = at(he, z0);
    if (pz < -hz) { float d = pz + hz; sq += d * d; set(q, z0, -hz); }
    else if (pz > hz) { float d = pz - hz; sq += d * d; set(q, z0, hz); }
    return sq;
}

// Region 4/5 and 1/2/3 helpers of the face case. "Region 5" keeps the reference's
// pme[y] + pme[y] term (src/GeomUtil.cpp:273,326).
__device__ __forceinline__ float region45(f3 p, f3 dir, f3 he, int x, int y, int z, f3 pme, f3 ppe, float npY,
                                          float& t, f3& q) {
    float dx = at(dir, x), dy = at(dir, y), dz = at(dir, z);
    float pmx = at(pme, x), pmy = at(pme, y), ppz = at(ppe, z);
    if (npY <= at(he, y)) {
        float tmp = at(p, y) - npY;
        float delta = dx * pmx + dy * tmp + dz * ppz;
        t = -delta;
        set(q, x, at(he, x)); set(q, y, npY); set(q, z, -at(he, z));
        return pmx * pmx + tmp * tmp + ppz * ppz - delta * delta;
    }
    float delta = dx * pmx + dy * pmy + dz * ppz;
    t = -delta;
    set(q, x, at(he, x)); set(q, y, at(he, y)); set(q, z, -at(he, z));
    return pmx * pmx + pmy + pmy + ppz * ppz - delta * delta;
}
__device__ __forceinline__ float region12(f3 p, f3 dir, f3 he, int x, int y, int z, f3 pme, f3 ppe, float npZ,
                                          float& t, f3& q) {
    float dx = at(dir, x), dy = at(dir, y), dz = at(dir, z);
    float pmx = at(pme, x), ppy = at(ppe, y), pmz = at(pme, z);
    if (npZ <= at(he, z)) {
        float tmp = at(p, z) - npZ;
        float delta = dx * pmx + dy * ppy + dz * tmp;
        t = -delta;
        set(q, x, at(he, x)); set(q, y, -at(he, y)); set(q, z, npZ);
        return pmx * pmx + ppy * ppy + tmp * tmp - delta * delta;
    }
    float delta = dx * pmx + dy * ppy + dz * pmz;
    t = -delta;
    set(q, x, at(he, x)); set(q, y, -at(he, y)); set(q, z, at(he, z));
    return pmx * pmx + ppy * ppy + pmz * pmz - delta * delta;
}

__device__ float line_aabb_face(f3 p, f3 dir, f3 he, int x, f3 pme, float& t, f3& q) {
    q = p;
    t = 0.f;
    int y = (x + 1) % 3, z = (y + 1) % 3;
    f3 ppe = add(p, he);
    float dx = at(dir, x), dy = at(dir, y), dz = at(dir, z);
    float pmx = at(pme, x);
    if (dx * at(ppe, y) >= dy * pmx) {
        if (dx * at(ppe, z) >= dz * pmx) {
            set(q, x, at(he, x));
            set(q, y, at(q, y) - pmx * dy / dx);
            set(q, z, at(q, z) - pmx * dz / dx);
            t = -pmx / dx;
            return 0.f;
        }
        float sqrLen = dx * dx + dz * dz;
        float npY = at(p, y) - dy * (dx * pmx + dz * at(ppe, z)) / sqrLen;
        return region45(p, dir, he, x, y, z, pme, ppe, npY, t, q);
    }
    if (dx * at(ppe, z) >= dz * pmx) {
        float sqrLen = dx * dx + dy * dy;
        float npZ = at(p, z) - dz * (dx * pmx + dy * at(ppe, y)) / sqrLen;
        return region12(p, dir, he, x, y, z, pme, ppe, npZ, t, q);
    }
    float npY = at(p, y) - dy * (dx * pmx + dz * at(ppe, z)) / (dx * dx + dz * dz);
    if (npY >= -at(he, y)) return region45(p, dir, he, x, y, z, pme, ppe, npY, t, q);
    float npZ = at(p, z) - dz * (dx * pmx + dy * at(ppe, y)) / (dx * dx + dy * dy);
    if (npZ >= -at(he, z)) return region12(p, dir, he, x, y, z, pme, ppe, npZ, t, q);
    float delta = dx * pmx + dy * at(ppe, y) + dz * at(ppe, z);
    t = -delta;
    set(q, x, at(he, x)); set(q, y, -at(he, y)); set(q, z, -at(he, z));
    return pmx * pmx + at(ppe, y) * at(ppe, y) + at(ppe, z) * at(ppe, z) - delta * delta;
}

__device__ float case_no_zeroes(f3 p, f3 dir, f3 he, float& t, f3& q) {
    f3 pme = sub(p, he);
    float dxEy = dir.x * pme.y, dyEx = dir.y * pme.x;
    if (dyEx >= dxEy) {
        float dzEx = dir.z * pme.x, dxEz = dir.x * pme.z;
        return line_aabb_face(p, dir, he, dzEx >= dxEz ? 0 : 2, pme, t, q);
    }
    float dzEy = dir.z * pme.y, dyEz = dir.y * pme.z;
    return line_aabb_face(p, dir, he, dzEy >= dyEz ? 1 : 2, pme, t, q);
}

__device__ float point_aabb(f3 p, f3 he, f3& q) {
    q = vclamp(p, neg(he), he);
    f3 d = sub(p, q);
    return dot(d, d);
}

__device__ float segment_aabb(f3 p, f3 dir, float mn, float mx, f3 he, float& t, f3& q) {
    bool refl[3];
    f3 pp = p, dd = dir;
    for (int i = 0; i < 3; ++i) {
        if (at(dd, i) < 0.f) { set(pp, i, -at(pp, i)); set(dd, i, -at(dd, i)); refl[i] = true; }
        else refl[i] = false;
    }
    float sq;
    bool px = dd.x > 0, py = dd.y > 0, pz = dd.z > 0;
    if (px && py && pz) sq = case_no_zeroes(pp, dd, he, t, q);
    else if (px && py) sq = case_one_zero(pp, 2, dd, he, t, q);
    else if (px && pz) sq = case_one_zero(pp, 1, dd, he, t, q);
    else if (py && pz) sq = case_one_zero(pp, 0, dd, he, t, q);
    else if (px) sq = case_two_zeros(pp, 0, he, t, q);
    else if (py) sq = case_two_zeros(pp, 1, he, t, q);
    else if (pz) sq = case_two_zeros(pp, 2, he, t, q);
    else { sq = point_aabb(pp, he, q); t = 0.f; }
    for (int i = 0; i < 3; ++i)
        if (refl[i]) set(q, i, -at(q, i));
    if (t < mn) { t = mn; sq = point_aabb(add(p, mul(dir, t)), he, q); }
    else if (t > mx) { t = mx; sq = point_aabb(add(p, mul(dir, t)), he, q); }
    return sq;
}

// ------------------------------------------------------------------ clipping
constexpr int MAXPOLY = 12;

__device__ __forceinline__ bool inside(f2 pt, f2 a, f2 b) {
    return (b.y - a.y) * (pt.x - a.x) - (b.x - a.x) * (pt.y - a.y) > 0;
}
__device__ __forceinline__ f2 intersect2(f2 a1, f2 b1, f2 a2, f2 b2) {
    f2 r1 = sub2(b1, a1), r2 = sub2(b2, a2);
    float t = det2(sub2(a1, a2), r2) / det2(mk2(-r1.x, -r1.y), r2);
    return add2(a1, mk2(t * r1.x, t * r1.y));
}
// Sutherland-Hodgman against an axis-aligned rectangle given as 4 corners (Clipping.cpp:21-53)
__device__ void clip_polygon(f2* poly, int& n, const f2* clip) {
    f2 out[MAXPOLY];
    for (int e = 0; e < 4; ++e) {
        f2 a = clip[e], b = clip[(e + 1) & 3];
        int m = 0;
        for (int i = 0; i < n; ++i) {
            int j = (i + 1) == n ? 0 : i + 1;
            bool ii = inside(poly[i], a, b), ji = inside(poly[j], a, b);
            if (ii && ji) { if (m < MAXPOLY) out[m++] = poly[j]; }
            else if (ii) { if (m < MAXPOLY) out[m++] = intersect2(poly[i], poly[j], a, b); }
            else if (ji) {
                if (m < MAXPOLY) out[m++] = intersect2(poly[i], poly[j], a, b);
                if (m < MAXPOLY) out[m++] = poly[j];
            }
        }
        n = m;
        for (int i = 0; i < m; ++i) poly[i] = out[i];
    }
}
__device__ bool clip_line(f2& p0, f2& p1, const f2* clip) {
    for (int i = 0; i < 4; ++i) {
        int j = (i + 1) & 3;
        bool in0 = inside(p0, clip[i], clip[j]), in1 = inside(p1, clip[i], clip[j]);
        if (in0 && in1) continue;
        if (in0) p1 = intersect2(p0, p1, clip[i], clip[j]);
        else if (in1) p0 = intersect2(p0, p1, clip[i], clip[j]);
        else return false;
    }
    return true;
}

// src/ContactsUtil.cpp:9-107
template <int CAP>
__device__ void polygon_box_face_contacts_n(f3 boxCenter, const m3& basis, int axis, int axisSign, f3 he,
                                            f3 incOrig, f3 incNormal, const f2* poly, int n, int cx, int cy,
                                            CPt* cps, int& numPoints) {
    f3 pen[CAP];
    int np = 0;
    f3 dir = s3(0.f);
    set(dir, axis, (float)axisSign);
    float denom = dot(dir, incNormal);
    float lim = at(he, axis) + 1e-4f;
    for (int i = 0; i < n; ++i) {
        f3 p3 = s3(0.f);
        set(p3, cx, poly[i].x);
        set(p3, cy, poly[i].y);
        float distance = dot(sub(incOrig, p3), incNormal) / denom;
        if (distance < lim) {
            set(p3, axis, axisSign * distance);
            pen[np++] = p3;
        }
    }
    auto emit = [&](int slot, int idx) {
        f3 on = pen[idx];
        set(on, axis, axisSign * at(he, axis));
        cps[slot].p0 = add(boxCenter, mulmv(basis, on));
        cps[slot].p1 = add(boxCenter, mulmv(basis, pen[idx]));
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
            f3 ca = sub(pen[0], pen[i]);
            f3 cb = sub(pen[maxDi], pen[i]);
            float area = det2(mk2(at(ca, cx), at(ca, cy)), mk2(at(cb, cx), at(cb, cy)));
            if (area > maxA) { maxA = area; maxAi = i; }
        }
        emit(2, maxAi);
        for (int i = 0; i < np; ++i) {
            f3 da = sub(pen[0], pen[i]);
            f3 db = sub(pen[maxDi], pen[i]);
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

__device__ __forceinline__ void polygon_box_face_contacts(f3 boxCenter, const m3& basis, int axis, int axisSign,
                                                          f3 he, f3 incOrig, f3 incNormal, const f2* poly, int n,
                                                          int cx, int cy, CPt* cps, int& numPoints) {
    polygon_box_face_contacts_n<MAXPOLY>(boxCenter, basis, axis, axisSign, he, incOrig, incNormal, poly, n, cx, cy,
                                         cps, numPoints);
}

// ------------------------------------------------------------------ pair routines
// src/Collision.cpp:54-107
__device__ void box_face_contacts(const m3& uRef, f3 posRef, f3 heRef, const m3& uInc, f3 posInc, f3 heInc,
                                  int refAxis, CPt* cps, int& numPoints) {
    f3 axis = col(uRef, refAxis);
    float refSign = dot(axis, sub(posInc, posRef)) < 0 ? -1.f : 1.f;
    float maxDot = 0.f, incSign = 1.f;
    int incAxis = 0;
    for (int i = 0; i < 3; ++i) {
        float d = dot(mul(-refSign, axis), col(uInc, i));
        float ad = gabs(d);
        if (ad > maxDot) { maxDot = ad; incAxis = i; incSign = d < 0 ? -1.f : 1.f; }
    }
    int ia1 = (incAxis + 1) % 3, ia2 = (incAxis + 2) % 3;
    m3 inv = inverse(uRef);
    f3 ui = col(uInc, incAxis), u1 = col(uInc, ia1), u2 = col(uInc, ia2);
    float h1 = at(heInc, ia1), h2 = at(heInc, ia2);
    f3 incOrig = mulmv(inv, sub(add(posInc, mul(mul(ui, at(heInc, incAxis)), incSign)), posRef));
    f3 a = mul(u1, h1), b = mul(u2, h2);
    f3 na = mul(neg(u1), h1);
    f3 poly3[4] = {add(incOrig, mulmv(inv, add(a, b))), add(incOrig, mulmv(inv, add(na, b))),
                   add(incOrig, mulmv(inv, sub(na, b))), add(incOrig, mulmv(inv, sub(a, b)))};
    int cx = (refAxis + 1) % 3, cy = (refAxis + 2) % 3;
    f2 poly[MAXPOLY];
    for (int i = 0; i < 4; ++i) poly[i] = mk2(at(poly3[i], cx), at(poly3[i], cy));
    float hx = at(heRef, cx), hy = at(heRef, cy);
    f2 clip[4] = {mk2(hx, hy), mk2(hx, -hy), mk2(-hx, -hy), mk2(-hx, hy)};
    int n = 4;
    clip_polygon(poly, n, clip);
    f3 incNormal = mulmv(inv, ui);
    polygon_box_face_contacts(posRef, uRef, refAxis, (int)refSign, heRef, incOrig, incNormal, poly, n, cx, cy, cps,
                              numPoints);
}

__device__ bool sphere_sphere(f3 p0, float r0, f3 p1, float r1, Mf& m) {
    f3 d = sub(p1, p0);
    float rs = r0 + r1;
    if (dot(d, d) > rs * rs) return false;
    float dl = length(d);
    m.normal = dl != 0.f ? divs(d, dl) : mk3(0.f, 1.f, 0.f);
    m.numPoints = 1;
    m.pts[0].p0 = add(p0, mul(m.normal, r0));
    m.pts[0].p1 = sub(p1, mul(m.normal, r1));
    return true;
}

__device__ bool capsule_capsule(f3 p0, qf q0, float hh0, float r0, f3 p1, qf q1, float hh1, float r1, Mf& m) {
    f3 up = mk3(0.f, 1.f, 0.f);
    f3 v0 = qrot(q0, up), v1 = qrot(q1, up);
    f3 a, b;
    closest_points_segments(p0, v0, -hh0, hh0, p1, v1, -hh1, hh1, a, b);
    f3 d = sub(b, a);
    float rs = r0 + r1;
    if (dot(d, d) > rs * rs) return false;
    float dl = length(d);
    m.normal = dl != 0.f ? divs(d, dl) : up;
    m.numPoints = 1;
    m.pts[0].p0 = add(a, mul(m.normal, r0));
    m.pts[0].p1 = sub(b, mul(m.normal, r1));
    return true;
}

__device__ bool sphere_capsule(f3 p0, float r0, f3 p1, qf q1, float hh1, float r1, Mf& m) {
    f3 up = mk3(0.f, 1.f, 0.f);
    f3 dir = qrot(q1, up);
    f3 q = closest_point_on_segment(p0, p1, dir, -hh1, hh1);
    f3 v = sub(q, p0);
    float rs = r0 + r1;
    if (dot(v, v) > rs * rs) return false;
    float vl = length(v);
    m.normal = vl != 0.f ? divs(v, vl) : up;
    m.numPoints = 1;
    m.pts[0].p0 = add(p0, mul(m.normal, r0));
    m.pts[0].p1 = sub(q, mul(m.normal, r1));
    return true;
}

__device__ bool sphere_box(f3 p0, float r0, f3 p1, qf q1, f3 he, Mf& m) {
    m3 u = mat3_cast(q1);
    f3 d = sub(p0, p1);
    d = mk3(dot(d, u.c0), dot(d, u.c1), dot(d, u.c2));
    f3 q = add(p1, mulmv(u, vclamp(d, neg(he), he)));
    f3 v = sub(q, p0);
    if (dot(v, v) > r0 * r0) return false;
    float vl = length(v);
    m.numPoints = 1;
    if (vl != 0.f) {
        m.normal = divs(v, vl);
        m.pts[0].p0 = add(p0, mul(m.normal, r0));
        m.pts[0].p1 = q;
    } else {
        float mn = 3.402823466e+38f;
        int axis = 0;
        for (int i = 0; i < 3; ++i) {
            float depth = at(he, i) - gabs(at(d, i));
            if (depth < mn) { mn = depth; axis = i; }
        }
        float sign = at(d, axis) != 0.f ? gsign(at(d, axis)) : 1.f;
        f3 bp = d;
        set(bp, axis, sign * at(he, axis));
        m.normal = mul(-sign, col(u, axis));
        m.pts[0].p0 = p0;
        m.pts[0].p1 = add(p1, mulmv(u, bp));
    }
    return true;
}

__device__ void capsule_box_contacts(f3 p0L, f3 p1L, float radius, f3 normal, f3 boxCenter, f3 he,
                                     const m3& basis, Mf& m) {
    int axis = 0;
    float axisSign = 0.f, maxDot = 0.f;
    for (int i = 0; i < 3; ++i) {
        float d = dot(normal, col(basis, i));
        float ad = gabs(d);
        if (ad > maxDot) { maxDot = ad; axis = i; axisSign = d < 0 ? 1.f : -1.f; }
    }
    int cx = (axis + 1) % 3, cy = (axis + 2) % 3;
    f2 l0 = mk2(at(p0L, cx), at(p0L, cy)), l1 = mk2(at(p1L, cx), at(p1L, cy));
    float hx = at(he, cx), hy = at(he, cy);
    f2 clip[4] = {mk2(hx, hy), mk2(hx, -hy), mk2(-hx, -hy), mk2(-hx, hy)};
    if (!clip_line(l0, l1, clip)) { m.numPoints = 0; return; }
    float onAxis = axisSign * at(he, axis);
    f3 a = s3(0.f), b = s3(0.f);
    float distX = at(p0L, cx) - at(p1L, cx), distY = at(p0L, cy) - at(p1L, cy);
    float adx = gabs(distX), ady = gabs(distY);
    if (adx > ady) {
        set(a, axis, gmix(at(p0L, axis), at(p1L, axis), (at(p0L, cx) - l0.x) / distX));
        set(b, axis, gmix(at(p1L, axis), at(p0L, axis), (at(p1L, cx) - l1.x) / -distX));
    } else if (ady > adx) {
        set(a, axis, gmix(at(p0L, axis), at(p1L, axis), (at(p0L, cy) - l0.y) / distY));
        set(b, axis, gmix(at(p1L, axis), at(p0L, axis), (at(p1L, cy) - l1.y) / -distY));
    } else {
        set(a, axis, at(p0L, axis));
        set(b, axis, at(p1L, axis));
    }
    set(a, axis, at(a, axis) - axisSign * radius);
    set(b, axis, at(b, axis) - axisSign * radius);
    int np = 0;
    float ha = at(he, axis);
    if (gabs(at(a, axis)) < ha) {
        set(a, cx, l0.x); set(a, cy, l0.y);
        f3 ob = a; set(ob, axis, onAxis);
        m.pts[np].p0 = add(boxCenter, mulmv(basis, a));
        m.pts[np].p1 = add(boxCenter, mulmv(basis, ob));
        ++np;
    }
    if (gabs(at(b, axis)) < ha) {
        set(b, cx, l1.x); set(b, cy, l1.y);
        f3 ob = b; set(ob, axis, onAxis);
        m.pts[np].p0 = add(boxCenter, mulmv(basis, b));
        m.pts[np].p1 = add(boxCenter, mulmv(basis, ob));
        ++np;
    }
    m.numPoints = np;
}

__device__ bool capsule_box(f3 p0, qf q0, float hh0, float r0, f3 p1, qf q1, f3 he, Mf& m) {
    m3 u = mat3_cast(q1);
    f3 p = sub(p0, p1);
    p = mk3(dot(p, u.c0), dot(p, u.c1), dot(p, u.c2));
    f3 dir = qrot(q0, mk3(0.f, 1.f, 0.f));
    f3 dl = mk3(dot(dir, u.c0), dot(dir, u.c1), dot(dir, u.c2));
    float t = 0.f;
    f3 q = s3(0.f);
    float sq = segment_aabb(p, dl, -hh0, hh0, he, t, q);
    if (sq >= r0 * r0) return false;
    f3 onSeg = add(p0, mul(dir, t));
    f3 onBox = add(p1, mulmv(u, q));
    f3 nrm = sub(onBox, onSeg);
    float nl = length(nrm);
    if (nl != 0.f) {
        m.normal = divs(nrm, nl);
    } else {
        f3 r, ar;
        r = mk3(dot(dir, u.c0), dot(dir, u.c1), dot(dir, u.c2));
        ar = vabs(r);
        float mx = -3.402823466e+38f;
        bool edge = false;
        int axis = 0;
        for (int i = 0; i < 3; ++i) {
            float d = gabs(at(p, i)) - (hh0 * at(ar, i) + r0) - at(he, i);
            if (d > mx) { mx = d; axis = i; }
        }
        float edgeOffset = 0.1f;
        {
            float rb = he.y * ar.z + he.z * ar.y;
            float d = gabs(p.z * r.y - p.y * r.z) - r0 - rb;
            if (ar.x < 0.999f && d > mx + edgeOffset) { mx = d; edge = true; axis = 0; edgeOffset = 0.f; }
        }
        {
            float rb = he.x * ar.z + he.z * ar.x;
            float d = gabs(p.x * r.z - p.z * r.x) - r0 - rb;
            if (ar.y < 0.999f && d > mx + edgeOffset) { mx = d; edge = true; axis = 1; edgeOffset = 0.f; }
        }
        {
            float rb = he.x * ar.y + he.y * ar.x;
            float d = gabs(p.y * r.x - p.x * r.y) - r0 - rb;
            if (ar.z < 0.999f && d > mx + edgeOffset) { mx = d; edge = true; axis = 2; }
        }
        f3 sep = edge ? cross(dir, col(u, axis)) : col(u, axis);
        m.normal = normalize(dot(sep, sub(p1, p0)) > 0 ? sep : neg(sep));
    }
    capsule_box_contacts(sub(p, mul(dl, hh0)), add(p, mul(dl, hh0)), r0, m.normal, p1, he, u, m);
    if (!m.numPoints) {
        m.numPoints = 1;
        m.pts[0].p0 = add(onSeg, mul(m.normal, r0));
        m.pts[0].p1 = onBox;
    }
    return true;
}

// src/Collision.cpp:135-350. LATER: a face contact's polygon is left to k_box_faces: face is
// set to 3 * the face's box + its axis, m untouched.
template <bool LATER>
__device__ bool box_box(f3 p0, qf q0, f3 he0, f3 p1, qf q1, f3 he1, Mf& m, int& face) {
    float edgeOffset = 0.1f;
    const float edgeLimit = 0.999f;
    bool isEdge = false;
    int faceBox = 0, faceAxis = 0, e0 = 0, e1 = 0;
    float mx = -3.402823466e+38f;
    m3 u0 = mat3_cast(q0), u1 = mat3_cast(q1);
    f3 t = sub(p1, p0);
    t = mk3(dot(t, u0.c0), dot(t, u0.c1), dot(t, u0.c2));
    float r[3][3], ar[3][3];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) {
            r[i][j] = dot(col(u0, i), col(u1, j));
            ar[i][j] = gabs(r[i][j]);
        }
    float h0[3] = {he0.x, he0.y, he0.z}, h1[3] = {he1.x, he1.y, he1.z}, tt[3] = {t.x, t.y, t.z};
    for (int i = 0; i < 3; ++i) {
        float rb = h1[0] * ar[i][0] + h1[1] * ar[i][1] + h1[2] * ar[i][2];
        float d = gabs(tt[i]) - h0[i] - rb;
        if (d > 0) return false;
        if (d > mx) { mx = d; faceBox = 0; faceAxis = i; }
    }
    for (int i = 0; i < 3; ++i) {
        float ra = h0[0] * ar[0][i] + h0[1] * ar[1][i] + h0[2] * ar[2][i];
        float l = gabs(tt[0] * r[0][i] + tt[1] * r[1][i] + tt[2] * r[2][i]);
        float d = l - ra - h1[i];
        if (d > 0) return false;
        if (d > mx) { mx = d; faceBox = 1; faceAxis = i; }
    }
    // A_i x B_j in the reference's order; each radius sum lists the lower axis first
    for (int i = 0; i < 3; ++i) {
        int i1 = (i + 1) % 3, i2 = (i + 2) % 3;
        int lo = i1 < i2 ? i1 : i2, hi = i1 < i2 ? i2 : i1;
        for (int j = 0; j < 3; ++j) {
            int j1 = (j + 1) % 3, j2 = (j + 2) % 3;
            int jlo = j1 < j2 ? j1 : j2, jhi = j1 < j2 ? j2 : j1;
            float ra = h0[lo] * ar[lo == i1 ? i2 : i1][j] + h0[hi] * ar[hi == i1 ? i2 : i1][j];
            float rb = h1[jlo] * ar[i][jlo == j1 ? j2 : j1] + h1[jhi] * ar[i][jhi == j1 ? j2 : j1];
            float l = gabs(tt[i2] * r[i1][j] - tt[i1] * r[i2][j]);
            float d = l - ra - rb;
            if (d > 0) return false;
            if (ar[i][j] < edgeLimit && d > mx + edgeOffset) {
                mx = d; isEdge = true; e0 = i; e1 = j; edgeOffset = 0.f;
            }
        }
    }
    if (LATER && !isEdge) {
        face = 3 * faceBox + faceAxis;
    } else if (!isEdge) {
        CPt cps[4];
        int np = 0;
        f3 axis;
        if (faceBox) {
            axis = col(u1, faceAxis);
            box_face_contacts(u1, p1, he1, u0, p0, he0, faceAxis, cps, np);
            for (int i = 0; i < np; ++i) { m.pts[i].p0 = cps[i].p1; m.pts[i].p1 = cps[i].p0; }
        } else {
            axis = col(u0, faceAxis);
            box_face_contacts(u0, p0, he0, u1, p1, he1, faceAxis, cps, np);
            for (int i = 0; i < np; ++i) m.pts[i] = cps[i];
        }
        m.numPoints = np;
        m.normal = dot(axis, sub(p1, p0)) < 0 ? neg(axis) : axis;
    } else {
        f3 a0 = col(u0, e0), a1 = col(u1, e1);
        f3 axis = cross(a0, a1);
        m.normal = normalize(dot(axis, sub(p1, p0)) < 0 ? neg(axis) : axis);
        float s0[3], s1[3];   // the edges' start corners
        for (int i = 0; i < 3; ++i) {
            s0[i] = i == e0 || dot(col(u0, i), m.normal) < 0 ? -1.f : 1.f;
            s1[i] = i == e1 || dot(col(u1, i), m.normal) > 0 ? -1.f : 1.f;
        }
        f3 c0 = add(add(add(p0, mul(s0[0] * h0[0], u0.c0)), mul(s0[1] * h0[1], u0.c1)), mul(s0[2] * h0[2], u0.c2));
        f3 c1 = add(add(add(p1, mul(s1[0] * h1[0], u1.c0)), mul(s1[1] * h1[1], u1.c1)), mul(s1[2] * h1[2], u1.c2));
        m.numPoints = 1;
        f3 a, b;
        closest_points_segments(c0, a0, 0.f, at(he0, e0) * 2, c1, a1, 0.f, at(he1, e1) * 2, a, b);
        m.pts[0].p0 = a;
        m.pts[0].p1 = b;
    }
    return true;
}

__device__ void flip(Mf& m) {
    m.normal = neg(m.normal);
    for (int i = 0; i < m.numPoints; ++i) { f3 a = m.pts[i].p0; m.pts[i].p0 = m.pts[i].p1; m.pts[i].p1 = a; }
}

// src/Collision.cpp:895-1016 for primitive shapes; face and LATER as box_box
template <bool LATER>
__device__ bool collide(int t0, float4 g0, f3 p0, qf q0, int t1, float4 g1, f3 p1, qf q1, Mf& m, int& face) {
    m.numPoints = 0;
    bool hit = false;
    f3 he0 = mk3(g0.x, g0.y, g0.z), he1 = mk3(g1.x, g1.y, g1.z);
    if (t0 == PGX_SPHERE) {
        if (t1 == PGX_SPHERE) return sphere_sphere(p0, g0.x, p1, g1.x, m);
        if (t1 == PGX_CAPSULE) return sphere_capsule(p0, g0.x, p1, q1, g1.x, g1.y, m);
        return sphere_box(p0, g0.x, p1, q1, he1, m);
    }
    if (t0 == PGX_CAPSULE) {
        if (t1 == PGX_SPHERE) { hit = sphere_capsule(p1, g1.x, p0, q0, g0.x, g0.y, m); flip(m); return hit; }
        if (t1 == PGX_CAPSULE) return capsule_capsule(p0, q0, g0.x, g0.y, p1, q1, g1.x, g1.y, m);
        return capsule_box(p0, q0, g0.x, g0.y, p1, q1, he1, m);
    }
    if (t1 == PGX_SPHERE) { hit = sphere_box(p1, g1.x, p0, q0, he0, m); flip(m); return hit; }
    if (t1 == PGX_CAPSULE) { hit = capsule_box(p1, q1, g1.x, g1.y, p0, q0, he0, m); flip(m); return hit; }
    return box_box<LATER>(p0, q0, he0, p1, q1, he1, m, face);
}

}  // namespace pgx

#include "np_convex.h"
#include "np_wave.h"
#include "np_trimesh.h"

namespace pgx {

// ------------------------------------------------------------------ kernel
__device__ __forceinline__ bool in_sorted(const uint64_t* __restrict__ a, int n, uint64_t key) {
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (a[mid] < key) lo = mid + 1; else hi = mid;
    }
    return lo < n && a[lo] == key;
}

// Index in a list of this lane's entry when the lanes with `want` append one entry each:
// one atomic on the list's counter per wave.
__device__ __forceinline__ int wave_append(int32_t* counter, bool want) {
    const uint64_t m = __ballot(want);
    const int lane = threadIdx.x & (WAVE - 1);
    const int leader = __ffsll((long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(counter, __popcll(m));
    base = __shfl(base, leader);
    return base + __popcll(m & ((1ull << lane) - 1ull));
}

// Shape-pair class of every pair: the unordered pair of primitive types (6 classes), or
// 15 for pairs that leave this kernel's collision routines (triangle or convex meshes,
// triggers, non-colliding pairs route or skip quickly). Sorted by class, a wave of the
// narrowphase runs one collision routine instead of every routine its pairs need.
__device__ __forceinline__ uint64_t pair_class(uint64_t key, int localBits, const int32_t* __restrict__ worldColStart,
                                               const int32_t* __restrict__ colOfLocal, const int32_t* __restrict__ ctype) {
    uint64_t lmask = (1ull << localBits) - 1;
    int base = worldColStart[(int)(key >> (2 * localBits))];
    int t0 = ctype[colOfLocal[base + (int)((key >> localBits) & lmask)]];
    int t1 = ctype[colOfLocal[base + (int)(key & lmask)]];
    bool prim = t0 <= PGX_BOX && t1 <= PGX_BOX;
    return prim ? (uint64_t)(min(t0, t1) * 3 + max(t0, t1)) : 15ull;
}
__global__ void k_pair_class(int nPairs, const uint64_t* __restrict__ pkeys, int localBits,
                             const int32_t* __restrict__ worldColStart, const int32_t* __restrict__ colOfLocal,
                             const int32_t* __restrict__ ctype, uint64_t* __restrict__ cls,
                             int32_t* __restrict__ order) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nPairs) return;
    cls[p] = pair_class(pkeys[p], localBits, worldColStart, colOfLocal, ctype);
    order[p] = p;
}

// The pairs' canonical order and their class order in one workgroup, one launch instead of
// two sorts and k_pair_class: 585 pairs 7.7 us instead of 11 us and two launches more;
// 4,315 pairs 24 us.
__global__ __launch_bounds__(RS_SINGLE_THREADS) void k_pair_order(int n, int items, int bits, uint64_t* __restrict__ pkeys,
                                                                  int localBits, const int32_t* __restrict__ worldColStart,
                                                                  const int32_t* __restrict__ colOfLocal,
                                                                  const int32_t* __restrict__ ctype,
                                                                  int32_t* __restrict__ order) {
    __shared__ RsBlock B;
    RsItems x;
#pragma unroll
    for (int k = 0; k < RS_SINGLE_ITEMS; ++k) {
        const int i = rs_index(items, k);
        if (k >= items || i >= n) continue;
        x.key[k] = pkeys[i];
        x.val[k] = 0;
    }
    rs_block_sort(B, x, n, bits, items);
    rs_block_exchange(B, x, n, items);
#pragma unroll
    for (int k = 0; k < RS_SINGLE_ITEMS; ++k) {
        const int i = rs_index(items, k);
        if (k >= items || i >= n) continue;
        pkeys[i] = x.key[k];
        x.key[k] = pair_class(x.key[k], localBits, worldColStart, colOfLocal, ctype);
    }
    rs_block_pass(B, x, n, 0, 4, items);   // stable: slot order within a class
#pragma unroll
    for (int k = 0; k < RS_SINGLE_ITEMS; ++k) {
        const int i = rs_index(items, k);
        if (k < items && i < n) order[x.pos[k]] = i;
    }
}

__global__ __launch_bounds__(256) void k_narrowphase(
    int nPairs, const int32_t* __restrict__ order, const uint64_t* __restrict__ pkeys, int localBits, const int32_t* __restrict__ worldColStart,
    const int32_t* __restrict__ colOfLocal, const int32_t* __restrict__ cbody, const int32_t* __restrict__ ctype,
    const int32_t* __restrict__ cflags, const float4* __restrict__ cparams, const float4* __restrict__ clpos,
    const float4* __restrict__ clquat, const uint32_t* __restrict__ centity, const float4* __restrict__ bpos,
    const float4* __restrict__ bquat, const uint64_t* __restrict__ nonColliding, int nNonColliding,
    int32_t* __restrict__ npNum, float4* __restrict__ npNormal, float4* __restrict__ npPts,
    int32_t* __restrict__ heavy, int32_t* __restrict__ nHeavy, int32_t* __restrict__ meshPairs,
    int32_t* __restrict__ nMesh, int32_t* __restrict__ meshCount, int32_t* __restrict__ trigList,
    int32_t* __restrict__ nTrig, const int32_t* __restrict__ filterClass, const uint8_t* __restrict__ filterTable,
    int filterK, int32_t* __restrict__ nFaces, int32_t* __restrict__ facesEnd) {
    // pairs per lane = pairs / (grid size): a lane takes every grid-size'th pair of the
    // class order; results are stored at the pair's own slot
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nPairs; i += gridDim.x * blockDim.x) {
        const int p = order[i];
        meshCount[p] = 0;
        uint64_t key = pkeys[p];
        uint64_t lmask = (1ull << localBits) - 1;
        int wd = (int)(key >> (2 * localBits));
        int base = worldColStart[wd];
        int c0 = colOfLocal[base + (int)((key >> localBits) & lmask)];
        int c1 = colOfLocal[base + (int)(key & lmask)];
        int num = 0, face = -1;
        // the contact filter on (collider of the lower entity, other collider): TRIGGER makes
        // a trigger pair, not a contact (src/Physecs.cpp:200-207); defaultContactFilter is a
        // trigger on either side (:20-23). Joint-connected / setCanCollide pairs are skipped (:209)
        bool skip = filterK ? filterTable[filterClass[c0] * filterK + filterClass[c1]] != 0
                            : ((cflags[c0] | cflags[c1]) & CF_TRIGGER) != 0;
        // trigger pairs go to k_triggers (before the non-colliding test, as in the reference)
        const bool toTrig = skip && trigList != nullptr;
        if (__ballot(toTrig)) {
            int i = wave_append(nTrig, toTrig);
            if (toTrig) trigList[i] = p;
        }
        if (!skip && nNonColliding) {
            uint64_t ek = ((uint64_t)centity[c0] << 32) | centity[c1];
            skip = in_sorted(nonColliding, nNonColliding, ek);
        }
        Mf m;
        m.numPoints = 0;
        // pairs with a triangle mesh go to the mesh passes, pairs with a convex mesh to
        // k_narrowphase_convex: appended with one atomic per wave
        const bool toMesh = !skip && (ctype[c0] == PGX_TRIANGLE_MESH || ctype[c1] == PGX_TRIANGLE_MESH);
        const bool toHeavy = !skip && !toMesh && (ctype[c0] == PGX_CONVEX_MESH || ctype[c1] == PGX_CONVEX_MESH);
        if (__ballot(toMesh)) {
            int i = wave_append(nMesh, toMesh);
            if (toMesh) meshPairs[i] = p;
        }
        if (__ballot(toHeavy)) {
            int i = wave_append(nHeavy, toHeavy);
            if (toHeavy) heavy[i] = p;
        }
        skip = skip || toMesh || toHeavy;
        if (!skip) {
            int b0 = cbody[c0], b1 = cbody[c1];
            f3 bp0 = xyz(bpos[b0]), bp1 = xyz(bpos[b1]);
            qf bq0 = q4(bquat[b0]), bq1 = q4(bquat[b1]);
            f3 p0 = add(bp0, qrot(bq0, xyz(clpos[c0])));
            qf q0 = qmul(bq0, q4(clquat[c0]));
            f3 p1 = add(bp1, qrot(bq1, xyz(clpos[c1])));
            qf q1 = qmul(bq1, q4(clquat[c1]));
            bool hit = collide<true>(ctype[c0], cparams[c0], p0, q0, ctype[c1], cparams[c1], p1, q1, m, face);
            num = hit ? m.numPoints : 0;
        }
        if (__ballot(face >= 0)) {
            const int k = wave_append(nFaces, face >= 0);
            if (face >= 0) facesEnd[-1 - k] = p;
        }
        npNum[p] = face >= 0 ? face : num;
        if (num) {
            npNormal[p] = f4(m.normal, 0.f);
            for (int k = 0; k < 4; ++k) {
                if (k < num) {
                    npPts[8 * (size_t)p + 2 * k] = f4(m.pts[k].p0, 0.f);
                    npPts[8 * (size_t)p + 2 * k + 1] = f4(m.pts[k].p1, 0.f);
                }
            }
        }
    }
}

// Pairs with a convex mesh, a wave per pair (np_wave.h): a fixed grid of CONVEX_WAVES waves,
// what the chip holds of their 14 KB of LDS each, walks the list. The list length is read on
// the device, so no host round trip.
constexpr int CONVEX_WAVES = 2816;
// The face contacts of box pairs (box_face_contacts and polygon_box_face_contacts_n,
// operation for operation): the other box's face clipped by the four sides of the reference
// face, its penetrating corners, four of them picked. Eight lanes per pair, a polygon corner
// each (a second round of corners where a clip leaves more than eight), the corners in LDS.
// With a lane per pair in k_narrowphase this was a chain of some thirty corners, each with a
// branch and a division, on polygons in scratch memory: 58 us for the 585 pairs of a pyramid
// of boxes however few they were, 17 us now with k_narrowphase; 177 and 111 us for 662k mixed
// pairs.
constexpr int BOX_LANES = 8, BOX_GROUPS = 256 / BOX_LANES, BOX_BLOCKS = 2048;
struct BoxClip { f2 poly[2][MAXPOLY]; f3 pen[MAXPOLY]; };
__device__ __forceinline__ uint32_t group_ballot(bool b) {
    return (uint32_t)(__ballot(b) >> (threadIdx.x & (WAVE - BOX_LANES))) & ((1u << BOX_LANES) - 1);
}
template <int CTRL>
__device__ __forceinline__ float larger_lane(float x) {
    const float y = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, true));
    return y > x ? y : x;
}
// the first index whose value (v[c] of lane l: element 8 c + l, below n) is the largest and
// above 0, else 0: the sequential loop that keeps what is greater than the best so far
__device__ __forceinline__ int first_largest(const float (&v)[2], int n) {
    const int l = threadIdx.x & (BOX_LANES - 1);
    float best = l < n && v[0] > 0.f ? v[0] : 0.f;
    if (BOX_LANES + l < n && v[1] > best) best = v[1];
    best = larger_lane<0xB1>(best);    // quad_perm 1,0,3,2
    best = larger_lane<0x4E>(best);    // quad_perm 2,3,0,1
    best = larger_lane<0x141>(best);   // row_half_mirror
    const uint32_t e0 = group_ballot(l < n && v[0] == best), e1 = group_ballot(BOX_LANES + l < n && v[1] == best);
    if (!(best > 0.f)) return 0;
    return e0 ? __ffs(e0) - 1 : BOX_LANES + __ffs(e1) - 1;
}
__global__ __launch_bounds__(256) void k_box_faces(
    const int32_t* __restrict__ nFacesP, const int32_t* __restrict__ facesEnd, const uint64_t* __restrict__ pkeys,
    int localBits, const int32_t* __restrict__ worldColStart, const int32_t* __restrict__ colOfLocal,
    const int32_t* __restrict__ cbody, const float4* __restrict__ cparams, const float4* __restrict__ clpos,
    const float4* __restrict__ clquat, const float4* __restrict__ bpos, const float4* __restrict__ bquat,
    int32_t* __restrict__ npNum, float4* __restrict__ npNormal, float4* __restrict__ npPts) {
    __shared__ BoxClip clips[BOX_GROUPS];
    const int group = threadIdx.x / BOX_LANES, l = threadIdx.x & (BOX_LANES - 1);
    BoxClip& C = clips[group];
    const uint32_t before = (1u << l) - 1;
    const int nFaces = *nFacesP;
    const uint64_t lmask = (1ull << localBits) - 1;
    for (int base = blockIdx.x * BOX_GROUPS; base < nFaces; base += gridDim.x * BOX_GROUPS) {
        const bool live = base + group < nFaces;   // the block's last groups repeat its first pair, unstored
        const int p = facesEnd[-1 - (live ? base + group : base)];
        const int code = live ? npNum[p] : 0;
        const uint64_t key = pkeys[p];
        const int cols = worldColStart[(int)(key >> (2 * localBits))];
        const int c0 = colOfLocal[cols + (int)((key >> localBits) & lmask)], c1 = colOfLocal[cols + (int)(key & lmask)];
        const int b0 = cbody[c0], b1 = cbody[c1];
        const qf bq0 = q4(bquat[b0]), bq1 = q4(bquat[b1]);
        const f3 p0 = add(xyz(bpos[b0]), qrot(bq0, xyz(clpos[c0]))), p1 = add(xyz(bpos[b1]), qrot(bq1, xyz(clpos[c1])));
        const m3 m0 = mat3_cast(qmul(bq0, q4(clquat[c0]))), m1 = mat3_cast(qmul(bq1, q4(clquat[c1])));
        const bool second = code >= 3;   // the reference face's box
        const int refAxis = second ? code - 3 : code;
        auto of = [&](f3 x, f3 y) { return mk3(second ? y.x : x.x, second ? y.y : x.y, second ? y.z : x.z); };
        const m3 uRef = mk_m3(of(m0.c0, m1.c0), of(m0.c1, m1.c1), of(m0.c2, m1.c2));
        const m3 uInc = mk_m3(of(m1.c0, m0.c0), of(m1.c1, m0.c1), of(m1.c2, m0.c2));
        const f3 posRef = of(p0, p1), posInc = of(p1, p0);
        const f3 heRef = xyz(cparams[second ? c1 : c0]), heInc = xyz(cparams[second ? c0 : c1]);
        // box_face_contacts: the incident face
        const f3 axis = col(uRef, refAxis);
        const float refSign = dot(axis, sub(posInc, posRef)) < 0 ? -1.f : 1.f;
        float maxDot = 0.f, incSign = 1.f;
        int incAxis = 0;
        for (int i = 0; i < 3; ++i) {
            const float d = dot(mul(-refSign, axis), col(uInc, i)), ad = gabs(d);
            if (ad > maxDot) { maxDot = ad; incAxis = i; incSign = d < 0 ? -1.f : 1.f; }
        }
        const int ia1 = incAxis == 2 ? 0 : incAxis + 1, ia2 = incAxis == 0 ? 2 : incAxis - 1;
        const m3 inv = inverse(uRef);
        const f3 ui = col(uInc, incAxis), u1 = col(uInc, ia1), u2 = col(uInc, ia2);
        const float h1 = at(heInc, ia1), h2 = at(heInc, ia2);
        const f3 incOrig = mulmv(inv, sub(add(posInc, mul(mul(ui, at(heInc, incAxis)), incSign)), posRef));
        const f3 a = mul(u1, h1), b = mul(u2, h2), na = mul(neg(u1), h1);
        const int cx = refAxis == 2 ? 0 : refAxis + 1, cy = refAxis == 0 ? 2 : refAxis - 1;
        {
            const f3 x = l == 1 || l == 2 ? na : a;
            const f3 corner = add(incOrig, mulmv(inv, l < 2 ? add(x, b) : sub(x, b)));
            if (l < 4) C.poly[0][l] = mk2(at(corner, cx), at(corner, cy));
        }
        wave_sync();
        // clip_polygon: an edge's outputs, in the order of the corners
        const float hx = at(heRef, cx), hy = at(heRef, cy);
        int n = 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const f2 ca = mk2(e < 2 ? hx : -hx, e == 0 || e == 3 ? hy : -hy);
            const f2 cb = mk2(e == 0 || e == 3 ? hx : -hx, e < 2 ? -hy : hy);
            const f2* in = C.poly[e & 1];
            f2* out = C.poly[1 - (e & 1)];
            int m = 0;
            for (int k = 0; k < MAXPOLY && __ballot(k < n); k += BOX_LANES) {
                const int i = k + l;
                const bool have = i < n;
                const f2 me = in[have ? i : 0], next = in[have && i + 1 < n ? i + 1 : 0];
                const bool ii = have && inside(me, ca, cb), ji = have && inside(next, ca, cb);
                const uint32_t one = group_ballot(ii || ji), two = group_ballot(!ii && ji);
                int at_ = m + __popc(one & before) + __popc(two & before);
                if (ii != ji) {
                    if (at_ < MAXPOLY) out[at_] = intersect2(me, next, ca, cb);
                    ++at_;
                }
                if (ji && at_ < MAXPOLY) out[at_] = next;
                m += __popc(one) + __popc(two);
            }
            n = min(m, MAXPOLY);
            wave_sync();
        }
        // polygon_box_face_contacts_n: the corners under the face
        const f3 incNormal = mulmv(inv, ui);
        const int axisSign = (int)refSign;
        f3 dir = s3(0.f);
        set(dir, refAxis, (float)axisSign);
        const float denom = dot(dir, incNormal), heAxis = at(heRef, refAxis), lim = heAxis + 1e-4f;
        int np = 0;
        for (int k = 0; k < MAXPOLY && __ballot(k < n); k += BOX_LANES) {
            const bool have = k + l < n;
            const f2 q = C.poly[0][have ? k + l : 0];
            f3 p3 = s3(0.f);
            set(p3, cx, q.x);
            set(p3, cy, q.y);
            const float distance = dot(sub(incOrig, p3), incNormal) / denom;
            const bool keep = have && distance < lim;
            const uint32_t kept = group_ballot(keep);
            set(p3, refAxis, axisSign * distance);
            if (keep) C.pen[np + __popc(kept & before)] = p3;
            np += __popc(kept);
        }
        wave_sync();
        int pick = l;   // the corner of contact l
        if (np > 4) {
            const f3 first = C.pen[0];
            f3 pen[2];
            float v[2];
            for (int c = 0; c < 2; ++c) {
                pen[c] = C.pen[min(BOX_LANES * c + l, np - 1)];
                const f3 d = sub(pen[c], first);
                v[c] = dot(d, d);
            }
            const int far = first_largest(v, np);
            const f3 second_ = C.pen[far];
            for (int c = 0; c < 2; ++c) {
                const f3 da = sub(first, pen[c]), db = sub(second_, pen[c]);
                v[c] = det2(mk2(at(da, cx), at(da, cy)), mk2(at(db, cx), at(db, cy)));
            }
            const int left = first_largest(v, np);
            for (int c = 0; c < 2; ++c) v[c] = -v[c];
            const int right = first_largest(v, np);
            pick = l == 0 ? 0 : l == 1 ? far : l == 2 ? left : right;
            np = 4;
        }
        if (live && l < np) {
            const f3 pen = C.pen[pick];
            f3 on = pen;
            set(on, refAxis, axisSign * heAxis);
            const f3 onRef = add(posRef, mulmv(uRef, on)), onInc = add(posRef, mulmv(uRef, pen));
            npPts[8 * (size_t)p + 2 * l] = f4(second ? onInc : onRef, 0.f);
            npPts[8 * (size_t)p + 2 * l + 1] = f4(second ? onRef : onInc, 0.f);
        }
        if (live && l == 0) {
            npNum[p] = np;
            if (np) npNormal[p] = f4(dot(axis, sub(p1, p0)) < 0 ? neg(axis) : axis, 0.f);
        }
        wave_sync();
    }
}

__global__ __launch_bounds__(64) void k_narrowphase_convex(
    const int32_t* __restrict__ nHeavyP, const int32_t* __restrict__ heavy, const uint64_t* __restrict__ pkeys,
    int localBits, const int32_t* __restrict__ worldColStart, const int32_t* __restrict__ colOfLocal,
    const int32_t* __restrict__ cbody, const int32_t* __restrict__ ctype, const float4* __restrict__ cparams,
    const float4* __restrict__ clpos, const float4* __restrict__ clquat, const float4* __restrict__ bpos,
    const float4* __restrict__ bquat, ConvexView cv, int32_t* __restrict__ npNum, float4* __restrict__ npNormal,
    float4* __restrict__ npPts, int32_t* __restrict__ errors) {
    __shared__ WaveMem M;
    const int nHeavy = *nHeavyP;
    const uint64_t lmask = (1ull << localBits) - 1;
    for (int h = blockIdx.x; h < nHeavy; h += gridDim.x) {
        const int p = heavy[h];
        const uint64_t key = pkeys[p];
        const int base = worldColStart[(int)(key >> (2 * localBits))];
        const int c0 = colOfLocal[base + (int)((key >> localBits) & lmask)];
        const int c1 = colOfLocal[base + (int)(key & lmask)];
        const int b0 = cbody[c0], b1 = cbody[c1];
        const qf bq0 = q4(bquat[b0]), bq1 = q4(bquat[b1]);
        const f3 p0 = add(xyz(bpos[b0]), qrot(bq0, xyz(clpos[c0])));
        const qf q0 = qmul(bq0, q4(clquat[c0]));
        const f3 p1 = add(xyz(bpos[b1]), qrot(bq1, xyz(clpos[c1])));
        const qf q1 = qmul(bq1, q4(clquat[c1]));
        Mf m;
        bool ovf;
        const bool hit = collide_convex_w(ctype[c0], cparams[c0], p0, q0, ctype[c1], cparams[c1], p1, q1, cv, M, m, ovf);
        if (threadIdx.x != 0) continue;
        if (ovf) atomicAdd(errors, 1);
        const int num = hit ? m.numPoints : 0;
        npNum[p] = num;
        if (num) {
            npNormal[p] = f4(m.normal, 0.f);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (k < num) {
                    npPts[8 * (size_t)p + 2 * k] = f4(m.pts[k].p0, 0.f);
                    npPts[8 * (size_t)p + 2 * k + 1] = f4(m.pts[k].p1, 0.f);
                }
        }
    }
}

// ------------------------------------------------------------------ overlap queries
// physecs::overlap (src/Overlap.cpp): the pair tests as yes/no answers, no manifold.
__device__ __forceinline__ bool ov_sphere_sphere(f3 p0, float r0, f3 p1, float r1) {   // Overlap.cpp:19-24
    f3 d = sub(p1, p0);
    float rs = r0 + r1;
    return !(dot(d, d) > rs * rs);
}

__device__ bool ov_capsule_capsule(f3 p0, qf q0, float hh0, float r0, f3 p1, qf q1, float hh1,   // :26-35
                                   float r1) {
    const f3 up = mk3(0.f, 1.f, 0.f);
    f3 a, b;
    closest_points_segments(p0, qrot(q0, up), -hh0, hh0, p1, qrot(q1, up), -hh1, hh1, a, b);
    f3 d = sub(b, a);
    float rs = r0 + r1;
    return !(dot(d, d) > rs * rs);
}

// Overlap.cpp:37-139: the 15 separating axes, separated when |t.L| - rA - rB > 0. For the
// edge axes Ai x Bj the radius sums take the other two axes of each box, lower index first.
__device__ bool ov_box_box(f3 p0, qf q0, f3 he0, f3 p1, qf q1, f3 he1) {
    const m3 u0 = mat3_cast(q0), u1 = mat3_cast(q1);
    f3 tv = sub(p1, p0);
    tv = mk3(dot(tv, u0.c0), dot(tv, u0.c1), dot(tv, u0.c2));
    float r[3][3], ar[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            r[i][j] = dot(col(u0, i), col(u1, j));
            ar[i][j] = gabs(r[i][j]);
        }
    const float a[3] = {he0.x, he0.y, he0.z}, b[3] = {he1.x, he1.y, he1.z}, t[3] = {tv.x, tv.y, tv.z};
#pragma unroll
    for (int i = 0; i < 3; ++i)
        if (gabs(t[i]) - a[i] - (b[0] * ar[i][0] + b[1] * ar[i][1] + b[2] * ar[i][2]) > 0) return false;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        float ra = a[0] * ar[0][i] + a[1] * ar[1][i] + a[2] * ar[2][i];
        if (gabs(t[0] * r[0][i] + t[1] * r[1][i] + t[2] * r[2][i]) - ra - b[i] > 0) return false;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int i1 = (i + 1) % 3, i2 = (i + 2) % 3;
        const int lo = i1 < i2 ? i1 : i2, hi = i1 < i2 ? i2 : i1;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int j1 = (j + 1) % 3, j2 = (j + 2) % 3;
            const int blo = j1 < j2 ? j1 : j2, bhi = j1 < j2 ? j2 : j1;
            float ra = a[lo] * ar[hi][j] + a[hi] * ar[lo][j];
            float rb = b[blo] * ar[i][bhi] + b[bhi] * ar[i][blo];
            if (gabs(t[i2] * r[i1][j] - t[i1] * r[i2][j]) - ra - rb > 0) return false;
        }
    }
    return true;
}

__device__ bool ov_sphere_capsule(f3 p0, float r0, f3 p1, qf q1, float hh1, float r1) {   // :145-153
    f3 q = closest_point_on_segment(p0, p1, qrot(q1, mk3(0.f, 1.f, 0.f)), -hh1, hh1);
    f3 v = sub(q, p0);
    float rs = r0 + r1;
    return !(dot(v, v) > rs * rs);
}

__device__ bool ov_sphere_box(f3 p0, float r0, f3 p1, qf q1, f3 he) {   // :155-169
    m3 u = mat3_cast(q1);
    f3 d = sub(p0, p1);
    d = mk3(dot(d, u.c0), dot(d, u.c1), dot(d, u.c2));
    f3 q = add(p1, mulmv(u, vclamp(d, neg(he), he)));
    f3 v = sub(q, p0);
    return !(dot(v, v) > r0 * r0);
}

// :175-193; separated when the squared distance reaches r^2 (>=, where the others use >)
__device__ bool ov_capsule_box(f3 p0, qf q0, float hh0, float r0, f3 p1, qf q1, f3 he) {
    m3 u = mat3_cast(q1);
    f3 p = sub(p0, p1);
    p = mk3(dot(p, u.c0), dot(p, u.c1), dot(p, u.c2));
    f3 dir = qrot(q0, mk3(0.f, 1.f, 0.f));
    f3 dl = mk3(dot(dir, u.c0), dot(dir, u.c1), dot(dir, u.c2));
    float t = 0.f;
    f3 q = s3(0.f);
    return !(segment_aabb(p, dl, -hh0, hh0, he, t, q) >= r0 * r0);
}

__device__ __forceinline__ SupConvex ov_convex(const ConvexView& cv, float4 g, f3 pos, qf q) {
    const int4 mi = cv.mesh[(int)g.w];
    return SupConvex{pos, mat3_cast(q), mk3(g.x, g.y, g.z), cv.verts + mi.x, mi.y};
}

// physecs::overlap (src/Overlap.cpp:203-235). A triangle mesh on either side never
// overlaps. The convex cases run GJK (Overlap.cpp:141-200); the box-convex case places the
// convex support at the box's position, as the reference does (Overlap.cpp:200).
__device__ bool overlap_shapes(int t0, float4 g0, f3 p0, qf q0, int t1, float4 g1, f3 p1, qf q1,
                               const ConvexView& cv) {
    if (t0 > PGX_CONVEX_MESH || t1 > PGX_CONVEX_MESH) return false;
    const f3 he0 = mk3(g0.x, g0.y, g0.z), he1 = mk3(g1.x, g1.y, g1.z);
    const f3 up = mk3(0.f, 1.f, 0.f);
    GjkV s[4];
    switch (t0) {
        case PGX_SPHERE:
            switch (t1) {
                case PGX_SPHERE: return ov_sphere_sphere(p0, g0.x, p1, g1.x);
                case PGX_CAPSULE: return ov_sphere_capsule(p0, g0.x, p1, q1, g1.x, g1.y);
                case PGX_BOX: return ov_sphere_box(p0, g0.x, p1, q1, he1);
                default: return gjk(SupSphere{p0, g0.x}, ov_convex(cv, g1, p1, q1), sub(p1, p0), s);
            }
        case PGX_CAPSULE:
            switch (t1) {
                case PGX_SPHERE: return ov_sphere_capsule(p1, g1.x, p0, q0, g0.x, g0.y);
                case PGX_CAPSULE: return ov_capsule_capsule(p0, q0, g0.x, g0.y, p1, q1, g1.x, g1.y);
                case PGX_BOX: return ov_capsule_box(p0, q0, g0.x, g0.y, p1, q1, he1);
                default:
                    return gjk(SupCapsule{p0, qrot(q0, up), g0.x, g0.y}, ov_convex(cv, g1, p1, q1), sub(p1, p0), s);
            }
        case PGX_BOX:
            switch (t1) {
                case PGX_SPHERE: return ov_sphere_box(p1, g1.x, p0, q0, he0);
                case PGX_CAPSULE: return ov_capsule_box(p1, q1, g1.x, g1.y, p0, q0, he0);
                case PGX_BOX: return ov_box_box(p0, q0, he0, p1, q1, he1);
                default: return gjk(SupBox{p0, mat3_cast(q0), he0}, ov_convex(cv, g1, p0, q1), sub(p1, p0), s);
            }
        default:
            switch (t1) {
                case PGX_SPHERE: return gjk(SupSphere{p1, g1.x}, ov_convex(cv, g0, p0, q0), sub(p0, p1), s);
                case PGX_CAPSULE:
                    return gjk(SupCapsule{p1, qrot(q1, up), g1.x, g1.y}, ov_convex(cv, g0, p0, q0), sub(p0, p1), s);
                case PGX_BOX: return gjk(SupBox{p1, mat3_cast(q1), he1}, ov_convex(cv, g0, p1, q0), sub(p0, p1), s);
                default: return gjk(ov_convex(cv, g0, p0, q0), ov_convex(cv, g1, p1, q1), sub(p1, p0), s);
            }
    }
}

// the primitive pairs of physecs::overlap (sphere, capsule, box on both sides), no GJK
__device__ bool overlap_prims(int t0, float4 g0, f3 p0, qf q0, int t1, float4 g1, f3 p1, qf q1) {
    const f3 he0 = mk3(g0.x, g0.y, g0.z), he1 = mk3(g1.x, g1.y, g1.z);
    if (t0 == PGX_SPHERE) {
        if (t1 == PGX_SPHERE) return ov_sphere_sphere(p0, g0.x, p1, g1.x);
        if (t1 == PGX_CAPSULE) return ov_sphere_capsule(p0, g0.x, p1, q1, g1.x, g1.y);
        return ov_sphere_box(p0, g0.x, p1, q1, he1);
    }
    if (t0 == PGX_CAPSULE) {
        if (t1 == PGX_SPHERE) return ov_sphere_capsule(p1, g1.x, p0, q0, g0.x, g0.y);
        if (t1 == PGX_CAPSULE) return ov_capsule_capsule(p0, q0, g0.x, g0.y, p1, q1, g1.x, g1.y);
        return ov_capsule_box(p0, q0, g0.x, g0.y, p1, q1, he1);
    }
    if (t1 == PGX_SPHERE) return ov_sphere_box(p1, g1.x, p0, q0, he0);
    if (t1 == PGX_CAPSULE) return ov_capsule_box(p1, q1, g1.x, g1.y, p0, q0, he0);
    return ov_box_box(p0, q0, he0, p1, q1, he1);
}

// intersects (src/BoundsUtil.cpp:87-92): inclusive on every axis
__device__ __forceinline__ bool boxes_meet(f3 amn, f3 amx, float4 bmn, float4 bmx) {
    return !(amx.x < bmn.x || amn.x > bmx.x || amx.y < bmn.y || amn.y > bmx.y || amx.z < bmn.z || amn.z > bmx.z);
}

// one collider of the query's world: the reference's leaf test (bounds, filter, shape).
// 0: no overlap; 1: overlap; 2: a pair with a convex mesh, left to k_overlap_convex (the
// walk keeps no GJK state, so it needs far fewer registers)
__device__ __forceinline__ int overlap_collider(const OverlapArgs& A, int c, int t, float4 g, f3 pos, qf q, f3 mn,
                                                f3 mx, int filter) {
    if (!boxes_meet(mn, mx, A.cbmin[c], A.cbmax[c])) return 0;
    if (filter && !(A.cdata[c] & filter)) return 0;
    const int ct = A.ctype[c];
    if (ct == PGX_TRIANGLE_MESH) return 0;   // overlaps nothing (src/Overlap.cpp:203-235)
    if (ct == PGX_CONVEX_MESH || t == PGX_CONVEX_MESH) return 2;
    const int b = A.cbody[c];
    const qf bq = q4(A.bquat[b]);
    const f3 cp = add(xyz(A.bpos[b]), qrot(bq, xyz(A.clpos[c])));
    return overlap_prims(t, g, pos, q, ct, A.cparams[c], cp, qmul(bq, q4(A.clquat[c]))) ? 1 : 0;
}

// One query per thread: its bounds, the walk of its world's LBVH (boxes tested inclusive,
// as the reference's recursion does) and its world's static colliders. Each hit appends the
// key (query << cbits | collider) with one atomic per wave; keys beyond the capacity are
// counted, not written. count[i] = the query's hits.
__global__ __launch_bounds__(64) void k_overlap(OverlapArgs A) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < A.n;
    int t = PGX_TRIANGLE_MESH, filter = 0, wd = 0;
    float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
    f3 pos = s3(0.f), mn = s3(0.f), mx = s3(0.f);
    qf q = q4(make_float4(0.f, 0.f, 0.f, 1.f));
    if (live) {
        t = A.qType[i];
        g = A.qPrm[i];
        const float4 pw = A.qPos[i];
        pos = xyz(pw);
        wd = __float_as_int(pw.w);
        q = q4(A.qQuat[i]);
        filter = A.qFilter[i];
        if (t <= PGX_CONVEX_MESH)
            shape_bounds(t, g, pos, q, A.cv.verts, A.cv.mesh, nullptr, nullptr, mn, mx);
    }
    // a triangle-mesh query overlaps nothing (src/Overlap.cpp:203-235)
    const bool active = live && t <= PGX_CONVEX_MESH;
    int hits = 0;
    int node = active ? A.worldRoot[wd] : -1;
    const int stop = active && node != -1 ? A.worldStop[wd] : -1;
    int visits = 0;
    int st = active ? A.worldStaticStart[wd] : 0;
    const int stEnd = active ? A.worldStaticStart[wd + 1] : 0;
    // the walk and then the static list, in one loop so that the wave's lanes append together
    while (true) {
        int c = -1;
        bool more = false;
        if (node != -1 && node != stop && visits < 2 * A.nLeaves) {   // a walk visits at most 2n - 1 nodes
            ++visits;
            more = true;
            if (node & LEAF_BIT) {
                const int l = node & ~LEAF_BIT;
                c = A.mvals[l];
                node = __float_as_int(A.leafA[l].w);
            } else {
                const float4 na = A.nodeA[node], nb = A.nodeB[node];
                node = boxes_meet(mn, mx, na, nb) ? __float_as_int(na.w) : __float_as_int(nb.w);
            }
        } else if (st < stEnd) {
            more = true;
            c = A.staticCols[st++];
        }
        const int r = c >= 0 ? overlap_collider(A, c, t, g, pos, q, mn, mx, filter) : 0;
        const bool hit = r == 1, toCvx = r == 2;
        if (__ballot(hit)) {
            const int slot = wave_append(A.total, hit);
            if (hit && slot < A.cap) A.keys[slot] = ((uint64_t)(uint32_t)i << A.cbits) | (uint32_t)c;
        }
        if (__ballot(toCvx)) {
            const int k = wave_append(A.nCvx, toCvx);
            if (toCvx && k < A.listCap) A.cvxPairs[k] = make_int2(i, c);
        }
        hits += hit;
        if (!__ballot(more)) break;
    }
    if (live) A.count[i] = hits;
}

// Trigger pairs: physecs::overlap of the two colliders (src/Physecs.cpp:199-206); the keys
// of the overlapping pairs are appended with one atomic per wave. A fixed grid walks the
// list, whose length is read on the device.
__global__ __launch_bounds__(64) void k_triggers(
    const int32_t* __restrict__ nTrigP, const int32_t* __restrict__ trigList, const uint64_t* __restrict__ pkeys,
    int localBits, const int32_t* __restrict__ worldColStart, const int32_t* __restrict__ colOfLocal,
    const int32_t* __restrict__ cbody, const int32_t* __restrict__ ctype, const float4* __restrict__ cparams,
    const float4* __restrict__ clpos, const float4* __restrict__ clquat, const float4* __restrict__ bpos,
    const float4* __restrict__ bquat, ConvexView cv, int32_t* __restrict__ nHits, uint64_t* __restrict__ hitKeys) {
    const int nTrig = *nTrigP;
    const uint64_t lmask = (1ull << localBits) - 1;
    // blocks are one wave, so the trip count is wave-uniform and the appends see whole waves
    for (int base = blockIdx.x * blockDim.x; base < nTrig; base += gridDim.x * blockDim.x) {
        const int h = base + (int)threadIdx.x;
        bool hit = false;
        uint64_t key = 0;
        if (h < nTrig) {
            key = pkeys[trigList[h]];
            const int b = worldColStart[(int)(key >> (2 * localBits))];
            const int c0 = colOfLocal[b + (int)((key >> localBits) & lmask)];
            const int c1 = colOfLocal[b + (int)(key & lmask)];
            const int b0 = cbody[c0], b1 = cbody[c1];
            const qf bq0 = q4(bquat[b0]), bq1 = q4(bquat[b1]);
            const f3 p0 = add(xyz(bpos[b0]), qrot(bq0, xyz(clpos[c0])));
            const f3 p1 = add(xyz(bpos[b1]), qrot(bq1, xyz(clpos[c1])));
            hit = overlap_shapes(ctype[c0], cparams[c0], p0, qmul(bq0, q4(clquat[c0])), ctype[c1], cparams[c1], p1,
                                 qmul(bq1, q4(clquat[c1])), cv);
        }
        if (__ballot(hit)) {
            const int slot = wave_append(nHits, hit);
            if (hit) hitKeys[slot] = key;
        }
    }
}

// ------------------------------------------------------------------ triangle-mesh pairs
// What the passes over mesh pairs read, for the step's pairs and the MTD queries' alike.
struct MeshArgs {
    const int32_t* nPairs;                 // number of mesh pairs (device)
    int maxPairs;                          // and how many of them are listed
    const int32_t* stepPairs;              // the step's: pair slots,
    const int2* queryPairs;                // or (query, collider)
    const uint64_t* pkeys;
    int localBits;
    const int32_t *worldColStart, *colOfLocal, *cbody, *ctype;
    const float4 *cparams, *clpos, *clquat, *bpos, *bquat;
    const float4 *qPrm, *qPos, *qQuat;
    const int32_t* qType;
    ConvexView cv;
    TriMeshView tv;
    int inOrder;                           // World::tmInOrder
    int32_t* errors;                       // capacity and EPA errors
    // candidates (triangle, pair), each pair's block of them, their records; the convex ones
    // that GJK hit, with their simplex (36 floats, word f of hit i at f * candCap + i)
    int32_t* candTotal;
    int candCap;
    int32_t *cand, *pairOf, *candOff, *candCount;
    MeshRecs recs;
    int32_t *hitTotal, *hitList;
    float* simplex;
};

struct MeshPair {
    int p, c, tb;                          // pair slot or query; the mesh's collider; the body's shape
    bool flip;
    float4 g;
    f3 pos0, pos1, lpos;
    qf or0, or1, lor;
    int4 mi;
};

__device__ __forceinline__ void collider_pose(const MeshArgs& A, int c, f3& pos, qf& q) {
    const int b = A.cbody[c];
    const qf bq = q4(A.bquat[b]);
    pos = add(xyz(A.bpos[b]), qrot(bq, xyz(A.clpos[c])));
    q = qmul(bq, q4(A.clquat[c]));
}

// mesh pair h: the body collider (or query shape) and the mesh, their world poses, the body
// in the mesh's frame. src/Collision.cpp:897-906: a mesh on side 0 is solved as (other, mesh)
// and flipped. False for a mesh-mesh pair (no routine).
template <bool QUERY>
__device__ __forceinline__ bool mesh_pair(const MeshArgs& A, int h, MeshPair& m, SupConvex& sc) {
    if (QUERY) {
        const int2 qc = A.queryPairs[h];
        m.p = qc.x;
        m.c = qc.y;
        m.flip = true;
        m.tb = A.qType[m.p];
        m.g = A.qPrm[m.p];
        m.pos0 = xyz(A.qPos[m.p]);
        m.or0 = q4(A.qQuat[m.p]);
    } else {
        m.p = A.stepPairs[h];
        const uint64_t key = A.pkeys[m.p];
        const uint64_t lmask = (1ull << A.localBits) - 1;
        const int base = A.worldColStart[(int)(key >> (2 * A.localBits))];
        const int c0 = A.colOfLocal[base + (int)((key >> A.localBits) & lmask)];
        const int c1 = A.colOfLocal[base + (int)(key & lmask)];
        const int t0 = A.ctype[c0], t1 = A.ctype[c1];
        if (t0 == PGX_TRIANGLE_MESH && t1 == PGX_TRIANGLE_MESH) return false;
        m.flip = t0 == PGX_TRIANGLE_MESH;
        const int cb = m.flip ? c1 : c0;
        m.c = m.flip ? c0 : c1;
        collider_pose(A, cb, m.pos0, m.or0);
        m.tb = A.ctype[cb];
        m.g = A.cparams[cb];
    }
    collider_pose(A, m.c, m.pos1, m.or1);
    m.mi = A.tv.mesh[(int)A.cparams[m.c].w];
    mesh_local(m.tb, m.g, m.pos0, m.or0, m.pos1, m.or1, A.cv, m.lpos, m.lor, sc);
    return true;
}

// Places in a list for the waves of a block, n[wave] each: one atomic per block. (One per
// wave, on one address, served some 65 per us: 47 us for the 3,071 pairs of 2,048 hulls and
// 1,024 capsules on a terrain, more than the query itself.) Every wave of the block calls it.
// A list counts on past its end, up to RESERVE_MAX places and what the blocks then at work ask
// for, so that places never wrap: a block that comes after takes its count back.
constexpr int RESERVE_MAX = 1 << 30;
template <int WAVES>
__device__ __forceinline__ int block_reserve(int32_t* counter, int n) {
    __shared__ int count[WAVES], first;
    const int wave = threadIdx.x / WAVE;
    if (wave_lane() == 0) count[wave] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        int total = 0;
        for (int k = 0; k < WAVES; ++k) total += count[k];
        first = total ? atomicAdd(counter, total) : 0;
        if (first > RESERVE_MAX) atomicSub(counter, total);
    }
    __syncthreads();
    int at = first;
    for (int k = 0; k < wave; ++k) at += count[k];
    __syncthreads();   // read before the block's next turn
    return at;
}

// pass 1, a wave per pair: the BVH query, and a block of candidate slots reserved for the
// pair. Queries without room are counted on (their caller provides it and asks again).
constexpr int MESH_BLOCK_WAVES = 8, MESH_BLOCKS = 512;
template <bool QUERY>
__global__ __launch_bounds__(MESH_BLOCK_WAVES * 64) void k_mesh_query(MeshArgs A, int32_t* __restrict__ meshCount) {
    __shared__ QueryMem mem[MESH_BLOCK_WAVES];
    const int n = min(*A.nPairs, A.maxPairs), lane = wave_lane(), wave = threadIdx.x / WAVE;
    QueryMem& S = mem[wave];
    for (int h0 = blockIdx.x * MESH_BLOCK_WAVES; h0 < n; h0 += gridDim.x * MESH_BLOCK_WAVES) {
        const int h = h0 + wave;
        int nc = 0;
        if (h < n) {
            MeshPair m;
            SupConvex sc;
            const bool ok = mesh_pair<QUERY>(A, h, m, sc);
            if (!QUERY && lane == 0) meshCount[m.p] = 0;
            if (ok) {
                const MeshCtx mc{&A.tv, m.mi};
                nc = mesh_query(m.tb, m.g, m.lpos, m.lor, A.cv, mc, A.inOrder != 0, S);
                if (nc < 0) {
                    if (lane == 0) atomicAdd(A.errors, 1);
                    nc = 0;
                }
            }
        }
        const int base = block_reserve<MESH_BLOCK_WAVES>(A.candTotal, nc);
        if (h >= n) continue;
        if (base + nc > A.candCap) {   // the last slots, some of the pair's, stay empty
            if (!QUERY && lane == 0) atomicAdd(A.errors, 1);
            for (int i = base + lane; i < A.candCap; i += WAVE) A.pairOf[i] = -1;
            nc = 0;
        }
        for (int i = lane; i < nc; i += WAVE) {
            A.cand[base + i] = S.cand[i];
            A.pairOf[base + i] = h;
        }
        if (lane == 0) {
            A.candOff[h] = base;
            A.candCount[h] = nc;
        }
    }
}

// pass 2, a lane per (pair, candidate triangle): the closed forms and their contact records;
// for a convex mesh GJK, its hits listed with their simplex. Slots without a candidate (pair
// -1) are skipped; no pair's records are among them.
constexpr int MESH_TEST_BLOCKS = 2048;
template <bool QUERY, bool CONVEX>
__global__ __launch_bounds__(64) void k_mesh_test(MeshArgs A) {
    const int total = min(*A.candTotal, A.candCap);
    // whole waves go round together, so the appends see whole waves
    for (int base = blockIdx.x * WAVE; base < total; base += gridDim.x * WAVE) {
        const int k = base + (int)threadIdx.x;
        const int h = k < total ? A.pairOf[k] : -1;
        bool solved = false;
        GV va, vb, vc, vd;
        if (h >= 0) {
            MeshPair m;
            SupConvex sc;
            mesh_pair<QUERY>(A, h, m, sc);
            const MeshCtx mc{&A.tv, m.mi};
            TCI ci;
            ci.tri = A.cand[k];
            const int4 ix = mc.tri(ci.tri);
            const f3 a = mc.vert(ix.x), b = mc.vert(ix.y), c = mc.vert(ix.z);
            bool hit;
            if (CONVEX && m.tb == PGX_CONVEX_MESH) {
                hit = solved = gjk_w(sc, SupTriangle{a, b, c}, sub(mc.c(ci.tri), sc.pos), va, vb, vc, vd);
            } else {
                hit = mesh_test_closed(m.tb, m.g, m.lpos, m.lor, a, b, c, mc.n(ci.tri), ci);
                if (hit) A.recs.store(k, ci);
            }
            A.recs.rec(k, TM_CI_WORDS) = hit ? 1 : 0;
        }
        if (CONVEX && __ballot(solved)) {
            const int i = wave_append(A.hitTotal, solved);
            if (solved) {
                A.hitList[i] = k;
                float* s = A.simplex + i;
                const size_t cap = (size_t)A.candCap;
                int f = 0;
                auto put = [&](const GV& g) {
                    for (const f3& v : {g.pos, g.sp0, g.sp1}) {
                        s[cap * f] = v.x; s[cap * (f + 1)] = v.y; s[cap * (f + 2)] = v.z;
                        f += 3;
                    }
                };
                put(va); put(vb); put(vc); put(vd);
            }
        }
    }
}

// pass 3, a wave per listed triangle: EPA and the contact record
template <bool QUERY>
__global__ __launch_bounds__(64) void k_mesh_epa(MeshArgs A) {
    __shared__ WaveMem M;
    const int n = *A.hitTotal;
    for (int i = blockIdx.x; i < n; i += gridDim.x) {
        const int k = A.hitList[i];
        MeshPair m;
        SupConvex sc;
        mesh_pair<QUERY>(A, A.pairOf[k], m, sc);
        const MeshCtx mc{&A.tv, m.mi};
        TCI ci;
        ci.tri = A.cand[k];
        ci.featureIndex = 0; ci.boxFeature = 0; ci.boxAxis = 0;
        const int4 ix = mc.tri(ci.tri);
        const f3 a = mc.vert(ix.x), b = mc.vert(ix.y), c = mc.vert(ix.z);
        // word `lane` of the simplex per lane, then in every lane
        const float word = A.simplex[(size_t)A.candCap * min((int)threadIdx.x, 35) + i];
        auto get = [&](int f) {
            return GV{mk3(lane_read(word, f), lane_read(word, f + 1), lane_read(word, f + 2)),
                      mk3(lane_read(word, f + 3), lane_read(word, f + 4), lane_read(word, f + 5)),
                      mk3(lane_read(word, f + 6), lane_read(word, f + 7), lane_read(word, f + 8))};
        };
        bool ovf;
        ci.normal = epa_w(hull_of(sc), SupTriangle{a, b, c}, get(0), get(9), get(18), get(27), M, ci.cpBody, ci.cpTri, ovf);
        convex_tri_feature(a, b, c, ci);
        if (threadIdx.x == 0) {
            if (ovf) atomicAdd(A.errors, 1);
            A.recs.store(k, ci);
        }
    }
}

// pass 4, a wave per pair: its hit records in candidate order into S; their number
__device__ __forceinline__ int mesh_hits(const MeshArgs& A, int off, int nc, EmitMem& S) {
    const int lane = wave_lane();
    int nct = 0;
    for (int first = 0; first < nc; first += WAVE) {
        const int i = first + lane;
        const bool hit = i < nc && A.recs.hit(off + i);
        const uint64_t hits = __ballot(hit);
        if (hit) {
            S.order[nct + __popcll(hits & lanes_below())] = i;
            S.feature[i] = A.recs.feature(off + i);
            S.dist[i] = A.recs.dist(off + i);
        }
        nct += (int)__popcll(hits);
    }
    wave_sync();
    return nct;
}

// and the emission passes: the step's manifolds go to a block of slots per pair
template <bool CONVEX>
__global__ __launch_bounds__(MESH_BLOCK_WAVES * 64) void k_mesh_emit(MeshArgs A, int32_t* __restrict__ npNum,
                                                  float4* __restrict__ npNormal, float4* __restrict__ npPts,
                                                  int32_t* __restrict__ npTri, int32_t* __restrict__ meshFirst,
                                                  int32_t* __restrict__ meshCount, int32_t* __restrict__ slotCounter,
                                                  int mmCap, int pairCap) {
    __shared__ EmitMem mem[MESH_BLOCK_WAVES];
    const int n = min(*A.nPairs, A.maxPairs), lane = wave_lane(), wave = threadIdx.x / WAVE;
    EmitMem& S = mem[wave];
    for (int h0 = blockIdx.x * MESH_BLOCK_WAVES; h0 < n; h0 += gridDim.x * MESH_BLOCK_WAVES) {
        const int h = h0 + wave;
        const int off = h < n ? A.candOff[h] : 0;
        const int nct = h < n ? mesh_hits(A, off, A.candCount[h], S) : 0;
        const int slot = block_reserve<MESH_BLOCK_WAVES>(slotCounter, nct);
        if (nct == 0) continue;
        if (slot + nct > mmCap) {
            if (lane == 0) atomicAdd(A.errors, 1);
            continue;
        }
        MeshPair m;
        SupConvex sc;
        mesh_pair<false>(A, h, m, sc);
        const MeshCtx mc{&A.tv, m.mi};
        MeshOut out{npNum, npNormal, npPts, npTri, pairCap + slot, slot, 0, m.flip};
        mesh_emit<CONVEX>(m.tb, m.g, m.lpos, m.lor, m.pos1, m.or1, mc, A.cv, S, A.recs, (size_t)off, nct, out);
        if (lane == 0) {
            meshFirst[m.p] = slot;
            meshCount[m.p] = out.n;
        }
    }
}

// ------------------------------------------------------------------ MTD overlap queries
// Scene::overlapWithMinTranslationalDistance (src/Physecs.cpp:653-688): collision(collider,
// query) for every collider whose bounds meet the query's; each manifold with points gives
// its normal and mtd. Results are appended with keys (query, collider, manifold index).
constexpr int MTD_MBITS = 8;   // manifold index within a pair: at most TM_MAXCAND

__device__ __forceinline__ float manifold_mtd(const Mf& m) {   // src/Physecs.cpp:663-670
    float mtd = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (i >= m.numPoints) break;
        float dist = dot(sub(m.pts[i].p0, m.pts[i].p1), m.normal);
        if (dist > mtd) mtd = dist;
    }
    return mtd;
}

__device__ __forceinline__ void mtd_store(const MtdArgs& A, int slot, int q, int c, int k, float4 res) {
    if (slot >= A.cap) return;
    A.keys[slot] = ((uint64_t)(uint32_t)q << (A.cbits + MTD_MBITS)) | ((uint64_t)(uint32_t)c << MTD_MBITS) |
                   (uint64_t)k;
    A.vals[slot] = slot;
    A.res[slot] = res;
}
__device__ __forceinline__ void mtd_put(const MtdArgs& A, int slot, int q, int c, int k, const Mf& m) {
    mtd_store(A, slot, q, c, k, f4(m.normal, manifold_mtd(m)));
}

__device__ __forceinline__ void mtd_query(const MtdArgs& A, int i, int& t, float4& g, f3& pos, qf& q, int& wd) {
    t = A.qType[i];
    g = A.qPrm[i];
    const float4 pw = A.qPos[i];
    pos = xyz(pw);
    wd = __float_as_int(pw.w);
    q = q4(A.qQuat[i]);
}

__device__ __forceinline__ void mtd_collider_pose(const MtdArgs& A, int c, f3& cp, qf& cq) {
    const int b = A.cbody[c];
    const qf bq = q4(A.bquat[b]);
    cp = add(xyz(A.bpos[b]), qrot(bq, xyz(A.clpos[c])));
    cq = qmul(bq, q4(A.clquat[c]));
}

// pass 1, one lane per query: the walk of its world's LBVH and static list (as k_overlap);
// pairs of primitives are solved here, pairs with a convex or triangle mesh are listed
__global__ __launch_bounds__(64) void k_mtd_walk(MtdArgs A, ConvexView cv) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < A.n;
    int t = PGX_SPHERE, wd = 0;
    float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
    f3 pos = s3(0.f), mn = s3(0.f), mx = s3(0.f);
    qf q = q4(make_float4(0.f, 0.f, 0.f, 1.f));
    if (live) {
        mtd_query(A, i, t, g, pos, q, wd);
        shape_bounds(t, g, pos, q, cv.verts, cv.mesh, nullptr, nullptr, mn, mx);
    }
    int node = live ? A.worldRoot[wd] : -1;
    const int stop = live && node != -1 ? A.worldStop[wd] : -1;
    int visits = 0;
    int st = live ? A.worldStaticStart[wd] : 0;
    const int stEnd = live ? A.worldStaticStart[wd + 1] : 0;
    while (true) {
        int c = -1;
        bool more = false;
        if (node != -1 && node != stop && visits < 2 * A.nLeaves) {   // a walk visits at most 2n - 1 nodes
            ++visits;
            more = true;
            if (node & LEAF_BIT) {
                const int l = node & ~LEAF_BIT;
                c = A.mvals[l];
                node = __float_as_int(A.leafA[l].w);
            } else {
                const float4 na = A.nodeA[node], nb = A.nodeB[node];
                node = boxes_meet(mn, mx, na, nb) ? __float_as_int(na.w) : __float_as_int(nb.w);
            }
        } else if (st < stEnd) {
            more = true;
            c = A.staticCols[st++];
        }
        bool hit = false, toCvx = false, toMesh = false;
        Mf m;
        m.numPoints = 0;
        if (c >= 0 && boxes_meet(mn, mx, A.cbmin[c], A.cbmax[c])) {
            const int ct = A.ctype[c];
            if (ct == PGX_TRIANGLE_MESH) {
                toMesh = true;
            } else if (ct == PGX_CONVEX_MESH || t == PGX_CONVEX_MESH) {
                toCvx = true;
            } else {   // collision(collider, query), src/Physecs.cpp:659
                f3 cp;
                qf cq;
                mtd_collider_pose(A, c, cp, cq);
                int face;
                hit = collide<false>(ct, A.cparams[c], cp, cq, t, g, pos, q, m, face) && m.numPoints > 0;
            }
        }
        if (__ballot(hit)) {
            const int slot = wave_append(A.counts, hit);
            if (hit) mtd_put(A, slot, i, c, 0, m);
        }
        if (__ballot(toCvx)) {
            const int k = wave_append(A.counts + 1, toCvx);
            if (toCvx && k < A.listCap) A.convexPairs[k] = make_int2(i, c);
        }
        if (__ballot(toMesh)) {
            const int k = wave_append(A.counts + 2, toMesh);
            if (toMesh && k < A.listCap) A.meshPairs[k] = make_int2(i, c);
        }
        if (!__ballot(more)) break;
    }
}

// pass 2: the pairs with a convex mesh, a wave per pair
__global__ __launch_bounds__(64) void k_mtd_convex(MtdArgs A, ConvexView cv) {
    __shared__ WaveMem M;
    const int n = min(A.counts[1], A.listCap);
    for (int h = blockIdx.x; h < n; h += gridDim.x) {
        const int2 qc = A.convexPairs[h];
        int t, wd;
        float4 g;
        f3 pos, cp;
        qf q, cq;
        mtd_query(A, qc.x, t, g, pos, q, wd);
        mtd_collider_pose(A, qc.y, cp, cq);
        Mf m;
        bool ovf;
        const bool hit = collide_convex_w(A.ctype[qc.y], A.cparams[qc.y], cp, cq, t, g, pos, q, cv, M, m, ovf);
        if (threadIdx.x != 0) continue;
        if (ovf) atomicAdd(A.counts + 3, 1);
        if (hit && m.numPoints > 0) mtd_put(A, atomicAdd(A.counts, 1), qc.x, qc.y, 0, m);
    }
}

// pass 3, the pairs with a triangle mesh, in the step's mesh passes: the manifolds of one
// (query, mesh) pair; the mesh is the collider, geom0, so the pair is
// solved as (query, mesh) and flipped (src/Collision.cpp:897-901)
struct MtdOut {
    float4* res;          // LDS: the pair's results
    int n;
    __device__ __forceinline__ void emit(Mf& m, int) {   // the same manifold in every lane
        if (m.numPoints <= 0) return;
        m.normal = neg(m.normal);
        swap_sides(m);
        if (wave_lane() == 0) res[n] = f4(m.normal, manifold_mtd(m));
        ++n;
    }
};

template <bool CONVEX>
__global__ __launch_bounds__(MESH_BLOCK_WAVES * 64) void k_mtd_mesh_emit(MeshArgs A, MtdArgs Q) {
    __shared__ EmitMem mem[MESH_BLOCK_WAVES];
    __shared__ float4 results[MESH_BLOCK_WAVES][TM_MAXCAND];
    const int n = min(*A.nPairs, A.maxPairs), wave = threadIdx.x / WAVE;
    EmitMem& S = mem[wave];
    for (int h0 = blockIdx.x * MESH_BLOCK_WAVES; h0 < n; h0 += gridDim.x * MESH_BLOCK_WAVES) {
        const int h = h0 + wave;
        const int off = h < n ? A.candOff[h] : 0;
        const int nct = h < n ? mesh_hits(A, off, A.candCount[h], S) : 0;
        MtdOut out{results[wave], 0};
        MeshPair m;
        if (nct) {
            SupConvex sc;
            mesh_pair<true>(A, h, m, sc);
            const MeshCtx mc{&A.tv, m.mi};
            mesh_emit<CONVEX>(m.tb, m.g, m.lpos, m.lor, m.pos1, m.or1, mc, A.cv, S, A.recs, (size_t)off, nct, out);
        }
        const int base = block_reserve<MESH_BLOCK_WAVES>(Q.counts, out.n);
        for (int k = wave_lane(); k < out.n; k += WAVE) mtd_store(Q, base + k, m.p, m.c, k, out.res[k]);
        wave_sync();   // the results are read before the wave's next pair overwrites them
    }
}

// the passes up to the emission
template <bool QUERY>
static void mesh_passes(World& w, const MeshArgs& A) {
    hipLaunchKernelGGL(k_mesh_query<QUERY>, dim3(MESH_BLOCKS), dim3(MESH_BLOCK_WAVES * 64), 0, w.stream, A, w.meshCount.p);
    if (w.nConvex > 0) {
        hipLaunchKernelGGL((k_mesh_test<QUERY, true>), dim3(MESH_TEST_BLOCKS), dim3(64), 0, w.stream, A);
        hipLaunchKernelGGL(k_mesh_epa<QUERY>, dim3(CONVEX_WAVES), dim3(64), 0, w.stream, A);
    } else {
        hipLaunchKernelGGL((k_mesh_test<QUERY, false>), dim3(MESH_TEST_BLOCKS), dim3(64), 0, w.stream, A);
    }
    PGX_LAUNCH_CHECK();
}

static MeshArgs mesh_args(World& w, MeshBuffers& b) {
    MeshArgs A{};
    A.pkeys = w.pkeys.p; A.localBits = w.localBits;
    A.worldColStart = w.worldColStart.p; A.colOfLocal = w.colOfLocal.p; A.cbody = w.cbody.p; A.ctype = w.ctype.p;
    A.cparams = w.cparams.p; A.clpos = w.clpos.p; A.clquat = w.clquat.p; A.bpos = w.bpos.p; A.bquat = w.bquat.p;
    A.cv = ConvexView{w.cvVerts.p, w.cvMesh.p, w.cvFace.p, w.cvFaceIdx.p, w.cvFaceN.p, w.cvFaceC.p};
    A.tv = TriMeshView{w.tmVerts.p, w.tmTris.p, w.tmTriN.p, w.tmTriC.p, w.tmNodes.p, w.tmMesh.p};
    A.inOrder = w.tmInOrder ? 1 : 0;
    A.candCap = b.candCap;
    A.cand = b.cand.p; A.pairOf = b.pairOf.p; A.candOff = b.candOff.p; A.candCount = b.candCount.p;
    A.recs = MeshRecs{b.recs.p, (size_t)b.candCap};
    A.hitList = b.hitList.p; A.simplex = b.simplex.p;
    return A;
}

// buffers for the mesh pairs' passes: `pairs` pairs, `cands` candidate triangles
void np_mesh_buffers(World& w, MeshBuffers& b, size_t pairs, size_t cands) {
    if (cands > (size_t)RESERVE_MAX)
        throw PgxError{PGX_ERR_CAPACITY, std::to_string(cands) + " candidate triangles are more than a call's list can hold"};
    b.reserve(pairs, cands, w.nConvex > 0);
}

void np_mtd_launch(World& w, const MtdArgs& A) {
    const ConvexView cv{w.cvVerts.p, w.cvMesh.p, w.cvFace.p, w.cvFaceIdx.p, w.cvFaceN.p, w.cvFaceC.p};
    hipLaunchKernelGGL(k_mtd_walk, dim3(div_up(A.n, 64)), dim3(64), 0, w.stream, A, cv);
    PGX_LAUNCH_CHECK();
    if (w.nConvex > 0) {
        hipLaunchKernelGGL(k_mtd_convex, dim3(CONVEX_WAVES), dim3(64), 0, w.stream, A, cv);
        PGX_LAUNCH_CHECK();
    }
    if (w.nTriMesh > 0) {
        MeshArgs M = mesh_args(w, w.qMesh);
        M.nPairs = A.counts + 2; M.maxPairs = A.listCap; M.queryPairs = A.meshPairs;
        M.qPrm = A.qPrm; M.qPos = A.qPos; M.qQuat = A.qQuat; M.qType = A.qType;
        M.errors = A.counts + 3; M.candTotal = A.counts + 4; M.hitTotal = A.counts + 5;
        mesh_passes<true>(w, M);
        hipLaunchKernelGGL(w.nConvex > 0 ? k_mtd_mesh_emit<true> : k_mtd_mesh_emit<false>, dim3(MESH_BLOCKS),
                           dim3(MESH_BLOCK_WAVES * 64), 0, w.stream, M, A);
        PGX_LAUNCH_CHECK();
    }
}

// the overlap queries' pairs with a convex mesh (GJK), a fixed grid of `lanes` threads;
// each hit appends its key and adds to its query's count
__global__ __launch_bounds__(64) void k_overlap_convex(OverlapArgs A, int lanes) {
    const int lane = blockIdx.x * blockDim.x + threadIdx.x;
    if (lane >= lanes) return;
    const int n = min(*A.nCvx, A.listCap);
    for (int h = lane; h < n; h += lanes) {
        const int2 qc = A.cvxPairs[h];
        const int i = qc.x, c = qc.y;
        const float4 pw = A.qPos[i];
        const int b = A.cbody[c];
        const qf bq = q4(A.bquat[b]);
        const f3 cp = add(xyz(A.bpos[b]), qrot(bq, xyz(A.clpos[c])));
        if (!overlap_shapes(A.qType[i], A.qPrm[i], xyz(pw), q4(A.qQuat[i]), A.ctype[c], A.cparams[c], cp,
                            qmul(bq, q4(A.clquat[c])), A.cv))
            continue;
        const int slot = atomicAdd(A.total, 1);
        if (slot < A.cap) A.keys[slot] = ((uint64_t)(uint32_t)i << A.cbits) | (uint32_t)c;
        atomicAdd(A.count + i, 1);
    }
}

void np_overlap_launch(hipStream_t s, const OverlapArgs& A, bool convex) {
    hipLaunchKernelGGL(k_overlap, dim3(div_up(A.n, 64)), dim3(64), 0, s, A);
    PGX_LAUNCH_CHECK();
    if (convex) {
        constexpr int lanes = 16384;
        hipLaunchKernelGGL(k_overlap_convex, dim3(lanes / 64), dim3(64), 0, s, A, lanes);
        PGX_LAUNCH_CHECK();
    }
}

void np_run(World& w, int nPairs) {
    if (w.hasTriggers) {   // this step's list: its pair and hit counts start at zero
        // every trigger pair and hit has a pair slot: the lists must hold pairCap entries
        if (w.trigList.n < (size_t)w.pairCap || w.trigKeys[0].n < (size_t)w.pairCap ||
            w.trigKeys[1].n < (size_t)w.pairCap || w.trigN.n < 4)
            throw PgxError{PGX_ERR_HIP, "trigger lists smaller than the pair capacity"};
        w.trigCur ^= 1;
        fill_i32(w.stream, w.trigN.p + 2 * w.trigCur, 0, 2);
    }
    if (nPairs == 0) return;
    const int ppl = std::max(1, w.tune.pairsPerLane);
    w.npOrder.alloc(w.pairCap);
    if (nPairs <= NP_ORDER_SMALL) {   // the pairs come unsorted (bp_find_pairs)
        hipLaunchKernelGGL(k_pair_order, dim3(1), dim3(rs_threads(nPairs)), 0, w.stream, nPairs, rs_item_count(nPairs),
                           w.worldBits + 2 * w.localBits, w.pkeys.p, w.localBits, w.worldColStart.p, w.colOfLocal.p,
                           w.ctype.p, w.npOrder.p);
        PGX_LAUNCH_CHECK();
    } else {
        w.npClass.alloc(w.pairCap);
        hipLaunchKernelGGL(k_pair_class, dim3(div_up(nPairs, 256)), dim3(256), 0, w.stream, nPairs, w.pkeys.p, w.localBits,
                           w.worldColStart.p, w.colOfLocal.p, w.ctype.p, w.npClass.p, w.npOrder.p);
        PGX_LAUNCH_CHECK();
        radix_sort_u64(w.stream, w.npClass.p, w.npOrder.p, nPairs, 4, w.sortT);   // stable: slot order within a class
    }
    hipLaunchKernelGGL(k_narrowphase, dim3(div_up(nPairs, 256 * ppl)), dim3(256), 0, w.stream, nPairs, w.npOrder.p,
                       w.pkeys.p,
                       w.localBits, w.worldColStart.p, w.colOfLocal.p, w.cbody.p, w.ctype.p, w.cflags.p,
                       w.cparams.p, w.clpos.p, w.clquat.p, w.centity.p, w.bpos.p, w.bquat.p, w.nonColliding.p,
                       w.nNonColliding, w.npNum.p, w.npNormal.p, w.npPts.p, w.heavy.p, w.counters.p + 8,
                       w.meshPairs.p, w.counters.p + 10, w.meshCount.p,
                       w.hasTriggers ? w.trigList.p : nullptr, w.trigN.p + 2 * w.trigCur, w.filterClass.p,
                       w.filterTable.p, w.filterK, w.counters.p + 4, w.heavy.p + w.pairCap);
    PGX_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_box_faces, dim3(std::min(div_up(nPairs, BOX_GROUPS), BOX_BLOCKS)), dim3(256), 0, w.stream,
                       w.counters.p + 4, w.heavy.p + w.pairCap, w.pkeys.p, w.localBits, w.worldColStart.p, w.colOfLocal.p,
                       w.cbody.p, w.cparams.p, w.clpos.p, w.clquat.p, w.bpos.p, w.bquat.p, w.npNum.p, w.npNormal.p,
                       w.npPts.p);
    PGX_LAUNCH_CHECK();
    if (w.hasTriggers) {
        ConvexView cv{w.cvVerts.p, w.cvMesh.p, w.cvFace.p, w.cvFaceIdx.p, w.cvFaceN.p, w.cvFaceC.p};
        hipLaunchKernelGGL(k_triggers, dim3(std::min(div_up(nPairs, 64), 1024)), dim3(64), 0, w.stream,
                           w.trigN.p + 2 * w.trigCur, w.trigList.p, w.pkeys.p, w.localBits, w.worldColStart.p,
                           w.colOfLocal.p, w.cbody.p, w.ctype.p, w.cparams.p, w.clpos.p, w.clquat.p, w.bpos.p,
                           w.bquat.p, cv, w.trigN.p + 2 * w.trigCur + 1, w.trigKeys[w.trigCur].p);
        PGX_LAUNCH_CHECK();
    }
    if (w.nConvex > 0) {
        ConvexView cv{w.cvVerts.p, w.cvMesh.p, w.cvFace.p, w.cvFaceIdx.p, w.cvFaceN.p, w.cvFaceC.p};
        hipLaunchKernelGGL(k_narrowphase_convex, dim3(CONVEX_WAVES), dim3(64), 0, w.stream,
                           w.counters.p + 8, w.heavy.p, w.pkeys.p, w.localBits, w.worldColStart.p, w.colOfLocal.p,
                           w.cbody.p, w.ctype.p, w.cparams.p, w.clpos.p, w.clquat.p, w.bpos.p, w.bquat.p, cv,
                           w.npNum.p, w.npNormal.p, w.npPts.p, w.counters.p + 9);
        PGX_LAUNCH_CHECK();
    }
    if (w.nTriMesh > 0) {
        MeshArgs A = mesh_args(w, w.stepMesh);
        A.nPairs = w.counters.p + 10; A.maxPairs = w.pairCap; A.stepPairs = w.meshPairs.p;
        A.errors = w.counters.p + 12; A.candTotal = w.counters.p + 13; A.hitTotal = w.counters.p + 2;
        mesh_passes<false>(w, A);
        hipLaunchKernelGGL(w.nConvex > 0 ? k_mesh_emit<true> : k_mesh_emit<false>, dim3(MESH_BLOCKS),
                           dim3(MESH_BLOCK_WAVES * 64), 0, w.stream, A,
                           w.npNum.p, w.npNormal.p, w.npPts.p, w.npTri.p, w.meshFirst.p, w.meshCount.p,
                           w.counters.p + 11, w.mmCap, w.pairCap);
        PGX_LAUNCH_CHECK();
    }
}

int np_trigger_events(World& w, int cap, int32_t* enter, int32_t* nEnter, int32_t* exit, int32_t* nExit) {
    *nEnter = 0;
    *nExit = 0;
    if (!w.hasTriggers) return PGX_OK;
    hipStream_t s = w.stream;
    int32_t n[4];
    PGX_HIP(hipMemcpyAsync(n, w.trigN.p, sizeof n, hipMemcpyDeviceToHost, s));
    PGX_HIP(hipStreamSynchronize(s));
    const int cur = w.trigCur, prev = cur ^ 1;
    std::vector<uint64_t> a((size_t)n[2 * cur + 1]), b((size_t)n[2 * prev + 1]);
    if (!a.empty()) PGX_HIP(hipMemcpyAsync(a.data(), w.trigKeys[cur].p, 8 * a.size(), hipMemcpyDeviceToHost, s));
    if (!b.empty()) PGX_HIP(hipMemcpyAsync(b.data(), w.trigKeys[prev].p, 8 * b.size(), hipMemcpyDeviceToHost, s));
    PGX_HIP(hipStreamSynchronize(s));
    std::sort(a.begin(), a.end());
    std::sort(b.begin(), b.end());
    std::vector<uint64_t> en, ex;
    std::set_difference(a.begin(), a.end(), b.begin(), b.end(), std::back_inserter(en));   // src/Physecs.cpp:538-544
    std::set_difference(b.begin(), b.end(), a.begin(), a.end(), std::back_inserter(ex));   // :545-551
    const uint64_t lmask = (1ull << w.localBits) - 1;
    auto decode = [&](const std::vector<uint64_t>& keys) {
        std::vector<std::pair<int32_t, int32_t>> out;
        for (uint64_t k : keys) {
            const int base = w.hostWorldColStart[(size_t)(k >> (2 * w.localBits))];
            out.push_back({w.hostColOfLocal[base + (int)((k >> w.localBits) & lmask)],
                           w.hostColOfLocal[base + (int)(k & lmask)]});
        }
        std::sort(out.begin(), out.end());
        return out;
    };
    const auto pe = decode(en), px = decode(ex);
    *nEnter = (int32_t)pe.size();
    *nExit = (int32_t)px.size();
    if ((int)pe.size() > cap || (int)px.size() > cap) return PGX_ERR_CAPACITY;
    for (size_t i = 0; i < pe.size(); ++i) { enter[2 * i] = pe[i].first; enter[2 * i + 1] = pe[i].second; }
    for (size_t i = 0; i < px.size(); ++i) { exit[2 * i] = px[i].first; exit[2 * i + 1] = px[i].second; }
    return PGX_OK;
}

}  // namespace pgx
