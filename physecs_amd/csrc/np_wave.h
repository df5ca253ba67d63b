// The convex narrowphase with one wave per pair: GJK, EPA and the convex contact generators,
// operation for operation with the reference, their loops spread over the wave's 64 lanes.
//
// A pair is a chain of some ten support queries (GJK), up to a hundred EPA insertions of one
// support query, one pass over all faces and one horizon each, then a search over the hulls'
// faces and a polygon clip. With a lane per pair every one of these loops ran in series on
// global memory (the polytope was a 17.7 KB workspace per lane) while a scene's few thousand
// pairs left most of the chip idle: 534 us for 2.4 k pairs of 24-point hulls, and 3.0 ms for
// a few hundred capsules against hulls, whose EPA runs its hundred insertions. Here
// - a hull's vertices sit in the lanes' registers, a support query is one dot product per
//   lane, a wave maximum and a lane read;
// - the polytope is in LDS (14 KB per wave, 11 waves per CU): distances and visibility of 64
//   faces at a time, new faces one per lane, the horizon's edges in registers;
// - faces of a hull are searched, and polygon corners clipped, one per lane.
// The same pairs then take 44 us and 134 us. What is left is the longest pair's chain: some
// 1.3 us per insertion, of LDS reads, wave maxima and 64-bit distances that wait on each other.
// What every lane needs (simplex, directions, normals) is computed by all lanes alike, so
// control flow is the same in the whole wave; a kernel using this has blocks of one wave.
//
// The sequential loops' ties are kept: the first of equal values wins (in SupConvex the
// lowest vertex of the lowest class i % 4), edges keep the list order of EpaPolytope, and
// findClosestFace's float running minimum is reproduced from its final value (closest_face).
// Included by narrowphase.hip after np_convex.h.
#pragma once

namespace pgx {

// ------------------------------------------------------------------ wave primitives
__device__ __forceinline__ int wave_lane() { return (int)threadIdx.x & (WAVE - 1); }
// The wave's LDS stores before it are seen by its loads after it: a wave's LDS operations
// are performed in order, so this only keeps the compiler from moving them. Everything here
// is inlined into its kernel: through a pointer that has lost its address space the same
// accesses would be flat ones, which are not ordered with each other.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ float lane_read(float x, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}
__device__ __forceinline__ f3 lane_read(f3 v, int lane) {
    return mk3(lane_read(v.x, lane), lane_read(v.y, lane), lane_read(v.z, lane));
}
// floats in the order of ints (-0 below 0), and back
__device__ __forceinline__ int ordered(int bits) { return bits ^ ((bits >> 31) & 0x7fffffff); }
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_max(int x) {
    return max(x, __builtin_amdgcn_update_dpp(-2147483647 - 1, x, CTRL, ROWS, 0xf, false));
}
// the largest of the lanes' values (none a NaN), in every lane; as ints, whose maximum takes
// its lane move as an operand
__device__ __forceinline__ float wave_max(float v) {
    int x = ordered(__float_as_int(v));
    x = dpp_max<0x111, 0xf>(x);   // row_shr 1, 2, 4, 8: a row's maximum in its last lane
    x = dpp_max<0x112, 0xf>(x);
    x = dpp_max<0x114, 0xf>(x);
    x = dpp_max<0x118, 0xf>(x);
    x = dpp_max<0x142, 0xa>(x);   // row_bcast 15, then 31: the wave's in lane 63
    x = dpp_max<0x143, 0xc>(x);
    return __int_as_float(ordered(__builtin_amdgcn_readlane(x, WAVE - 1)));
}
// x with lane l's value replaced
__device__ __forceinline__ int lane_write(int value, int l, int x) {
    return (int)(threadIdx.x & (WAVE - 1)) == l ? value : x;
}
// exclusive prefix of n over the wave and the wave's total
__device__ __forceinline__ int wave_scan(int n, int& total) {
    const int lane = wave_lane();
    int incl = n;
    for (int o = 1; o < WAVE; o <<= 1) {
        int t = __shfl_up(incl, o);
        if (lane >= o) incl += t;
    }
    total = __shfl(incl, WAVE - 1);
    return incl - n;
}
__device__ __forceinline__ uint64_t lanes_below() { return (1ull << wave_lane()) - 1ull; }
__device__ __forceinline__ int first_lane(uint64_t mask) { return __ffsll((unsigned long long)mask) - 1; }
__device__ __forceinline__ int last_lane(uint64_t mask) { return 63 - __clzll((long long)mask); }

// `for (i < n) if (v[i] > best) { best = v[i]; at = i; }` from best = 0, at = 0, with v[lane]
// of n <= 64 elements
__device__ __forceinline__ int wave_first_max(float v, bool in) {
    const float m = wave_max(in && v > 0.f ? v : 0.f);
    return m > 0.f ? first_lane(__ballot(in && v == m)) : 0;
}

// ------------------------------------------------------------------ support maps
// SupConvex with vertex `lane` of the hull in the lane's register (vertices from 64 on are
// read from memory). count: the padded count, a multiple of 4.
struct SupHull {
    f3 pos; m3 l2w; f3 scale; const float4* v; int count;
    f3 mine;
    __device__ __forceinline__ void load() { mine = wave_lane() < count ? xyz(v[wave_lane()]) : s3(0.f); }
    __device__ __forceinline__ f3 operator()(f3 dir) const {
        constexpr float LOWEST = -3.402823466e+38f;
        dir = mulv(scale, mk3(dot(dir, l2w.c0), dot(dir, l2w.c1), dot(dir, l2w.c2)));
        const int lane = wave_lane();
        float d = LOWEST;
        int at = lane;
        if (lane < count) {
            const float e = (mine.x * dir.x + mine.y * dir.y) + mine.z * dir.z;
            if (e > d) d = e;
        }
        for (int i = lane + WAVE; i < count; i += WAVE) {   // of one class i % 4, ascending: the first largest stays
            const float4 p = v[i];
            const float e = (p.x * dir.x + p.y * dir.y) + p.z * dir.z;
            if (e > d) { d = e; at = i; }
        }
        const float m = wave_max(d);
        int best = 0;
        if (m > LOWEST) {
            const uint64_t eq = __ballot(d == m);
            uint64_t cls = 0;
#pragma unroll
            for (int k = 3; k >= 0; --k) {
                const uint64_t c = eq & (0x1111111111111111ull << k);
                if (c) cls = c;
            }
            if (count <= WAVE) {
                best = first_lane(cls);
            } else {   // the lowest vertex among the class's lanes
                const bool in = (cls >> lane) & 1ull;
                best = -(int)wave_max(in ? -(float)at : LOWEST);
            }
        }
        const f3 p = best < WAVE ? lane_read(mine, best) : xyz(v[best]);
        return add(pos, mulmv(l2w, mulv(scale, p)));
    }
};
__device__ __forceinline__ SupHull hull_of(const SupConvex& s) {
    SupHull h{s.pos, s.l2w, s.scale, s.v, (s.count + 3) & ~3, s3(0.f)};
    h.load();
    return h;
}

// Any shape on side 0 of a pair (the same in the whole wave), so that a kernel holds one GJK
// and one EPA, not one per shape. g: sphere (r), capsule (half height, r; hull.l2w.c0 its
// axis), box (half extents).
struct SupSide {
    int type;
    SupHull hull;
    f3 g;
    __device__ __forceinline__ f3 operator()(f3 d) const {
        if (type == PGX_CONVEX_MESH) return hull(d);
        if (type == PGX_SPHERE) return SupSphere{hull.pos, g.x}(d);
        if (type == PGX_CAPSULE) return SupCapsule{hull.pos, hull.l2w.c0, g.x, g.y}(d);
        return SupBox{hull.pos, hull.l2w, g}(d);
    }
};

// ------------------------------------------------------------------ GJK
// a simplex vertex; every coordinate is a float widened to double where it is used
struct GV { f3 pos, sp0, sp1; };
__device__ __forceinline__ GV pick(bool c, const GV& a, const GV& b) {
    GV r;
    r.pos = mk3(c ? a.pos.x : b.pos.x, c ? a.pos.y : b.pos.y, c ? a.pos.z : b.pos.z);
    r.sp0 = mk3(c ? a.sp0.x : b.sp0.x, c ? a.sp0.y : b.sp0.y, c ? a.sp0.z : b.sp0.z);
    r.sp1 = mk3(c ? a.sp1.x : b.sp1.x, c ? a.sp1.y : b.sp1.y, c ? a.sp1.z : b.sp1.z);
    return r;
}
__device__ __forceinline__ GV lane_read(const GV& g, int lane) {
    return GV{lane_read(g.pos, lane), lane_read(g.sp0, lane), lane_read(g.sp1, lane)};
}
template <class S0, class S1>
__device__ __forceinline__ GV mdiff_w(const S0& s0, const S1& s1, f3 dir) {
    GV r;
    r.sp0 = s0(dir);
    r.sp1 = s1(neg(dir));
    r.pos = sub(r.sp0, r.sp1);
    return r;
}
// gjk (np_convex.h) with the simplex in named vertices (no indexed access, no scratch) and
// its support queries answered at one place in the code: written out where the algorithm asks
// them, they are eleven copies of both support maps, and as fast (both within 2 us of each
// other on 2.4 k hull pairs).
template <class S0, class S1>
__device__ __forceinline__ bool gjk_w(const S0& s0, const S1& s1, f3 startDir, GV& a, GV& b, GV& c, GV& d) {
    // what the answer is for
    enum { FIRST, SECOND_ZERO, SECOND, THIRD, LINE_THIRD, LINE_THIRD_BACK, LAST, LAST_BACK, FOURTH, LOOP };
    int ask = FIRST, fi = 0, rounds = 0;
    d3 dir = wide(normalize(startDir)), plain = dir;   // plain: a direction before its normalisation
    bool unit = true;                                  // dir is used as it is
    while (true) {
        if (!unit) dir = dnormalize(dir);
        const GV v = mdiff_w(s0, s1, narrow(dir));
        // checkDirection (src/GJK.h:162-167) of the queries that must pass the origin
        if ((ask == SECOND || ask == THIRD || ask == FOURTH || ask == LOOP) && !(ddot(wide(v.pos), dir) >= 0)) return false;
        unit = false;
        bool line = false, last = false;               // go on with the third vertex of a line, with the last one
        switch (ask) {
            case FIRST:
                a = v;
                if (is_zero(a.pos)) {
                    dir = dneg(dir);
                    unit = true;
                    ask = SECOND_ZERO;
                } else {
                    dir = dneg(wide(a.pos));
                    ask = SECOND;
                }
                break;
            case SECOND_ZERO:
                b = v;
                line = true;
                break;
            case SECOND: {
                b = v;
                const d3 ab = dsub(wide(a.pos), wide(b.pos));
                dir = dcross(dcross(ab, dneg(wide(b.pos))), ab);
                if (is_zero(narrow(dir))) line = true;
                else ask = THIRD;
                break;
            }
            case THIRD: {
                c = v;
                dir = dcross(dsub(wide(b.pos), wide(a.pos)), dsub(wide(c.pos), wide(a.pos)));
                const double sg = dsign(ddot(dneg(wide(a.pos)), dir));
                if (!sg) {
                    ask = LAST;
                } else {
                    dir = dmul(sg, dir);
                    ask = FOURTH;
                }
                break;
            }
            case LINE_THIRD:
                c = v;
                if (sqr_dist_point_line(c.pos, a.pos, b.pos) < 0.00001f) {
                    dir = dneg(plain);
                    unit = true;
                    ask = LINE_THIRD_BACK;
                } else {
                    last = true;
                }
                break;
            case LINE_THIRD_BACK:
                c = v;
                last = true;
                break;
            case LAST:
                d = v;
                if (!(dist_point_plane(d.pos, a.pos, narrow(dir)) < 0.0001f)) return true;
                dir = dneg(dir);
                unit = true;
                ask = LAST_BACK;
                break;
            case LAST_BACK:
                d = v;
                return true;
            case FOURTH:
                d = v;
                ask = LOOP;
                break;
            default: {   // the new vertex replaces vertex fi, then changes places with vertex 3
                a = pick(fi == 0, d, a);
                b = pick(fi == 1, d, b);
                c = pick(fi == 2, d, c);
                d = v;
                break;
            }
        }
        if (line) {   // complete_from_line, src/GJK.h:233-243
            const d3 ab = dsub(wide(a.pos), wide(b.pos));
            dir = dcross(ab, mkd(0, 1, 0));
            if (is_zero(narrow(dir))) dir = dcross(ab, mkd(0, 0, 1));
            plain = dir;
            ask = LINE_THIRD;
        } else if (last) {
            dir = dcross(dsub(wide(b.pos), wide(a.pos)), dsub(wide(c.pos), wide(a.pos)));
            ask = LAST;
        } else if (ask == LOOP) {   // simplexContainsOrigin (src/GJK.h:175-181)
            if (rounds++ == 100) return false;
            const d3 pa = wide(a.pos), pb = wide(b.pos), pc = wide(c.pos), pd = wide(d.pos);
            fi = 2;
            bool outside = check_face(pd, pa, pb, pc, dir);
            if (!outside) { fi = 1; outside = check_face(pd, pc, pa, pb, dir); }
            if (!outside) { fi = 0; outside = check_face(pd, pb, pc, pa, dir); }
            if (!outside) return true;
        }
    }
}

// ------------------------------------------------------------------ EPA
// a clipped polygon's corners
struct WavePoly {
    f2 poly[CVX_MAXPOLY];
    f3 pen[CVX_MAXPOLY];
};
// and EPA's polytope
struct WaveMem : WavePoly {
    double n[4][EPA_MAXF];        // per face: unit normal, and its distance (EPA.h:41-43)
    float v[EPA_MAXV * 9];        // per vertex: pos, sp0, sp1
    int fi[EPA_MAXF];             // per face: its vertices, a byte each
};
static_assert(EPA_MAXV < 256 && EPA_MAXE == 2 * WAVE, "a vertex in a byte, edges in two registers");

__device__ __forceinline__ d3 mem_pos(const WaveMem& M, int i) {
    return mkd(M.v[9 * i], M.v[9 * i + 1], M.v[9 * i + 2]);
}
__device__ __forceinline__ GV mem_vertex(const WaveMem& M, int i) {
    const float* p = M.v + 9 * i;
    return GV{mk3(p[0], p[1], p[2]), mk3(p[3], p[4], p[5]), mk3(p[6], p[7], p[8])};
}
__device__ __forceinline__ void mem_put(WaveMem& M, int i, const GV& g) {
    float* p = M.v + 9 * i;
    p[0] = g.pos.x; p[1] = g.pos.y; p[2] = g.pos.z;
    p[3] = g.sp0.x; p[4] = g.sp0.y; p[5] = g.sp0.z;
    p[6] = g.sp1.x; p[7] = g.sp1.y; p[8] = g.sp1.z;
}
__device__ __forceinline__ d3 mem_normal(const WaveMem& M, int f) { return mkd(M.n[0][f], M.n[1][f], M.n[2][f]); }
// EPA.h:24-34, one face per lane
__device__ __forceinline__ void mem_face(WaveMem& M, int f, int i0, int i1, int i2) {
    const d3 p0 = mem_pos(M, i0), p1 = mem_pos(M, i1), p2 = mem_pos(M, i2);
    d3 n = dcross(dsub(p0, p1), dsub(p2, p1));
    const double len = dlength(n);
    if (len) n = ddivs(n, len);
    M.fi[f] = i0 | (i1 << 8) | (i2 << 16);
    M.n[0][f] = n.x; M.n[1][f] = n.y; M.n[2][f] = n.z;
    M.n[3][f] = ddot(p0, n);
}

// src/EPA.h:9-186 over the wave
template <class S0, class S1>
__device__ __forceinline__ f3 epa_w(const S0& s0, const S1& s1, const GV& a, const GV& b, const GV& c, const GV& d, WaveMem& M,
                    f3& cp0, f3& cp1, bool& overflow) {
    const int lane = wave_lane();
    overflow = false;
    int nv = 4, nf = 4;
    if (lane < 4) mem_put(M, lane, pick(lane < 2, pick(lane == 0, a, b), pick(lane == 2, c, d)));
    wave_sync();
    {   // EpaPolytope(GjkSimplex&), src/EPA.h:50-66: a vertex index per byte, a face per lane
        const d3 pa = wide(a.pos), pb = wide(b.pos);
        const d3 n = dcross(dsub(pa, pb), dsub(wide(c.pos), pb));
        const bool in = ddot(dsub(wide(d.pos), pa), n) < 0;
        const int faces[4] = {in ? 0x020100 : 0x010200, in ? 0x000103 : 0x000203, in ? 0x010203 : 0x020103,
                              in ? 0x020003 : 0x010003};
        const int f = lane == 0 ? faces[0] : lane == 1 ? faces[1] : lane == 2 ? faces[2] : faces[3];
        if (lane < 4) mem_face(M, lane, f & 255, (f >> 8) & 255, f >> 16);
    }
    wave_sync();
    float minDist = 0.f;
    d3 normal = mkd(0, 0, 0);
    int faceIndex = 0;
    for (int it = 0; it < 100 && !overflow; ++it) {
        // findClosestFace (:68-79): a float running minimum m, a face taken when its double
        // distance is below m, m then rounded from it. m only falls and ends at the least
        // rounded distance; a face of that rounded distance is taken when it is the first
        // (m was above) or when its distance itself is below m (rounding was upward): the
        // last of these, or else the first, is the one left. None when nothing is below inf.
        float low = __builtin_inff();
        int taken = -1, first = -1;
        double dist = __builtin_inf();
        if (lane < nf) dist = M.n[3][lane];
        low = fminf(low, (float)dist);
        for (int f = WAVE + lane; f < nf; f += WAVE) low = fminf(low, (float)M.n[3][f]);
        minDist = -wave_max(-low);
        for (int k = 0; k < nf; k += WAVE) {
            if (k) dist = k + lane < nf ? M.n[3][k + lane] : __builtin_inf();
            const uint64_t below = __ballot(dist < (double)minDist);
            if (below) taken = k + last_lane(below);
            const uint64_t same = __ballot(k + lane < nf && (float)dist == minDist);
            if (same && first < 0) first = k + first_lane(same);
        }
        if (taken < 0 && minDist < __builtin_inff()) taken = first;
        if (taken >= 0) {
            faceIndex = taken;
            normal = mem_normal(M, taken);
        }
        const GV v = mdiff_w(s0, s1, narrow(normal));
        if (__ballot(ddot(wide(v.pos), normal) - (double)minDist < (double)0.00001f)) break;
        // insertVertex (:81-120)
        if (nv >= EPA_MAXV) { overflow = true; break; }
        // the faces that see the vertex, from the last to the first; the last face fills each
        // one's place (it comes later, so it has been looked at: the faces still to come are in
        // their places). Up to 64 faces only note where each place's face comes from.
        int ne = 0, e0 = -1, e1 = -1;   // edge k in lane k & 63 of e0 or e1: first | second << 8
        const bool small = nf <= WAVE;
        int source = lane;
        for (int k = (nf - 1) & ~(WAVE - 1); k >= 0; k -= WAVE) {
            bool see = false;
            int ixs = 0;
            if (k + lane < nf) {
                ixs = M.fi[k + lane];
                see = ddot(mem_normal(M, k + lane), dsub(wide(v.pos), mem_pos(M, ixs & 255))) > 0;
            }
            for (uint64_t seen = __ballot(see); seen;) {
                const int l = last_lane(seen);
                seen &= ~(1ull << l);
                const int f = k + l, ix = __builtin_amdgcn_readlane(ixs, l);
                const int v0 = ix & 255, v1 = (ix >> 8) & 255, v2 = ix >> 16;
                const int edge[3] = {v0 | (v1 << 8), v1 | (v2 << 8), v2 | (v0 << 8)};
                const int back[3] = {v1 | (v0 << 8), v2 | (v1 << 8), v0 | (v2 << 8)};
                bool found[3];
#pragma unroll
                for (int j = 0; j < 3; ++j) {   // a found edge's place is taken by the last one
                    const uint64_t lo = __ballot(e0 == back[j]);
                    if (ne <= WAVE) {
                        found[j] = lo != 0;
                        if (lo) {
                            --ne;
                            e0 = lane_write(__builtin_amdgcn_readlane(e0, ne), last_lane(lo), e0);
                            e0 = lane_write(-1, ne, e0);
                        }
                    } else {
                        const uint64_t hi = __ballot(e1 == back[j]);
                        found[j] = (hi | lo) != 0;
                        if (hi | lo) {
                            --ne;
                            const int end = __builtin_amdgcn_readlane(e1, ne - WAVE);
                            if (hi) e1 = lane_write(end, last_lane(hi), e1);
                            else e0 = lane_write(end, last_lane(lo), e0);
                            e1 = lane_write(-1, ne - WAVE, e1);
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    if (found[j]) continue;
                    if (ne >= EPA_MAXE) { overflow = true; break; }
                    if (ne < WAVE) e0 = lane_write(edge[j], ne, e0);
                    else e1 = lane_write(edge[j], ne - WAVE, e1);
                    ++ne;
                }
                --nf;
                if (f == nf) continue;
                if (small) {
                    source = lane_write(__builtin_amdgcn_readlane(source, nf), f, source);
                } else {
                    if (lane < 4) M.n[lane][f] = M.n[lane][nf];
                    else if (lane == 4) M.fi[f] = M.fi[nf];
                    wave_sync();
                }
            }
        }
        if (small && __ballot(lane < nf && source != lane)) {
            const bool moved = lane < nf && source != lane;
            const d3 n = mem_normal(M, source);
            const double dn = M.n[3][source];
            const int ix = M.fi[source];
            wave_sync();
            if (moved) {
                M.n[0][lane] = n.x; M.n[1][lane] = n.y; M.n[2][lane] = n.z;
                M.n[3][lane] = dn;
                M.fi[lane] = ix;
            }
        }
        const int vi = nv++;
        if (lane == 0) mem_put(M, vi, v);
        wave_sync();
        if (nf + ne > EPA_MAXF) { overflow = true; break; }
        for (int k = lane; k < ne; k += WAVE) {
            const int e = k < WAVE ? e0 : e1;
            mem_face(M, nf + k, vi, e & 255, e >> 8);
        }
        nf += ne;
        wave_sync();
    }
    // getClosestPoints (:122-168), including proj = normal + distance (:133)
    const int ix = M.fi[faceIndex];
    const GV ga = mem_vertex(M, ix & 255), gb = mem_vertex(M, (ix >> 8) & 255), gc = mem_vertex(M, ix >> 16);
    const d3 pa = wide(ga.pos);
    const d3 proj = dadds(mem_normal(M, faceIndex), M.n[3][faceIndex]);
    const f3 v0 = narrow(dsub(wide(gb.pos), pa)), v1 = narrow(dsub(wide(gc.pos), pa)), v2 = narrow(dsub(proj, pa));
    const double d00 = dot(v0, v0), d01 = dot(v0, v1), d11 = dot(v1, v1), d20 = dot(v2, v0), d21 = dot(v2, v1);
    const double denom = d00 * d11 - d01 * d01;
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
    cp0 = narrow(dadd(dadd(dmul(u, wide(ga.sp0)), dmul(vv, wide(gb.sp0))), dmul(w, wide(gc.sp0))));
    cp1 = narrow(dadd(dadd(dmul(u, wide(ga.sp1)), dmul(vv, wide(gb.sp1))), dmul(w, wide(gc.sp1))));
    wave_sync();   // the polytope is read before the wave's next pair overwrites it
    return narrow(normal);
}

// ------------------------------------------------------------------ contact generation
// the face of a hull whose value(face) is largest and above 0, the first of equals (0 if none)
template <class F>
__device__ __forceinline__ int wave_face(int n, F value) {
    float best = 0.f;
    int at = 0;
    for (int i = wave_lane(); i < n; i += WAVE) {
        const float d = value(i);
        if (d > best) { best = d; at = i; }
    }
    const float m = wave_max(best);
    if (!(m > 0.f)) return 0;
    if (n <= WAVE) return first_lane(__ballot(best == m));
    return -(int)wave_max(best == m ? -(float)at : -3.402823466e+38f);
}

// clipPolygon (src/Clipping.cpp:21-53), at most CVX_MAXPOLY corners, with corner `lane` of the polygon (n of them)
// and of the clip polygon (nclip) in the lanes
__device__ __forceinline__ void wave_clip(f2& p, int& n, f2 clip, int nclip, WavePoly& M) {
    const int lane = wave_lane();
    const uint64_t lt = lanes_below();
    for (int e = 0; e < nclip; ++e) {
        const int e2 = e + 1 == nclip ? 0 : e + 1;
        const f2 a = mk2(lane_read(clip.x, e), lane_read(clip.y, e));
        const f2 b = mk2(lane_read(clip.x, e2), lane_read(clip.y, e2));
        const int j = lane + 1 >= n ? 0 : lane + 1;
        const f2 q = mk2(__shfl(p.x, j), __shfl(p.y, j));
        const bool in = lane < n, ii = in && inside(p, a, b), ji = in && inside(q, a, b);
        const uint64_t one = __ballot(ii || ji), two = __ballot(!ii && ji);
        const int at = (int)__popcll(one & lt) + (int)__popcll(two & lt);
        if (ii || ji) {
            const f2 x = intersect2(p, q, a, b);
            if (at < CVX_MAXPOLY) M.poly[at] = ii && ji ? q : x;
            if (!ii && at + 1 < CVX_MAXPOLY) M.poly[at + 1] = q;
        }
        n = min((int)__popcll(one) + (int)__popcll(two), CVX_MAXPOLY);
        wave_sync();
        if (lane < n) p = M.poly[lane];
        wave_sync();
    }
}

// A face of one shape clipped against a face of the other: corner `lane` of the incident
// polygon and of the clip polygon in the reference face's plane, and the frame that the
// contacts are taken back from. polygon_box_face_contacts (src/ContactsUtil.cpp:9-107) takes
// the plane of a box's axis; polygon_polygon_face_contacts (:109-204) is the same arithmetic
// for axis y, sign 1, plane (z, x) and the face's distance in place of the half extent.
struct FaceClip {
    f2 p, clip;
    int n, nclip;
    f3 refPos, incOrig, incNormal, he;
    m3 basis;
    int axis, axisSign;
    __device__ __forceinline__ void polygon_frame(f3 pos, const m3& refToWorld, f3 refOrig, f3 refNormal) {
        refPos = pos;
        basis = refToWorld;
        he = s3(dot(refOrig, refNormal));
        axis = 1;
        axisSign = 1;
    }
};

__device__ __forceinline__ void wave_contacts(FaceClip& F, WavePoly& M, CPt* cps, int& numPoints) {
    wave_clip(F.p, F.n, F.clip, F.nclip, M);
    const int axis = F.axis, cx = (axis + 1) % 3, cy = (axis + 2) % 3, lane = wave_lane();
    const float lim = at(F.he, axis);
    f3 dir = s3(0.f), p3 = s3(0.f);
    set(dir, axis, (float)F.axisSign);
    const float denom = dot(dir, F.incNormal);
    set(p3, cx, F.p.x);
    set(p3, cy, F.p.y);
    const float distance = dot(sub(F.incOrig, p3), F.incNormal) / denom;
    const bool keep = lane < F.n && distance < lim + 1e-4f;
    set(p3, axis, F.axisSign * distance);
    // the penetrating corners, in order
    const uint64_t mask = __ballot(keep);
    const int np = (int)__popcll(mask);
    if (keep) M.pen[__popcll(mask & lanes_below())] = p3;
    wave_sync();
    const f3 pen = lane < np ? M.pen[lane] : s3(0.f);
    wave_sync();
    int pick0 = 0, pick1 = 1, pick2 = 2, pick3 = 3;   // the up to four that become contacts
    numPoints = np;
    if (np > 4) {
        const f3 p0 = lane_read(pen, 0), d = sub(pen, p0);
        pick1 = wave_first_max(dot(d, d), lane < np);
        const f3 ca = sub(p0, pen), cb = sub(lane_read(pen, pick1), pen);
        const float area = det2(mk2(at(ca, cx), at(ca, cy)), mk2(at(cb, cx), at(cb, cy)));
        pick2 = wave_first_max(area, lane < np);
        pick3 = wave_first_max(-area, lane < np);
        numPoints = 4;
    }
    // contact `lane` in lanes 0-3, then in every lane
    const f3 c = mk3(__shfl(pen.x, lane == 0 ? pick0 : lane == 1 ? pick1 : lane == 2 ? pick2 : pick3),
                     __shfl(pen.y, lane == 0 ? pick0 : lane == 1 ? pick1 : lane == 2 ? pick2 : pick3),
                     __shfl(pen.z, lane == 0 ? pick0 : lane == 1 ? pick1 : lane == 2 ? pick2 : pick3));
    f3 on = c;
    set(on, axis, F.axisSign * lim);
    const f3 a = add(F.refPos, mulmv(F.basis, on)), b = add(F.refPos, mulmv(F.basis, c));
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < numPoints) {
            cps[i].p0 = lane_read(a, i);
            cps[i].p1 = lane_read(b, i);
        }
}

// vertex `lane` of a face (face vertices beyond the face's count are not read)
__device__ __forceinline__ f3 lane_face_vert(const MeshRef& m, int2 F, int n) {
    return m.face_vert(F, wave_lane() < n ? wave_lane() : 0);
}

// convex_convex_contacts, src/Collision.cpp:352-410
__device__ __forceinline__ void convex_convex_clip(f3 pos0, qf or0, const MeshRef& m0, f3 s0, f3 pos1, qf or1,
                                                   const MeshRef& m1, f3 s1, f3 normal, FaceClip& F) {
    const int f0 = wave_face(m0.nfaces(), [&](int i) { return dot(normal, world_face_normal(or0, m0.fnormal(i), s0)); });
    const int f1 = wave_face(m1.nfaces(), [&](int i) { return -dot(normal, world_face_normal(or1, m1.fnormal(i), s1)); });
    const int2 F0 = m0.face(f0), F1 = m1.face(f1);
    const m3 worldToC0 = transpose(mat3_cast(or0));
    const f3 refOrig = mulv(s0, m0.fcentroid(f0));
    const f3 u0 = normalize(sub(mulv(s0, m0.face_vert(F0, 0)), refOrig));
    const f3 u1 = normalize(divv(m0.fnormal(f0), s0));
    const f3 u2 = cross(u0, u1);
    const m3 c0ToRef = transpose(mk_m3(u0, u1, u2));
    const m3 worldToRef = mulmm(c0ToRef, worldToC0);
    F.nclip = F0.y < 16 ? F0.y : 16;
    F.n = F1.y < 16 ? F1.y : 16;
    const f3 cv = mulmv(c0ToRef, mulv(s0, lane_face_vert(m0, F0, F.nclip)));
    const f3 pv = mulmv(worldToRef, sub(add(pos1, qrot(or1, mulv(s1, lane_face_vert(m1, F1, F.n)))), pos0));
    F.p = mk2(pv.z, pv.x);
    F.clip = mk2(cv.z, cv.x);
    F.incOrig = mulmv(worldToRef, sub(add(pos1, qrot(or1, mulv(s1, m1.fcentroid(f1)))), pos0));
    F.incNormal = mulmv(worldToRef, qrot(or1, normalize(divv(m1.fnormal(f1), s1))));
    F.polygon_frame(pos0, transpose(worldToRef), refOrig, u1);
}

// capsule_convex_contacts, src/Collision.cpp:694-785
__device__ __forceinline__ void capsule_convex_contacts_w(f3 p0L, f3 p1L, float radius, f3 meshPos, const m3& c2w, const MeshRef& m,
                                          f3 scale, Mf& res) {
    const int fi = wave_face(m.nfaces(), [&](int i) { return -dot(res.normal, normalize(mulmv(c2w, divv(m.fnormal(i), scale)))); });
    const int2 F = m.face(fi);
    const f3 refOrig = mulv(scale, m.fcentroid(fi));
    const f3 u0 = normalize(sub(mulv(scale, m.face_vert(F, 0)), refOrig));
    const f3 u1 = normalize(divv(m.fnormal(fi), scale));
    const f3 u2 = cross(u0, u1);
    const m3 convexToRef = transpose(mk_m3(u0, u1, u2));
    const int nc = F.y < 16 ? F.y : 16;
    const f3 cv = mulmv(convexToRef, mulv(scale, lane_face_vert(m, F, nc)));
    const f3 p0Ref = mulmv(convexToRef, p0L), p1Ref = mulmv(convexToRef, p1L);
    f2 line0 = mk2(p0Ref.z, p0Ref.x), line1 = mk2(p1Ref.z, p1Ref.x);
    bool kept = true;   // clip_line_n
    for (int i = 0; i < nc && kept; ++i) {
        const int j = i + 1 == nc ? 0 : i + 1;
        const f2 a = mk2(lane_read(cv.z, i), lane_read(cv.x, i)), b = mk2(lane_read(cv.z, j), lane_read(cv.x, j));
        const bool in0 = inside(line0, a, b), in1 = inside(line1, a, b);
        if (in0 && in1) continue;
        if (in0) line1 = intersect2(line0, line1, a, b);
        else if (in1) line0 = intersect2(line0, line1, a, b);
        else kept = false;
    }
    res.numPoints = 0;
    if (!kept) return;
    const m3 refToWorld = mulmm(c2w, transpose(convexToRef));
    const float distToPlane = dot(refOrig, u1);
    float y0, y1;
    const float distX = p0Ref.z - p1Ref.z, distY = p0Ref.x - p1Ref.x;
    const float adx = gabs(distX), ady = gabs(distY);
    if (adx && adx >= ady) {
        y0 = gmix(p0Ref.y, p1Ref.y, (p0Ref.z - line0.x) / distX);
        y1 = gmix(p1Ref.y, p0Ref.y, (p1Ref.z - line1.x) / -distX);
    } else if (ady > adx) {
        y0 = gmix(p0Ref.y, p1Ref.y, (p0Ref.x - line0.y) / distY);
        y1 = gmix(p1Ref.y, p0Ref.y, (p1Ref.x - line1.y) / -distY);
    } else {
        y0 = p0Ref.y;
        y1 = p1Ref.y;
    }
    y0 -= radius;
    y1 -= radius;
    const bool k0 = y0 < distToPlane, k1 = y1 < distToPlane;
    const f3 a0 = add(meshPos, mulmv(refToWorld, mk3(line0.y, y0, line0.x)));
    const f3 a1 = add(meshPos, mulmv(refToWorld, mk3(line0.y, distToPlane, line0.x)));
    const f3 b0 = add(meshPos, mulmv(refToWorld, mk3(line1.y, y1, line1.x)));
    const f3 b1 = add(meshPos, mulmv(refToWorld, mk3(line1.y, distToPlane, line1.x)));
    if (k0) { res.pts[0].p0 = a0; res.pts[0].p1 = a1; }
    else if (k1) { res.pts[0].p0 = b0; res.pts[0].p1 = b1; }
    if (k0 && k1) { res.pts[1].p0 = b0; res.pts[1].p1 = b1; }
    res.numPoints = (k0 ? 1 : 0) + (k1 ? 1 : 0);
}

// the clip rectangle (hx, hy), (hx, -hy), (-hx, -hy), (-hx, hy) of a box's face
__device__ __forceinline__ f2 lane_rectangle(float hx, float hy) {
    const int lane = wave_lane();
    return mk2(lane < 2 ? hx : -hx, lane == 0 || lane == 3 ? hy : -hy);
}

// box_convex_contacts, src/Collision.cpp:808-871
__device__ __forceinline__ void box_convex_clip(f3 boxCenter, const m3& basis, f3 he, f3 cpos, qf cor, const MeshRef& m,
                                                f3 scale, f3 normal, FaceClip& F) {
    int boxAxis = 0;
    float boxAxisSign = 0.f, maxDot = 0.f;
    for (int i = 0; i < 3; ++i) {
        float d = dot(normal, col(basis, i));
        float ad = gabs(d);
        if (ad > maxDot) { maxDot = ad; boxAxis = i; boxAxisSign = d < 0 ? -1.f : 1.f; }
    }
    const int fi = wave_face(m.nfaces(), [&](int i) { return -dot(normal, world_face_normal(cor, m.fnormal(i), scale)); });
    const int2 Fc = m.face(fi);
    const int cx = (boxAxis + 1) % 3, cy = (boxAxis + 2) % 3;
    const m3 worldToBox = transpose(basis);
    F.n = Fc.y < 16 ? Fc.y : 16;
    const f3 v = mulmv(worldToBox, sub(add(cpos, qrot(cor, mulv(scale, lane_face_vert(m, Fc, F.n)))), boxCenter));
    F.p = mk2(at(v, cx), at(v, cy));
    F.clip = lane_rectangle(at(he, cx), at(he, cy));
    F.nclip = 4;
    F.incOrig = mulmv(worldToBox, sub(add(cpos, qrot(cor, mulv(scale, m.fcentroid(fi)))), boxCenter));
    F.incNormal = normalize(mulmv(worldToBox, qrot(cor, divv(m.fnormal(fi), scale))));
    F.refPos = boxCenter;
    F.basis = basis;
    F.he = he;
    F.axis = boxAxis;
    F.axisSign = (int)boxAxisSign;
}

// one pair with a convex mesh on either side (src/Collision.cpp:895-1016); flips as the
// reference's dispatcher does. The result is the same in every lane.
__device__ __forceinline__ bool collide_convex_w(int t0, float4 g0, f3 p0, qf q0, int t1, float4 g1, f3 p1, qf q1, const ConvexView& cv,
                                 WaveMem& M, Mf& m, bool& overflow) {
    m.numPoints = 0;
    overflow = false;
    const bool flipRes = t0 == PGX_CONVEX_MESH && t1 != PGX_CONVEX_MESH;
    if (flipRes) {   // mirrored: solve (other, convex) and flip
        const int tt = t0; t0 = t1; t1 = tt;
        const float4 gg = g0; g0 = g1; g1 = gg;
        const f3 pp = p0; p0 = p1; p1 = pp;
        const qf qq = q0; q0 = q1; q1 = qq;
    }
    const MeshRef m1{&cv, cv.mesh[(int)g1.w]};
    const SupHull b = hull_of(SupConvex{p1, mat3_cast(q1), mk3(g1.x, g1.y, g1.z), cv.verts + m1.info.x, m1.info.y});
    SupSide a{t0, SupHull{p0, m3{}, s3(1.f), nullptr, 0, s3(0.f)}, mk3(g0.x, g0.y, g0.z)};
    MeshRef m0{&cv, make_int4(0, 0, 0, 0)};
    if (t0 == PGX_CAPSULE) a.hull.l2w.c0 = qrot(q0, mk3(0.f, 1.f, 0.f));
    else if (t0 != PGX_SPHERE) a.hull.l2w = mat3_cast(q0);
    if (t0 == PGX_CONVEX_MESH) {
        m0.info = cv.mesh[(int)g0.w];
        a.hull = hull_of(SupConvex{p0, a.hull.l2w, a.g, cv.verts + m0.info.x, m0.info.y});
    }
    GV va, vb, vc, vd;
    const bool hit = gjk_w(a, b, sub(p1, p0), va, vb, vc, vd);
    if (hit) {
        m.normal = epa_w(a, b, va, vb, vc, vd, M, m.pts[0].p0, m.pts[0].p1, overflow);
        if (t0 == PGX_SPHERE) {                              // src/Collision.cpp:488-499
            m.numPoints = 1;
        } else if (t0 == PGX_CAPSULE) {                      // src/Collision.cpp:787-806
            const f3 axis = a.hull.l2w.c0;
            const m3 w2c = inverse(b.l2w);
            const f3 p = mulmv(w2c, sub(p0, p1));
            const f3 axisLc = mulmv(w2c, axis);
            capsule_convex_contacts_w(add(p, mul(axisLc, g0.x)), sub(p, mul(axisLc, g0.x)), g0.y, p1, b.l2w, m1, b.scale,
                                      m);
        } else {                                             // src/Collision.cpp:412-426,873-887
            FaceClip F;
            if (t0 == PGX_BOX) box_convex_clip(p0, a.hull.l2w, a.g, p1, q1, m1, b.scale, m.normal, F);
            else convex_convex_clip(p0, q0, m0, a.hull.scale, p1, q1, m1, b.scale, m.normal, F);
            int n;
            CPt pts[4];
            wave_contacts(F, M, pts, n);
            if (n) {
#pragma unroll
                for (int i = 0; i < 4; ++i) m.pts[i] = pts[i];
                m.numPoints = n;
            }
        }
        if (!m.numPoints) m.numPoints = 1;                   // the points of EPA
    }
    if (flipRes) {
        m.normal = neg(m.normal);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i < m.numPoints) { const f3 t = m.pts[i].p0; m.pts[i].p0 = m.pts[i].p1; m.pts[i].p1 = t; }
    }
    return hit;
}

}  // namespace pgx
