// walls_geom.h -- distance from a point to an STL triangle and the nearest-wall search, shared
// by the wall kernels and the sphere kernels.
#pragma once
#include "mpsr_internal.h"

namespace mpsr {

template <typename R> struct P3 { R x, y, z; };
template <typename R> __device__ inline P3<R> p3(R x, R y, R z) { return P3<R>{x, y, z}; }
template <typename R> __device__ inline P3<R> psub(P3<R> a, P3<R> b) { return p3(a.x - b.x, a.y - b.y, a.z - b.z); }
template <typename R> __device__ inline P3<R> padd(P3<R> a, P3<R> b) { return p3(a.x + b.x, a.y + b.y, a.z + b.z); }
template <typename R> __device__ inline R pdot(P3<R> a, P3<R> b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
template <typename R> __device__ inline R pmag(P3<R> a) { return build_sqrt(a.x * a.x + a.y * a.y + a.z * a.z); }

// ---------------------------------------------------------------------------------------------
// distance to a triangle, Utility_Inline.h:46-170
// ---------------------------------------------------------------------------------------------
template <typename R> __device__ inline R segment_ratio(P3<R> p1, P3<R> p2, P3<R> p3_) {
    const P3<R> dv = psub(p2, p1);
    R den = dv.x * dv.x + dv.y * dv.y + dv.z * dv.z;
    const R num = (p3_.x - p1.x) * (p2.x - p1.x) + (p3_.y - p1.y) * (p2.y - p1.y) + (p3_.z - p1.z) * (p2.z - p1.z);
    if (den == 0.0) den = (R)1e-5;
    return num / den;
}
// CalcDistanceVectorLine: beyond the ends it returns L1 - P (u < 0) and L0 - P (u > 1)
template <typename R> __device__ inline P3<R> line_vec(P3<R> l0, P3<R> l1, P3<R> p) {
    const R u = segment_ratio(l0, l1, p);
    P3<R> d = p3<R>(0, 0, 0);
    if (u >= 0 && u <= 1) {
        const P3<R> m = psub(l1, l0);
        const P3<R> q = p3(l0.x + u * m.x, l0.y + u * m.y, l0.z + u * m.z);
        d = psub(p, q);
    }
    if (u < 0) d = psub(l1, p);
    if (u > 1) d = psub(l0, p);
    return d;
}
template <typename R> __device__ inline R tri_distance(const TriD<R>& t, P3<R> p, P3<R>* out) {
    const P3<R> v0 = p3(t.v[0], t.v[1], t.v[2]), v1 = p3(t.v[3], t.v[4], t.v[5]), v2 = p3(t.v[6], t.v[7], t.v[8]);
    // CalcNormalDistance with the stored normal and the centroid divided by the double 3.0
    const P3<R> n = p3(t.nrm[0], t.nrm[1], t.nrm[2]);
    P3<R> cc = p3<R>(0, 0, 0);
    cc.x += v0.x; cc.y += v0.y; cc.z += v0.z;
    cc.x += v1.x; cc.y += v1.y; cc.z += v1.z;
    cc.x += v2.x; cc.y += v2.y; cc.z += v2.z;
    cc.x = (R)((double)cc.x / 3.0);
    cc.y = (R)((double)cc.y / 3.0);
    cc.z = (R)((double)cc.z / 3.0);
    const R ln = n.x * cc.x + n.y * cc.y + n.z * cc.z;
    const R rn = n.x * p.x + n.y * p.y + n.z * p.z;
    const R den = n.x * n.x + n.y * n.y + n.z * n.z;
    const R sden = build_sqrt(den);
    P3<R> dv = p3<R>(0, 0, 0);
    if (!(sden == 0.0)) {
        const R coef = (rn - ln) / sden;
        dv.x = coef / sden * n.x;
        dv.y = coef / sden * n.y;
        dv.z = coef / sden * n.z;
    }
    const P3<R> P = p3(p.x - dv.x, p.y - dv.y, p.z - dv.z);
    const P3<R> e0 = psub(v2, v0), e1 = psub(v1, v0), e2 = psub(P, v0);
    const R d00 = pdot(e0, e0), d01 = pdot(e0, e1), d02 = pdot(e0, e2), d11 = pdot(e1, e1), d12 = pdot(e1, e2);
    const R inv = 1 / (d00 * d11 - d01 * d01);
    const R u = (d11 * d02 - d01 * d12) * inv;
    const R v = (d00 * d12 - d01 * d02) * inv;
    if (u >= 0 && v >= 0 && u + v > 1) dv = line_vec(v1, v2, p);
    if (u < 0) dv = line_vec(v0, v1, p);
    if (v < 0) dv = line_vec(v0, v2, p);
    *out = dv;
    return pmag(dv);
}

// nearest triangle of the wanted kind (drag or not) over the 27-cell stencil
template <typename R>
__device__ inline int nearest_triangle(const Consts<R>& c, R x, R y, R z, const int* __restrict__ tstart,
                                       const int* __restrict__ tcount, const int* __restrict__ tids,
                                       const TriD<R>* __restrict__ tris, int want_drag, R* best, P3<R>* bdir) {
    *best = (R)1e8;
    *bdir = p3<R>(0, 0, 0);
    int bid = -1;
    int ci, cj, ck;
    if (!cell_coords(c, x, y, z, ci, cj, ck)) return bid;
    const long long cid = cell_of(c, ci, cj, ck);
    if (cid < 0 || cid >= c.ncell) return bid;
    const P3<R> p = p3(x, y, z);
    for (int k = -1; k <= 1; ++k)
        for (int j = -1; j <= 1; ++j)
            for (int i = -1; i <= 1; ++i) {
                const long long m = cell_of(c, ci + i, cj + j, ck + k);
                if (m < 0 || m >= c.ncell) continue;
                const int n = tcount[m];
                const int a = tstart[m];
                for (int e = 0; e < n; ++e) {
                    const int tid = tids[a + e];
                    const TriD<R>& tr = tris[tid];
                    if (tr.is_drag != want_drag) continue;
                    if (tid != bid) {
                        P3<R> dv;
                        const R dm = tri_distance(tr, p, &dv);
                        if (dm < *best) {
                            *best = dm;
                            *bdir = dv;
                            bid = tid;
                        }
                    }
                }
            }
    return bid;
}

// Bounds on tri_distance(t, p).  It ends on a point of an edge, a vertex, or the point P = p - (distance
// along the stored normal) when the barycentric coordinates of P put it inside the triangle.  The stored
// normal need not be the triangle's own (rotating walls keep the one they were read with): tilted by theta,
// P lies in the plane through the centroid across the stored normal, above or below a point of the
// triangle, so at most rad tan(theta) off it, and |P - centroid| <= rad / cos(theta), with rad the largest
// distance of a vertex from the centroid.  The build's root, up to 0.18 % low, divides the distance along
// the normal twice, so P overshoots that plane by up to 0.37 % of the distance d, which moves the point of
// the triangle below it by up to 0.37 % d / cos(theta), and shortens the result by 0.18 % once: with
// cos(theta) >= 0.2 the result is at least 0.975 times the bound, and at most 1.005 times |p - centroid|
// + rad.  tri_tilt is 1 / cos(theta), infinite where no bound is drawn: a larger tilt or a degenerate
// triangle (twice its area below 1 % of the longest edge squared), whose barycentric coordinates say
// little.  The margins, 1 % of the cell size and of rad, are for the rounding of the rest, and kFarRounding
// coordinate roundings (Consts::far_eps) for that of the coordinates themselves, which outgrows them far
// from the origin: the dot products of the normal with the point and the centroid err by up to 9, the
// point's way to float, the box's corner and the points of the edges by 2 each.
static constexpr float kFarRounding = 16.0f;
template <typename R> __device__ inline double tri_tilt(const TriD<R>& t) {
    const double ax = t.v[0], ay = t.v[1], az = t.v[2], bx = t.v[3], by = t.v[4], bz = t.v[5], cx = t.v[6],
                 cy = t.v[7], cz = t.v[8];
    const double e1x = bx - ax, e1y = by - ay, e1z = bz - az, e2x = cx - ax, e2y = cy - ay, e2z = cz - az;
    const double e3x = cx - bx, e3y = cy - by, e3z = cz - bz;
    const double gx = e1y * e2z - e1z * e2y, gy = e1z * e2x - e1x * e2z, gz = e1x * e2y - e1y * e2x;
    const double nx = t.nrm[0], ny = t.nrm[1], nz = t.nrm[2];
    const double gg = gx * gx + gy * gy + gz * gz, nn = nx * nx + ny * ny + nz * nz, ng = nx * gx + ny * gy + nz * gz;
    const double L2 = fmax(e1x * e1x + e1y * e1y + e1z * e1z,
                           fmax(e2x * e2x + e2y * e2y + e2z * e2z, e3x * e3x + e3y * e3y + e3z * e3z));
    if (!(gg >= 1e-4 * L2 * L2 && L2 > 0.0 && nn > 0.0 && ng * ng >= 0.04 * nn * gg)) return INFINITY;
    return fmax(1.0, sqrt(nn * gg / (ng * ng)));
}
// the centroid, rounded to float, and the largest distance of a vertex from it
template <typename R> __device__ inline double tri_centre(const TriD<R>& t, float* c) {
    for (int a = 0; a < 3; ++a) c[a] = (float)(((double)t.v[a] + (double)t.v[3 + a] + (double)t.v[6 + a]) / 3.0);
    double r2 = 0;
    for (int k = 0; k < 3; ++k) {
        const double dx = (double)t.v[3 * k] - c[0], dy = (double)t.v[3 * k + 1] - c[1], dz = (double)t.v[3 * k + 2] - c[2];
        r2 = fmax(r2, dx * dx + dy * dy + dz * dz);
    }
    return sqrt(r2);
}
// A lower bound of tri_distance(t, p) over the points p of the box [lo, lo + size]^3 (0 where none is
// drawn), as a float no larger than the bound: the distance between the box and the triangle's bounding
// box, less the margins and what the tilt takes P off the triangle.
template <typename R>
__device__ inline float tri_box_bound(const TriD<R>& t, R lox, R loy, R loz, R size, float far_eps) {
    const double sz = (double)size, tilt = tri_tilt(t);
    if (!(tilt < 1e3)) return 0.0f;
    float cc[3];
    const double rad = tri_centre(t, cc);
    const double lx = lox, ly = loy, lz = loz;
    auto gap = [&](double a, double b, double c, double lo) {
        const double tmin = fmin(a, fmin(b, c)), tmax = fmax(a, fmax(b, c));
        return fmax(0.0, fmax(tmin - (lo + sz), lo - tmax));
    };
    const double dx = gap(t.v[0], t.v[3], t.v[6], lx), dy = gap(t.v[1], t.v[4], t.v[7], ly),
                 dz = gap(t.v[2], t.v[5], t.v[8], lz);
    const double lb = 0.975 * (sqrt(dx * dx + dy * dy + dz * dz) - rad * (0.01 + sqrt(tilt * tilt - 1.0))) - 0.01 * sz -
                      kFarRounding * far_eps;
    if (!(lb > 0.0)) return 0.0f;
    return (float)(lb * 0.999999);
}
// A sphere around every point tri_distance can end on: |p - centre| less its radius, times 0.975, less 1 %
// of the cell size and the coordinates' rounding, is a lower bound.  The radius is infinite where no bound is drawn, and negated for a
// drag triangle.
template <typename R> __device__ inline float4 tri_sphere(const TriD<R>& t) {
    float cc[3];
    const double rad = tri_centre(t, cc), tilt = tri_tilt(t);
    const float r = tilt < 1e3 ? (float)(rad * 1.01 * tilt) : INFINITY;
    return make_float4(cc[0], cc[1], cc[2], t.is_drag ? -r : r);
}

// A triangle spans several cells, so the 27-cell walk of nearest_triangle meets it in several
// lists.  Met again, its distance is the same and only a strictly nearer triangle replaces the
// running nearest, so the result is the triangle of least distance, the first met of those of
// equal distance: the least (distance, position of first meeting).  The cell walk kernels write
// each cell's triangles once (head[cell] = (pool offset, count)), with their positions of first
// meeting, ordered by tri_box_bound over the cell's box; a particle inside that box (to within half the bound's margin) stops at the
// first triangle whose bound exceeds its nearest distance so far, as no later one can be nearer or
// as near.  A particle outside it (the grid's truncating cell index puts particles up to one cell
// below the grid into the first cell) takes every listed triangle.  A cell without a list (count
// -1: no particles when the lists were written, or more than kStencilTris triangles) takes the
// full walk.
//
// Both bounds are those of the walls as they were binned: where the triangles have moved since (`moved`),
// every lane walks its whole list.
//
// the walk of a point's cell, and whether its bounds hold for the point
struct TriWalk {
    int2 h;
    int cut;
};
template <typename R>
__device__ inline TriWalk walk_of(const Consts<R>& c, bool want, R x, R y, R z, const int2* __restrict__ uhead, int moved) {
    int ci = 0, cj = 0, ck = 0;
    long long cid = -1;
    if (want && cell_coords(c, x, y, z, ci, cj, ck)) cid = cell_of(c, ci, cj, ck);
    TriWalk w;
    w.h = (cid >= 0 && cid < c.ncell) ? uhead[cid] : make_int2(0, -1);
    const R slack = c.cell * (R)0.005;
    const R lox = c.bminx + (R)ci * c.cell, loy = c.bminy + (R)cj * c.cell, loz = c.bminz + (R)ck * c.cell;
    w.cut = !moved && x >= lox - slack && x <= lox + c.cell + slack && y >= loy - slack &&
            y <= loy + c.cell + slack && z >= loz - slack && z <= loz + c.cell + slack;
    return w;
}

// Each lane (of those with `want`) walks its own list, if it has one: the drag search, and lists so short that
// the wave's search costs more.
template <typename R>
__device__ inline int nearest_in_lane(bool want, P3<R> p, const TriWalk& w, const int2* __restrict__ ulist,
                                      const TriD<R>* __restrict__ tris, int want_drag, R* best, P3<R>* bdir) {
    *best = (R)1e8;
    *bdir = p3<R>(0, 0, 0);
    int bid = -1, bpos = 0;
    const int n = want ? w.h.y : 0;
    int2 next = n > 0 ? ulist[w.h.x] : make_int2(0, 0);
    for (int e = 0; e < n; ++e) {
        const int2 en = next;
        next = ulist[w.h.x + min(e + 1, n - 1)];   // on its way while this triangle's record is
        if (w.cut && (R)__uint_as_float((unsigned)en.y & ~kWalkPosMask) > *best) break;
        const TriD<R>& tr = tris[en.x];
        if (tr.is_drag != want_drag) continue;
        P3<R> dv;
        const R dm = tri_distance(tr, p, &dv);
        const int pos = (int)((unsigned)en.y & kWalkPosMask);
        if (dm < *best || (dm == *best && bid >= 0 && pos < bpos)) {
            *best = dm;
            *bdir = dv;
            bid = en.x;
            bpos = pos;
        }
    }
    return bid;
}

// The nearest listed wall (no drag triangle) by one wave, a point per lane (`want` lanes only; every lane of the
// wave calls it).  A full distance is a
// chain of about 250 instructions, and a particle near a fine wall has 70-130 listed triangles, of which a
// few are near it.  So the points with a list are taken eight at a time, eight lanes to a point (lane
// 8 j + q takes entries j, j + 8, ... of point q; the points of a cell read the same entries).  A first
// pass over the spheres (tri_sphere, written when the triangles were binned) bounds each point's distance
// from above, a second puts the (point, entry) pairs whose spheres are not farther into a queue, and the
// queue is tested 64 pairs at a time.  A triangle left out is farther than the nearest, so it is neither
// nearer nor as near, and the least (distance, position) does not depend on who tests what.
// Per pass, each lane walking its own list / this (rotating drums): 141 / 41 us at 62k particles, 102 / 45 at
// 126k, 75 / 60 at 517k, FP64 142 / 76 at 126k; 16 buckets of 730k particles 279 / 179.
template <typename R> struct NearestLds {
    unsigned long long best[64];   // bits of the nearest distance as a double
    P3<R> dir[64];
    int pos[64], id[64], who[64];
    unsigned queue[kNearestQueue + 64];
};
template <typename R>
__device__ inline int nearest_in_wave(const Consts<R>& c, bool want, P3<R> pt, const TriWalk& wk,
                                      const int2* __restrict__ ulist, const TriD<R>* __restrict__ tris,
                                      const float4* __restrict__ sph, R* best, P3<R>* bdir, NearestLds<R>& L) {
    const int lane = lane_id();
    const R x = pt.x, y = pt.y, z = pt.z;
    const int2 h = wk.h;
    const int cut = wk.cut;
    *best = (R)1e8;
    *bdir = p3<R>(0, 0, 0);
    const bool listed = want && h.y > 0;
    const unsigned long long mask = __ballot(listed);
    const int count = __popcll(mask), q = lane & 7, j = lane >> 3;
    L.best[lane] = (unsigned long long)__double_as_longlong(1e8);
    L.pos[lane] = 0x7fffffff;
    L.id[lane] = -1;
    if (listed) L.who[__popcll(mask & ((1ull << lane) - 1ull))] = lane;
    wave_lds_sync();
    int queued = 0;   // pairs in the queue: source lane in the high 6 bits, entry
    // the full distances of the queue's pairs; the points keep the least (distance, position)
    auto flush = [&]() {
        wave_lds_sync();
        for (int base = 0; base < queued; base += 64) {
            const bool on = base + lane < queued;
            const unsigned pair = on ? L.queue[base + lane] : 0u;
            const int src = (int)(pair >> 26), e = (int)(pair & 0x3ffffffu);
            const P3<R> p = p3(__shfl(x, src, 64), __shfl(y, src, 64), __shfl(z, src, 64));
            const int off = __shfl(h.x, src, 64);
            P3<R> dv = p3<R>(0, 0, 0);
            R dm = (R)1e8;
            int2 en = make_int2(0, 0);
            if (on) {
                en = ulist[off + e];
                dm = tri_distance(tris[en.x], p, &dv);
            }
            const bool near = on && dm < (R)1e8;
            const unsigned long long bits = (unsigned long long)__double_as_longlong((double)dm);
            const unsigned long long old = near ? L.best[src] : 0ull;
            if (near) atomicMin(&L.best[src], bits);
            wave_lds_sync();
            const bool least = near && L.best[src] == bits;
            if (least && bits < old) L.pos[src] = 0x7fffffff;   // the positions kept were of a farther one
            wave_lds_sync();
            const int pos = (int)((unsigned)en.y & kWalkPosMask);
            if (least) atomicMin(&L.pos[src], pos);
            wave_lds_sync();
            if (least && L.pos[src] == pos) {
                L.dir[src] = dv;
                L.id[src] = en.x;
            }
            wave_lds_sync();
        }
        queued = 0;
    };
    for (int g = 0; g < count; g += 8) {
        const int src = g + q < count ? L.who[g + q] : 0;
        const float px = (float)__shfl(x, src, 64), py = (float)__shfl(y, src, 64), pz = (float)__shfl(z, src, 64);
        const int off = __shfl(h.x, src, 64), n0 = __shfl(h.y, src, 64), cutq = __shfl(cut, src, 64);
        const int n = g + q < count ? n0 : 0;
        const float margin = 0.01f * (float)c.cell + kFarRounding * c.far_eps;
        const int2* const list = ulist + off;
        // f(on, e, sphere) for this lane's entries, four at a time (their loads are issued together: a
        // round waits for two loads, one after the other), until the list ends or, for a point inside its
        // cell, the entries' box bounds (ascending) exceed `up`; the lanes of the wave stay together
        auto walk = [&](const float& up, auto&& f) {
            bool go = j < n;
            for (int e0 = j; __any(go); e0 += 32) {
                int2 en[4];
                float4 sp[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) en[u] = go && e0 + 8 * u < n ? list[e0 + 8 * u] : make_int2(0, 0x7f800000);
#pragma unroll
                for (int u = 0; u < 4; ++u) sp[u] = sph[en[u].x];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const bool far = cutq && __uint_as_float((unsigned)en[u].y & ~kWalkPosMask) > up;
                    go = go && e0 + 8 * u < n && !far;
                    f(go, e0 + 8 * u, sp[u]);
                }
            }
        };
        auto push = [&](bool take, int e) {
            const unsigned long long m = __ballot(take);
            if (take) L.queue[queued + __popcll(m & ((1ull << lane) - 1ull))] = ((unsigned)src << 26) | (unsigned)e;
            queued += __popcll(m);
        };
        // the sphere's radius is negative for a drag triangle
        float up = 1e8f;
        int eup = -1;
        walk(up, [&](bool on, int e, const float4& sp) {
            const float dx = px - sp.x, dy = py - sp.y, dz = pz - sp.z;
            const float u = (sqrtf(dx * dx + dy * dy + dz * dz) + fabsf(sp.w)) * 1.005f + margin;
            if (on && !(sp.w < 0.f) && u < up) {
                up = u;
                eup = e;
            }
        });
        // each lane's nearest sphere is tested at once: the point's distance so far is a bound several
        // times tighter than the spheres'
        push(eup >= 0, eup);
        flush();
        if (n > 0) up = fminf(up, (float)__longlong_as_double((long long)L.best[src]) * 1.00001f);
#pragma unroll
        for (int o = 8; o < 64; o <<= 1) up = fminf(up, __shfl_xor(up, o, 64));
        walk(up, [&](bool on, int e, const float4& sp) {
            const float dx = px - sp.x, dy = py - sp.y, dz = pz - sp.z;
            const float far = (up + margin) * 1.026f + fabsf(sp.w);
            const bool take = on && e != eup && !(sp.w < 0.f) && !(dx * dx + dy * dy + dz * dz > far * far);
            push(take, e);
            if (queued > kNearestQueue) flush();
        });
    }
    flush();
    int bid = -1;
    if (listed) {
        bid = L.id[lane];
        if (bid >= 0) {
            *best = (R)__longlong_as_double((long long)L.best[lane]);
            *bdir = L.dir[lane];
        }
    }
    return bid;
}

// The wall of the negative-pressure term (radix DeviceProcess_Kernel.h:1110-1134): over the triangle
// lists of the 27 stencil cells, drag or not, the first listed triangle of each cell replaces the running
// nearest (the reference's l == 0 branch) unless it is that triangle already, the others replace it when
// strictly nearer.  The running distance is always that of the running triangle, so a first triangle that
// is the running one leaves the state it would set, and every cell with a list starts anew: the result is
// that of the last such cell alone, which is all that is walked (the corrector with the term, 126k
// particles: 290 -> 37 us).  Returns the id (-1 for none) and the distance in *best.
template <typename R>
__device__ inline int negp_triangle(const Consts<R>& c, R x, R y, R z, const int* __restrict__ tstart,
                                    const int* __restrict__ tcount, const int* __restrict__ tids,
                                    const TriD<R>* __restrict__ tris, R* best) {
    *best = (R)1e8;
    int nid = -1;
    int ci, cj, ck;
    if (!cell_coords(c, x, y, z, ci, cj, ck)) return nid;
    const long long cid = cell_of(c, ci, cj, ck);
    if (cid < 0 || cid >= c.ncell) return nid;
    const P3<R> p = p3(x, y, z);
    int n = 0, a = 0;
    for (int s = 26; s >= 0 && n == 0; --s) {
        const long long m = cell_of(c, ci + s % 3 - 1, cj + (s / 3) % 3 - 1, ck + s / 9 - 1);
        if (m < 0 || m >= c.ncell) continue;
        n = tcount[m];
        a = tstart[m];
    }
    for (int l = 0; l < n; ++l) {
        const int tid = tids[a + l];
        P3<R> dv;
        const R dm = tri_distance(tris[tid], p, &dv);
        if (l == 0 || dm < *best) { *best = dm; nid = tid; }
    }
    return nid;
}

// Deterministic pow, exp(y log x) in double rounded once to R, from IEEE-exact operations only
// (+ - * /, frexp, ldexp, floor) so that host and device give the same bits whatever their libm:
//   log x = e ln2 + 2 atanh(s), s = (m - 1)/(m + 1), m in [sqrt(1/2), sqrt(2)), series to s^23
//   exp z = 2^k exp(r), z = k ln2 + r (Cody-Waite split of ln2), |r| <= ln2/2, Taylor to r^15
__device__ inline double det_log(double x) {
    int e = 0;
    double m = frexp(x, &e);
    if (m < 0.70710678118654752440) {
        m = m * 2.0;
        e = e - 1;
    }
    const double s = (m - 1.0) / (m + 1.0), s2 = s * s;
    double p = 1.0 / 23.0;
    for (int k = 10; k >= 0; --k) p = p * s2 + 1.0 / (double)(2 * k + 1);
    const double ln2_hi = 6.93147180369123816490e-01, ln2_lo = 1.90821492927058770002e-10;
    return (double)e * ln2_hi + ((double)e * ln2_lo + 2.0 * s * p);
}
__device__ inline double det_exp(double z) {
    if (z > 709.0) return INFINITY;
    if (z < -745.0) return 0.0;
    const double ln2_hi = 6.93147180369123816490e-01, ln2_lo = 1.90821492927058770002e-10;
    const double k = floor(z / 0.69314718055994530942 + 0.5);
    const double r = (z - k * ln2_hi) - k * ln2_lo;
    double p = 1.0;
    for (int j = 15; j >= 1; --j) p = 1.0 + p * r / (double)j;
    return ldexp(p, (int)k);
}
template <typename R> __device__ inline R powd(R x, R y) {
    if (y == R(0)) return R(1);
    if (x == R(0)) return y > R(0) ? R(0) : (R)INFINITY;
    return (R)det_exp((double)y * det_log((double)x));
}

}  // namespace mpsr
