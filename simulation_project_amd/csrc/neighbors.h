// neighbors.h -- the canonical 27-cell neighbour walk shared by the particle and PPE kernels.
#pragma once
#include <type_traits>
#include "mpsr_internal.h"

namespace mpsr {

template <typename R> __device__ inline R4<R> mk4(R x, R y, R z, R w);
template <> __device__ inline float4 mk4<float>(float x, float y, float z, float w) { return make_float4(x, y, z, w); }
template <> __device__ inline double4 mk4<double>(double x, double y, double z, double w) { return make_double4(x, y, z, w); }

// every candidate t != self in the 27-cell stencil around (x, y, z), canonical order
template <typename R, typename F>
__device__ inline void for_candidates(const Consts<R>& c, const int* __restrict__ cs, const int* __restrict__ ce,
                                      R x, R y, R z, int self, F&& f) {
    int ci, cj, ck;
    if (!cell_coords(c, x, y, z, ci, cj, ck)) return;
    const long long cid = cell_of(c, ci, cj, ck);
    if (cid < 0 || cid >= c.ncell) return;
    for (int k = -1; k <= 1; ++k)
        for (int j = -1; j <= 1; ++j)
            for (int i = -1; i <= 1; ++i) {
                const long long m = cell_of(c, ci + i, cj + j, ck + k);
                if (m < 0 || m >= c.ncell) continue;
                const int a = cs[m];
                if (a < 0) continue;
                const int b = ce[m];
                for (int t = a; t < b; ++t)
                    if (t != self) f(t);
            }
}

// for_candidates restricted to the stencil cells whose box lies within `reach` of (x, y, z), with
// a 1 % margin over the build's distance (sqrt14 errs by at most 0.18 %, the cell boxes by a few
// ulp): a skipped cell holds no particle closer than `reach`, and the cells that remain are
// visited in the same order, so every sum over the neighbours within `reach` is unchanged
template <typename R, typename F>
__device__ inline void for_candidates_within(const Consts<R>& c, const int* __restrict__ cs,
                                             const int* __restrict__ ce, R x, R y, R z, int self, R reach,
                                             F&& f) {
    int ci, cj, ck;
    if (!cell_coords(c, x, y, z, ci, cj, ck)) return;
    const long long cid = cell_of(c, ci, cj, ck);
    if (cid < 0 || cid >= c.ncell) return;
    const R m = reach * (R)1.01;
    const R m2 = m * m;
    // squared distance to the cell slabs at offsets -1 and +1 per axis (0 for the own slab)
    const R lx = c.bminx + (R)ci * c.cell, ly = c.bminy + (R)cj * c.cell, lz = c.bminz + (R)ck * c.cell;
    const R xm = x - lx, xp = lx + c.cell - x, ym = y - ly, yp = ly + c.cell - y, zm = z - lz, zp = lz + c.cell - z;
    const R xm2 = xm * xm, xp2 = xp * xp, ym2 = ym * ym, yp2 = yp * yp, zm2 = zm * zm, zp2 = zp * zp;
    for (int k = -1; k <= 1; ++k) {
        const R dz2 = k < 0 ? zm2 : (k > 0 ? zp2 : (R)0);
        for (int j = -1; j <= 1; ++j) {
            const R dyz2 = dz2 + (j < 0 ? ym2 : (j > 0 ? yp2 : (R)0));
            if (dyz2 > m2) continue;
            for (int i = -1; i <= 1; ++i) {
                if (dyz2 + (i < 0 ? xm2 : (i > 0 ? xp2 : (R)0)) > m2) continue;
                const long long mm = cell_of(c, ci + i, cj + j, ck + k);
                if (mm < 0 || mm >= c.ncell) continue;
                const int a = cs[mm];
                if (a < 0) continue;
                const int b = ce[mm];
                for (int t = a; t < b; ++t)
                    if (t != self) f(t);
            }
        }
    }
}

template <typename R>
__device__ inline R dist3(R x, R y, R z, R qx, R qy, R qz) {
    return build_sqrt((x - qx) * (x - qx) + (y - qy) * (y - qy) + (z - qz) * (z - qz));
}

// for_candidates in groups: g(t0, Q, m) for runs of up to 4 consecutive candidates t0 ..
// t0 + m - 1 of one stencil cell, in the canonical order, with Q[u] = spos[t0 + u] (Q[u] for u >= m
// repeats the last record and is to be ignored; self is not skipped: the caller tests it).  A
// caller that reads a second record of its neighbours loads them for the whole group before it
// uses them, so one wait covers the group instead of one per neighbour.
template <typename R, typename F>
__device__ inline void for_candidate_groups(const Consts<R>& c, const int* __restrict__ cs,
                                            const int* __restrict__ ce, const R4<R>* __restrict__ spos, R x, R y,
                                            R z, F&& g) {
    int ci, cj, ck;
    if (!cell_coords(c, x, y, z, ci, cj, ck)) return;
    const long long cid = cell_of(c, ci, cj, ck);
    if (cid < 0 || cid >= c.ncell) return;
    for (int k = -1; k <= 1; ++k)
        for (int j = -1; j <= 1; ++j)
            for (int i = -1; i <= 1; ++i) {
                const long long mcell = cell_of(c, ci + i, cj + j, ck + k);
                if (mcell < 0 || mcell >= c.ncell) continue;
                const int a = cs[mcell];
                if (a < 0) continue;
                const int b = ce[mcell];
                int t = a;
                for (; t + 4 <= b; t += 4) {
                    R4<R> Q[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) Q[u] = spos[t + u];
                    g(t, Q, 4);
                }
                if (t < b) {
                    const int m = b - t;
                    R4<R> Q[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) Q[u] = spos[t + (u < m ? u : m - 1)];
                    g(t, Q, m);
                }
            }
}

// ---- the canonical walk with its distance test on the matrix cores ---------------------------
// A walk meets about 800 candidates per particle and keeps 120 (Laplacian radius) or 32; with one
// lane per particle every candidate costs its load, the exact distance and, as some lane of the
// wave always hits, the neighbour work.  Here one wave takes 64 consecutive sorted particles in two
// phases.
//
// Phase 1 tests all pairs of a cell's particles and its stencil's candidates by a product: with q' the
// candidate relative to the centre of its own cell, X the particle relative to that of its own and D
// the difference of the centres, half of |X - q|^2 - T is
//     (qx', qy', qz', 1) . (-(X - D), (|X - D|^2 - T) / 2) + |q'|^2 / 2,
// the 16 x 16 x 4 FP32 product of 16 candidates and 16 particles plus its accumulator, whose sign is
// the test.  The binning writes q' (an array per component, as a load costs a cycle for every lane that
// is not next to its neighbour) and |q'|^2 / 2, the accumulator, which is the same for all particles.  Each lane shifts the signs of its 8 results of a run of 32 candidates into a byte
// of the particle's bit word in LDS (one VALU instruction per 64 pairs, against nine).
// T holds (1.004 reach + e)^2 + 1e-4 cell^2: the build's root errs by at most 0.18 %, and the product, of
// values up to 6 cells, by less than 1e-4 cell^2.  e = 6 far_eps is for the centres: a float centre is off by
// up to 1.5 far_eps an axis (the product with the cell size and the sum are rounded), so the particle's and
// the candidate's leave X - D - q' off by up to 3 an axis; far from the origin that outgrows the rest (l0 =
// 10 mm, 10 km out: 2 mm, with which a tenth of the pressures went wrong).  So every neighbour within
// reach has its bit.
//
// Phase 2 runs over each lane's own bits in walk order, f(q, record) with the record of the next one
// loaded ahead; f tests the exact distance, so the sums are those of the plain walk.
//
// What bounds it: phase 1 the issue of about 30 instructions per word of 32 candidates and 16 particles
// and the slowest waves (sparse cells at the fluid's rim are tested one by one); phase 2 the gathers, at
// a lane a cycle when they hit L1.  Against the plain walks it replaced (FP32): PND pass of the EOS
// pressure 121 -> 63 us at 4k particles, 154 -> 99 at 126k, 386 -> 295 at 517k; of the PPE 267 -> 130 at
// 62k, 1037 -> 960 at 1M; heat conduction 210 -> 96 at 120k; turbulence 237 -> 103 at 126k; FP64 PND
// pass 396 -> 205 at 126k.
//
// The bit words of a wave take 14 KB of LDS (10 waves on a CU).  kNearWords holds the stencil of any
// cells of up to 64 particles; denser ones are taken in three passes, one per z plane of the stencil, and
// a wave of many sparse cells in groups of cells whose words fit the table.  (40 words sent a fifth of a
// drum's cells into three passes: 520 -> 651 us in the predictor at 517k.)  Lanes whose particle lies
// over 4 cells from its cell (aliased by the truncating cell index) or whose key is not its cell (a dead
// slot) take the plain walk, as do those of a stencil plane of more than kNearWords words; the candidates
// of a stencil cell that the cell index wraps to the other side of the grid all get their bit.
// The cells of a wave are tested one after the other, so a wave of many cells (a spray, the rim of the
// fluid) takes the plain walk too, its lanes side by side, where that is shorter: a cell of W words costs
// 2 + W / 4 us, a plain walk of S candidates 20 + S / 5 us (waves alone on a SIMD).  Above kNearCells cells a
// wave compares them, with the stencils of its first and last particle's cells, and above kNearCellsMost it
// does not ask.  (Counted for every lane, S and W took 10 us; with S / 10 dense fluids lost 15-50 % at their
// rims.)  PND pass of particles strewn at random, without the rule / with it: 264 / 34 us at 64k and one a
// cell, 181 / 59 at four, 108 / 97 at eight, 91 / 93 at fifteen, 1,149 / 117 at 500k and one a cell; predictor
// in FP64 1,213 / 213 there.  (Plain kernels, whose waves have no bit words to hold, take 45, 64, 82, 108,
// 133 and 206.)
static constexpr int kNearCells = 7, kNearCellsMost = 16;
// g(q0, Q, m) for runs of up to 4 candidates as for_candidate_groups, over the stencil cells within `reach`
// (as for_candidates_within, its margin with the cell boxes' rounding, up to 1.5 far_eps an axis, and the
// offsets' own), the ranges of a row of cells loaded together
static constexpr float kCullRounding = 5.0f;
template <typename R, typename F>
__device__ inline void for_candidates_sparse(const Consts<R>& c, const int* __restrict__ cs, const int* __restrict__ ce,
                                             const R4<R>* __restrict__ spos, R x, R y, R z, R reach, F&& g) {
    int ci, cj, ck;
    if (!cell_coords(c, x, y, z, ci, cj, ck)) return;
    const long long cid = cell_of(c, ci, cj, ck);
    if (cid < 0 || cid >= c.ncell) return;
    const R m = reach * (R)1.01 + (R)(kCullRounding * c.far_eps);
    const R m2 = m * m;
    const R lx = c.bminx + (R)ci * c.cell, ly = c.bminy + (R)cj * c.cell, lz = c.bminz + (R)ck * c.cell;
    const R xm = x - lx, xp = lx + c.cell - x, ym = y - ly, yp = ly + c.cell - y, zm = z - lz, zp = lz + c.cell - z;
    const R dx2[3] = {xm * xm, (R)0, xp * xp};
    const bool inside = m < c.cell && cj >= 0 && cj < c.gy && ck >= 0 && ck < c.gz;   // and worth it
    for (int k = -1; k <= 1; ++k) {
        const R dz2 = k < 0 ? zm * zm : (k > 0 ? zp * zp : (R)0);
        for (int j = -1; j <= 1; ++j) {
            const R dyz2 = dz2 + (j < 0 ? ym * ym : (j > 0 ? yp * yp : (R)0));
            // a cell that the index wraps to the other side of the grid is not where its offset says
            const bool cull = inside && cj + j >= 0 && cj + j < c.gy && ck + k >= 0 && ck + k < c.gz;
            if (cull && dyz2 > m2) continue;
            int a[3], b[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const long long n = cell_of(c, ci + i - 1, cj + j, ck + k);
                const bool in = n >= 0 && n < c.ncell && !(cull && dyz2 + dx2[i] > m2);
                a[i] = in ? cs[n] : -1;
                b[i] = in ? ce[n] : -1;
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                if (a[i] < 0) continue;
                const int last = b[i] - 1;
                for (int q = a[i]; q <= last; q += 4) {
                    R4<R> Q[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) Q[u] = spos[min(q + u, last)];
                    g(q, Q, min(4, last + 1 - q));
                }
            }
        }
    }
}

// f(q, Q) for each candidate of a run but `self`
template <typename R, typename F> __device__ inline auto each_of(int self, F f) {
    return [=](int q0, const R4<R> (&Q)[4], int m) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (u < m && q0 + u != self) f(q0 + u, Q[u]);
    };
}

typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v2fu __attribute__((ext_vector_type(2), aligned(4)));
typedef float v4fu __attribute__((ext_vector_type(4), aligned(4)));
static constexpr int kNearWords = 54;
static constexpr int kNearTable = 432;
static constexpr int kNearRow = kNearWords + 1;   // odd: the lanes' rows start in different banks
struct NearLds {
    uint32_t bits[65 * kNearRow];                 // row 64 takes the bytes of padding lanes
    int first[kNearTable];                        // sorted index of a word's first candidate, by cell
    int meta[kNearWords];
};

// use(q, load(q)) for the neighbours by their bits; plain(q0, Q, m) for the candidates of a plain walk, in
// runs (for_candidate_groups: self among them).  Both test the exact distance.
template <typename R, typename Load, typename Use, typename Plain>
__device__ inline void for_near_mfma(const Consts<R>& c, const int* __restrict__ cs, const int* __restrict__ ce,
                                     const RelPos& rel, const uint32_t* __restrict__ skeys, int t0,
                                     int N, bool want, const R4<R>* __restrict__ spos, R x, R y, R z, R reach, NearLds& L,
                                     Load&& load, Use&& use, Plain&& plain) {
    const int lane = lane_id(), t = t0 + lane;
    const int gz = c.gz, gyz = c.gy * c.gz;
    const uint32_t key = t < N ? skeys[t] : (uint32_t)c.ncell;
    const float cell = (float)c.cell;
    const double rt = 1.004 * (double)reach + 6.0 * (double)c.far_eps;
    const float T = (float)(rt * rt + 1e-4 * (double)c.cell * (double)c.cell);
    bool mine = false, walk = false;
    if (want) {
        int ci, cj, ck;
        if (cell_coords(c, x, y, z, ci, cj, ck)) {
            const long long cid = cell_of(c, ci, cj, ck);
            if (cid >= 0 && cid < c.ncell) {
                mine = (uint32_t)cid == key && rel.half_sq(t) <= 8.0f * cell * cell;
                walk = !mine;
            }
        }
    }
    // lane s < 27 of a cell: its stencil cell's range (z outer, x inner); len 0 outside the grid
    const int di = lane % 3 - 1, dj = (lane / 3) % 3 - 1, dk = lane / 9 - 1;
    const int doff = di * gyz + dj * gz + dk;
    auto range = [&](int K, int& a, int& b) {
        const int m = max(0, min(c.ncell - 1, (int)min((long long)K + doff, (long long)c.ncell)));
        a = cs[m];
        b = ce[m];
    };
    auto length = [&](int K, int a, int b) {
        const long long m = (long long)K + doff;
        return lane < 27 && m >= 0 && m < c.ncell && a >= 0 ? b - a : 0;
    };
    // the cell index wraps at the grid's y and z faces: such a stencil cell is not at its offset
    auto wraps = [&](int K) {
        const int r = K % gyz, j = r / gz + dj, k = r % gz + dk;
        return j < 0 || j >= c.gy || k < 0 || k >= gz;
    };
    const int k4 = lane >> 4, n16 = lane & 15;
    uint8_t* const bytes = reinterpret_cast<uint8_t*>(L.bits);
    // candidate 2 n16 + tau of a run of 32 is row n16 of product tau (0, 1); the results of a lane are
    // then those of candidates 8 k4 .. 8 k4 + 7
    const uint32_t aoff = ((uint32_t)k4 * (uint32_t)rel.stride + 2u * n16) * 4u, woff = 16u * k4;
    unsigned long long left = __ballot(mine);
    int K = 0, ca = 0, cb = 0, s0 = 0;   // the next cell, its stencil's ranges, its first stencil cell not done
    if (left) {
        K = __builtin_amdgcn_readlane((int)key, __ffsll(left) - 1);
        range(K, ca, cb);
    }
    const int cells = __popcll(__ballot(lane == 0 || (int)key != __shfl_up((int)key, 1, 64)));
    if (left && cells > kNearCells) {
        bool strewn = cells > kNearCellsMost;
        if (!strewn) {
            const int K1 = __builtin_amdgcn_readlane((int)key, 63 - __clzll(left));
            int a1, b1;
            range(K1, a1, b1);
            // candidates in the low 17 bits, words above them
            auto count = [&](int len) {
                const int l = min(len, 4095);
                return __builtin_amdgcn_readlane(wave_inclusive_scan(l | (((l + 31) >> 5) << 17)), 63);
            };
            const int n0 = count(length(K, ca, cb)), n1 = count(length(K1, a1, b1));
            const int S = max(n0 & 0x1ffff, n1 & 0x1ffff), W = (n0 >> 17) + (n1 >> 17);   // W of both
            strewn = cells * (80 + 5 * W) > 800 + 8 * S;
        }
        if (strewn) {
            walk = walk || mine;
            mine = false;
            left = 0;
        }
    }
    while (left) {
        int nw = 0, tab = 0, at = 0;
        bool full = false;
        while (left && !full) {
            const unsigned long long mem = __ballot(mine && (int)key == K);
            const int l0 = __ffsll(mem) - 1, l1 = 63 - __clzll(mem);
            const int len = length(K, ca, cb);
            const int all = (len + 31) >> 5;
            const int sum = wave_inclusive_scan(all);
            const int w0 = __builtin_amdgcn_readlane(sum, 8), w1 = __builtin_amdgcn_readlane(sum, 17),
                      w2 = __builtin_amdgcn_readlane(sum, 26);
            const bool skip = max(w0, max(w1 - w0, w2 - w1)) > kNearWords;
            const int s1 = w2 > kNearWords && !skip ? s0 + 9 : 27;   // all, or a plane at a time
            const int before = s0 > 0 ? __builtin_amdgcn_readlane(sum, max(0, s0 - 1)) : 0;
            const int words = skip ? 0 : __builtin_amdgcn_readlane(sum, s1 - 1) - before;
            if (at > 0 && (at + words > kNearTable || s1 - s0 < 27)) break;
            if (skip && mine && (int)key == K) walk = true;
            const int a = ca, cell0 = s0, K0 = K;
            full = s1 - s0 < 27;
            s0 = s1;
            if (s1 == 27) {   // on to the next cell, its ranges loaded while this one is tested
                left &= ~mem;
                s0 = 0;
                if (left) {
                    K = __builtin_amdgcn_readlane((int)key, __ffsll(left) - 1);
                    range(K, ca, cb);
                }
            }
            // the words of this cell: lane w < words holds word w's first candidate, length and shift
            const int ws = lane >= cell0 && lane < s1 && words > 0 ? all : 0;
            const int w00 = sum - all - before;
            const int id = lane | (wraps(K0) ? 128 : 0);
            for (int r = 0; r < ws; ++r) {
                L.first[at + w00 + r] = a + 32 * r;
                L.meta[w00 + r] = id | (min(32, len - 32 * r) << 8);
            }
            wave_lds_sync();
            const bool has = lane < words;
            const int vfirst = has ? L.first[at + lane] : 0, vmeta = has ? L.meta[lane] : 0;
            const int vs = vmeta & 127;
            const float vx = (float)(vs % 3 - 1) * cell, vy = (float)((vs / 3) % 3 - 1) * cell,
                        vz = (float)(vs / 9 - 1) * cell;
            const int vlen = vmeta >> 8;
            const float vh = vmeta & 128 ? -1e30f : 0.5f * (vx * vx + vy * vy + vz * vz - T);
            if (mine && (int)key == K0) {
                nw = words;
                tab = at;
            }
            at += words;
            const int tiles = (l1 - l0 + 16) >> 4;
            auto test = [&](auto nt) {
                constexpr int NT = decltype(nt)::value;
                // the particles' operands, 16 to a tile: bits of pb + sx p1 + sy p2 + sz p3 + sh p4
                float pb[NT], p1[NT], p2[NT], p3[NT];
                const float p4 = k4 == 3 ? 1.0f : 0.0f;
                uint8_t* pa[NT];
#pragma unroll
                for (int p = 0; p < NT; ++p) {
                    const int pl = l0 + 16 * p + n16;
                    const float* const v = rel.x + (t0 + min(pl, l1));
                    const float vx_ = v[0], vy_ = v[rel.stride], vz_ = v[2 * (size_t)rel.stride];
                    pb[p] = k4 == 0 ? -vx_ : (k4 == 1 ? -vy_ : (k4 == 2 ? -vz_ : rel.half_sq(t0 + min(pl, l1))));
                    p1[p] = k4 == 3 ? -vx_ : (k4 == 0 ? 1.0f : 0.0f);
                    p2[p] = k4 == 3 ? -vy_ : (k4 == 1 ? 1.0f : 0.0f);
                    p3[p] = k4 == 3 ? -vz_ : (k4 == 2 ? 1.0f : 0.0f);
                    pa[p] = bytes + (pl <= l1 ? pl : 64) * kNearRow * 4 + k4;
                }
                // operands of a word, loaded kAhead words ahead: a load takes longer than a word's test
                constexpr int kAhead = 4;
                v2f A[kAhead];
                v4f C0[kAhead], C1[kAhead];
                auto fetch = [&](int w, v2f& av, v4f& c0, v4f& c1) {
                    const int f = __builtin_amdgcn_readlane(vfirst, min(w, words - 1)), odd = f & 1;
                    const char* const bx = reinterpret_cast<const char*>(rel.x + f);
                    const char* const b0 = reinterpret_cast<const char*>(rel.w + (odd ? rel.half : 0) + (f >> 1));
                    const char* const b1 = reinterpret_cast<const char*>(rel.w + (odd ? 0 : rel.half) + ((f + 1) >> 1));
                    av = *reinterpret_cast<const v2fu*>(bx + aoff);
                    c0 = *reinterpret_cast<const v4fu*>(b0 + woff);
                    c1 = *reinterpret_cast<const v4fu*>(b1 + woff);
                };
                auto word = [&](int w, const v2f& av, const v4f& c0, const v4f& c1) {
                    auto sf = [&](float v) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), w)); };
                    const float sx = sf(vx), sy = sf(vy), sz = sf(vz), sh = sf(vh);
                    const uint32_t valid = (uint32_t)((1ull << __builtin_amdgcn_readlane(vlen, w)) - 1ull) >> (8 * k4);
                    v4f lo[NT], hi[NT];
#pragma unroll
                    for (int p = 0; p < NT; ++p) {
                        const float bb = __builtin_fmaf(sx, p1[p], __builtin_fmaf(sy, p2[p],
                                         __builtin_fmaf(sz, p3[p], __builtin_fmaf(sh, p4, pb[p]))));
                        lo[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.x, bb, c0, 0, 0, 0);
                        hi[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.y, bb, c1, 0, 0, 0);
                    }
#pragma unroll
                    for (int p = 0; p < NT; ++p) {
                        uint32_t m = 0;
#pragma unroll
                        for (int v = 3; v >= 0; --v) {
                            m = __builtin_amdgcn_alignbit(m, __float_as_uint(hi[p][v]), 31);
                            m = __builtin_amdgcn_alignbit(m, __float_as_uint(lo[p][v]), 31);
                        }
                        pa[p][4 * w] = (uint8_t)(m & valid);
                    }
                };
                if (words > 0) {
#pragma unroll
                    for (int u = 0; u < kAhead; ++u) fetch(u, A[u], C0[u], C1[u]);
                    for (int w = 0; w < words; w += kAhead) {
#pragma unroll
                        for (int u = 0; u < kAhead; ++u) {
                            if (w + u < words) word(w + u, A[u], C0[u], C1[u]);
                            fetch(w + u + kAhead, A[u], C0[u], C1[u]);
                        }
                    }
                }
            };
            if (tiles == 1) test(std::integral_constant<int, 1>{});
            else if (tiles == 2) test(std::integral_constant<int, 2>{});
            else if (tiles == 3) test(std::integral_constant<int, 3>{});
            else test(std::integral_constant<int, 4>{});
            wave_lds_sync();   // meta is rewritten for the next cell
        }
        // phase 2
        const uint32_t* const row = L.bits + lane * kNearRow;
        const int* const first = L.first + tab;
        int w = 0;
        uint32_t bits = 0, nbits = nw > 0 ? row[0] : 0u;   // this word's rest, and the next word
        int base = 0, nbase = nw > 0 ? first[0] : 0;
        auto next = [&]() {
            while (bits == 0 && w < nw) {
                bits = nbits;
                base = nbase;
                ++w;
                nbits = row[w];                             // row[nw] exists, and is not used
                nbase = w < nw ? first[w] : 0;
            }
            if (bits == 0) return -1;
            const int q = base + __builtin_ctz(bits);
            bits &= bits - 1u;
            return q;
        };
        // a ring of three records: two loads are in flight while a third record is used
        int q0 = next(), q1 = next(), q2 = next();
        auto r0 = load(q0 >= 0 ? q0 : 0), r1 = load(q1 >= 0 ? q1 : 0), r2 = load(q2 >= 0 ? q2 : 0);
        while (q0 >= 0) {
            if (q0 != t) use(q0, r0);
            q0 = next();
            if (q0 >= 0) r0 = load(q0);
            if (q1 >= 0 && q1 != t) use(q1, r1);
            q1 = next();
            if (q1 >= 0) r1 = load(q1);
            if (q2 >= 0 && q2 != t) use(q2, r2);
            q2 = next();
            if (q2 >= 0) r2 = load(q2);
        }
        wave_lds_sync();
    }
    if (walk) for_candidates_sparse(c, cs, ce, spos, x, y, z, reach, plain);
}

}  // namespace mpsr
