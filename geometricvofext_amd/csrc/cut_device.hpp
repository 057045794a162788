// Plane cuts of cells and faces shared between the lanes of a wave: one face
// per lane, its points and crossings in LDS, the sums over a cell's faces read
// from LDS in face order.  Same operations in the same order as the one-lane
// routines of simplic_device.hpp, so the same bits.
#pragma once
#include "simplic_device.hpp"
#include "simplic_types.hpp"

namespace svp {

// Division by one divisor of several numerators: the reciprocal is refined
// once (two Newton steps from v_rcp_f64), each quotient then takes a product
// and one exact-residual correction.  These are the steps of the compiler's
// own FP64 division without its range scaling, so a quotient has the same
// bits as '/' wherever that scaling does nothing: divisor within
// [1e-250, 1e250] and numerator zero (the sign of a zero is not kept) or of
// magnitude 1e-290 and above; a smaller numerator can differ in the last place.
struct Rcp {
    double b, y;
};
__device__ inline Rcp rcp_of(double b) {
    double y = __builtin_amdgcn_rcp(b);
    y = __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
    y = __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
    return Rcp{b, y};
}
__device__ inline double div_by(double a, Rcp r) {
    const double q = a * r.y;
    return __builtin_fma(__builtin_fma(-r.b, q, a), r.y, q);
}
__device__ inline V3 div_by(V3 a, Rcp r) { return v3(div_by(a.x, r), div_by(a.y, r), div_by(a.z, r)); }

// x with the sign of s changed when s < 0 (sgn(s) * x for s >= 0 or s < 0;
// like sgn, a NaN counts as negative)
__device__ inline V3 flip_if_neg(V3 x, double s) {
    const bool keep = s >= 0.0;
    return v3(keep ? x.x : -x.x, keep ? x.y : -x.y, keep ? x.z : -x.z);
}

// The walk of cutFace::calcSubFace around a face of 3 or 4 points for every
// sign pattern of its vertex distances (bit i set: vertex i submerged): the
// sub-face's points in the order the walk emits them.  code(k): 0..3 a vertex,
// 4.. the crossings in walk order; past the last one the first point again,
// which closes the polygon and makes the triangles after it empty.
struct CutWalk {
    unsigned codes;   // 7 entries of 4 bits
    unsigned info;    // points (4 bits), crossings (4 bits), then per crossing the edge's first vertex (2 bits each)
};
constexpr CutWalk cut_walk(int n, int mask) {
    CutWalk w{0u, 0u};
    int first = -1;
    for (int i = 0; i < n; ++i)
        if (((mask >> i) & 1) && first < 0) first = i;
    if (first < 0 || mask == (1 << n) - 1) return w;
    int np = 0, nx = 0;
    unsigned edges = 0u;
    for (int k = 0; k < n; ++k) {
        const int cur = (first + k) % n, nxt = (cur + 1) % n;
        const int a = (mask >> cur) & 1, b = (mask >> nxt) & 1;
        if (a) w.codes |= (unsigned)cur << (4 * np++);
        if (a != b) {
            w.codes |= (unsigned)(4 + nx) << (4 * np++);
            edges |= (unsigned)cur << (2 * nx++);
        }
    }
    for (int k = np; k < 7; ++k) w.codes |= (unsigned)first << (4 * k);
    w.info = (unsigned)np | ((unsigned)nx << 4) | (edges << 8);
    return w;
}
struct CutWalks {
    CutWalk w[24];   // masks of 4-point faces, then of 3-point faces
};
constexpr CutWalks make_cut_walks() {
    CutWalks t{};
    for (int m = 0; m < 16; ++m) t.w[m] = cut_walk(4, m);
    for (int m = 0; m < 8; ++m) t.w[16 + m] = cut_walk(3, m);
    return t;
}
static __device__ const CutWalks kCutWalks = make_cut_walks();

// One of four values by index.  The values are arguments, so they are in
// registers before the choice: a choice between elements of an array can
// become a load through a chosen address, which moves the array to scratch.
__device__ inline double pick4(double a, double b, double c, double d, int e) {
    const double lo = (e & 1) ? b : a, hi = (e & 1) ? d : c;
    return (e & 2) ? hi : lo;
}
__device__ inline double choose(bool c, double a, double b) { return c ? a : b; }

__device__ inline V3 lds3(const double (&a)[3][64], int t) { return v3(a[0][t], a[1][t], a[2][t]); }
__device__ inline void lds3_put(double (&a)[3][64], int t, V3 v) {
    a[0][t] = v.x;
    a[1][t] = v.y;
    a[2][t] = v.z;
}

// cutFace::calcSubFace (cutFace.C:136-259) of a lane's face at one plane
// distance.  ps: the wave's LDS, places 0..FP-1 the points of the lane's
// face, FP.. its plane crossings (written here, in walk order); dots: point .
// normal of its n points.  Faces of 3 or 4 points look the walk up by their
// sign pattern, so each crossing is divided once and the triangles come from
// a list; larger faces walk their points twice.
template <int FP>
struct FaceWalk {
    double (&ps)[FP + MAX_IF_POINTS][3][64];
    const CutWalk (&walks)[24];
    const int t, n;
    double d[FP];
    unsigned mask = 0u;   // submerged vertices
    int nIf = 0;

    __device__ __attribute__((always_inline)) inline FaceWalk(double (&ps_)[FP + MAX_IF_POINTS][3][64],
                                                              const CutWalk (&walks_)[24], int t_, int n_,
                                                              const double (&dots)[FP], double dist)
        : ps(ps_), walks(walks_), t(t_), n(n_) {
        double least = 1.0;
#pragma unroll
        for (int i = 0; i < FP; ++i) {
            d[i] = dots[i] + dist;
            least = fmin(least, fabs(d[i]));
        }
        if (least < SVP_TSMALL) {
#pragma unroll
            for (int i = 0; i < FP; ++i)
                if (fabs(d[i]) < SVP_TSMALL) d[i] += sgn(d[i]) * SVP_TSMALL;
        }
#pragma unroll
        for (int i = 0; i < FP; ++i)
            if (i < n && d[i] < 0.0) mask |= 1u << i;
    }
    // -1 submerged, 0 cut, 1 empty
    __device__ inline int status() const { return mask == 0u ? 1 : (mask == (1u << n) - 1u ? -1 : 0); }

    __device__ inline V3 crossPoint(int e, int e1, double dc, double dn) const {
        const double w = div_by(dc, rcp_of(dc - dn));
        const V3 a = lds3(ps[e], t), b = lds3(ps[e1], t);
        return a + w * (b - a);
    }
    __device__ __attribute__((always_inline)) inline void listCrossing(const CutWalk& w, int k) const {
        const int e = (int)((w.info >> (8 + 2 * k)) & 3u);
        const int e1 = e + 1 == n ? 0 : e + 1;
        lds3_put(ps[FP + k], t,
                 crossPoint(e, e1, pick4(d[0], d[1], d[2], d[3], e), pick4(d[0], d[1], d[2], d[3], e1)));
    }
    __device__ inline V3 listEntry(const CutWalk& w, int k) const {
        const int c = (int)((w.codes >> (4 * k)) & 15u);
        return lds3(ps[c < 4 ? c : FP + c - 4], t);
    }
    __device__ inline double distOf(int e) const {
        double v = d[0];
#pragma unroll
        for (int k = 1; k < FP; ++k) v = choose(e == k, d[k], v);
        return v;
    }
    // the walk of a face of more than 4 points; record: its crossings to ps
    template <class Emit>
    __device__ inline bool walkPoints(Emit emit, bool record) {
        bool ok = true;
        int cur = __ffs((int)mask) - 1, nx = 0;
        double dc = distOf(cur);
        V3 pc = lds3(ps[cur], t);
        for (int k = 0; k < n; ++k) {
            const int nxt = cur + 1 == n ? 0 : cur + 1;
            const double dn = distOf(nxt);
            const V3 pn = lds3(ps[nxt], t);
            if (dc < 0.0) emit(pc);
            if ((dc < 0.0) != (dn < 0.0)) {
                const double w = div_by(dc, rcp_of(dc - dn));
                const V3 q = pc + w * (pn - pc);
                emit(q);
                if (record) {
                    if (nx < MAX_IF_POINTS) lds3_put(ps[FP + nx], t, q);
                    else ok = false;
                    nx++;
                }
            }
            cur = nxt;
            dc = dn;
            pc = pn;
        }
        if (record) nIf = nx > MAX_IF_POINTS ? MAX_IF_POINTS : nx;
        return ok;
    }

    // the plane's crossings of the cut face alone; false as for subFace
    __device__ __attribute__((always_inline)) inline bool crossings() {
        if (FP == 4 || n <= 4) {
            const CutWalk w = walks[(n == 3 ? 16u : 0u) + mask];
            nIf = (int)((w.info >> 4) & 15u);
            listCrossing(w, 0);
            listCrossing(w, 1);
            if (nIf > 2) {
                listCrossing(w, 2);
                listCrossing(w, 3);
            }
            return true;
        }
        return walkPoints([](V3) {}, true);
    }

    // centre and area of the cut face (calcSubFaceCentreAndArea,
    // cutFace.C:37-96); false when the plane crosses it more than
    // MAX_IF_POINTS times
    __device__ __attribute__((always_inline)) inline bool subFace(V3& centre, V3& area) {
        bool ok = true;
        V3 fC = VZERO, sumN = VZERO, sumAc = VZERO;
        double sumA = 0.0;
        auto tri = [&](V3 a, V3 b) {
            const V3 c = a + b + fC;
            const V3 nv = cross(b - a, fC - a);
            const double ar = mag(nv);
            sumN = sumN + nv;
            sumA += ar;
            sumAc = sumAc + ar * c;
        };
        int np;
        V3 q0, q1, q2;
        if (FP == 4 || n <= 4) {
            const CutWalk w = walks[(n == 3 ? 16u : 0u) + mask];
            np = (int)(w.info & 15u);
            nIf = (int)((w.info >> 4) & 15u);
            listCrossing(w, 0);
            listCrossing(w, 1);
            if (nIf > 2) {
                listCrossing(w, 2);
                listCrossing(w, 3);
            }
            q0 = listEntry(w, 0);
            q1 = listEntry(w, 1);
            q2 = listEntry(w, 2);
            const V3 q3 = listEntry(w, 3), q4 = listEntry(w, 4);
            fC = q0 + q1 + q2;
            fC = vsel(np > 3, fC + q3, fC);
            fC = vsel(np > 4, fC + q4, fC);
            if (np > 5) fC = fC + listEntry(w, 5);
            // RN(1/4), RN(1/5), RN(1/6): with a correctly rounded reciprocal
            // the corrected quotient is the correctly rounded one
            fC = div_by(fC, Rcp{(double)np, np == 4 ? 0.25 : (np == 5 ? 0.2 : 1.0 / 6.0)});
            tri(q0, q1);
            tri(q1, q2);
            tri(q2, q3);
            if (np > 3) tri(q3, q4);
            if (np > 4) {
                const V3 q5 = listEntry(w, 5);
                tri(q4, q5);
                if (np > 5) tri(q5, q0);
            }
        } else {
            np = 0;
            q0 = q1 = q2 = VZERO;
            ok = walkPoints([&](V3 q) {
                fC = fC + q;
                q0 = vsel(np == 0, q, q0);
                q1 = vsel(np == 1, q, q1);
                q2 = vsel(np == 2, q, q2);
                np++;
            }, true);
            fC = div_by(fC, rcp_of((double)np));
            V3 prev = q0;
            int k = 0;
            walkPoints([&](V3 q) {
                if (k++ > 0) tri(prev, q);
                prev = q;
            }, false);
            tri(prev, q0);
        }
        const bool small = sumA < SVP_ROOTVSMALL;
        const V3 quot = div_by((1.0 / 3.0) * sumAc, rcp_of(sumA));
        centre = vsel(small, fC, quot);
        area = vsel(small, VZERO, 0.5 * sumN);
        if (np == 3) {
            centre = (1.0 / 3.0) * (q0 + q1 + q2);
            area = 0.5 * cross(q1 - q0, q2 - q0);
        }
        return ok;
    }

    // magnitude of the cut face's area alone: the triangles' own magnitudes,
    // which calcSubFaceCentreAndArea only compares with ROOTVSMALL there, are
    // taken where the area vector does not settle that (their sum is at least
    // its length)
    __device__ __attribute__((always_inline)) inline double subArea(bool& ok) {
        V3 fC = VZERO, sumN = VZERO;
        auto tri = [&](V3 a, V3 b) { sumN = sumN + cross(b - a, fC - a); };
        if (FP == 4 || n <= 4) {
            const CutWalk w = walks[(n == 3 ? 16u : 0u) + mask];
            const int np = (int)(w.info & 15u);
            nIf = (int)((w.info >> 4) & 15u);
            listCrossing(w, 0);
            listCrossing(w, 1);
            if (nIf > 2) {
                listCrossing(w, 2);
                listCrossing(w, 3);
            }
            const V3 q0 = listEntry(w, 0), q1 = listEntry(w, 1), q2 = listEntry(w, 2);
            if (np == 3) return mag(0.5 * cross(q1 - q0, q2 - q0));
            const V3 q3 = listEntry(w, 3), q4 = listEntry(w, 4);
            fC = q0 + q1 + q2 + q3;
            fC = vsel(np > 4, fC + q4, fC);
            if (np > 5) fC = fC + listEntry(w, 5);
            fC = div_by(fC, Rcp{(double)np, np == 4 ? 0.25 : (np == 5 ? 0.2 : 1.0 / 6.0)});
            tri(q0, q1);
            tri(q1, q2);
            tri(q2, q3);
            tri(q3, q4);
            if (np > 4) {
                const V3 q5 = listEntry(w, 5);
                tri(q4, q5);
                if (np > 5) tri(q5, q0);
            }
            const double a2 = magSqr(0.5 * sumN);
            if (a2 > 1e-290) return sqrt(a2);
        }
        V3 centre, area;
        ok &= subFace(centre, area);
        return mag(area);
    }
};

}  // namespace svp
