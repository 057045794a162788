// Plane placement (cutCell::findSignedDistance, cutCell.C:611-799) and the
// interface velocity Un0 (advection.C:126) of every mixed cell: one lane per
// cell face, a group of G lanes per cell.
#include <algorithm>

#include "cut_device.hpp"
#include "mesh_device.hpp"

namespace svp {

// waves per SIMD the register allocation targets (build-time tuning; results
// do not depend on it)
#ifndef SVP_FSD_WAVES
#define SVP_FSD_WAVES 2
#endif

// One wave's LDS.  The arrays over lanes hold one value per lane of the wave
// (the lane of a cell's face), components apart, so neither a lane's own
// indexed reads nor the reads of a whole group's values meet in a bank.  The
// crossings' places are used again within a cut (place_cut), which keeps the
// LDS at three waves per SIMD.
template <int G, int FP>
struct PlaceLds {
    static constexpr int NG = 64 / G;
    static constexpr int NP = G <= 8 ? NS_CELL_POINTS : GEN_CELL_POINTS;
    double ps[FP + MAX_IF_POINTS][3][64];   // the face's points, then its plane crossings in walk order
    double ar[64];                          // first interface segment's area, then the face's pyramid
    double vof[NG];                         // volume fraction of the group's cut
    CutWalk walk[24];
};

// The lane's face
template <int FP>
struct PlaceFace {
    int n;              // points, 0 for a lane without a face
    double dots[FP];    // point . normal
    V3 fullC, fullA;    // the face as a fully submerged sub-face
};

struct PlaceCut {
    int status;
    double VOF;
    V3 C, S;
    unsigned cut, sub;  // faces cut and fully submerged, one bit per face
    int nEdge;          // plane crossings on the cut faces
};

// cutCell::calcSubCell (cutCell.C:343-542) for one cell per group: every lane
// cuts its face and leaves what the cell's sums take from it in LDS; every
// lane of the group then takes the sums, in face order, and holds the result.
// A face that adds nothing to a sum (empty, not cut, or a lane without a face)
// leaves -0.0, which changes no partial sum, so the sums need no test per face.
template <int G, int FP>
__device__ __attribute__((always_inline)) inline void place_cut(PlaceLds<G, FP>& L, int t, int g, int l, int nF,
                                                                const PlaceFace<FP>& F, double dist, double Vc,
                                                                Rcp rV, bool vcPlain, PlaceCut& out, bool& ok) {
    constexpr unsigned long long GM = G == 64 ? ~0ull : ((1ull << G) - 1ull);
    // faces per cell the sums run over: all lanes of a small group (unrolled),
    // the cell's own faces in a large one
    const int nS = G <= 8 ? G : nF;
    const int gb = g * G;
    int status = 1, nIf = 0;
    V3 centre = VZERO, area = VZERO;
    if (l < nF) {
        FaceWalk<FP> w(L.ps, L.walk, t, F.n, F.dots, dist);
        status = w.status();
        centre = vsel(status == 1, VZERO, F.fullC);
        area = vsel(status == 1, VZERO, F.fullA);
        if (status == 0) {
            ok &= w.subFace(centre, area);
            nIf = w.nIf;
        }
    }
    const V3 NEG = v3(-0.0, -0.0, -0.0);
    const bool isCut = l < nF && status == 0;
    const bool isSub = l < nF && status == -1;
    if (!isCut) {
        lds3_put(L.ps[FP], t, NEG);
        lds3_put(L.ps[FP + 1], t, NEG);
    }
    const unsigned cut = (unsigned)((__ballot(isCut) >> gb) & GM);
    const unsigned sub = (unsigned)((__ballot(isSub) >> gb) & GM);
    const bool isFour = isCut && nIf > 2;
    const unsigned long long fourAll = __ballot(isFour);
    const unsigned four = (unsigned)((fourAll >> gb) & GM);
    out.cut = cut;
    out.sub = sub;
    out.nEdge = 2 * (__popc(cut) + __popc(four));
    __builtin_amdgcn_wave_barrier();
    // calcInterfaceCentreAndArea (cutCell.C:37-100)
    V3 fC = VZERO;
    if (fourAll == 0ull) {
#pragma unroll
        for (int f = 0; f < nS; ++f) fC = fC + lds3(L.ps[FP], gb + f) + lds3(L.ps[FP + 1], gb + f);
    } else {
        for (int f = 0; f < nF; ++f) {
            fC = fC + lds3(L.ps[FP], gb + f) + lds3(L.ps[FP + 1], gb + f);
            if ((four >> f) & 1u) fC = fC + lds3(L.ps[FP + 2], gb + f) + lds3(L.ps[FP + 3], gb + f);
        }
    }
    if (out.nEdge > 0) fC = div_by(fC, rcp_of((double)out.nEdge));
    V3 nv = NEG, arc = NEG;
    double ar = -0.0;
    V3 x1 = VZERO, x2 = VZERO, x3 = VZERO;
    if (isCut) {
        const V3 a = lds3(L.ps[FP], t);
        x1 = lds3(L.ps[FP + 1], t);
        nv = cross(x1 - a, fC - a);
        ar = mag(nv);
        arc = ar * (a + x1 + fC);
    }
    if (fourAll != 0ull) {
        x2 = lds3(L.ps[FP + 2], t);
        x3 = lds3(L.ps[FP + 3], t);
    }
    __builtin_amdgcn_wave_barrier();
    // the crossings are in registers now: their places take the segments'
    // normals and area moments and the sub-faces' centres
    double(&sCtr)[3][64] = L.ps[FP];
    double(&sNn)[3][64] = L.ps[FP + 2];
    double(&sArc)[3][64] = L.ps[FP + 3];
    lds3_put(sNn, t, nv);
    L.ar[t] = ar;
    lds3_put(sArc, t, arc);
    lds3_put(sCtr, t, vsel(isCut || isSub, centre, NEG));
    __builtin_amdgcn_wave_barrier();
    V3 sumN = VZERO, sumAc = VZERO;
    double sumA = 0.0;
    auto segment = [&](V3 n1, double a1, V3 c1) {
        sumN = sumN + flip_if_neg(n1, dot(n1, sumN));
        sumA += a1;
        sumAc = sumAc + c1;
    };
    if (fourAll == 0ull) {
#pragma unroll
        for (int f = 0; f < nS; ++f) segment(lds3(sNn, gb + f), L.ar[gb + f], lds3(sArc, gb + f));
    } else {
        // a face the plane crosses four times has two more segments, which
        // the lanes take from its lane's crossings
        for (int f = 0; f < nF; ++f) {
            segment(lds3(sNn, gb + f), L.ar[gb + f], lds3(sArc, gb + f));
            const V3 p1 = v3(__shfl(x1.x, gb + f), __shfl(x1.y, gb + f), __shfl(x1.z, gb + f));
            const V3 p2 = v3(__shfl(x2.x, gb + f), __shfl(x2.y, gb + f), __shfl(x2.z, gb + f));
            const V3 p3 = v3(__shfl(x3.x, gb + f), __shfl(x3.y, gb + f), __shfl(x3.z, gb + f));
            if ((four >> f) & 1u) {
                const V3 n1 = cross(p2 - p1, fC - p1);
                const double a1 = mag(n1);
                segment(n1, a1, a1 * (p1 + p2 + fC));
                const V3 n2 = cross(p3 - p2, fC - p2);
                const double a2 = mag(n2);
                segment(n2, a2, a2 * (p2 + p3 + fC));
            }
        }
    }
    const bool small = sumA < SVP_ROOTVSMALL;
    const V3 quot = div_by((1.0 / 3.0) * sumAc, rcp_of(sumA));
    V3 C = vsel(small, fC, quot), S = vsel(small, VZERO, 0.5 * sumN);
    if (dot(S, C) < 0.0) S = (-1.0) * S;
    // mag(S) < TSMALL: the root only where its square does not settle it
    const double s2 = magSqr(S);
    bool tiny = false;
    if (!(s2 > 1.01e-28)) tiny = sqrt(s2) < SVP_TSMALL;
    // calcSubCellCentreAndVolume (cutCell.C:103-137)
    V3 sum = VZERO;
#pragma unroll
    for (int f = 0; f < nS; ++f) sum = sum + lds3(sCtr, gb + f);
    sum = sum + C;
    const V3 cEst = div_by(sum, rcp_of((double)(__popc(cut | sub) + 1)));
    L.ar[t] = (isCut || isSub) ? fmax(fabs(dot(area, centre - cEst)), SVP_VSMALL) : -0.0;
    __builtin_amdgcn_wave_barrier();
    double vol = 0.0;
#pragma unroll
    for (int f = 0; f < nS; ++f) vol += L.ar[gb + f];
    vol += fmax(fabs(dot(S, C - cEst)), SVP_VSMALL);
    vol = div_by(vol, Rcp{3.0, 1.0 / 3.0});
    const double VOF = vcPlain ? div_by(vol, rV) : vol / Vc;
    const unsigned all = nF >= 32 ? ~0u : ((1u << nF) - 1u);
    const bool empty = (cut | sub) == 0u, full = sub == all;
    const bool inside = !empty && !full;
    const bool one = full || (inside && tiny && sub != 0u);
    out.status = (inside && !tiny) ? 0 : (one ? -1 : 1);
    out.VOF = (inside && !tiny) ? VOF : (one ? 1.0 : 0.0);
    out.C = vsel(inside, C, VZERO);
    out.S = vsel(inside, S, VZERO);
    __builtin_amdgcn_wave_barrier();
}

// Un0 = U(interface centre) . n of a cut cell (advection.C:126):
// interpolationCellPoint's tet search with one lane per face (point(k), pl:
// the face's points and their labels) and its cell-point interpolation
template <int G, int FP, class Point>
__device__ __attribute__((always_inline)) inline double group_un0(const DevMesh& m, const DevState& st, int g, int l,
                                                                  int nF, int c, V3 Cc, int fsz, Point point,
                                                                  const int (&pl)[FP], bool ownFace, V3 pos,
                                                                  V3 normalI) {
    const double tol = SVP_SMALL;
    bool found = false;
    double bw[4] = {0, 0, 0, 0}, bestMin = -1e300;
    int bp[3] = {0, 0, 0};
    if (l < nF) {
#pragma unroll
        for (int k = 1; k < FP - 1; ++k) {
            if (k >= fsz - 1 || found) continue;
            const V3 b0 = point(0), qa = point(k), qb = point(k + 1);
            const V3 b1 = vsel(ownFace, qa, qb), b2 = vsel(ownFace, qb, qa);
            const V3 e0 = Cc - b2, e1 = b0 - b2, e2 = b1 - b2;
            const double detT = dot(e0, cross(e1, e2));
            double w[4];
            if (fabs(detT) < SVP_SMALL) {
                w[0] = w[1] = w[2] = w[3] = -1.0;
            } else {
                const V3 r = pos - b2;
                w[0] = dot(r, cross(e1, e2)) / detT;
                w[1] = dot(e0, cross(r, e2)) / detT;
                w[2] = dot(e0, cross(e1, r)) / detT;
                w[3] = 1.0 - w[0] - w[1] - w[2];
            }
            const double mn = fmin(fmin(w[0], w[1]), fmin(w[2], w[3]));
            const bool in = mn + tol > 0.0;
            if (in || mn > bestMin) {
                found = in;
                bestMin = mn;
#pragma unroll
                for (int s = 0; s < 4; ++s) bw[s] = w[s];
                bp[0] = pl[0];
                bp[1] = ownFace ? pl[k] : pl[k + 1];
                bp[2] = ownFace ? pl[k + 1] : pl[k];
            }
        }
    }
    // first face (in cell-face order) with a containing tet, else the tet of
    // largest minimum weight, earliest on ties
    const unsigned long long grpMask = ((1ull << G) - 1ull) << (g * G);
    const unsigned long long foundMask = __ballot(found && l < nF) & grpMask;
    int src = 0;
    if (foundMask) {
        src = __ffsll((long long)foundMask) - 1 - g * G;
    } else {
        double best = -1e300;
        for (int k = 0; k < nF; ++k) {
            const double v = __shfl(bestMin, g * G + k);
            if (v > best) {
                best = v;
                src = k;
            }
        }
    }
    double w[4];
    int pp[3];
#pragma unroll
    for (int s = 0; s < 4; ++s) w[s] = __shfl(bw[s], g * G + src);
#pragma unroll
    for (int s = 0; s < 3; ++s) pp[s] = __shfl(bp[s], g * G + src);
    // point values: lane s of the group evaluates point s
    V3 pu = VZERO;
    if (l < 3) pu = point_u(m, st, (l == 0) ? pp[0] : (l == 1 ? pp[1] : pp[2]));
    V3 pv[3];
#pragma unroll
    for (int s = 0; s < 3; ++s)
        pv[s] = v3(__shfl(pu.x, g * G + s), __shfl(pu.y, g * G + s), __shfl(pu.z, g * G + s));
    const V3 Ui = w[0] * ld3(st.U, c) + w[1] * pv[0] + w[2] * pv[1] + w[3] * pv[2];
    return dot(Ui, normalI);
}

// Groups that cut one cell at different distances at the same time: with few
// mixed cells a wave has its SIMD to itself and the kernel takes one wave's
// chain of cuts (34 us for 270 hexahedra), so lanes left over go into trying several vertex levels (and
// both thirds of the last bracket) at once: 6 groups take a hexahedron's
// seven dependent cuts to three, 3 to four, 2 to four or five.  The widest
// split is taken whose waves all have a SIMD each (3.5k hexahedra: 38.4 us
// with 2 groups on 707 waves, 42.3 with 3 on 1177, 42.1 with 1 on 354).
constexpr int PLACE_WAVES = 1024;
template <int G>
__device__ inline int place_split(int nWork) {
    constexpr int NG = 64 / G;
    const int waves = min(PLACE_WAVES / (int)gridDim.y, (int)gridDim.x);   // a batch's cases share the chip
    auto fits = [&](int s) { return s <= NG && (nWork + NG / s - 1) / (NG / s) <= waves; };
    if constexpr (G == 6) {
        if (fits(6)) return 6;
        if (fits(3)) return 3;
    }
    if constexpr (G == 8) {
        if (fits(8)) return 8;
        if (fits(4)) return 4;
    }
    return fits(2) ? 2 : 1;
}

// findSignedDistance and Un0 of one mixed cell per S groups of G lanes, one
// lane per cell face (cells of at most G faces; FP: points per face).  All
// lanes of a cell hold the same volume fractions, so they follow the same
// bracketing and Newton steps as one lane would.  One wave per workgroup: the
// LDS traffic of a wave is in order.
//
// Bound by issue where every SIMD has two waves (about 1350 instructions per
// cut, 700 of them FP64) and by the chain of dependent cuts, each a chain of
// divisions, square roots and sums in the reference's order, below that.
// Against records of whole faces in LDS, tested face by face, with each
// crossing divided twice and one cut at a time: 21k hexahedra (128^3,
// perturbed) 141 -> 85 us, 3.5k (64^3) 76 -> 38, 270 (16^3) 69 -> 25, 1.2k
// tetrahedra 59 -> 36; 3.9k cells of a 2:1 refined mesh 1416 -> 105 us (one
// lane per cell before), their Un0 75 -> 7.6.
template <int G, int FP>
__device__ __attribute__((always_inline)) inline void k_fsd_group_body(const DevMesh& m, const DevState& st, const int* wl, const int* wn) {
    using Lds = PlaceLds<G, FP>;
    constexpr int NG = Lds::NG, NP = Lds::NP;
    constexpr int PPL = (NP + G - 1) / G;  // cell points per lane
    static_assert((FP + MAX_IF_POINTS) * 3 * 64 >= 2 * NG * NP, "the levels fit over the points");
    __shared__ Lds L;
    const int t = threadIdx.x;
    if (t < 24) L.walk[t] = kCutWalks.w[t];
    __syncthreads();
    const int nWork = wl ? *wn : *st.nMixed;
    const int S = place_split<G>(nWork);
    const int cells = NG / S;                 // per wave
    const int g = t / G, l = t % G;           // group of the wave, face of the cell
    const int slot = g / S, s = g % S;        // cell of the wave, its group
    if (slot >= cells) return;
    for (int wi = blockIdx.x * cells + slot; wi < nWork; wi += gridDim.x * cells) {
        const int i = wl ? wl[wi] : wi;
        const int c = st.mixed[i];
        int nF, np;
        const int fb = cell_faces(m, c, nF), pb = cell_points(m, c, np);
        const V3 normalI = ld3(st.ifN, i);
        const double alphaI = st.alpha[c];
        const V3 Cc = ld3(m.C, c);
        const double Vc = m.V[c];
        // (a cell without faces has no loads to make and no plane)
        if (nF == 0 || mag(normalI) < SVP_TSMALL) {
            if (l == 0 && s == 0) {
                st.status[i] = (int)sgn(0.5 - alphaI);
                st.nCutPts[i] = 0;
                st.faceClass[i] = 0ull;
                if (!st.fsdKeep) {
                    st.ifD[i] = 0.0;
                    st3(st.ifC, i, VZERO);
                    st3(st.ifS, i, VZERO);
                }
                st.un0[i] = 0.0;
            }
            continue;
        }
        // The lane's face and cell points, every load unconditional (slots
        // past the cell's faces or points, or past the face's points, repeat
        // the last one): the face chain and the point chain go out together,
        // where loads under a lane condition would each wait for all the
        // loads before them.
        const int fL = m.cFaces[fb + min(l, nF - 1)];
        int cp[PPL];
#pragma unroll
        for (int k = 0; k < PPL; ++k) cp[k] = m.cPts[pb + min(l + k * G, np - 1)];
        int fsz;
        const int s0 = face_points(m, fL, fsz);
        int pl[FP];
#pragma unroll
        for (int k = 0; k < FP; ++k) pl[k] = m.fPts[s0 + min(k, fsz - 1)];
        V3 q[FP];
#pragma unroll
        for (int k = 0; k < FP; ++k) q[k] = ld3(m.pts, pl[k]);
        V3 cpt[PPL];
#pragma unroll
        for (int k = 0; k < PPL; ++k) cpt[k] = ld3(m.pts, cp[k]);
        PlaceFace<FP> F;
        F.fullC = ld3(m.fullCS, 2 * fL);
        F.fullA = ld3(m.fullCS, 2 * fL + 1);
        F.n = l < nF ? fsz : 0;
        const bool ownFace = m.own[fL] == c;
        // vertex levels -n.x of the cell points, sorted descending by rank
        // (over the points' LDS, which is filled after); lane l of the group
        // keeps the levels of rank l, l + G, ...
        double lev[PPL];
        {
            double* raw = &L.ps[0][0][0] + g * NP;
            double* srt = &L.ps[0][0][0] + (NG + g) * NP;
            double v[PPL];
            int rank[PPL];
#pragma unroll
            for (int k = 0; k < PPL; ++k) {
                v[k] = -dot(normalI, cpt[k]);
                rank[k] = 0;
                if (l + k * G < np) raw[l + k * G] = v[k];
            }
            __builtin_amdgcn_wave_barrier();
            for (int j = 0; j < np; ++j) {
                const double x = raw[j];
#pragma unroll
                for (int k = 0; k < PPL; ++k) rank[k] += (x > v[k]) || (x == v[k] && j < l + k * G);
            }
#pragma unroll
            for (int k = 0; k < PPL; ++k)
                if (l + k * G < np) srt[rank[k]] = v[k];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int k = 0; k < PPL; ++k) lev[k] = srt[min(l + k * G, np - 1)];
            __builtin_amdgcn_wave_barrier();
        }
        auto level = [&](int r) {
            double x = __shfl(lev[0], g * G + r % G);
#pragma unroll
            for (int k = 1; k < PPL; ++k) {
                const double y = __shfl(lev[k], g * G + r % G);
                x = r >= k * G ? y : x;
            }
            return x;
        };
        // the plane's normal is fixed for the cell: dot(point, n) once
#pragma unroll
        for (int k = 0; k < FP; ++k) {
            lds3_put(L.ps[k], t, q[k]);
            F.dots[k] = dot(q[k], normalI);
        }
        __builtin_amdgcn_wave_barrier();
        bool ok = true;
        const Rcp rV = rcp_of(Vc);
        const bool vcPlain = fabs(Vc) > 1e-250 && fabs(Vc) < 1e250;
        // one loop around a single cut, so that the cut's code exists once:
        // phase 0 bisects over the vertex levels, 1 and 2 cut at a third and
        // two thirds of the last bracket, 3 is the final cut at the plane found
        double lowDistance = level(0), upDistance = level(np - 1);
        int lowLabel = 0, upLabel = np - 1;
        double lowAlpha = 0.0, upAlpha = 1.0;
        PlaceCut cc;
        double dOut = 0.0, deltaDistance = 0.0, alphaOneThird = 0.0;
        int phase = 0, owner = 0;   // group holding the final cut
        while (true) {
            double dist;
            int lab0 = 0, lab1 = -1, lab2 = -1, from = -1;   // labels cut this round (from + 1 + s when from >= 0)
            if (phase == 0) {
                const int inner = upLabel - lowLabel - 1;
                if (inner > 0) {
                    int lab;
                    if (FP <= 4 && inner <= S) {
                        from = lowLabel;
                        lab = lowLabel + 1 + min(s, inner - 1);
                    } else {
                        // the middle level (0.5 (up + low), halves away from
                        // zero) and, with groups to spare, what follows it on
                        // either side; two groups try the side where alpha
                        // would lie if it grew evenly over the bracket
                        lab0 = (upLabel + lowLabel + 1) >> 1;
                        const int below = (lowLabel + lab0 + 1) >> 1, above = (lab0 + upLabel + 1) >> 1;
                        // (not for faces of more than 4 points, whose cut can
                        // fail: only the levels the bisection visits count)
                        if (FP > 4) {
                        } else if (S >= 3) {
                            lab1 = below;
                            lab2 = above;
                        } else if (S == 2) {
                            lab1 = 2.0 * (alphaI - lowAlpha) > upAlpha - lowAlpha ? above : below;
                        }
                        lab = s == 1 && lab1 >= 0 ? lab1 : (s == 2 && lab2 >= 0 ? lab2 : lab0);
                    }
                    dist = level(lab);
                } else if (fabs(lowDistance - upDistance) < SVP_TSMALL) {
                    dOut = 0.5 * (lowDistance + upDistance);
                    dist = dOut;
                    phase = 3;
                } else {
                    deltaDistance = (upDistance - lowDistance) / 3.0;
                    phase = 1;
                }
            }
            if (phase == 1) dist = s == 1 ? lowDistance + 2.0 * deltaDistance : lowDistance + deltaDistance;
            else if (phase == 2) dist = lowDistance + 2.0 * deltaDistance;
            else if (phase == 3) dist = dOut;
            place_cut<G, FP>(L, t, g, l, nF, F, dist, Vc, rV, vcPlain, cc, ok);
            if (phase == 3) break;
            if (l == 0) L.vof[g] = cc.VOF;
            __builtin_amdgcn_wave_barrier();
            const int base = g - s;
            if (phase == 0) {
                bool hit = false;
                while (upLabel - lowLabel > 1) {
                    const int mid = (upLabel + lowLabel + 1) >> 1;
                    const int at = from >= 0 ? mid - from - 1
                                             : (mid == lab0 ? 0 : (mid == lab1 ? 1 : (mid == lab2 ? 2 : -1)));
                    if (at < 0) break;
                    const double midDistance = level(mid);
                    const double midAlpha = L.vof[base + at];
                    if (fabs(midAlpha - alphaI) < SVP_TSMALL) {
                        dOut = midDistance;
                        owner = at;
                        hit = true;
                        break;
                    }
                    if (midAlpha > alphaI) {
                        upLabel = mid;
                        upDistance = midDistance;
                        upAlpha = midAlpha;
                    } else {
                        lowLabel = mid;
                        lowDistance = midDistance;
                        lowAlpha = midAlpha;
                    }
                }
                if (hit) break;
            } else if (phase == 1 && S == 1) {
                alphaOneThird = cc.VOF - lowAlpha;
                phase = 2;
            } else {
                if (S > 1) alphaOneThird = L.vof[base] - lowAlpha;
                const double alphaPrismatoid = upAlpha - lowAlpha;
                const double alphaTwoThirds = L.vof[base + (S > 1 ? 1 : 0)] - lowAlpha;
                const double a = 13.5 * alphaOneThird - 13.5 * alphaTwoThirds + 4.5 * alphaPrismatoid;
                const double b = -22.5 * alphaOneThird + 18.0 * alphaTwoThirds - 4.5 * alphaPrismatoid;
                const double cq = 9.0 * alphaOneThird - 4.5 * alphaTwoThirds + 1.0 * alphaPrismatoid;
                const double d = lowAlpha - alphaI;
                double lambda = 0.5;
                for (int iter = 0; iter < 100; iter++) {
                    const double func = a * (lambda * lambda * lambda) + b * (lambda * lambda) + cq * lambda + d;
                    const double funcPrime = 3.0 * a * (lambda * lambda) + 2.0 * b * lambda + cq;
                    const double lambdaNew = lambda - (func / funcPrime);
                    if (fabs(lambdaNew - lambda) < SVP_TSMALL) break;
                    lambda = lambdaNew;
                }
                dOut = lowDistance - lambda * (lowDistance - upDistance);
                phase = 3;
            }
            __builtin_amdgcn_wave_barrier();
        }
        // (every group's: a group without the final cut may have cut the last
        // bracket at two thirds)
        if (!ok) atomicOr(st.errFlag, ERR_TOO_MANY_CROSSINGS);
        if (s != owner) continue;
        if (l == 0) {
            unsigned long long fcls = 0ull;
            for (int k = 0; k < nF; ++k) {
                const unsigned long long s1 = ((cc.cut >> k) & 1u) ? 1ull : (((cc.sub >> k) & 1u) ? 0ull : 2ull);
                fcls |= s1 << (2 * k);
            }
            st.status[i] = cc.status;
            st.nCutPts[i] = cc.nEdge;
            st.faceClass[i] = fcls;
            st.ifD[i] = dOut;
            st3(st.ifC, i, cc.C);
            st3(st.ifS, i, cc.S);
        }
        // (a large group's Un0 waits for the advect, k_un0_group)
        if constexpr (G <= 8) {
            double un0 = 0.0;
            if (cc.status == 0) un0 = group_un0<G, FP>(m, st, g, l, nF, c, Cc, fsz, [&](int k) { return lds3(L.ps[k], t); },
                                                        pl, ownFace, cc.C, normalI);
            if (l == 0) st.un0[i] = un0;
        }
        __builtin_amdgcn_wave_barrier();
    }
}

template <int G, int FP>
__global__ void __launch_bounds__(64, SVP_FSD_WAVES) k_fsd_group(DevMesh m, DevState st, const int* wl, const int* wn) {
    k_fsd_group_body<G, FP>(m, st, wl, wn);
    if (threadIdx.x == 0) stage_stop(st, 0);
}

template <int G, int FP>
__global__ void __launch_bounds__(64, SVP_FSD_WAVES) kb_fsd_group(const BatchCase* __restrict__ bc,
                                                                  const BatchStepInfo* __restrict__ info) {
    const BatchCase& c = bc[blockIdx.y];
    const BatchStepInfo si = info[blockIdx.y];
    if (!(si.dt > 0.0)) return;
    const DevMesh m = c.m;
    k_fsd_group_body<G, FP>(m, batch_view(c, si, 0, 0), nullptr, nullptr);
}

// Un0 of every mixed cell by the same lane groups, where the plane placement
// leaves it to the advect (the velocity may be set in between)
template <int G, int FP>
__global__ void __launch_bounds__(64, 1) k_un0_group(DevMesh m, DevState st) {
    constexpr int NG = 64 / G;
    const int g = threadIdx.x / G, l = threadIdx.x % G;
    const int nMixed = *st.nMixed;
    for (int i = blockIdx.x * NG + g; i < nMixed; i += gridDim.x * NG) {
        double un0 = 0.0;
        if (st.status[i] == 0) {
            const int c = st.mixed[i];
            int nF, fsz;
            const int fb = cell_faces(m, c, nF);
            const int fL = m.cFaces[fb + min(l, nF - 1)];
            const int s0 = face_points(m, fL, fsz);
            int pl[FP];
#pragma unroll
            for (int k = 0; k < FP; ++k) pl[k] = m.fPts[s0 + min(k, fsz - 1)];
            V3 q[FP];
#pragma unroll
            for (int k = 0; k < FP; ++k) q[k] = ld3(m.pts, pl[k]);
            un0 = group_un0<G, FP>(m, st, g, l, nF, c, ld3(m.C, c), fsz, [&](int k) { return q[k]; }, pl,
                                   m.own[fL] == c, ld3(st.ifC, i), ld3(st.ifN, i));
        }
        if (l == 0) st.un0[i] = un0;
    }
}

void launch_un0_group(const DevMesh& m, const DevState& st, hipStream_t s) {
    k_un0_group<32, MAX_FACE_POINTS><<<2048, 64, 0, s>>>(m, st);
}

// 4 lanes per cell take a tetrahedron (16 cells per wave), 6 a hexahedron (10
// cells, 4 lanes idle), 8 any cell of at most 8 faces and 16 points; 32 the
// other polyhedra (up to 24 faces of up to 8 points).  More workgroups than
// the chip holds at once (2048) are queued rather than looped over, so that
// the last cells start as soon as a place is free.
void launch_fsd_group(const DevMesh& m, const DevState& st, hipStream_t s, const int* wl, const int* wn) {
    const int grid = std::max(1, std::min(4 * PLACE_WAVES, m.nC));
    switch (st.placeGroup) {
        case 4: k_fsd_group<4, 4><<<grid, 64, 0, s>>>(m, st, wl, wn); break;
        case 6: k_fsd_group<6, 4><<<grid, 64, 0, s>>>(m, st, wl, wn); break;
        case 8: k_fsd_group<8, 4><<<grid, 64, 0, s>>>(m, st, wl, wn); break;
        default: k_fsd_group<32, MAX_FACE_POINTS><<<grid, 64, 0, s>>>(m, st, wl, wn); break;
    }
}

void launch_batch_fsd_group(const BatchCase* bc, const BatchStepInfo* info, int n, int x, int G, hipStream_t s) {
    if (G == 4) kb_fsd_group<4, 4><<<dim3(x, n), 64, 0, s>>>(bc, info);
    else if (G == 6) kb_fsd_group<6, 4><<<dim3(x, n), 64, 0, s>>>(bc, info);
    else kb_fsd_group<8, 4><<<dim3(x, n), 64, 0, s>>>(bc, info);
}

// ---------------------------------------------------------------------------
// PLIC surface: reconstruction::interface (reconstruction.C:787-835) with
// cutCell::interfacePoints (cutCell.C:545-608)
// ---------------------------------------------------------------------------
// Vector::normalise of OpenFOAM: zero below ROOTVSMALL, else divided by its
// magnitude component by component
__device__ inline V3 normalised(V3 v) {
    const double s = mag(v);
    return s < SVP_ROOTVSMALL ? VZERO : v / s;
}

// One wave's LDS: per lane of a wave (a cell face) its points, crossings and
// interface segments, per group the angles of all its crossings.
template <int G, int FP>
struct PlicLds {
    static constexpr int NG = 64 / G;
    static constexpr int NX = MAX_IF_POINTS * G;
    double ps[FP + MAX_IF_POINTS][3][64];
    double sn[MAX_IF_POINTS - 1][3][64], sc[MAX_IF_POINTS - 1][3][64], sa[MAX_IF_POINTS - 1][64];
    double ang[NG][NX], sorted[NG][NX];   // crossing order, angle order
    unsigned char drop[NG][NX];           // angle order: the crossing repeats the one before it
    CutWalk walk[24];
};

// The polygon of every mixed cell, its plane cut through the mesh faces again
// (no warped-face split), as the reference does: the crossings of the cut
// faces (face order, crossing order) sorted by their angle about the interface
// centre, in a frame with z along the interface area vector and x towards the
// first crossing; a crossing whose angle lies within 1e-8 of the previous one
// in that order is dropped.  The sort is stable, like sortedOrder.
// Count mode (pts == nullptr): ptOff[i] = polygon size of mixed cell i,
// faceIdx[i] = 1 if it has a polygon.  Write mode: ptOff and faceIdx hold the
// exclusive scans of those; the polygon goes to pts[ptOff[i]..], its cell and
// first point to faceCells / faceOff at faceIdx[i].
//
// A lane per cell face, G lanes per cell, as for the plane placement: a lane
// takes its face's crossings, their angles and their places in the order;
// neither the cut faces' areas nor the volume are needed.  Bound by its chain
// of divisions, roots and sums (3.5k hexahedra are 350 waves): 136 -> 10.4 us
// a launch at 64^3 against one lane per cell with its records in scratch.
template <int G, int FP>
__global__ void __launch_bounds__(64, 1) k_plic_group(DevMesh m, DevState st, int nMixed, int* ptOff, int* faceIdx,
                                                      double* pts, int* faceCells, int* faceOff) {
    using Lds = PlicLds<G, FP>;
    constexpr int NG = Lds::NG;
    constexpr unsigned long long GM = (1ull << G) - 1ull;
    __shared__ Lds L;
    const int t = threadIdx.x;
    if (t < 24) L.walk[t] = kCutWalks.w[t];
    __syncthreads();
    const int g = t / G, l = t % G, gb = g * G;
    if (g >= NG) return;
    for (int i = blockIdx.x * NG + g; i < nMixed; i += gridDim.x * NG) {
        const int c = st.mixed[i];
        int nF, n;
        const int fb = cell_faces(m, c, nF);
        if (nF == 0) {   // no face to load, no polygon
            if (l == 0 && !pts) ptOff[i] = faceIdx[i] = 0;
            continue;
        }
        const V3 normalI = ld3(st.ifN, i);
        const double dist = st.ifD[i];
        const int fL = m.cFaces[fb + min(l, nF - 1)];
        const int s0 = face_points(m, fL, n);
        int pl[FP];
#pragma unroll
        for (int k = 0; k < FP; ++k) pl[k] = m.fPts[s0 + min(k, n - 1)];
        V3 q[FP];
#pragma unroll
        for (int k = 0; k < FP; ++k) q[k] = ld3(m.pts, pl[k]);
        double dots[FP];
#pragma unroll
        for (int k = 0; k < FP; ++k) {
            lds3_put(L.ps[k], t, q[k]);
            dots[k] = dot(q[k], normalI);
        }
        int status = 1, nIf = 0;
        bool ok = true;
        if (l < nF) {
            FaceWalk<FP> w(L.ps, L.walk, t, n, dots, dist);
            status = w.status();
            if (status == 0) {
                ok = w.crossings();
                nIf = w.nIf;
            }
        }
        if (!ok) atomicOr(st.errFlag, ERR_TOO_MANY_CROSSINGS);
        const V3 NEG = v3(-0.0, -0.0, -0.0);   // changes no sum
        if (nIf == 0) {
            lds3_put(L.ps[FP], t, NEG);
            lds3_put(L.ps[FP + 1], t, NEG);
        }
        const unsigned cut = (unsigned)((__ballot(nIf > 0) >> gb) & GM);
        const unsigned sub = (unsigned)((__ballot(l < nF && status == -1) >> gb) & GM);
        const unsigned long long fourAll = __ballot(nIf > 2);
        const unsigned four = (unsigned)((fourAll >> gb) & GM);
        const int nX = 2 * (__popc(cut) + __popc(four));
        __builtin_amdgcn_wave_barrier();
        // calcInterfaceCentreAndArea (cutCell.C:37-100)
        V3 fC = VZERO;
        for (int f = 0; f < nF; ++f) {
            fC = fC + lds3(L.ps[FP], gb + f) + lds3(L.ps[FP + 1], gb + f);
            if ((four >> f) & 1u) fC = fC + lds3(L.ps[FP + 2], gb + f) + lds3(L.ps[FP + 3], gb + f);
        }
        if (nX > 0) fC = fC / (double)nX;
        if (nIf == 0) {
            lds3_put(L.sn[0], t, NEG);
            lds3_put(L.sc[0], t, NEG);
            L.sa[0][t] = -0.0;
        }
        for (int k = 0; k + 1 < nIf; ++k) {
            const V3 a = lds3(L.ps[FP + k], t), b = lds3(L.ps[FP + k + 1], t);
            const V3 nn = cross(b - a, fC - a);
            const double ar = mag(nn);
            lds3_put(L.sn[k], t, nn);
            lds3_put(L.sc[k], t, ar * (a + b + fC));
            L.sa[k][t] = ar;
        }
        __builtin_amdgcn_wave_barrier();
        V3 sumN = VZERO, sumAc = VZERO;
        double sumA = 0.0;
        for (int f = 0; f < nF; ++f) {
            const int nSeg = ((four >> f) & 1u) ? MAX_IF_POINTS - 1 : 1;
            for (int k = 0; k < nSeg; ++k) {
                const V3 nn = lds3(L.sn[k], gb + f);
                sumN = sumN + flip_if_neg(nn, dot(nn, sumN));
                sumA += L.sa[k][gb + f];
                sumAc = sumAc + lds3(L.sc[k], gb + f);
            }
        }
        const bool small = sumA < SVP_ROOTVSMALL;
        const V3 quot = (1.0 / 3.0) * sumAc / sumA;
        V3 C = vsel(small, fC, quot), S = vsel(small, VZERO, 0.5 * sumN);
        if (dot(S, C) < 0.0) S = (-1.0) * S;
        const double magS = mag(S);
        const unsigned all = nF >= 32 ? ~0u : ((1u << nF) - 1u);
        const bool isCut = (cut | sub) != 0u && sub != all && !(magS < SVP_TSMALL) && nX > 0;
        int out = 0;   // polygon size
        if (isCut) {
            const V3 zhat = S / magS;
            V3 xhat = lds3(L.ps[FP], gb + __ffs((int)cut) - 1) - C;
            xhat = xhat - dot(xhat, zhat) * zhat;
            xhat = normalised(xhat);
            const V3 yhat = normalised(cross(zhat, xhat));
            const unsigned before = (1u << l) - 1u;
            const int first = 2 * (__popc(cut & before) + __popc(four & before));   // place of the lane's crossings
            for (int k = 0; k < nIf; ++k) {
                const V3 r = lds3(L.ps[FP + k], t) - C;
                L.ang[g][first + k] = atan2(dot(r, yhat), dot(r, xhat));
            }
            __builtin_amdgcn_wave_barrier();
            int rank[MAX_IF_POINTS];
#pragma unroll
            for (int k = 0; k < MAX_IF_POINTS; ++k) {
                if (k >= nIf) break;
                const double a = L.ang[g][first + k];
                int r = 0;
                for (int j = 0; j < nX; ++j) {
                    const double b = L.ang[g][j];
                    r += j < first + k ? !(b > a) : (a > b);
                }
                rank[k] = r;
                L.sorted[g][r] = a;
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int k = 0; k < MAX_IF_POINTS; ++k) {
                if (k >= nIf) break;
                const int r = rank[k];
                L.drop[g][r] = r > 0 && !(fabs(L.sorted[g][r] - L.sorted[g][r - 1]) > 1e-8);
            }
            __builtin_amdgcn_wave_barrier();
            for (int j = 0; j < nX; ++j) out += !L.drop[g][j];
            if (pts) {
                const int o = ptOff[i];
#pragma unroll
                for (int k = 0; k < MAX_IF_POINTS; ++k) {
                    if (k >= nIf || L.drop[g][rank[k]]) continue;
                    int at = 0;
                    for (int j = 0; j < rank[k]; ++j) at += !L.drop[g][j];
                    st3(pts, o + at, lds3(L.ps[FP + k], t));
                }
            }
        }
        if (l == 0) {
            if (!pts) {
                ptOff[i] = out;
                faceIdx[i] = out > 0 ? 1 : 0;
            } else if (out > 0) {
                faceCells[faceIdx[i]] = c;
                faceOff[faceIdx[i]] = ptOff[i];
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// lanes per cell as for the plane placement of unsplit cells
void launch_plic_polygons(const DevMesh& m, const DevState& st, int nMixed, int* ptOff, int* faceIdx, double* pts,
                          int* faceCells, int* faceOff, hipStream_t s) {
    const int grid = std::min(4 * PLACE_WAVES, cdiv(nMixed, 64 / st.plicGroup));
    switch (st.plicGroup) {
        case 4: k_plic_group<4, 4><<<grid, 64, 0, s>>>(m, st, nMixed, ptOff, faceIdx, pts, faceCells, faceOff); break;
        case 6: k_plic_group<6, 4><<<grid, 64, 0, s>>>(m, st, nMixed, ptOff, faceIdx, pts, faceCells, faceOff); break;
        case 8: k_plic_group<8, 4><<<grid, 64, 0, s>>>(m, st, nMixed, ptOff, faceIdx, pts, faceCells, faceOff); break;
        default:
            k_plic_group<32, MAX_FACE_POINTS><<<grid, 64, 0, s>>>(m, st, nMixed, ptOff, faceIdx, pts, faceCells,
                                                                  faceOff);
    }
}

}  // namespace svp
