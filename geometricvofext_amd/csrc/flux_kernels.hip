// Interface face volumes of the advection: timeIntegratedFlux
// (advection.C:85-140) over the downwind faces of the cut cells, with
// cutFace::timeIntegratedFaceFlux / timeIntegratedArea (cutFace.C:262-506).
//
// A face's swept area is Simpson's rule over the sub-intervals between its
// points' arrival times; every cut it needs (the start, each sub-interval's
// end and its middle) depends on the times alone, so a group of lanes can take
// one cut each: 2 (n - 1) + 1 lanes for a face of n points, 5 for each
// triangle of a warped face's fan.  The sub-intervals are then added in time
// order, the reference's order.
#include <algorithm>
#include <cmath>

#include "cut_device.hpp"
#include "mesh_device.hpp"

namespace svp {

// waves per SIMD the register allocation targets (build-time tuning; results
// do not depend on it)
#ifndef SVP_FLUX_WAVES
#define SVP_FLUX_WAVES 3
#endif

// lanes per face: 5 for triangles, 7 for faces of up to 4 points, 15 for
// faces of up to 8, 20 (4 triangles of 5 lanes) where most faces are warped
constexpr int FLUX_TRI = 5, FLUX_QUAD = 7, FLUX_GEN = 2 * (MAX_FACE_POINTS - 1) + 1, FLUX_FAN = 20;

template <int FP>
struct FluxLds {
    double ps[FP + MAX_IF_POINTS][3][64];   // the points of the lane's polygon, then its crossings
    CutWalk walk[24];
};

// The times of timeIntegratedArea (cutFace.C:392-506) for a polygon of n
// points (dots = point . normal): the first and last arrival and the ends of
// the sub-intervals Simpson's rule takes, node[0] their start.
template <int FP>
struct SweptTimes {
    double node[FP + 1];
    int cnt;            // sub-intervals
    double first, last;

    __device__ __attribute__((always_inline)) inline SweptTimes(const double (&dots)[FP], int n, double distance,
                                                                Rcp rU, double dt) {
        double pt[FP];
#pragma unroll
        for (int k = 0; k < FP; ++k) {
            double x = div_by(dots[k] + distance, rU);
            x = fabs(x) < SVP_TSMALL ? 0.0 : x;
            pt[k] = k < n ? x : 1.7e308;
        }
        // ascending sort (values only): odd-even transposition, static
        // indices; the places past n stay last
#pragma unroll
        for (int r = 0; r < FP; ++r)
#pragma unroll
            for (int k = r & 1; k + 1 < FP; k += 2) {
                const double x = pt[k], y = pt[k + 1];
                pt[k] = fmin(x, y);
                pt[k + 1] = fmax(x, y);
            }
        first = pt[0];
        last = pt[2];
#pragma unroll
        for (int k = 3; k < FP; ++k) last = choose(k < n, pt[k], last);
        const double smallTime = fmax(fabs(div_by(SVP_TSMALL, rU)), SVP_TSMALL);
        double prev = first > 0.0 ? first : 0.0;
#pragma unroll
        for (int k = 0; k <= FP; ++k) node[k] = prev;
        cnt = 0;
        auto add = [&](double x) {
            cnt++;
#pragma unroll
            for (int k = 1; k <= FP; ++k) node[k] = choose(cnt == k, x, node[k]);
        };
        // the first point never ends a sub-interval: it starts the first one
        // or lies before it
#pragma unroll
        for (int k = 1; k < FP; ++k) {
            if (k < n && pt[k] > (prev + smallTime) && pt[k] < dt) {
                add(pt[k]);
                prev = pt[k];
            }
        }
        if (last > dt) add(dt);
    }
    __device__ inline double at(int i) const {
        double x = node[0];
#pragma unroll
        for (int k = 1; k <= FP; ++k) x = choose(i == k, node[k], x);
        return x;
    }
};

// One cut of timeIntegratedArea: number 0 at the start, 2k - 1 at the end of
// sub-interval k, 2k at its middle.  fullMag: the whole polygon's area as
// calcSubFace forms it; deltaTau: half of the sub-interval.
template <int FP>
__device__ __attribute__((always_inline)) inline double swept_cut(FluxLds<FP>& L, int t, int c, int n,
                                                                  const double (&dots)[FP], double distance,
                                                                  double fullMag, double Un0,
                                                                  const SweptTimes<FP>& T, double& deltaTau, bool& ok) {
    const int k = (c + 1) >> 1;
    const double tauOld = T.at(k - 1), tauNew = T.at(k);
    deltaTau = 0.5 * (tauNew - tauOld);
    double dist = distance;
    if (c > 0) dist = (c & 1) ? distance - tauNew * Un0 : distance - (tauOld + deltaTau) * Un0;
    FaceWalk<FP> w(L.ps, L.walk, t, n, dots, dist);
    const int s = w.status();
    return s == 0 ? w.subArea(ok) : (s == 1 ? 0.0 : fullMag);
}

// timeIntegratedArea of a polygon whose points are in ps, by the lanes base,
// base + 1, ... (this lane is number c), one cut each.  Every lane returns the
// result.
template <int FP>
__device__ __attribute__((always_inline)) inline double group_tia(FluxLds<FP>& L, int t, int base, int c, int n,
                                                                  const double (&dots)[FP], double distance,
                                                                  double fullMag, double Un0, double dt, double magSf,
                                                                  bool& ok) {
    const SweptTimes<FP> T(dots, n, distance, rcp_of(Un0), dt);
    if (T.last <= 0.0) return magSf * dt * pos0(Un0);
    if (T.first >= dt) return magSf * dt * (1.0 - pos0(Un0));
    const bool late = T.first > 0.0;
    const double before = magSf * (1.0 - pos0(Un0));
    double area = before, deltaTau = 0.0;
    if (c == 0 ? !late : ((c + 1) >> 1) <= T.cnt)
        area = swept_cut<FP>(L, t, c, n, dots, distance, fullMag, Un0, T, deltaTau, ok);
    const double subNew = __shfl(area, t - 1), subOld = __shfl(area, c == 2 ? t - 2 : t - 3);
    const double term = div_by(deltaTau, Rcp{3.0, 1.0 / 3.0}) * (subOld + 4.0 * area + subNew);
    double sum = late ? before * T.first : 0.0;
    if (!(T.last > dt)) sum += magSf * (dt - T.last) * pos0(Un0);
    for (int k = 1; k <= T.cnt; ++k) sum += __shfl(term, base + 2 * k);
    return sum;
}

// The same by one lane, cut after cut.
template <int FP>
__device__ __attribute__((always_inline)) inline double lane_tia(FluxLds<FP>& L, int t, int n,
                                                                 const double (&dots)[FP], double distance,
                                                                 double fullMag, double Un0, double dt, double magSf,
                                                                 bool& ok) {
    const SweptTimes<FP> T(dots, n, distance, rcp_of(Un0), dt);
    if (T.last <= 0.0) return magSf * dt * pos0(Un0);
    if (T.first >= dt) return magSf * dt * (1.0 - pos0(Un0));
    const bool late = T.first > 0.0;
    const double before = magSf * (1.0 - pos0(Un0));
    double sum = late ? before * T.first : 0.0;
    if (!(T.last > dt)) sum += magSf * (dt - T.last) * pos0(Un0);
    double subOld = before, subNew = 0.0;
    for (int c = late ? 1 : 0; c <= 2 * T.cnt; ++c) {
        double deltaTau;
        const double area = swept_cut<FP>(L, t, c, n, dots, distance, fullMag, Un0, T, deltaTau, ok);
        if (c == 0) {
            subOld = area;
        } else if (c & 1) {
            subNew = area;
        } else {
            sum += div_by(deltaTau, Rcp{3.0, 1.0 / 3.0}) * (subOld + 4.0 * area + subNew);
            subOld = subNew;
        }
    }
    return sum;
}

// One face's volume.  CUTS: FG lanes take it, one lane per cut (this lane is
// number c of them, lane t of the wave), with FLUX_FAN of them four fan
// triangles at a time; else one lane takes a polygon with all its cuts, and 4
// lanes a face where most are warped (FG = FLUX_FAN).  Every lane reaches the
// same shuffles as the others of its face; the result is lane c = 0's.
template <int FG, int FP, bool CUTS>
__device__ __attribute__((always_inline)) inline double face_flux(const DevMesh& m, FluxLds<FP>& L, int t, int c,
                                                                  int f, double phi, V3 normal, double distance,
                                                                  double Un0, double dt, bool& ok) {
    const int base = t - c;
    int n;
    const int fs = face_points(m, f, n);
    const double magSf = m.magSf[f];
    const bool moving = fabs(Un0 * dt) > SVP_TSMALL;
    auto swept = [&](int from, int number, int points, const double (&dots)[FP], double full, double mg) {
        if constexpr (CUTS) return group_tia<FP>(L, t, from, number, points, dots, distance, full, Un0, dt, mg, ok);
        else return lane_tia<FP>(L, t, points, dots, distance, full, Un0, dt, mg, ok);
    };
    auto still = [&](int points, const double (&dots)[FP], double full) {
        FaceWalk<FP> w(L.ps, L.walk, t, points, dots, distance);
        const int s = w.status();
        return s == 0 ? w.subArea(ok) : (s == 1 ? 0.0 : full);
    };
    if (FG == FLUX_TRI || m.flat[f] > (1.0 - SVP_TSMALL)) {
        if (!CUTS && c > 0) return 0.0;
        int pl[FP];
        V3 q[FP];
        double dots[FP];
#pragma unroll
        for (int k = 0; k < FP; ++k) pl[k] = m.fPts[fs + min(k, n - 1)];
#pragma unroll
        for (int k = 0; k < FP; ++k) q[k] = ld3(m.pts, pl[k]);
        const double fullMag = mag(ld3(m.fullCS, 2 * f + 1));
#pragma unroll
        for (int k = 0; k < FP; ++k) {
            lds3_put(L.ps[k], t, q[k]);
            dots[k] = dot(q[k], normal);
        }
        if (moving) return phi / magSf * swept(base, c, n, dots, fullMag, magSf);
        const double alphaf = still(n, dots, fullMag) / magSf;
        return (phi * dt * alphaf);
    }
    // a warped face is the fan of triangles (centre, point j, point j + 1)
    constexpr int PAR = FG == FLUX_FAN ? 4 : 1;    // triangles at a time
    constexpr int W = CUTS ? FLUX_TRI : 1;         // lanes per triangle
    const int sub = c / W;
    const V3 fc = ld3(m.Cf, f);
    double dVf = 0.0;
    for (int j0 = 0; j0 < n; j0 += PAR) {
        const int j = j0 + sub;
        double term = 0.0;
        if (sub < PAR && j < n) {
            const V3 pa = ld3(m.pts, m.fPts[fs + j]);
            const V3 pb = ld3(m.pts, m.fPts[fs + (j + 1 == n ? 0 : j + 1)]);
            lds3_put(L.ps[0], t, fc);
            lds3_put(L.ps[1], t, pa);
            lds3_put(L.ps[2], t, pb);
            double dots[FP];
#pragma unroll
            for (int k = 0; k < FP; ++k) dots[k] = dot(k == 0 ? fc : (k == 1 ? pa : pb), normal);
            const double magSfTri = mag(triAreaNormal(fc, pa, pb));
            const double phiTri = phi * magSfTri / magSf;
            if (moving) {
                term = phiTri / magSfTri * swept(base + W * sub, c % W, 3, dots, magSfTri, magSfTri);
            } else {
                const double alphafTri = still(3, dots, magSfTri) / magSfTri;
                term = (phiTri * dt * alphafTri);
            }
        }
#pragma unroll
        for (int k = 0; k < PAR; ++k) {
            const double x = __shfl(term, base + W * k);
            if (j0 + k < n) dVf += x;
        }
    }
    return dVf;
}

// timeIntegratedFlux over the (cut cell, downwind face) pairs of the work
// list, or (tetrahedra, whose light faces do not repay the list) over every
// (mixed cell, face) pair, the upwind ones dropping out; that form also writes
// the needBounding tags the list kernel writes otherwise.  One wave per
// workgroup, LANES lanes per pair.
template <int FG, int FP, bool LISTED, bool CUTS>
__device__ __attribute__((always_inline)) inline void interface_flux_pairs(const DevMesh& m, const DevState& st,
                                                                           FluxLds<FP>& L, double dt, int slots,
                                                                           int epoch, long nWork) {
    constexpr int LANES = CUTS ? FG : (FG == FLUX_FAN ? 4 : 1);
    constexpr int PER_WAVE = 64 / LANES;
    const int t = threadIdx.x;
    const int g = t / LANES, c = t % LANES;
    if (g >= PER_WAVE) return;
    for (long wi = (long)blockIdx.x * PER_WAVE + g; wi < nWork; wi += (long)gridDim.x * PER_WAVE) {
        int i, f;
        double ph;
        if (LISTED) {
            const int2 e = st.fluxList[wi];
            i = e.x;
            f = e.y;
            ph = st.phi[f];
        } else {
            i = (int)(wi / slots);
            const int k = (int)(wi % slots);
            // the pair's cell and face loaded once, before the needBounding
            // stores (after which reloads of them would wait)
            const int cell = st.mixed[i];
            int nf;
            const int fb = cell_faces(m, cell, nf);
            if (k >= nf) continue;
            f = m.cFaces[fb + k];
            ph = st.phi[f];
            const int status = st.status[i];
            const int fo = m.own[f];
            const int fn = f < m.nIF ? m.nbr[f] : -1;
            const unsigned char em = empty_flag(m, f);
            if (c == 0) {
                if (k == 0) st.nbTag[cell] = epoch;
                if (f < m.nIF) st.nbTag[fo == cell ? fn : fo] = epoch;
            }
            if (status != 0) continue;
            bool down;
            if (f < m.nIF) down = (fo == cell) ? (ph >= 0.0) : (ph < 0.0);
            else down = !em && (ph >= 0.0);
            if (!down) continue;
        }
        bool ok = true;
        double v = 0.0;
        if (!(fabs(ph) <= SVP_TSMALL))
            v = face_flux<FG, FP, CUTS>(m, L, t, c, f, ph, ld3(st.ifN, i), st.ifD[i], st.un0[i], dt, ok);
        if (c == 0) st.dVf[f] = v;
        if (!ok) atomicOr(st.errFlag, ERR_TOO_MANY_CROSSINGS);
    }
}

// With few pairs the launch takes one chain, so a pair's cuts go to separate
// lanes; past FLUX_CUT_WAVES waves of that form the chip is full and the lanes
// that repeat a pair's loads and times cost more than the shorter chain gives:
// a lane then takes all cuts of its polygon.  Against one lane per face (or 4
// per warped face) with a copy of the walk for every cut: 16^3 27.5 -> 5.8 us,
// 64^3 31.6 -> 7.9, 33^3 perturbed (warped) 19.5 -> 7.2, 28^3 tetrahedra 18.6
// -> 8.0, refined 20^3 (larger polygons) 111 -> 14; with about 60k warped faces
// (128^3 perturbed) 55.7 with a lane per cut, 27.7 with a lane per triangle
// (50.5 before).
constexpr int FLUX_CUT_WAVES = 4096;

template <int FG, int FP, bool LISTED>
__device__ __attribute__((always_inline)) inline void k_interface_flux_body(const DevMesh& m, const DevState& st,
                                                                            double dt, int slots, int epoch) {
    __shared__ FluxLds<FP> L;
    if (threadIdx.x < 24) L.walk[threadIdx.x] = kCutWalks.w[threadIdx.x];
    __syncthreads();
    const long nWork = LISTED ? (long)*st.fluxCount : (long)*st.nMixed * slots;
    if (nWork <= (long)(FLUX_CUT_WAVES / (int)gridDim.y) * (64 / FG))
        interface_flux_pairs<FG, FP, LISTED, true>(m, st, L, dt, slots, epoch, nWork);
    else
        interface_flux_pairs<FG, FP, LISTED, false>(m, st, L, dt, slots, epoch, nWork);
}

template <int FG, int FP, bool LISTED>
__global__ void __launch_bounds__(64, FP > 4 ? 2 : SVP_FLUX_WAVES) k_interface_flux(DevMesh m, DevState st, double dt, int slots) {
    k_interface_flux_body<FG, FP, LISTED>(m, st, dt, slots, st.epoch);
}

template <int FG, int FP, bool LISTED>
__global__ void __launch_bounds__(64, FP > 4 ? 2 : SVP_FLUX_WAVES) kb_interface_flux(const BatchCase* __restrict__ bc,
                                                                        const BatchStepInfo* __restrict__ info) {
    const BatchCase& c = bc[blockIdx.y];
    const BatchStepInfo si = info[blockIdx.y];
    if (!(si.dt > 0.0)) return;
    const DevMesh m = c.m;
    const DevState st = batch_view(c, si, 1, 0);
    k_interface_flux_body<FG, FP, LISTED>(m, st, si.dt, st.maxCellFaces, si.epoch);
}

// lanes per face, by the mesh: triangles only (and cells of at most 4 faces,
// which take no work list), faces of more than 4 points, mostly warped faces,
// else mostly flat ones
int flux_kind(const DevMesh& m, int maxCellFaces, int fluxFan) {
    if (m.facePoints == 3 && maxCellFaces <= 4) return FLUX_TRI;
    if (!m.triQuadFaces) return FLUX_GEN;
    return fluxFan ? FLUX_FAN : FLUX_QUAD;
}
bool flux_listed(const DevMesh& m, int maxCellFaces) { return flux_kind(m, maxCellFaces, 0) != FLUX_TRI; }

void launch_interface_flux(const DevMesh& m, const DevState& st, double dt, hipStream_t s) {
    const int slots = st.maxCellFaces;
    const int kind = flux_kind(m, slots, st.fluxFan);
    // a wave for every few faces of an interface of twice nC^(2/3) cells (a
    // sphere's or a wavy sheet's; larger ones loop): workgroups that find no
    // face cost a few ns each
    const double faces = 2.0 * std::cbrt((double)m.nC) * std::cbrt((double)m.nC) * slots / (kind == FLUX_TRI ? 1 : 2);
    const int grid = (int)std::max(256.0, std::min((double)FLUX_CUT_WAVES, faces / (64 / kind)));
    if (kind == FLUX_TRI) k_interface_flux<FLUX_TRI, 4, false><<<grid, 64, 0, s>>>(m, st, dt, slots);
    else if (kind == FLUX_GEN) k_interface_flux<FLUX_GEN, MAX_FACE_POINTS, true><<<grid, 64, 0, s>>>(m, st, dt, slots);
    else if (kind == FLUX_FAN) k_interface_flux<FLUX_FAN, 4, true><<<grid, 64, 0, s>>>(m, st, dt, slots);
    else k_interface_flux<FLUX_QUAD, 4, true><<<grid, 64, 0, s>>>(m, st, dt, slots);
}

void launch_batch_interface_flux(const BatchCase* bc, const BatchStepInfo* info, int n, int x, int kind,
                                 hipStream_t s) {
    const dim3 grid(x, n);
    if (kind == FLUX_TRI) kb_interface_flux<FLUX_TRI, 4, false><<<grid, 64, 0, s>>>(bc, info);
    else if (kind == FLUX_GEN) kb_interface_flux<FLUX_GEN, MAX_FACE_POINTS, true><<<grid, 64, 0, s>>>(bc, info);
    else if (kind == FLUX_FAN) kb_interface_flux<FLUX_FAN, 4, true><<<grid, 64, 0, s>>>(bc, info);
    else kb_interface_flux<FLUX_QUAD, 4, true><<<grid, 64, 0, s>>>(bc, info);
}

}  // namespace svp
