// Device helpers shared by the kernel translation units: mesh gathers and the
// batched kernels' view of a case.
#pragma once
#include "simplic_device.hpp"
#include "simplic_types.hpp"

namespace svp {

static inline int cdiv(long a, long b) { return (int)((a + b - 1) / b); }

// where a gathered empty-patch flag of face f is read: f itself for a
// boundary face; for an interior face (never empty, and its flag unused) the
// first boundary face's, clamped into the array when there is none
__device__ inline int empty_slot(const DevMesh& m, int f) { return min(max(f, m.nIF), m.nF - 1); }

// the flags of N gathered faces; a mesh without empty patches reads none (at
// 128^3 cells the alpha update, with a flag for each of six faces, took 39.5 us
// and takes 33.3, the Courant sums 36.1 and 31.4)
template <int N>
__device__ __attribute__((always_inline)) inline void empty_flags(const DevMesh& m, const int (&f)[N],
                                                                  unsigned char (&em)[N]) {
    if (m.hasEmpty) {
#pragma unroll
        for (int k = 0; k < N; ++k) em[k] = m.fEmpty[empty_slot(m, f[k])];
    } else {
#pragma unroll
        for (int k = 0; k < N; ++k) em[k] = 0;
    }
}
__device__ inline unsigned char empty_flag(const DevMesh& m, int f) {
    return m.hasEmpty ? m.fEmpty[empty_slot(m, f)] : (unsigned char)0;
}

// First entry and length of an element's list in a CSR.  A mesh whose elements
// all have the same number of entries (hexahedra, tetrahedra) needs no load for
// them: in the interface kernels, which follow chains of labels, each such load
// is a memory round trip (64^3 cells, four steps: 1130 -> 1113 us; at 128^3 the
// alpha update and the upwind pass, which stream the lists, 41 -> 40 us each).
__device__ inline int csr_range(const int* off, int same, int e, int& n) {
    if (same) {
        n = same;
        return e * same;
    }
    const int b = off[e];
    n = off[e + 1] - b;
    return b;
}
__device__ inline int cell_faces(const DevMesh& m, int c, int& nf) { return csr_range(m.cOff, m.cellFaces, c, nf); }
__device__ inline int cell_points(const DevMesh& m, int c, int& np) { return csr_range(m.cpOff, m.cellPoints, c, np); }
__device__ inline int face_points(const DevMesh& m, int f, int& n) { return csr_range(m.fOff, m.facePoints, f, n); }

// volPointInterpolation value at a point: the weighted sum of its source
// values in source order.  A point of up to PU_SLOTS sources (every interior
// point of a hexahedral mesh) loads all source labels and weights, then all
// their values, before the sum, instead of waiting on two loads per source.
constexpr int PU_SLOTS = 8;
__device__ inline V3 point_u(const DevMesh& m, const DevState& st, int p) {
    const int o0 = m.psOff[p], n = m.psOff[p + 1] - o0;
    V3 t = VZERO;
    if (n >= 1 && n <= PU_SLOTS) {
        int src[PU_SLOTS];
        double w[PU_SLOTS];
        V3 u[PU_SLOTS];
#pragma unroll
        for (int k = 0; k < PU_SLOTS; ++k) {
            src[k] = m.psSrc[o0 + min(k, n - 1)];
            w[k] = m.psW[o0 + min(k, n - 1)];
        }
#pragma unroll
        for (int k = 0; k < PU_SLOTS; ++k) {
            // a source is a cell (>= 0) or a boundary face (~face)
            const double* base = src[k] >= 0 ? st.U : st.Ub;
            const int idx = src[k] >= 0 ? src[k] : (~src[k]) - m.nIF;
            u[k] = ld3(base, idx);
        }
#pragma unroll
        for (int k = 0; k < PU_SLOTS; ++k)
            if (k < n) t = t + w[k] * u[k];
        return t;
    }
    for (int k = o0; k < o0 + n; ++k) {
        const int s = m.psSrc[k];
        const V3 u = (s >= 0) ? ld3(st.U, s) : ld3(st.Ub, (~s) - m.nIF);
        t = t + m.psW[k] * u;
    }
    return t;
}

// state view of a batched case: buffers as they are (swapped 0) or with alpha
// and alphaOld exchanged, bounding half of pass number `pass` of the step
__device__ inline DevState batch_view(const BatchCase& c, const BatchStepInfo& si, int swapped, int pass) {
    return c.st[((si.aPar ^ swapped) << 1) | (si.hPar ^ (pass & 1))];
}

// The GPU times of reconstruct and advect, taken by their own kernels: an event
// record before and after each (four commands that the kernels of a step
// queue behind) took 14 us of a 125 us step at 16^3 cells, 12 at 64^3 (four
// steps 888 -> 838 us).  The first kernel of a stage adds up what has
// ended before it and notes its start; every block of the kernels that can be
// the stage's last notes its end, in one of CLOCK_SLOTS words, by a maximum that
// nothing waits for.  So a time runs from the first block of the first kernel
// to the last block of the last one, without the command processor's work before and
// after, which events around the call include: 331 us a step at 128^3 where they
// give 342.
// adds the finished stages to their sums (one wave)
__device__ inline void stage_fold(const DevState& st, int lane) {
    for (int k = 0; k < 2; ++k) {
        unsigned long long end = st.clock[CLOCK_STRIDE + (k * CLOCK_SLOTS + lane) * CLOCK_STRIDE];
        for (int o = 32; o > 0; o >>= 1) {
            const unsigned long long x = __shfl_xor(end, o);
            end = x > end ? x : end;
        }
        if (lane == 0) {
            const unsigned long long start = st.clock[k];
            if (start != 0ull && end > start) st.clock[2 + k] += end - start;
            st.clock[k] = 0ull;
        }
    }
}
__device__ inline void stage_start(const DevState& st, int stage, int lane) {
    const unsigned long long now = wall_clock64();
    stage_fold(st, lane);
    if (lane == 0) st.clock[stage] = now;
}
// (one lane per wave)
__device__ inline void stage_stop(const DevState& st, int stage) {
    const int slot = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) & (CLOCK_SLOTS - 1);
    atomicMax(&st.clock[CLOCK_STRIDE + (stage * CLOCK_SLOTS + slot) * CLOCK_STRIDE],
              (unsigned long long)wall_clock64());
}
// the same by one lane of every block, once all its waves are done
__device__ inline void stage_stop_block(const DevState& st, int stage) {
    __syncthreads();
    if (threadIdx.x == 0) stage_stop(st, stage);
}

}  // namespace svp
