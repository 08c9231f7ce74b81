// Arguments and box lookups of the per-voxel design kernels (design.hip,
// design_pass.hip).
#pragma once

#include "fdtd_common.hpp"

namespace fdtd_amd {

constexpr int kDesignMaxProbes = 8;

// (r, kappa) of a voxel and the four Kahan words of its gradients, loaded
// and stored whole
typedef float f2v __attribute__((ext_vector_type(2)));
typedef float f4v __attribute__((ext_vector_type(4)));
struct DesignArgs {
    // fields: ping-pong sets {p, vx, vy, vz}; step s reads set s & 1
    float* f[2][4];
    const uint8_t* flags;
    const float* dec[3];
    int nx, ny, nz;
    float cv0, cp0;
    // design box [lo, hi) with r = rho/rho0 and kappa = K/K0 (float32)
    int lo[3], hi[3];
    const f2v* rk;                   // device [box][2]: (r, kappa) per voxel, or NULL (air)
    // source (one point source; -1 none) and probes
    int src_i, src_j, src_k;
    const double* wave;              // device [steps]
    int n_probe;
    const int32_t* probe;            // device [n_probe][3] (i, j, k)
    float* trace;                    // device [steps][n_probe] (forward)
    const float* g;                  // device [steps][n_probe] (adjoint: dL/dy)
    // history: p on [lo-1, hi+1), div on [lo, hi); slot of step s = s - hist0
    float* hist_p;
    float* hist_div;
    int64_t hist0;
    int64_t hist_steps;
    // their rows along k: p_nk elements from cell p_k0 on (d_nk, d_k0: div). As
    // long as the boxes, or whole 4-cell lanes for passes (a lane cut by the box's
    // edge takes five stores instead of one: with 9 of them per plane they were a
    // third of a pass)
    int p_k0, p_nk, d_k0, d_nk;
    // gradient accumulators on the box: Kahan (sum, compensation) of dL/dr,
    // then of dL/dkappa, per voxel
    f4v* acc;
    // pb of every box voxel (the adjoint sweep of step n writes pbb[n & 1]),
    // read by the gradient pass of step n after the next step's sweep
    float* pbb[2];
    // gradient factor -cv / (r_lo + r_hi) of every face of the box, formed once
    // per adjoint call: x faces of cells [lo0, hi0] x [lo1, hi1) x [lo2, hi2)
    // (the face below each cell), likewise y and z; see face_offsets()
    float* face_e;
    // tiling; the strips that meet the design box form the sub-grid
    // [b_seg0, b_seg1) x [b_sj0, b_sj1) x [b_si0, b_si1)
    int planes, nseg, nstrip_j, nwaves, blocks_per_xcd;
    int b_seg0, b_seg1, b_sj0, b_sj1, b_si0, b_si1, b_blocks_per_xcd;
    int rows;  // rows per plain strip; the box strips split them
    // multi-step passes: face coefficients along x, y, z and the cell coefficient
    // of the box grown by one cell below, its lanes whole ([4][coef_cells()]), the
    // updated velocities of an adjoint pass's first steps there ([steps - 1][3]
    // [coef_cells()]) and the pb of its steps ([steps][dbox_cells()])
    const float* coef;
    float* pass_w;
    float* pass_pb;
    // the box launch: planes [b_i0, b_i1) in nb_i strips of box_planes planes
    int box_planes, b_i0, b_i1, nb_i;
};

__host__ __device__ inline int64_t ebox_cells(const DesignArgs& a) {
    return static_cast<int64_t>(a.hi[0] - a.lo[0] + 2) * (a.hi[1] - a.lo[1] + 2) * a.p_nk;
}

__host__ __device__ inline int64_t dbox_cells(const DesignArgs& a) {
    return static_cast<int64_t>(a.hi[0] - a.lo[0]) * (a.hi[1] - a.lo[1]) * a.d_nk;
}

__device__ __forceinline__ float cvf(const DesignArgs& a, float r_lo, float r_hi) {
    return a.cv0 / ((r_lo + r_hi) * 0.5f);
}

template <typename T>
__device__ __forceinline__ GMEM T* gm(T* p) { return gmem(p); }
template <typename T>
__device__ __forceinline__ const GMEM T* gm(const T* p) { return gmem(p); }

__device__ __forceinline__ uint32_t cix(int i, int j, int k, int ny, int nz) { return lidx<uint32_t>(i, j, k, ny, nz); }
template <typename T>
__device__ __forceinline__ T ldo(const GMEM T* base, uint32_t idx) { return ldx(base, idx); }
template <typename T>
__device__ __forceinline__ void sto(GMEM T* base, uint32_t idx, T v) { stx(base, idx, v); }
// An absent (r, kappa) array means (1, 1) everywhere: its loads read this.
static __device__ __align__(8) float kDesignOne[2] = {1.0f, 1.0f};

struct BoxTab {
    const GMEM f2v* p;
    uint32_t mask;  // offsets are masked to 0 when the array is absent
    bool has;
};
__device__ __forceinline__ BoxTab box_tab(const f2v* p) {
    if (p) return {gm(p), 0xffffffffu, true};
    return {gm(reinterpret_cast<const f2v*>(kDesignOne)), 0u, false};
}
// (r, kappa) of a voxel, (1, 1) outside the box
__device__ __forceinline__ f2v box_val(const BoxTab& t, int off, bool in) {
    const f2v v = ldo(t.p, static_cast<uint32_t>(off) & t.mask);
    const f2v one = {1.0f, 1.0f};
    return (in && t.has) ? v : one;
}

__host__ __device__ inline int64_t face_count(int bx, int by, int bz, int d) {
    return static_cast<int64_t>(bx + (d == 0)) * (by + (d == 1)) * (bz + (d == 2));
}

// The region of the pass coefficients: cells whose own faces or pressure differ
// from air's, from coef_k0 (a multiple of 4) in whole lanes along k.
__host__ __device__ inline int coef_k0(const DesignArgs& a) { return (a.lo[2] - 1) & ~3; }
__host__ __device__ inline int coef_nk(const DesignArgs& a) { return ((a.hi[2] + 3) & ~3) - coef_k0(a); }
__host__ __device__ inline int64_t coef_cells(const DesignArgs& a) {
    return static_cast<int64_t>(a.hi[0] - a.lo[0] + 1) * (a.hi[1] - a.lo[1] + 1) * coef_nk(a);
}
// The history's rows: the boxes' own, or whole lanes.
inline void history_rows(DesignArgs& a, bool lanes) {
    a.p_k0 = a.lo[2] - 1;
    a.d_k0 = a.lo[2];
    int p_end = a.hi[2] + 1, d_end = a.hi[2];
    if (lanes) {
        a.p_k0 &= ~3;
        a.d_k0 &= ~3;
        p_end = (p_end + 3) & ~3;
        d_end = (d_end + 3) & ~3;
    }
    a.p_nk = p_end - a.p_k0;
    a.d_nk = d_end - a.d_k0;
}

}  // namespace fdtd_amd
