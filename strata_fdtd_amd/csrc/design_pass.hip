// Multi-step passes of the per-voxel design solve (gfx950): the forward step and
// the time-reversed adjoint step three at a time, as k_multi_step takes the plain
// step (windows of 4-cell lanes marched along i as a pipeline of stages; see
// there). Cell by cell the operations and their order are those of the one-step
// sweeps in design.hip, so the results are the same bit for bit.
//
// A voxel's face and cell coefficients (k_design_coefs, formed once per call by the
// same division of the same two r values; in the stages it would be three IEEE
// divisions per cell and step) are loaded with its plane and stay in LDS, a slot
// per plane in flight, until the last stage has used them. With the stages'
// exchange that is the LDS of a CU for one workgroup of 512 threads.
//
// What bounds them at 192^3 with a 128^3 box (both sets, coefficients and flags in
// the Infinity Cache): the latency of a plane's two LDS phases and its vector
// work at this occupancy; the one-step sweeps moved 320 MB per step. Per three
// steps: forward with history 103-108 us, adjoint 117, gradient terms 51, where the
// one-step kernels took 141, 215 and 56.

#include <algorithm>

#include "design_common.hpp"
#include "pass_device.hpp"

namespace fdtd_amd {

constexpr int kDesignPassThreads = 512;

// cv of the three upper faces and cp of every cell of the coefficient region.
__global__ __launch_bounds__(256) void k_design_coefs(const DesignArgs a, float* __restrict__ coef) {
    const int bx = a.hi[0] - a.lo[0], by = a.hi[1] - a.lo[1], bz = a.hi[2] - a.lo[2];
    const int nk = coef_nk(a), k0 = coef_k0(a);
    const int64_t cells = coef_cells(a);
    const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= cells) return;
    const int ck = static_cast<int>(e % nk) + k0 - a.lo[2];
    const int cj = static_cast<int>((e / nk) % (by + 1)) - 1;
    const int ci = static_cast<int>(e / (static_cast<int64_t>(nk) * (by + 1))) - 1;
    const BoxTab RK = box_tab(a.rk);
    auto at = [&](int i, int j, int k) {
        const bool in = i >= 0 && i < bx && j >= 0 && j < by && k >= 0 && k < bz;
        return box_val(RK, in ? (i * by + j) * bz + k : 0, in);
    };
    const f2v v = at(ci, cj, ck);
    coef[e] = cvf(a, v.x, at(ci + 1, cj, ck).x);
    coef[cells + e] = cvf(a, v.x, at(ci, cj + 1, ck).x);
    coef[2 * cells + e] = cvf(a, v.x, at(ci, cj, ck + 1).x);
    coef[3 * cells + e] = a.cp0 * v.y;
}

// A thread's place in the coefficient region: its lane is in it or not, whole.
struct CoefLane {
    const GMEM float* base;
    uint32_t off, plane, cells;
    int i_lo, i_hi;
    bool in;
};
__device__ __forceinline__ CoefLane coef_lane(const DesignArgs& a, const PassWindow& w) {
    CoefLane c;
    const int nk = coef_nk(a), k0 = coef_k0(a);
    c.base = gmem(a.coef);
    c.plane = static_cast<uint32_t>(a.hi[1] - a.lo[1] + 1) * nk;
    c.cells = static_cast<uint32_t>(coef_cells(a));
    c.i_lo = a.lo[0] - 1;
    c.i_hi = a.hi[0];
    c.in = a.coef && w.ld && w.j >= a.lo[1] - 1 && w.j < a.hi[1] && w.k >= k0 && w.k < k0 + nk;
    c.off = c.in ? static_cast<uint32_t>(w.j - a.lo[1] + 1) * nk + (w.k - k0) : 0u;
    return c;
}
// coefficient q (0..2 faces along x, y, z, 3 cell) of plane i, `air` off the region
__device__ __forceinline__ f4v coef_at(const CoefLane& c, int q, int i, float air) {
    f4v v = {air, air, air, air};
    if (c.in && i >= c.i_lo && i < c.i_hi)
        v = ld4(c.base, q * c.cells + static_cast<uint32_t>(i - c.i_lo) * c.plane + c.off);
    return v;
}

// A thread's place in the planes of a box array whose rows are whole lanes, n cells
// from cell k0 (a multiple of 4) on: row `row` of `rows`.
struct BoxLane {
    uint32_t off;
    bool in;
};
__device__ __forceinline__ BoxLane box_lane(const PassWindow& w, int row, int rows, int k0, int n) {
    BoxLane b{0u, w.out && row >= 0 && row < rows && w.k >= k0 && w.k < k0 + n};
    if (b.in) b.off = static_cast<uint32_t>(row * n + (w.k - k0));
    return b;
}
template <bool NT>
__device__ __forceinline__ void st_box(GMEM float* plane, const BoxLane& b, f4v v) {
    if (b.in) st4<NT>(plane, b.off, v);
}

// Lane q of a wave holds probe q's plane if the probe lies in the given rows and
// cells (kNowhere otherwise).
__device__ __forceinline__ int probe_plane(const DesignArgs& a, int lane, int j0, int j1, int k0, int k1) {
    if (lane >= a.n_probe) return kNowhere;
    const int pj = a.probe[3 * lane + 1], pk = a.probe[3 * lane + 2];
    return pj >= j0 && pj < j1 && pk >= k0 && pk < k1 ? a.probe[3 * lane] : kNowhere;
}

struct ForwardStage {
    f4v vx, vy, vz, vxp;
    uint32_t f;
};

// Steps s .. s + kPassSteps - 1 of the forward solve.
template <bool NTS>
__global__ __launch_bounds__(kDesignPassThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_design_forward_pass(
    const DesignArgs a, const PassTile mt, int64_t s) {
    constexpr int T = kPassSteps, NT = kDesignPassThreads;
    __shared__ f4v sP[T][NT];
    __shared__ f4v sY[T][NT + 1];
    __shared__ float sX[T][NT];
    __shared__ float sZ[T][NT + 1];
    // the coefficients of the stages' planes (plane i in slot i mod T), each thread's own
    __shared__ f4v sC[T][4][NT];
    const int lb = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (lb >= mt.nwg) return;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const f4v zero = {0.f, 0.f, 0.f, 0.f};
    if (tid < T) {
        sY[tid][NT] = zero;
        sZ[tid][NT] = 0.f;
    }
    const int par = static_cast<int>(s & 1);
    const GMEM float* __restrict__ P = gmem(a.f[par][0]);
    const GMEM float* __restrict__ VX = gmem(a.f[par][1]);
    const GMEM float* __restrict__ VY = gmem(a.f[par][2]);
    const GMEM float* __restrict__ VZ = gmem(a.f[par][3]);
    const GMEM uint8_t* __restrict__ FL = gmem(a.flags);
    const uint32_t sx = static_cast<uint32_t>(ny) * static_cast<uint32_t>(nz);
    const PassWindow w = pass_window(mt, NT, tid, lb, nx, ny, nz);
    const CoefLane cl = coef_lane(a, w);
    const float dy = w.ld ? a.dec[1][w.j] : 1.f;
    f4v dz = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (w.ld && w.k + e < nz) dz[e] = a.dec[2][w.k + e];
    const int probe_i = probe_plane(a, lane, w.jlo, w.jhi, w.klo, w.khi);
    // history: p on the box grown by one cell, div on the box
    const int bx = a.hi[0] - a.lo[0], by = a.hi[1] - a.lo[1], bz = a.hi[2] - a.lo[2];
    const uint32_t p_plane = static_cast<uint32_t>((by + 2) * a.p_nk), d_plane = static_cast<uint32_t>(by * a.d_nk);
    const BoxLane pl = box_lane(w, w.j - a.lo[1] + 1, by + 2, a.p_k0, a.p_nk);
    const BoxLane dl = box_lane(w, w.j - a.lo[1], by, a.d_k0, a.d_nk);

    ForwardStage st[T];
#pragma unroll
    for (int t = 0; t < T; ++t) st[t] = ForwardStage{zero, zero, zero, zero, 0u};
    const int m0 = max(w.i0 - T, 0), m1 = w.i1 + T - 1;
    auto at = [&](int i) { return static_cast<uint32_t>(i) * sx + w.c0; };
    auto flags = [&](uint32_t c) -> uint32_t { return *reinterpret_cast<const GMEM u32u*>(at32(FL, c)); };
    f4v p0 = zero, pn = zero;
    if (w.ld) {
        const uint32_t c = at(m0);
        p0 = ld4(P, c);
        st[0].vx = ld4(VX, c);
        st[0].vy = ld4(VY, c);
        st[0].vz = ld4(VZ, c);
        st[0].f = flags(c);
        if (m0 + 1 < nx) pn = ld4(P, c + sx);
    }
    int slot[T];  // of the stages' planes
#pragma unroll
    for (int t = 0; t < T; ++t) {
        slot[t] = (T - t) % T;
#pragma unroll
        for (int q = 0; q < 4; ++q) sC[slot[t]][q][tid] = t ? zero : coef_at(cl, q, m0, q < 3 ? a.cv0 : a.cp0);
    }
    float dxs[T], dxn;
#pragma unroll
    for (int t = 1; t < T; ++t) dxs[t] = 1.f;
    dxs[0] = uni(a.dec[0], m0);
    // history of the pass's steps that are recorded (null: none)
    GMEM float *hps[T], *hds[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int64_t h = s + t - a.hist0;
        const bool on = a.hist_p && h >= 0 && h < a.hist_steps;
        hps[t] = on ? gmem(a.hist_p + h * ebox_cells(a)) : nullptr;
        hds[t] = on ? gmem(a.hist_div + h * dbox_cells(a)) : nullptr;
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        sP[t][tid] = t ? zero : p0;
        sX[t][tid] = t ? 0.f : p0.x;
    }
    __builtin_amdgcn_s_waitcnt(kWaitLoads);
    for (int m = m0; m < m1; ++m) {
        lds_barrier();  // the stages' pressures are posted
        // ---- next plane's loads
        f4v qp = zero, qx = zero, qy = zero, qz = zero;
        uint32_t qf = 0;
        if (w.ld && m + 1 < m1 && m + 1 < nx) {
            const uint32_t c = at(m + 1);
            if (m + 2 < nx) qp = ld4(P, c + sx);
            qx = ld4(VX, c);
            qy = ld4(VY, c);
            qz = ld4(VZ, c);
            qf = flags(c);
        }
        f4v qc[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) qc[q] = coef_at(cl, q, m + 1, q < 3 ? a.cv0 : a.cp0);
        dxn = uni(a.dec[0], min(m + 1, nx - 1));
        // ---- y and z faces of every stage's plane
#pragma unroll
        for (int t = 0; t < T; ++t) {
            ForwardStage& S = st[t];
            const f4v p = sP[t][tid];
            const f4v pu = sP[t][w.iu];
            const float pr = sX[t][w.ir];
            f4v vy = keep(S.vy + sC[slot[t]][1][tid] * (pu - p), S.f, 2);
            const f4v pk = {p.y, p.z, p.w, pr};
            f4v vz = keep(S.vz + sC[slot[t]][2][tid] * (pk - p), S.f, 3);
            // the last faces keep their velocity
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                vy[e] = w.jlast ? S.vy[e] : vy[e];
                vz[e] = w.vlast == e ? S.vz[e] : vz[e];
            }
            S.vz = vz;
            sY[t][tid] = vy;
            sZ[t][tid] = vz.w;
        }
        lds_barrier();
        // ---- x faces and pressures, stage by stage
        f4v cpn = pn, cx = qx, cy = qy, cz = qz;
        uint32_t cf = qf;
        f4v p = sP[0][tid];
        f4v hp[T], hd[T];  // the history's p and div
#pragma unroll
        for (int t = 0; t < T; ++t) {
            ForwardStage& S = st[t];
            const int i = m - t;
            const f4v vy = sY[t][tid];
            const f4v yb = sY[t][w.id];
            const float zb = sZ[t][w.il];
            const float dx = dxs[t];
            f4v vx = S.vx;
            if (i < nx - 1) vx = keep(S.vx + sC[slot[t]][0][tid] * (cpn - p), S.f, 1);
            const f4v zl = {zb, S.vz.x, S.vz.y, S.vz.z};
            const f4v div = ((vx - S.vxp) + (vy - yb)) + (S.vz - zl);
            f4v ps = ((keep(p + sC[slot[t]][3][tid] * div, S.f, 0) * dx) * dy) * dz;
            if (i == a.src_i && w.j == a.src_j && a.src_k >= w.k && a.src_k < w.k + 4) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (w.k + e == a.src_k && ((S.f >> (8 * e)) & FDTD_FLAG_AIR))
                        ps[e] = static_cast<float>(static_cast<double>(ps[e]) + a.wave[s + t]);
            }
            const f4v ox = vx * dx, oy = vy * dy, oz = S.vz * dz;
            const bool mine = i >= w.i0 && i < w.i1;
            for (uint64_t pm = __builtin_amdgcn_ballot_w64(probe_i == i && mine); pm; pm &= pm - 1) {
                const int q = __builtin_ctzll(pm);
                const int pj = a.probe[3 * q + 1], pk = a.probe[3 * q + 2];
                if (w.in_win && w.j == pj && pk >= w.k && pk < w.k + 4) {
                    const int e = pk - w.k;
                    a.trace[(s + t) * a.n_probe + q] = e == 0 ? ps.x : (e == 1 ? ps.y : (e == 2 ? ps.z : ps.w));
                }
            }
            hp[t] = p;
            hd[t] = div;
            // this stage's next plane: what came in (loads, or the stage before)
            const uint32_t f = S.f;
            S = ForwardStage{cx, cy, cz, vx, cf};
            if (t + 1 < T) p = sP[t + 1][tid];  // read before the next stage's p is posted
            sP[t][tid] = cpn;
            sX[t][tid] = cpn.x;
            cpn = ps;
            cx = ox;
            cy = oy;
            cz = oz;
            cf = f;
        }
        pn = qp;
        // Every store of the plane comes after the wait for the next one's loads:
        // a wait behind them would be for the stores as well (with the history
        // stored stage by stage, box or not, a step took 10 us longer).
        __builtin_amdgcn_s_waitcnt(kWaitLoads);
        {
            const int i = m - (T - 1);
            if (w.out && i >= w.i0) {
                const uint32_t c = at(i);
                st_lane<NTS>(gmem(a.f[par ^ 1][0]), c, cpn, w.nv);
                st_lane<NTS>(gmem(a.f[par ^ 1][1]), c, cx, w.nv);
                st_lane<NTS>(gmem(a.f[par ^ 1][2]), c, cy, w.nv);
                st_lane<NTS>(gmem(a.f[par ^ 1][3]), c, cz, w.nv);
            }
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int i = m - t, ei = i - a.lo[0] + 1;
            if (!hps[t] || i < w.i0 || i >= w.i1 || ei < 0 || ei >= bx + 2) continue;  // uniform
            st_box<true>(hps[t] + ei * p_plane, pl, hp[t]);
            if (ei > 0 && ei <= bx) st_box<true>(hds[t] + (ei - 1) * d_plane, dl, hd[t]);
        }
        // the slot of the plane that left the last stage takes the next plane's
        const int free_slot = slot[T - 1];
#pragma unroll
        for (int q = 0; q < 4; ++q) sC[free_slot][q][tid] = qc[q];
#pragma unroll
        for (int t = T - 1; t > 0; --t) {
            slot[t] = slot[t - 1];
            dxs[t] = dxs[t - 1];
        }
        slot[0] = free_slot;
        dxs[0] = dxn;
    }
}

struct AdjointStage {
    f4v vx, vy, vz;                 // lambda's velocities at the stage's plane
    f4v cwx;                        // cv w of the x face below it
    f4v pb;                         // its pb (q is in LDS)
    uint32_t f;
};

// Adjoint steps n, n - 1, .. n - kPassSteps + 1: lambda_{n+1} in set (n + 1) & 1
// to lambda_{n-2} in the other. q = air cp pb takes the pressure's place in the
// stages' exchange, and the products cv w of the y and z faces that of the
// velocities. What k_design_grad3 needs of each step is stored beside the
// fields: pb on the box and, but for the last step, the updated velocities.
template <bool NTS>
__global__ __launch_bounds__(kDesignPassThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_design_adjoint_pass(
    const DesignArgs a, const PassTile mt, int64_t n) {
    constexpr int T = kPassSteps, NT = kDesignPassThreads;
    __shared__ f4v sQ[T][NT];
    __shared__ f4v sY[T][NT + 1];
    __shared__ float sX[T][NT];
    __shared__ float sZ[T][NT + 1];
    // the coefficients of the stages' planes (plane i in slot i mod T), each
    // thread's own; a cell's own coefficient was used a plane ahead
    __shared__ f4v sC[T][4][NT];
    const int lb = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (lb >= mt.nwg) return;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const f4v zero = {0.f, 0.f, 0.f, 0.f};
    if (tid < T) {
        sY[tid][NT] = zero;
        sZ[tid][NT] = 0.f;
    }
    const int src = static_cast<int>((n + 1) & 1);
    const GMEM float* __restrict__ P = gmem(a.f[src][0]);
    const GMEM float* __restrict__ VX = gmem(a.f[src][1]);
    const GMEM float* __restrict__ VY = gmem(a.f[src][2]);
    const GMEM float* __restrict__ VZ = gmem(a.f[src][3]);
    const GMEM uint8_t* __restrict__ FL = gmem(a.flags);
    const uint32_t sx = static_cast<uint32_t>(ny) * static_cast<uint32_t>(nz);
    const PassWindow w = pass_window(mt, NT, tid, lb, nx, ny, nz);
    const CoefLane cl = coef_lane(a, w);
    const float dy = w.ld ? a.dec[1][w.j] : 1.f;
    f4v dz = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (w.ld && w.k + e < nz) dz[e] = a.dec[2][w.k + e];
    const int probe_i = probe_plane(a, lane, w.w0, w.w0 + mt.rows, w.k0, w.k0 + 4 * mt.kt);
    const int bx = a.hi[0] - a.lo[0], by = a.hi[1] - a.lo[1], bz = a.hi[2] - a.lo[2];
    const uint32_t b_plane = static_cast<uint32_t>(by * a.d_nk), w_plane = static_cast<uint32_t>((by + 1) * coef_nk(a));
    const BoxLane pl = box_lane(w, w.j - a.lo[1], by, a.d_k0, a.d_nk);
    const BoxLane wl = box_lane(w, w.j - a.lo[1] + 1, by + 1, coef_k0(a), coef_nk(a));

    auto at = [&](int i) { return static_cast<uint32_t>(i) * sx + w.c0; };
    auto flags = [&](uint32_t c) -> uint32_t { return *reinterpret_cast<const GMEM u32u*>(at32(FL, c)); };
    // pb of plane i from its pressure at adjoint step n - t
    auto pb_of = [&](f4v p, int i, int t, float dx) -> f4v {
        for (uint64_t pm = __builtin_amdgcn_ballot_w64(probe_i == i); pm; pm &= pm - 1) {
            const int q = __builtin_ctzll(pm);
            const int pj = a.probe[3 * q + 1], pk = a.probe[3 * q + 2];
            if (w.j == pj)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (w.k + e == pk) p[e] += a.g[(n - t) * a.n_probe + q];
        }
        return ((dx * dy) * dz) * p;
    };

    AdjointStage st[T];
#pragma unroll
    for (int t = 0; t < T; ++t) st[t] = AdjointStage{zero, zero, zero, zero, zero, 0u};
    const int m0 = max(w.i0 - T, 0), m1 = w.i1 + T - 1;
    f4v p0 = zero, pn = zero, cpl = zero;   // cpl: cp of plane m + 1
    uint32_t fn = 0;                        // flags of plane m + 1
    if (w.ld) {
        const uint32_t c = at(m0);
        p0 = ld4(P, c);
        st[0].vx = ld4(VX, c);
        st[0].vy = ld4(VY, c);
        st[0].vz = ld4(VZ, c);
        st[0].f = flags(c);
        if (m0 + 1 < nx) {
            pn = ld4(P, c + sx);
            fn = flags(c + sx);
        }
    }
    int slot[T];  // of the stages' planes
#pragma unroll
    for (int t = 0; t < T; ++t) {
        slot[t] = (T - t) % T;
#pragma unroll
        for (int q = 0; q < 4; ++q) sC[slot[t]][q][tid] = t ? zero : coef_at(cl, q, m0, q < 3 ? a.cv0 : a.cp0);
    }
    cpl = coef_at(cl, 3, m0 + 1, a.cp0);
    // the damping of the stages' planes along x, and of the plane ahead of stage 0
    float dxs[T + 1], dxn;
#pragma unroll
    for (int t = 2; t <= T; ++t) dxs[t] = 1.f;
    dxs[1] = uni(a.dec[0], m0);
    dxs[0] = uni(a.dec[0], min(m0 + 1, nx - 1));
    st[0].pb = pb_of(p0, m0, 0, dxs[1]);
    {
        const f4v q0 = keep(sC[slot[0]][3][tid] * st[0].pb, st[0].f, 0);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            sQ[t][tid] = t ? zero : q0;
            sX[t][tid] = t ? 0.f : q0.x;
        }
    }
    __builtin_amdgcn_s_waitcnt(kWaitLoads);
    for (int m = m0; m < m1; ++m) {
        lds_barrier();  // the stages' q are posted
        // ---- next plane's loads: velocities, pressure and flags one further
        f4v qp = zero, qx = zero, qy = zero, qz = zero;
        uint32_t qf = 0;
        if (w.ld && m + 1 < m1 && m + 1 < nx) {
            const uint32_t c = at(m + 1);
            if (m + 2 < nx) {
                qp = ld4(P, c + sx);
                qf = flags(c + sx);
            }
            qx = ld4(VX, c);
            qy = ld4(VY, c);
            qz = ld4(VZ, c);
        }
        f4v qc[4];
#pragma unroll
        for (int q = 0; q < 3; ++q) qc[q] = coef_at(cl, q, m + 1, a.cv0);
        qc[3] = coef_at(cl, 3, m + 2, a.cp0);
        dxn = uni(a.dec[0], min(m + 2, nx - 1));
        // ---- y and z faces of every stage's plane
#pragma unroll
        for (int t = 0; t < T; ++t) {
            AdjointStage& S = st[t];
            const f4v q = sQ[t][tid];
            const f4v qu = sQ[t][w.iu];
            const float qr = sX[t][w.ir];
            const f4v ty = dy * S.vy + q, tz = dz * S.vz + q;
            const f4v qk = {q.y, q.z, q.w, qr};
            f4v wy = keep(ty - qu, S.f, 2), wz = keep(tz - qk, S.f, 3);
            // the last faces have no upper cell
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                wy[e] = w.jlast ? ty[e] : wy[e];
                wz[e] = w.vlast == e ? tz[e] : wz[e];
            }
            S.vy = wy;
            S.vz = wz;
            sY[t][tid] = sC[slot[t]][1][tid] * wy;
            sZ[t][tid] = sC[slot[t]][2][tid].w * wz.w;
        }
        lds_barrier();
        // ---- x faces and pressures, stage by stage
        f4v cpn = pn, cx = qx, cy = qy, cz = qz, ccp = cpl;
        uint32_t cf = fn;
        f4v q = sQ[0][tid];
        f4v pbs[T], ws[T - 1][3];  // what the gradient needs of the stages' planes
#pragma unroll
        for (int t = 0; t < T; ++t) {
            AdjointStage& S = st[t];
            const int i = m - t;
            const f4v yo = sY[t][tid], yb = sY[t][w.id];
            const float zb = sZ[t][w.il];
            const float dx = dxs[t + 1];
            const f4v pbn = pb_of(cpn, i + 1, t, dxs[t]);
            const f4v qn = keep(ccp * pbn, cf, 0);
            f4v wx = dx * S.vx + q;
            f4v acc = keep(S.pb, S.f, 0), cwx = zero;
            if (i < nx - 1) {
                wx = keep(wx - qn, S.f, 1);
                cwx = sC[slot[t]][0][tid] * wx;
                acc -= cwx;
            }
            const f4v zo = sC[slot[t]][2][tid] * S.vz;
            const f4v zl = {zb, zo.x, zo.y, zo.z};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[e] = w.jlast ? acc[e] : acc[e] - yo[e];
                acc[e] = w.vlast == e ? acc[e] : acc[e] - zo[e];
            }
            if (i > 0) acc += S.cwx;
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = w.j > 0 ? acc[e] + yb[e] : acc[e];
            acc.x = w.k > 0 ? acc.x + zl.x : acc.x;
            acc.y += zl.y;
            acc.z += zl.z;
            acc.w += zl.w;
            pbs[t] = S.pb;
            if (t < T - 1) {
                ws[t][0] = wx;
                ws[t][1] = S.vy;
                ws[t][2] = S.vz;
            }
            // this stage's next plane: what came in (loads, or the stage before)
            const AdjointStage old = S;
            S = AdjointStage{cx, cy, cz, cwx, pbn, cf};
            // the next stage's plane ahead is this one's own
            if (t + 1 < T) ccp = sC[slot[t]][3][tid];
            if (t + 1 < T) q = sQ[t + 1][tid];  // read before the next stage's q is posted
            sQ[t][tid] = qn;
            sX[t][tid] = qn.x;
            cpn = acc;
            cx = wx;
            cy = old.vy;
            cz = old.vz;
            cf = old.f;
        }
        pn = qp;
        fn = qf;
        // every store of the plane comes after the wait for the next one's loads
        __builtin_amdgcn_s_waitcnt(kWaitLoads);
        {
            const int i = m - (T - 1);
            if (w.out && i >= w.i0) {
                const uint32_t c = at(i);
                st_lane<NTS>(gmem(a.f[src ^ 1][0]), c, cpn, w.nv);
                st_lane<NTS>(gmem(a.f[src ^ 1][1]), c, cx, w.nv);
                st_lane<NTS>(gmem(a.f[src ^ 1][2]), c, cy, w.nv);
                st_lane<NTS>(gmem(a.f[src ^ 1][3]), c, cz, w.nv);
            }
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int i = m - t, wi = i - a.lo[0] + 1;
            if (i < w.i0 || i >= w.i1 || wi < 0 || wi > bx) continue;  // uniform
            if (wi > 0) st_box<false>(gmem(a.pass_pb) + (t * dbox_cells(a) + (wi - 1) * b_plane), pl, pbs[t]);
            if (t < T - 1)
#pragma unroll
                for (int x = 0; x < 3; ++x)
                    st_box<false>(gmem(a.pass_w) + ((3 * t + x) * coef_cells(a) + wi * w_plane), wl, ws[t][x]);
        }
        // The slot of the plane that left the last stage takes the next plane's:
        // its cell coefficient is the one read a plane ahead.
        const int free_slot = slot[T - 1];
#pragma unroll
        for (int q = 0; q < 3; ++q) sC[free_slot][q][tid] = qc[q];
        sC[free_slot][3][tid] = cpl;
        cpl = qc[3];
#pragma unroll
        for (int t = T - 1; t > 0; --t) slot[t] = slot[t - 1];
        slot[0] = free_slot;
#pragma unroll
        for (int t = T; t > 0; --t) dxs[t] = dxs[t - 1];
        dxs[0] = dxn;
    }
}

// Gradient terms of the kPassSteps adjoint steps n, n - 1, .. of a pass, as
// k_design_grad forms and adds them (same terms, same order).
__global__ __launch_bounds__(256) void k_design_grad3(const DesignArgs a, int64_t n) {
    const int bx = a.hi[0] - a.lo[0], by = a.hi[1] - a.lo[1], bz = a.hi[2] - a.lo[2];
    const uint32_t b = blockIdx.x * 256u + threadIdx.x;
    if (b >= static_cast<uint32_t>(bx) * by * bz) return;
    const int bk = static_cast<int>(b % bz), t = static_cast<int>(b / bz);
    const int bj = t % by, bi = t / by;
    const int nz = a.nz;
    const uint32_t sx = static_cast<uint32_t>(a.ny) * static_cast<uint32_t>(nz);
    const uint32_t c = cix(a.lo[0] + bi, a.lo[1] + bj, a.lo[2] + bk, a.ny, nz);
    GMEM f4v* __restrict__ ACC = gm(a.acc);
    const int ey = by + 2, ez = a.p_nk, k = a.lo[2] + bk;
    const uint32_t e = static_cast<uint32_t>(((bi + 1) * ey + (bj + 1)) * ez + (k - a.p_k0));
    const uint32_t d = static_cast<uint32_t>((bi * by + bj) * a.d_nk + (k - a.d_k0));
    const uint32_t wy = static_cast<uint32_t>(by + 1), wz = static_cast<uint32_t>(coef_nk(a));
    const uint32_t cw = ((bi + 1) * wy + (bj + 1)) * wz + static_cast<uint32_t>(k - coef_k0(a));
    const GMEM float* __restrict__ EX = gm(a.face_e);
    const GMEM float* __restrict__ EY = EX + face_count(bx, by, bz, 0);
    const GMEM float* __restrict__ EZ = EY + face_count(bx, by, bz, 1);
    const uint32_t fx = static_cast<uint32_t>((bi * by + bj) * bz + bk);
    const uint32_t fy = static_cast<uint32_t>((bi * (by + 1) + bj) * bz + bk);
    const uint32_t fz = static_cast<uint32_t>((bi * by + bj) * (bz + 1) + bk);
    const float exm = ldo(EX, fx), exp_ = ldo(EX, fx + static_cast<uint32_t>(by * bz));
    const float eym = ldo(EY, fy), eyp = ldo(EY, fy + static_cast<uint32_t>(bz));
    const float ezm = ldo(EZ, fz), ezp = ldo(EZ, fz + 1u);
    const bool air = ldo(gm(a.flags), c) & FDTD_FLAG_AIR;
    f4v g = ldo(ACC, b);
#pragma unroll
    for (int q = 0; q < kPassSteps; ++q) {
        const int64_t m = n - q;
        // the last step's velocities are in the fields, the others' beside them
        const bool last = q == kPassSteps - 1;
        const int64_t wc = coef_cells(a);
        const GMEM float* __restrict__ WX = gm(last ? a.f[m & 1][1] : a.pass_w + 3 * q * wc);
        const GMEM float* __restrict__ WY = gm(last ? a.f[m & 1][2] : a.pass_w + (3 * q + 1) * wc);
        const GMEM float* __restrict__ WZ = gm(last ? a.f[m & 1][3] : a.pass_w + (3 * q + 2) * wc);
        const uint32_t o = last ? c : cw, ox = last ? sx : wy * wz, oy = last ? static_cast<uint32_t>(nz) : wz;
        const GMEM float* __restrict__ hp = gm(a.hist_p + (m - a.hist0) * ebox_cells(a));
        const float hpc = ldo(hp, e);
        const float hxp = ldo(hp, e + static_cast<uint32_t>(ey * ez)), hyp = ldo(hp, e + static_cast<uint32_t>(ez)),
                    hzp = ldo(hp, e + 1u);
        const float hxm = ldo(hp, e - static_cast<uint32_t>(ey * ez)), hym = ldo(hp, e - static_cast<uint32_t>(ez)),
                    hzm = ldo(hp, e - 1u);
        const float pb = ldo(gm(a.pass_pb + q * dbox_cells(a)), d);
        const float dv = ldo(gm(a.hist_div + (m - a.hist0) * dbox_cells(a)), d);
        float gr = 0.f;
        gr += ldo(WX, o) * (hxp - hpc) * exp_;
        gr += ldo(WY, o) * (hyp - hpc) * eyp;
        gr += ldo(WZ, o) * (hzp - hpc) * ezp;
        gr += ldo(WX, o - ox) * (hpc - hxm) * exm;
        gr += ldo(WY, o - oy) * (hpc - hym) * eym;
        gr += ldo(WZ, o - 1u) * (hpc - hzm) * ezm;
        float y = gr - g.y;
        float s = g.x + y;
        g.y = (s - g.x) - y;
        g.x = s;
        if (air) {
            y = pb * a.cp0 * dv - g.w;
            s = g.z + y;
            g.w = (s - g.z) - y;
            g.z = s;
        }
    }
    sto(ACC, b, g);
}

// ---- host side -------------------------------------------------------------------
bool pick_pass_tile(int nx, int ny, int nz, int only_nt, double share, PassTile& best);

// The windows of a design pass: one workgroup per CU, so half of what the split
// of the chip assumes for this workgroup size.
bool design_pass_tile(const DesignArgs& a, PassTile& m) {
    return pick_pass_tile(a.nx, a.ny, a.nz, kDesignPassThreads, 0.5, m);
}

hipError_t launch_design_coefs(const DesignArgs& a, float* coef, hipStream_t st) {
    const int64_t cells = coef_cells(a);
    hipLaunchKernelGGL(k_design_coefs, dim3(static_cast<unsigned>((cells + 255) / 256)), dim3(256), 0, st, a, coef);
    return hipGetLastError();
}

hipError_t launch_design_forward_pass(const DesignArgs& a, const PassTile& m, int64_t s, bool nts, hipStream_t st) {
    const dim3 grid((m.nwg + 7) & ~7), block(kDesignPassThreads);
    if (nts) hipLaunchKernelGGL(k_design_forward_pass<true>, grid, block, 0, st, a, m, s);
    else hipLaunchKernelGGL(k_design_forward_pass<false>, grid, block, 0, st, a, m, s);
    return hipGetLastError();
}

// The adjoint steps n .. n - kPassSteps + 1 and their gradient terms.
hipError_t launch_design_adjoint_pass(const DesignArgs& a, const PassTile& m, int64_t n, bool nts, hipStream_t st) {
    const dim3 grid((m.nwg + 7) & ~7), block(kDesignPassThreads);
    if (nts) hipLaunchKernelGGL(k_design_adjoint_pass<true>, grid, block, 0, st, a, m, n);
    else hipLaunchKernelGGL(k_design_adjoint_pass<false>, grid, block, 0, st, a, m, n);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    const int64_t box = static_cast<int64_t>(a.hi[0] - a.lo[0]) * (a.hi[1] - a.lo[1]) * (a.hi[2] - a.lo[2]);
    hipLaunchKernelGGL(k_design_grad3, dim3(static_cast<unsigned>((box + 255) / 256)), dim3(256), 0, st, a, n);
    return hipGetLastError();
}

}  // namespace fdtd_amd
