// Several time steps in one pass over HBM (temporal blocking), gfx950.
//
// k_fused_step reads and writes every field once per step and runs at the rate
// of a streaming pass, so a step that is not to cost 33 B per cell has to share
// its pass with others. k_multi_step takes T steps per pass: a workgroup owns a
// window of rows (j) and 4-cell lanes (k) and marches along i as a pipeline of
// T stages, stage t taking step s + t on plane m - t while stage 0 is at plane
// m. What stage t makes of a plane is what stage t + 1 reads, in registers; only
// stage 0 loads from memory and only stage T - 1 stores.
//
// A thread owns 4 consecutive k cells of one row (16-byte accesses). Its row
// above (p) and below (the updated vy) and its lane neighbours (p, vz) come from
// LDS, posted in two phases per plane: the stages' pressures, then, once the y
// and z faces are updated, their vy and vz. The outermost row and cell of a
// window lack a neighbour, so each stage's valid cells shrink by one on every
// interior side; neighbouring windows overlap by what T stages lose and store
// only what is valid after the last one. Per cell the operations and their order
// are k_fused_step's, so the results are the same bit for bit.
//
// What bounds it: at 512^3 HBM (a pass moves 4.65 GB, 1.05 times the 33 B per
// cell of one step, since windows next to each other march the same planes at
// the same time and share their halos in L2), with the vector units busy half
// the time; on small grids the latency of its planes (1.2 us and 0.12 us per
// resident wave), of which a pass over even one plane takes six. Held to 128
// VGPRs (one workgroup of 1024 per CU) without spills in the loop: pressures and
// updated vy stay in LDS only (with them in registers the spills made 512^3
// 20% slower). Per step, air boxes: 512^3 850 us with k_fused_step, 335-360
// here; 261x243x307 196, 61; 192^3 38.8, 18.5; 100^3 9.3, 7.2; 64^3 5.6, 5.4.

#include <algorithm>

#include "ade_device.hpp"
#include "fdtd_common.hpp"
#include "pass_device.hpp"

namespace fdtd_amd {

// The kernel's arguments where they lie (FusedArgs is the first), for code that
// rarely runs: rare() hides the pointer's value, so its loads stay there and
// hold no scalar registers across the loop.
__device__ __forceinline__ const CMEM FusedArgs* kernargs() {
#if defined(__HIP_DEVICE_COMPILE__)
    return (const CMEM FusedArgs*)__builtin_amdgcn_kernarg_segment_ptr();
#else
    return nullptr;
#endif
}
__device__ __forceinline__ const CMEM FusedArgs* rare(const CMEM FusedArgs* p) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(p));
#endif
    return p;
}

// One stage's state of a thread: velocities at the stage's plane (its pressure is
// in LDS), the updated and not yet damped vx of the plane below, the plane's flags.
struct Stage {
    f4v vx, vy, vz, vxp;
    uint32_t f;
};

// The pass of steps s .. s + kPassSteps - 1 over one workgroup's windows: number
// lb of the windows-by-chunks of `mt`, of the solve described at `ka`.
template <bool NU, int NT, bool NTS>
__device__ __forceinline__ void pass_workgroup(const CMEM FusedArgs* ka, const PassTile& mt, int64_t s, int lb) {
    const CMEM FusedArgs& a = *ka;
    constexpr int T = kPassSteps;
    __shared__ f4v sP[T][NT];
    __shared__ f4v sY[T][NT + 1];
    // vz: nonuniform grids keep it in LDS as well (with their coefficients it would
    // not fit the registers), uniform ones the last element and p's first alone
    __shared__ f4v sV[NU ? T : 1][NU ? NT + 1 : 1];
    __shared__ float sX[NU ? 1 : T][NU ? 1 : NT];
    __shared__ float sZ[NU ? 1 : T][NU ? 1 : NT + 1];
    // nonuniform grids: damping, face and cell coefficients along k, per lane
    __shared__ f4v sK[NU ? 3 : 1][NU ? kMaxLanes : 1];
    // the window's sources: their samples of the pass's steps, and the row and cell
    // they act on (-1: any)
    __shared__ double sW[NU ? FDTD_MAX_SOURCES : 1][T];
    __shared__ int sOn[NU ? FDTD_MAX_SOURCES : 1][2];
    const int tid = threadIdx.x;
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    if (tid < T) {
        sY[tid][NT] = f4v{0.f, 0.f, 0.f, 0.f};  // the row below the window's first
        if constexpr (NU) sV[tid][NT] = f4v{0.f, 0.f, 0.f, 0.f};  // the cell before its first lane
        else sZ[tid][NT] = 0.f;
    }
    const int par = static_cast<int>(s & 1);
    const GMEM float* __restrict__ P = gmem(par ? a.f[1][0] : a.f[0][0]);
    const GMEM float* __restrict__ VX = gmem(par ? a.f[1][1] : a.f[0][1]);
    const GMEM float* __restrict__ VY = gmem(par ? a.f[1][2] : a.f[0][2]);
    const GMEM float* __restrict__ VZ = gmem(par ? a.f[1][3] : a.f[0][3]);
    GMEM float* __restrict__ Po = gmem(par ? a.f[0][0] : a.f[1][0]);
    GMEM float* __restrict__ VXo = gmem(par ? a.f[0][1] : a.f[1][1]);
    GMEM float* __restrict__ VYo = gmem(par ? a.f[0][2] : a.f[1][2]);
    GMEM float* __restrict__ VZo = gmem(par ? a.f[0][3] : a.f[1][3]);
    const GMEM uint8_t* __restrict__ FL = gmem(a.flags);
    const uint32_t sx = static_cast<uint32_t>(ny) * static_cast<uint32_t>(nz);
    const float cv = a.cv, cp = a.cp;

    const int row = tid / mt.kt;
    const int kl = tid - row * mt.kt;
    const bool in_win = row < mt.rows;
    const int iu = row + 1 < mt.rows ? tid + mt.kt : tid;  // row above
    const int id = (row > 0 && in_win) ? tid - mt.kt : NT; // row below
    const int ir = tid + 1 < NT ? tid + 1 : tid;           // next lane
    const int il = kl > 0 ? tid - 1 : NT;                  // previous lane

    const int nwin = mt.nseg * mt.njt;
    const int chunk = lb / nwin, win = lb - chunk * nwin;
    const int i0 = chunk * mt.units;
    const int i1 = min(nx, i0 + mt.units);
    const int seg = win % mt.nseg, jt = win / mt.nseg;
    // window origin and the rows / lanes it stores
    const int w0 = jt * (mt.rows - 2 * T);
    const int jlo = jt == 0 ? 0 : w0 + T;
    const int jhi = jt == mt.njt - 1 ? ny : w0 + mt.rows - T;
    const int k0 = 4 * (seg == 0 ? 0 : seg * mt.ko - 1);
    const int klo = 4 * seg * mt.ko;
    const int khi = seg == mt.nseg - 1 ? nz : 4 * (seg + 1) * mt.ko;
    const int j = w0 + row;
    const int k = k0 + 4 * kl;
    const bool ld = in_win && j < ny && k < nz;
    const bool out = ld && j >= jlo && j < jhi && k >= klo && k < khi;
    const int nv = nz - k;                               // 4 or more: a whole lane
    const uint32_t c0 = static_cast<uint32_t>(j) * static_cast<uint32_t>(nz) + static_cast<uint32_t>(k);
    const bool jlast = j == ny - 1;
    const bool jlast_win = w0 + mt.rows >= ny;           // uniform
    const bool klast_win = k0 + 4 * mt.kt >= nz;         // uniform
    const int vlast = nz - 1 - k;                        // element of the last z face (0..3 in one lane)
    const float dy = ld ? gmem(a.dec[1])[j] : 1.f;
    float cvy = cv, icy = 1.f;
    if (NU && ld) {
        icy = gmem(a.icl[1])[j];
        if (j + 1 < ny) cvy = cv * gmem(a.ifc[1])[j];
    }
    f4v dzr = {1.f, 1.f, 1.f, 1.f};
    auto lane_tables = [&](int kk, f4v& dz, f4v& cvz, f4v& icz) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (kk + e < nz) {
                dz[e] = gmem(a.dec[2])[kk + e];
                if (NU) {
                    icz[e] = gmem(a.icl[2])[kk + e];
                    if (kk + e + 1 < nz) cvz[e] = cv * gmem(a.ifc[2])[kk + e];
                }
            }
    };
    if constexpr (NU) {
        if (tid < mt.kt) {
            f4v dz = {1.f, 1.f, 1.f, 1.f}, cz = {cv, cv, cv, cv}, iz = {1.f, 1.f, 1.f, 1.f};
            lane_tables(k0 + 4 * tid, dz, cz, iz);
            sK[0][tid] = dz;
            sK[1][tid] = cz;
            sK[2][tid] = iz;
        }
    } else {
        f4v none = {};
        lane_tables(k, dzr, none, none);
    }
    // Flag bits that say nothing about walls: the last faces, which keep their
    // velocity, cells past the row and lanes past the window or grid.
    uint32_t ends = kOpen;
    if (ld) {
        ends = jlast ? kOpenY : 0u;
        if (vlast < 4) ends |= (FDTD_FLAG_OPEN_Z << (8 * vlast)) | static_cast<uint32_t>(uint64_t(kOpen) << (8 * vlast + 8));
    }
    // Sources that touch the window and probes it stores: lane q holds the
    // plane of source q (kEvery: a y or z plane source, on every plane) and
    // of probe q, kNowhere if it is elsewhere, so a stage finds what its
    // plane has with one compare. kNowhere is no plane: a stage's own plane
    // runs from -(T - 1) to nx + T - 2.
    int src_i = kNowhere, probe_i = kNowhere;
    {
        const int q = tid & (kWave - 1);
        const int jw = w0 + mt.rows, kw = k0 + 4 * mt.kt;
        if (q < a.n_src) {
            const int at = a.src_i[q], sj = a.src_j[q], sk = a.src_k[q];
            if (a.src_kind[q] == 0) {
                if (sj >= w0 && sj < jw && sk >= k0 && sk < kw) src_i = at;
            } else if (at == 0) {
                src_i = sj;
            } else if (at == 1 ? (sj >= w0 && sj < jw) : (sj >= k0 && sj < kw)) {
                src_i = kEvery;
            }
            if (NU && tid < kWave && src_i != kNowhere) {
                const bool point = a.src_kind[q] == 0;
                sOn[q][0] = point || at == 1 ? sj : -1;
                sOn[q][1] = point ? sk : (at == 2 ? sj : -1);
                for (int t = 0; t < T; ++t) {
                    const bool known = s + t < a.wave_len;
                    if (!known) atomicOr(a.health, 2u);
                    sW[q][t] = known ? gmem(a.wave)[q * a.wave_len + s + t] : 0.0;
                }
            }
        }
        if (q < a.n_sweep_probe) {
            const GMEM int32_t* __restrict__ PIJK = gmem(a.probe_ijk);
            const int pi = PIJK[3 * q], pj = PIJK[3 * q + 1], pk = PIJK[3 * q + 2];
            if (pj >= jlo && pj < jhi && pk >= klo && pk < khi && pi >= i0 && pi < i1) probe_i = pi;
        }
    }

    // A lane past its row's last cell reads on into the next row (or the pad
    // past the last one): those cells feed nothing that is stored.
    auto at = [&](int i) { return static_cast<uint32_t>(i) * sx + c0; };
    auto flags = [&](uint32_t c) -> uint32_t { return *reinterpret_cast<const GMEM u32u*>(at32(FL, c)); };

    const f4v zero = {0.f, 0.f, 0.f, 0.f};
    Stage st[T];
#pragma unroll
    for (int t = 0; t < T; ++t) st[t] = Stage{zero, zero, zero, zero, 0u};
    const int m0 = max(i0 - T, 0);
    const int m1 = i1 + T - 1;
    // plane m0, and p of the one after it
    f4v p0 = zero, pn = zero;
    if (ld) {
        const uint32_t c = at(m0);
        p0 = ld4(P, c);
        st[0].vx = ld4(VX, c);
        st[0].vy = ld4(VY, c);
        st[0].vz = ld4(VZ, c);
        st[0].f = flags(c);
        if (m0 + 1 < nx) pn = ld4(P, c + sx);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        sP[t][tid] = t ? zero : p0;
        if constexpr (!NU) sX[t][tid] = t ? 0.f : p0.x;
    }
    // the stages' damping (and coefficients) along x: read one plane ahead and
    // handed on from stage to stage, so that no stage waits for a scalar load
    float dxs[T], ifs[T], ics[T];
    auto x_tables = [&](int i, float& dx, float& ifx, float& icx) {
        const int ic = min(i, nx - 1);
        dx = uni(a.dec[0], ic);
        ifx = icx = 1.f;
        if (NU) {
            ifx = uni(a.ifc[0], min(i, nx - 2));
            icx = uni(a.icl[0], ic);
        }
    };
#pragma unroll
    for (int t = 1; t < T; ++t) dxs[t] = ifs[t] = ics[t] = 1.f;
    x_tables(m0, dxs[0], ifs[0], ics[0]);
    __builtin_amdgcn_s_waitcnt(kWaitLoads);
    for (int m = m0; m < m1; ++m) {
        lds_barrier();  // the stages' pressures are posted
        // ---- next plane's loads
        f4v qp = zero, qx = zero, qy = zero, qz = zero;
        uint32_t qf = 0;
        if (ld && m + 1 < m1 && m + 1 < nx) {
            const uint32_t c = at(m + 1);
            if (m + 2 < nx) qp = ld4(P, c + sx);
            qx = ld4(VX, c);
            qy = ld4(VY, c);
            qz = ld4(VZ, c);
            qf = flags(c);
        }
        float dxn, ifn, icn;
        x_tables(m + 1, dxn, ifn, icn);
        // ---- y and z faces of every stage's plane
#pragma unroll
        for (int t = 0; t < T; ++t) {
            Stage& S = st[t];
            const f4v p = sP[t][tid];
            const f4v pu = sP[t][iu];
            float pr;
            if constexpr (NU) pr = sP[t][ir].x;
            else pr = sX[t][ir];
            f4v vy = S.vy + cvy * (pu - p);
            const f4v pk = {p.y, p.z, p.w, pr};
            f4v vz;
            if constexpr (NU) vz = S.vz + sK[1][again(kl)] * (pk - p);
            else vz = S.vz + cv * (pk - p);
            const bool walls = __builtin_amdgcn_ballot_w64(((S.f | ends) & kOpen) != kOpen) != 0;
            if (walls) {
                vy = keep(vy, S.f, 2);
                vz = keep(vz, S.f, 3);
            }
            if (jlast_win) {
#pragma unroll
                for (int e = 0; e < 4; ++e) vy[e] = jlast ? S.vy[e] : vy[e];
            }
            if (klast_win) {
#pragma unroll
                for (int e = 0; e < 4; ++e) vz[e] = vlast == e ? S.vz[e] : vz[e];
            }
            sY[t][tid] = vy;
            if constexpr (NU) {
                sV[t][tid] = vz;
            } else {
                S.vz = vz;
                sZ[t][tid] = vz.w;
            }
        }
        lds_barrier();
        // ---- x faces and pressures, stage by stage: what stage t makes of
        // its plane is p(i + 1) of stage t + 1, and its state of the next round
        f4v cpn = pn, cx = qx, cy = qy, cz = qz;
        uint32_t cf = qf;
        f4v p = sP[0][tid];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            Stage& S = st[t];
            const int i = m - t;
            const f4v vy = sY[t][tid];
            const f4v yb = sY[t][id];
            f4v vz;
            float zb;
            if constexpr (NU) {
                vz = sV[t][tid];
                zb = sV[t][il].w;
            } else {
                vz = S.vz;
                zb = sZ[t][il];
            }
            const float dx = dxs[t];
            f4v vx = S.vx;
            const bool walls = __builtin_amdgcn_ballot_w64(((S.f | ends) & kOpen) != kOpen) != 0;
            if (i < nx - 1) {
                const float cvx = NU ? cv * ifs[t] : cv;
                vx = S.vx + cvx * (cpn - p);
                if (walls) vx = keep(vx, S.f, 1);
            }
            const f4v zl = {zb, vz.x, vz.y, vz.z};
            const f4v dvx = vx - S.vxp, dvy = vy - yb, dvz = vz - zl;
            f4v pnew;
            if (NU) {
                const float icx = ics[t];
                pnew = p + cp * ((icx * dvx + icy * dvy) + sK[2][again(kl)] * dvz);
            } else {
                pnew = p + cp * ((dvx + dvy) + dvz);
            }
            if (walls) pnew = keep(pnew, S.f, 0);
            const f4v dz = NU ? sK[0][again(kl)] : dzr;
            f4v ps = ((pnew * dx) * dy) * dz;
            const f4v ox = vx * dx, oy = vy * dy, oz = vz * dz;
            const uint64_t adds = __builtin_amdgcn_ballot_w64(src_i == i || src_i == kEvery);
            if (adds) {
                // A z plane source acts on every plane of its windows: through the
                // scalar loads below it costs the 320x320x480 plate 9% of its step,
                // from LDS 3%. Uniform grids keep the loads: there the LDS form,
                // with or without sources, made every plane 2% slower.
                if constexpr (NU) {
                    for (uint32_t sm = static_cast<uint32_t>(adds); sm; sm &= sm - 1) {
                        const int q = __builtin_ctz(sm);
                        const double w = sW[q][t];
                        const int on_j = sOn[q][0], on_k = sOn[q][1];
                        const uint32_t hit = ((on_j == j) | (on_j < 0)) ? S.f : 0u;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float v = static_cast<float>(static_cast<double>(ps[e]) + w);
                            const bool on = (((hit >> (8 * e)) & FDTD_FLAG_AIR) != 0) & ((on_k == k + e) | (on_k < 0));
                            ps[e] = on ? v : ps[e];
                        }
                    }
                } else {
                    const CMEM FusedArgs* r = rare(ka);
                    for (uint32_t sm = static_cast<uint32_t>(adds); sm; sm &= sm - 1) {
                        const int q = __builtin_ctz(sm);
                        // the planes or point it acts on, -1: any (its i has matched)
                        const bool point = r->src_kind[q] == 0;
                        const int ax = r->src_i[q], aj = r->src_j[q], ak = r->src_k[q];
                        const int on_j = point || ax == 1 ? aj : -1;
                        const int on_k = point ? ak : (ax == 2 ? aj : -1);
                        const bool known = s + t < r->wave_len;
                        if (!known && tid == 0) atomicOr(r->health, 2u);
                        const double w = known ? uni(r->wave, q * r->wave_len + s + t) : 0.0;
                        const uint32_t hit = (known & ((on_j == j) | (on_j < 0))) ? S.f : 0u;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float v = static_cast<float>(static_cast<double>(ps[e]) + w);
                            const bool on = (((hit >> (8 * e)) & FDTD_FLAG_AIR) != 0) & ((on_k == k + e) | (on_k < 0));
                            ps[e] = on ? v : ps[e];
                        }
                    }
                }
            }
            const uint64_t hits = __builtin_amdgcn_ballot_w64(probe_i == i);
            if (hits) {
                const CMEM FusedArgs* r = rare(ka);
                for (uint64_t pm = hits; pm; pm &= pm - 1) {
                    const int q = __builtin_ctzll(pm);
                    const int pj = uni(r->probe_ijk, 3 * q + 1), pk = uni(r->probe_ijk, 3 * q + 2);
                    if (s + t >= r->trace_len) {
                        if (tid == 0) atomicOr(r->health, 2u);
                    } else if (in_win && j == pj && pk >= k && pk < k + 4) {
                        const int e = pk - k;
                        const float v = e == 0 ? ps.x : (e == 1 ? ps.y : (e == 2 ? ps.z : ps.w));
                        gmem(r->trace)[(s + t) * r->n_probe + q] = v;
                        if (!isfinite(v)) atomicOr(r->health, 1u);
                    }
                }
            }
            if (t == T - 1) {
                // The next plane's loads are waited for before the stores are
                // issued: later, the wait would be for the stores as well.
                __builtin_amdgcn_s_waitcnt(kWaitLoads);
                if (out && i >= i0) {
                    const uint32_t c = at(i);
                    if (nv >= 4) {
                        st4<NTS>(Po, c, ps);
                        st4<NTS>(VXo, c, ox);
                        st4<NTS>(VYo, c, oy);
                        st4<NTS>(VZo, c, oz);
                    } else {
#pragma unroll
                        for (int e = 0; e < 3; ++e)
                            if (e < nv) {
                                stx(Po, c + e, ps[e]);
                                stx(VXo, c + e, ox[e]);
                                stx(VYo, c + e, oy[e]);
                                stx(VZo, c + e, oz[e]);
                            }
                    }
                }
            }
            // this stage's next plane: what came in (loads, or the stage before)
            const uint32_t f = S.f;
            S = Stage{cx, cy, cz, vx, cf};
            if (t + 1 < T) p = sP[t + 1][tid];  // read before the next stage's p is posted
            sP[t][tid] = cpn;
            if constexpr (!NU) sX[t][tid] = cpn.x;
            cpn = ps;
            cx = ox;
            cy = oy;
            cz = oz;
            cf = f;
        }
        pn = qp;
#pragma unroll
        for (int t = T - 1; t > 0; --t) {
            dxs[t] = dxs[t - 1];
            ifs[t] = ifs[t - 1];
            ics[t] = ics[t - 1];
        }
        dxs[0] = dxn;
        ifs[0] = ifn;
        ics[0] = icn;
    }
}

template <bool NU, int NT, bool NTS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_multi_step(const FusedArgs a,
                                                                                             const PassTile mt) {
    // XCD-aware order: hardware block b runs on XCD b mod 8, which takes a
    // contiguous range of the windows
    const int lb = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (lb < mt.nwg) pass_workgroup<NU, NT, NTS>(kernargs(), mt, uni(a.step_ptr, 0) + a.koff, lb);
}

// A pass of every solve in a batch table: steps koff .. koff + kPassSteps - 1 of a
// chunk of `chunk` steps that starts at each solve's counter. A solve with fewer
// steps left, to its limit or the chunk's end, skips the pass (k_batch_step takes
// the rest). Workgroups are dealt out through the prefix sums `offsets`; the
// number of solves and the sums are read from device memory, as k_batch_step
// reads its own. Each solve's windows are picked for its share of the chip. 24
// enclosures of 64-192 cells a side, 1000-3000 steps, served in 709 ms with single
// steps and in 404 with passes (430 with workgroups of 256, 405 with 1024).
template <bool NTS>
__global__ __launch_bounds__(kBatchPassThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_batch_pass(
    const FusedArgs* __restrict__ table, const PassTile* __restrict__ tiles, const int* __restrict__ offsets,
    const int* __restrict__ n_ptr, int koff, int chunk) {
    const int n = uni(n_ptr, 0);
    const int total = uni(offsets, n);
    const int bpx = (total + 7) / 8;
    const int xb = blockIdx.x >> 3;
    if (xb >= bpx) return;
    const int g = (blockIdx.x & 7) * bpx + xb;
    if (g >= total) return;
    int lo = 0, hi = n;  // offsets[lo] <= g < offsets[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (uni(offsets, mid) <= g) lo = mid; else hi = mid;
    }
    const CMEM FusedArgs* ka = (const CMEM FusedArgs*)table + lo;
    const int64_t s0 = uni(ka->step_ptr, 0);
    if (s0 + koff + kPassSteps > min(ka->step_limit, s0 + chunk)) return;
    const PassTile mt = ((const CMEM PassTile*)tiles)[lo];
    pass_workgroup<false, kBatchPassThreads, NTS>(ka, mt, s0 + koff, g - uni(offsets, lo));
}

// a microphone whose cells lie within this of the material box is in the boxes of
// both of the patch's first steps (grown by 4 and 3 cells)
constexpr int kPatchMic = kPassSteps;

// ---- ADE patch ------------------------------------------------------------------
// A pass takes every cell as plain air. Poles change the cells of their material
// after one step and those up to t - 1 cells around them after t, so the pass is
// wrong on the material's box grown by two cells, and only there. Those cells are
// stepped one step at a time from the same input state: step 1 on the box grown by
// four cells into dense scratch, step 2 on it grown by three, step 3 on it grown by
// two into the output, over what the pass wrote. The scratch stays in the caches
// (the 512^3 enclosure's 81^3 box: 23 MB per step).
//
// A launch's first workgroups take the listed cells with poles, a thread each, the
// others the rows of the grown box without those cells, four cells a lane. With a
// thread for every cell of the box, those with poles scattered over its waves, a
// step of the 81^3 box took 20.2 us and of a lined room's 86 x 102 x 130 (a fifth of
// the cells with poles) 31; this way 16.4 and 23.4, the latter bound by the poles'
// lanes, whose rows are pieces of a few cells: 1.7 times the L1 accesses.

// The four cells from (i, j, k) of a step's input state as plain air, their sources
// among them; nk of them lie in the row.
template <bool NU>
__device__ __forceinline__ void air_cells(const FusedArgs& a, const FieldView& S, int i, int j, int k, int nk,
                                          int64_t s, f4v o[4]) {
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const uint32_t sy = S.nz, sx = static_cast<uint32_t>(S.ny) * S.nz;
    const uint32_t gy = nz, gx = static_cast<uint32_t>(ny) * nz;
    const uint32_t c = lidx<uint32_t>(i - S.oi, j - S.oj, k - S.ok, S.ny, S.nz), g = lidx<uint32_t>(i, j, k, ny, nz);
    const GMEM float *P = gmem(S.f[0]), *VX = gmem(S.f[1]), *VY = gmem(S.f[2]), *VZ = gmem(S.f[3]);
    const GMEM uint8_t* FL = gmem(a.flags);
    const auto ldf = [&](uint32_t at) { return *reinterpret_cast<const GMEM u32u*>(at32(FL, at)); };
    const f4v zero = {0.f, 0.f, 0.f, 0.f};
    const bool ux = i + 1 < nx, uy = j + 1 < ny, dx = i > 0, dy = j > 0, dz = k > 0;
    const f4v p = ld4(P, c), vx = ld4(VX, c), vy = ld4(VY, c), vz = ld4(VZ, c);
    // where there is no neighbour its loads read the cell itself
    const uint32_t cxl = dx ? c - sx : c, cyl = dy ? c - sy : c, czl = dz ? c - 1u : c;
    const f4v pxh = ld4(P, ux ? c + sx : c), pxl = ld4(P, cxl), pyh = ld4(P, uy ? c + sy : c), pyl = ld4(P, cyl);
    const f4v vxl = ld4(VX, cxl), vyl = ld4(VY, cyl);
    const float pzh = ldx(P, nk == 4 && k + 4 < nz ? c + 4u : c), pzl = ldx(P, czl), vzl = ldx(VZ, czl);
    const uint32_t f = ldf(g), fx = ldf(dx ? g - gx : g), fy = ldf(dy ? g - gy : g), fz = ldx(FL, dz ? g - 1u : g);
    const auto tab = [&](const float* v, int at) { return ldx(gmem(v), static_cast<uint32_t>(at)); };
    const float dxi = tab(a.dec[0], i), dyj = tab(a.dec[1], j);
    float dzk[4], iz[4], cz[5];
    const auto face = [&](int ax, int at, bool on) { return NU ? a.cv * (on ? tab(a.ifc[ax], at) : 1.f) : a.cv; };
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int ke = min(k + e, nz - 1);
        dzk[e] = tab(a.dec[2], ke);
        iz[e] = NU ? tab(a.icl[2], ke) : 1.f;
        cz[e + 1] = face(2, ke, ke + 1 < nz);
    }
    cz[0] = face(2, k - 1, dz);
    const float fxh = face(0, i, ux), fxl = face(0, i - 1, dx), fyh = face(1, j, uy), fyl = face(1, j - 1, dy);
    const float ix = NU ? tab(a.icl[0], i) : 1.f, iy = NU ? tab(a.icl[1], j) : 1.f;
    constexpr int bx = __builtin_ctz(FDTD_FLAG_OPEN_X), by = __builtin_ctz(FDTD_FLAG_OPEN_Y),
                  bz = __builtin_ctz(FDTD_FLAG_OPEN_Z);
    // the last face of an axis is neither updated nor masked
    const f4v hx = ux ? keep(vx + fxh * (pxh - p), f, bx) : vx, lx = dx ? keep(vxl + fxl * (p - pxl), fx, bx) : zero;
    const f4v hy = uy ? keep(vy + fyh * (pyh - p), f, by) : vy, ly = dy ? keep(vyl + fyl * (p - pyl), fy, by) : zero;
    f4v hz, lz;
    lz[0] = dz && (fz & FDTD_FLAG_OPEN_Z) ? vzl + cz[0] * (p[0] - pzl) : 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float up = e < 3 ? p[e < 3 ? e + 1 : 3] : pzh;
        const float v = vz[e] + cz[e + 1] * (up - p[e]);
        hz[e] = k + e + 1 < nz ? ((f >> (8 * e + bz)) & 1u ? v : 0.f) : vz[e];
        if (e < 3) lz[e < 3 ? e + 1 : 3] = hz[e];
    }
    const f4v ax = hx - lx, ay = hy - ly, az = hz - lz;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float q;
        if (NU) q = p[e] + a.cp * (((ix * ax[e]) + (iy * ay[e])) + (iz[e] * az[e]));
        else q = p[e] + a.cp * ((ax[e] + ay[e]) + az[e]);
        const bool air = (f >> (8 * e)) & FDTD_FLAG_AIR;
        if (!air) q = 0.f;
        o[0][e] = ((q * dxi) * dyj) * dzk[e];
        o[3][e] = hz[e] * dzk[e];
    }
    o[1] = hx * dxi;
    o[2] = hy * dyj;
    if (s < a.wave_len)
        for (int q = 0; q < a.n_src; ++q) {
            const int kind = a.src_kind[q], si = a.src_i[q], sj = a.src_j[q], sk = a.src_k[q];
            // from k: the source's cells, all four or one
            const int z = kind == 0 ? sk : si == 2 ? sj : -1;
            const bool row = kind == 0 ? (si == i) & (sj == j) : (si == 2) | (sj == (si == 0 ? i : j));
            if (!row) continue;
            const double w = a.wave[q * a.wave_len + s];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if ((z < 0 || z == k + e) && ((f >> (8 * e)) & FDTD_FLAG_AIR))
                    o[0][e] = static_cast<float>(static_cast<double>(o[0][e]) + w);
        }
}

template <bool NU>
__global__ __launch_bounds__(256) void k_patch_step(const FusedArgs a, const PatchArgs pt, int t, int pole_wgs) {
    const int64_t s = uni(a.step_ptr, 0) + a.koff + t;
    const int par = static_cast<int>((s - t) & 1);
    const int grow = 2 * kPassSteps - 2 - t;
    int lo[3], n[3];
    const int dim[3] = {a.nx, a.ny, a.nz};
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        lo[x] = max(a.box_lo[x] - grow, 0);
        n[x] = min(a.box_hi[x] + grow, dim[x]) - lo[x];
    }
    // the step's input: the state or the box of the step before, one cell larger
    FieldView S{{}, 0, 0, 0, a.ny, a.nz};
    if (t == 0) {
        for (int g = 0; g < 4; ++g) S.f[g] = a.f[par][g];
    } else {
        const int from = grow + 1;
        S.oi = max(a.box_lo[0] - from, 0);
        S.oj = max(a.box_lo[1] - from, 0);
        S.ok = max(a.box_lo[2] - from, 0);
        S.ny = min(a.box_hi[1] + from, a.ny) - S.oj;
        S.nz = min(a.box_hi[2] + from, a.nz) - S.ok;
        const int64_t cells = static_cast<int64_t>(min(a.box_hi[0] + from, a.nx) - S.oi) * S.ny * S.nz;
        for (int g = 0; g < 4; ++g) S.f[g] = pt.box[t - 1] + g * cells;
    }
    const int64_t cells = static_cast<int64_t>(n[0]) * n[1] * n[2];
    const auto out = [&](int g) { return gmem(t == kPassSteps - 1 ? a.f[par ^ 1][g] : pt.box[t] + g * cells); };
    const auto out_at = [&](int i, int j, int k) {
        return t == kPassSteps - 1 ? lidx<uint32_t>(i, j, k, a.ny, a.nz)
                                   : lidx<uint32_t>(i - lo[0], j - lo[1], k - lo[2], n[1], n[2]);
    };
    // probes in the region (the pass recorded what it made of them)
    const GMEM int32_t* __restrict__ PIJK = gmem(a.probe_ijk);
    const int lane = threadIdx.x & (kWave - 1);
    int at[3] = {kNowhere, kNowhere, kNowhere};
    if (lane < a.n_sweep_probe)
#pragma unroll
        for (int x = 0; x < 3; ++x) at[x] = PIJK[3 * lane + x];
    int i, j, k, nk = 0;            // nk: cells from (i, j, k); bit e of own: cell k + e is this lane's
    uint32_t own = 0;
    f4v o[4];
    if (static_cast<int>(blockIdx.x) < pole_wgs) {
        const int64_t q = blockIdx.x * int64_t(256) + threadIdx.x;
        const bool live = q < a.n_ade_cells;
        const uint32_t b = static_cast<uint32_t>(a.ade_cells[live ? q : 0]);
        const uint32_t by = a.box_hi[1] - a.box_lo[1], bz = a.box_hi[2] - a.box_lo[2], row = b / bz;
        k = a.box_lo[2] + static_cast<int>(b - row * bz);
        i = a.box_lo[0] + static_cast<int>(row / by);
        j = a.box_lo[1] + static_cast<int>(row % by);
        if (live) {
            const uint32_t c = lidx<uint32_t>(i, j, k, a.ny, a.nz);
            const int m = ldx(gmem(a.material), c);
            const bool air = ldx(gmem(a.flags), c) & FDTD_FLAG_AIR;
            const float p0 = ldx(gmem(S.f[0]), lidx<uint32_t>(i - S.oi, j - S.oj, k - S.ok, S.ny, S.nz));
            const DensityJ d{t == 1 ? pt.J : a.J, t == 1, t == 0 && !pt.density};
            float v[4];
            CellPoles cp;
            fetch_poles(a, d, 0, cp);
            ade_cell<NU, true, uint32_t>(a, S, d, i, j, k, m, b, cp, v);
            if (s < a.wave_len && air) v[0] = ade_sources(a, i, j, k, s, v[0]);
            const uint32_t at_out = out_at(i, j, k);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                stx(out(g), at_out, v[g]);
                o[g][0] = v[g];
            }
            // density poles' J of the next step, from this step's pressure: from
            // a.J into pt.J and back, since neighbours still read this step's
            if (t < kPassSteps - 1)
                ade_density_next(a, d, b, m, p0, v[0], cp, t == 1 ? a.J : pt.J);
            nk = 1;
            own = 1;
        }
    } else {
        const uint32_t lanes = static_cast<uint32_t>(n[2] + 3) >> 2;
        const uint32_t e = (blockIdx.x - pole_wgs) * 256u + threadIdx.x, row = e / lanes;
        const int in_row = 4 * static_cast<int>(e - row * lanes);
        i = lo[0] + static_cast<int>(row / static_cast<uint32_t>(n[1]));
        j = lo[1] + static_cast<int>(row % static_cast<uint32_t>(n[1]));
        k = lo[2] + in_row;
        if (row < static_cast<uint32_t>(n[0]) * static_cast<uint32_t>(n[1])) {
            nk = min(4, n[2] - in_row);
            own = (1u << nk) - 1u;
            if (i >= a.box_lo[0] && i < a.box_hi[0] && j >= a.box_lo[1] && j < a.box_hi[1]) {
                // the four cells' materials, those outside the box as 0; the array
                // ends with the grid
                const uint32_t c = lidx<uint32_t>(i, j, k, a.ny, a.nz);
                const uint32_t last = static_cast<uint32_t>(a.nx) * a.ny * a.nz - 4u, at4 = min(c, last);
                uint32_t m = *reinterpret_cast<const GMEM u32u*>(at32(gmem(a.material), at4)) >> (8u * (c - at4));
                const int skip = min(max(a.box_lo[2] - k, 0), 4), stop = min(max(a.box_hi[2] - k, 0), nk);
                m &= static_cast<uint32_t>((uint64_t(1) << (8 * stop)) - 1u) & static_cast<uint32_t>(~uint64_t(0) << (8 * skip));
                if (m) {
                    CellPoles cp;
                    fetch_poles(a, DensityJ{}, 0, cp);
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        const int mx = (m >> (8 * x)) & 255u;
                        if (mx && has_pole(a, cp, mx)) own &= ~(1u << x);
                    }
                }
            }
            if (own) {
                air_cells<NU>(a, S, i, j, k, nk, s, o);
                const uint32_t d = out_at(i, j, k);
                if (own == 15u) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) st4<false>(out(g), d, o[g]);
                } else {
#pragma unroll
                    for (int g = 0; g < 4; ++g)
#pragma unroll
                        for (int x = 0; x < 4; ++x)
                            if ((own >> x) & 1u) stx(out(g), d + static_cast<uint32_t>(x), o[g][x]);
                }
            }
        }
    }
    bool in = lane < a.n_sweep_probe;
#pragma unroll
    for (int x = 0; x < 3; ++x) in = in && at[x] >= lo[x] && at[x] < lo[x] + n[x];
    for (uint64_t pm = __builtin_amdgcn_ballot_w64(in); pm; pm &= pm - 1) {
        const int q = __builtin_ctzll(pm);
        const int x = uni(a.probe_ijk, 3 * q + 2) - k;
        if (uni(a.probe_ijk, 3 * q) != i || uni(a.probe_ijk, 3 * q + 1) != j || x < 0 || x >= nk || s >= a.trace_len)
            continue;
        if (!((own >> x) & 1u)) continue;
        const float v = x == 0 ? o[0][0] : x == 1 ? o[0][1] : x == 2 ? o[0][2] : o[0][3];
        a.trace[s * a.n_probe + q] = v;
        if (!isfinite(v)) atomicOr(a.health, 1u);
    }
}

// ---- stations --------------------------------------------------------------------
// The samples of a pass's steps, of which it stores the last one's state alone, of
// the microphones and of the probes past the 64 that the pass records itself: one
// workgroup per station steps the few cells around it from the pass's input
// state (step 1 on its cells grown by one, step 2 on them) and gathers; a
// station inside the patch's boxes gathers from those. Latency bounds it: two
// dependent steps and a gather, 8.1 us a pass for two microphones (three launches of
// k_mic_gather: 13.8). What it buys is the pass: a lined 131 x 157 x 203 room with
// two microphones took 48 us a step one by one and takes 42.6.
template <bool NU>
__global__ __launch_bounds__(256) void k_station_pass(const FusedArgs a, const PatchArgs pt, const StationPass mp) {
    const int m = blockIdx.x, tid = threadIdx.x;
    const int64_t s = uni(a.step_ptr, 0) + a.koff;
    const int par = static_cast<int>(s & 1);
    const int dim[3] = {a.nx, a.ny, a.nz};
    const bool probe = m >= a.n_mic;
    const int pq = a.n_sweep_probe + m - a.n_mic;
    int lo[3], hi[3];
    bool patched = a.n_pole > 0;
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        lo[x] = probe ? uni(a.probe_ijk, 3 * pq + x) : uni(mp.box, 6 * m + x);
        hi[x] = probe ? lo[x] + 1 : uni(mp.box, 6 * m + 3 + x);
        patched = patched && lo[x] >= a.box_lo[x] - kPatchMic && hi[x] <= a.box_hi[x] + kPatchMic;
    }
    float* scratch = mp.scratch + static_cast<int64_t>(m) * kMicScratch;
    FieldView S{{}, 0, 0, 0, a.ny, a.nz};
    for (int g = 0; g < 4; ++g) S.f[g] = a.f[par][g];
    for (int t = 0; t < kPassSteps; ++t) {
        // the box of the state after this step
        const int grow = patched ? 2 * kPassSteps - 2 - t : kPassSteps - 2 - t;
        int b0[3] = {}, n[3] = {dim[0], dim[1], dim[2]};
        if (t < kPassSteps - 1)
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                b0[x] = max((patched ? a.box_lo[x] : lo[x]) - grow, 0);
                n[x] = min((patched ? a.box_hi[x] : hi[x]) + grow, dim[x]) - b0[x];
            }
        const int64_t cells = static_cast<int64_t>(n[0]) * n[1] * n[2];
        FieldView D{{}, b0[0], b0[1], b0[2], n[1], n[2]};
        float* base = patched && t < kPassSteps - 1 ? pt.box[t] : scratch;
        for (int g = 0; g < 4; ++g) D.f[g] = t == kPassSteps - 1 ? a.f[par ^ 1][g] : base + g * cells;
        if (!patched && t < kPassSteps - 1) {
            if (tid < cells) {
                const int k = b0[2] + tid % n[2], r = tid / n[2];
                const int j = b0[1] + r % n[1], i = b0[0] + r / n[1];
                float o[4];
                CellPoles cp;
                ade_cell<NU, false, uint32_t>(a, S, DensityJ{}, i, j, k, 0, 0u, cp, o);
                if (s + t < a.wave_len && (a.flags[lin(i, j, k, a.ny, a.nz)] & FDTD_FLAG_AIR))
                    o[0] = ade_sources(a, i, j, k, s + t, o[0]);
                for (int g = 0; g < 4; ++g) base[g * cells + tid] = o[g];
            }
            __syncthreads();
            scratch += 4 * cells;
            S = D;
        }
        if (probe) {
            if (tid > 0) continue;
            if (s + t < a.trace_len) {
                const float v = D.f[0][D.at(lo[0], lo[1], lo[2])];
                a.trace[(s + t) * a.n_probe + pq] = v;
                if (!isfinite(v)) atomicOr(a.health, 1u);
            } else {
                atomicOr(a.health, 2u);
            }
        } else if (tid < 4 && s + t < a.mic_len) {
            const float* F = tid == 0 ? D.f[0] : tid == 1 ? D.f[1] : tid == 2 ? D.f[2] : D.f[3];
            a.mic_out[((s + t) * a.n_mic + m) * 4 + tid] = mic_sum(a, m, tid, [&](int c) {
                const int row = c / a.nz;
                return F[D.at(row / a.ny, row % a.ny, c % a.nz)];
            });
        }
    }
}

// ---- host side -------------------------------------------------------------------
constexpr int kCUs = 256;

// Windows of `nseg` k segments and workgroups of `nt` threads, marching `chunks`
// ranges of planes; false where they do not exist.
static bool pass_windows(int nx, int ny, int nz, int nt, int nseg, PassTile& m) {
    const int lanes = (nz + 3) / 4;
    m.nt = nt;
    m.nseg = nseg;
    if (nseg == 1) {
        m.ko = m.kt = lanes;
    } else {
        if (lanes < nseg) return false;
        m.ko = ((lanes - 1 + nseg - 1) / nseg + 3) & ~3;  // segments start on 64-byte blocks of the row
        m.kt = m.ko + 2;
        // every segment has lanes to store, and the last one's fit its window
        if ((nseg - 1) * m.ko >= lanes || lanes - (nseg - 1) * m.ko > m.ko + 1) return false;
    }
    if (m.kt > std::min(nt, kMaxLanes)) return false;
    m.rows = std::min(nt / m.kt, ny);
    const int inner = m.rows - 2 * kPassSteps;
    if (m.rows >= ny) m.njt = 1;
    else if (inner < 1) return false;
    else m.njt = (ny - 2 * kPassSteps + inner - 1) / inner;
    return true;
}

// The split of a pass over the chip with the least estimated time. The estimate
// is the marching time (plane rounds of the busiest CU: a plane takes 1.23 us of
// latency and 0.12 us per resident wave) and, beyond the Infinity Cache, the
// traffic at 5.2 TB/s times 1.2, the larger of the two and 0.3 of the smaller.
// Fitted to 3337 measured (workgroup, segments, chunks) triples of 14 grids from
// 40^3 to 400^3 (rms 16%): what it picks runs within 12% of the best triple.
// only_nt: that workgroup size alone (0: any). share: the part of the chip the
// pass has (a solve in a batch).
bool pick_pass_tile(int nx, int ny, int nz, int only_nt, double share, PassTile& best) {
    const int64_t cells = static_cast<int64_t>(nx) * ny * nz;
    if (cells >= kMaxCells32) return false;
    double low = 0.0;
    bool found = false;
    for (int nt : {1024, 512, 256}) {
        if (only_nt && nt != only_nt) continue;
        const int cus = std::max(1, static_cast<int>(kCUs * share));
        const int per_cu = 1024 / nt, slots = cus * per_cu;
        for (int nseg = 1; nseg <= 64; ++nseg) {
            PassTile m{};
            if (!pass_windows(nx, ny, nz, nt, nseg, m)) continue;
            const int nwin = m.nseg * m.njt;
            // chunks c: the fewest of each chunk length (2 sqrt(nx) of them at most)
            for (int c = 1, units = 0; c <= nx; c = units > 1 ? (nx + units - 2) / (units - 1) : nx + 1) {
                units = (nx + c - 1) / c;
                const int64_t n = static_cast<int64_t>(nwin) * ((nx + units - 1) / units);
                const double planes = units + 2 * kPassSteps - 1;
                auto plane_us = [&](int64_t wgs) {
                    return 1.23 + 0.12 * (static_cast<double>((wgs + cus - 1) / cus) * nt / kWave);
                };
                const int64_t full = n / slots, rest = n % slots;
                const double march = planes * (full * plane_us(slots) + (rest ? plane_us(rest) : 0.0));
                double cost = march;
                if (cells > kCacheResidentCells) {
                    const double traffic = 1.2 * cells * (16.0 + 17.0 * (units + 2.0 * kPassSteps) / units) / 5.2e6;
                    cost = std::max(march, traffic) + 0.3 * std::min(march, traffic);
                }
                if (!found || cost < low) {
                    found = true;
                    low = cost;
                    m.units = units;
                    m.nwg = static_cast<int>(n);
                    best = m;
                }
            }
        }
    }
    return found;
}

// The given split instead; false where the grid has no such windows.
bool pass_tile_of(int nx, int ny, int nz, int nt, int nseg, int units, PassTile& m) {
    m = PassTile{};
    const bool sizes = (nt == 256 || nt == 512 || nt == 1024) && nseg >= 1 && units >= 1 && units <= nx;
    if (static_cast<int64_t>(nx) * ny * nz >= kMaxCells32 || !sizes || !pass_windows(nx, ny, nz, nt, nseg, m)) return false;
    const int64_t n = static_cast<int64_t>(m.nseg) * m.njt * ((nx + units - 1) / units);
    m.units = units;
    m.nwg = static_cast<int>(n);
    return n < (1 << 30);
}

template <bool NU, int NT>
static hipError_t launch_pass_t(const FusedArgs& a, const PassTile& m, bool nts, hipStream_t st) {
    const int blocks = (m.nwg + 7) & ~7;
    if (nts) hipLaunchKernelGGL((k_multi_step<NU, NT, true>), dim3(blocks), dim3(NT), 0, st, a, m);
    else hipLaunchKernelGGL((k_multi_step<NU, NT, false>), dim3(blocks), dim3(NT), 0, st, a, m);
    return hipGetLastError();
}

static int64_t grown_cells(const FusedArgs& a, int grow) {
    const int dim[3] = {a.nx, a.ny, a.nz};
    int64_t n = 1;
    for (int x = 0; x < 3; ++x) n *= std::min(a.box_hi[x] + grow, dim[x]) - std::max(a.box_lo[x] - grow, 0);
    return n;
}

// Whether a pass and its patch take less than single steps with their fix-up. Cells
// with poles cost about the same either way, so what counts is the rest of the grown
// box, which the patch takes at the price of a plain step's cells (4.8 us per million
// and step in grids of 2 million cells, 6.2 at 4 million, 7.6 at 7, 7 to 8 beyond the
// cache), against what a pass saves on the whole grid: 2.9 us per million in the
// cache; beyond it 4 where rows are whole 64-byte blocks, 5 of 32 bytes, 6 to 7
// otherwise (there a single step's accesses cross lines, a pass's halos hit them);
// and a launch or two where a step is little more than those. The shares below are
// where the two ways meet, or a little under it. Both were timed on 633 solves of
// 40^3 to 390^3 with 1, 3 and 8 poles: pairs of small absorbers at opposite corners
// of a box of a tenth of the grid up to all of it, full boxes, shells and scattered
// cells. Pairs in a third, half and all of the grid, single steps and passes, us a
// step: 128^3 23.1 (21.5, 24.7, 27.6); 160^3 33.7 (30.0, 36.3, 45.7); 192^3 45.5 (49.0,
// 59.0, 81.2); 256^3 126 (97.6, 124, 165); 264^3 173 (115, 142, 193); 390^3 615 (351,
// 435, 659). Full boxes, three poles: 100^3 40, 31; 192^3 257, 178. Where this takes
// passes none of them was over 2% slower than single steps.
bool patch_pays(const FusedArgs& a) {
    const int64_t cells = static_cast<int64_t>(a.nx) * a.ny * a.nz;
    if (cells >= kMaxCells32) return false;  // no passes at all
    double share;
    if (cells <= 5000000) share = 0.45;
    else if (cells <= 6000000) share = 0.4;
    else if (cells <= 7500000) share = 0.33;
    else share = a.nz % 16 == 0 ? 0.45 : a.nz % 8 == 0 ? 0.58 : cells <= 17000000 ? 0.64 : 0.8;
    const int64_t air = grown_cells(a, 2 * kPassSteps - 2) - a.n_ade_cells;
    return static_cast<double>(air) <= 1e5 + share * static_cast<double>(cells);
}

// Scratch floats of the patch: the boxes of steps 1 and 2, then the n_density density
// poles' second J.
int64_t patch_floats(const FusedArgs& a, int n_density, int64_t off[3]) {
    const int64_t first = grown_cells(a, 2 * kPassSteps - 2), second = grown_cells(a, 2 * kPassSteps - 3);
    off[0] = 0;
    off[1] = 4 * first;
    off[2] = off[1] + 4 * second;
    return off[2] + n_density * grown_cells(a, 0) + 4;  // a lane reads up to three cells past its row
}

// Whether a pass can record a microphone with the cells [lo, hi): it lies in the
// patch's boxes, or no cell it depends on has poles. (A single cell does either.)
bool mic_in_pass(const FusedArgs& a, const int32_t box[6]) {
    bool inside = true, apart = false;
    for (int x = 0; x < 3; ++x) {
        const int lo = box[x], hi = box[3 + x];
        if (hi - lo > kMicCells) return false;
        inside = inside && lo >= a.box_lo[x] - kPatchMic && hi <= a.box_hi[x] + kPatchMic;
        apart = apart || hi + kPassSteps - 1 <= a.box_lo[x] || lo - (kPassSteps - 1) >= a.box_hi[x];
    }
    return a.n_pole == 0 || inside || apart;
}

// The stations' samples of a pass's steps (after it and its patch).
hipError_t launch_pass_stations(const FusedArgs& a, bool nu, const PatchArgs& pt, const StationPass& mp,
                                hipStream_t st) {
    const dim3 grid(a.n_mic + a.n_probe - a.n_sweep_probe);
    if (nu) hipLaunchKernelGGL(k_station_pass<true>, grid, dim3(256), 0, st, a, pt, mp);
    else hipLaunchKernelGGL(k_station_pass<false>, grid, dim3(256), 0, st, a, pt, mp);
    return hipGetLastError();
}

hipError_t launch_density(const FusedArgs& a, hipStream_t st);

// The cells a pass took wrongly (after it, on the same steps).
hipError_t launch_patch(const FusedArgs& a, bool nu, const PatchArgs& pt, hipStream_t st) {
    hipError_t e = pt.density ? launch_density(a, st) : hipSuccess;
    const int pole_wgs = static_cast<int>((a.n_ade_cells + 255) / 256);
    for (int t = 0; t < kPassSteps && e == hipSuccess; ++t) {
        const int grow = 2 * kPassSteps - 2 - t;
        const int64_t row = std::min(a.box_hi[2] + grow, a.nz) - std::max(a.box_lo[2] - grow, 0);
        const int64_t lanes = grown_cells(a, grow) / row * ((row + 3) / 4);
        const dim3 grid(static_cast<unsigned>(pole_wgs + (lanes + 255) / 256));
        if (nu) hipLaunchKernelGGL(k_patch_step<true>, grid, dim3(256), 0, st, a, pt, t, pole_wgs);
        else hipLaunchKernelGGL(k_patch_step<false>, grid, dim3(256), 0, st, a, pt, t, pole_wgs);
        e = hipGetLastError();
    }
    return e;
}

// Steps koff .. koff + kPassSteps - 1 of a chunk in one pass. nts: non-temporal stores.
hipError_t launch_pass(const FusedArgs& a, bool nu, const PassTile& m, bool nts, hipStream_t st) {
    switch (m.nt) {
        case 1024: return nu ? launch_pass_t<true, 1024>(a, m, nts, st) : launch_pass_t<false, 1024>(a, m, nts, st);
        case 512: return nu ? launch_pass_t<true, 512>(a, m, nts, st) : launch_pass_t<false, 512>(a, m, nts, st);
        case 256: return nu ? launch_pass_t<true, 256>(a, m, nts, st) : launch_pass_t<false, 256>(a, m, nts, st);
        default: return hipErrorInvalidValue;
    }
}

// Passes of a batch (workgroups up to cap_wgs, the grid covers the capacity).
hipError_t launch_batch_pass(const FusedArgs* table, const PassTile* tiles, const int* offsets, const int* n_ptr,
                             int cap_wgs, bool nts, int koff, int chunk, hipStream_t st) {
    const int blocks = std::max(8, (cap_wgs + 7) & ~7);
    if (nts)
        hipLaunchKernelGGL(k_batch_pass<true>, dim3(blocks), dim3(kBatchPassThreads), 0, st, table, tiles, offsets,
                           n_ptr, koff, chunk);
    else
        hipLaunchKernelGGL(k_batch_pass<false>, dim3(blocks), dim3(kBatchPassThreads), 0, st, table, tiles, offsets,
                           n_ptr, koff, chunk);
    return hipGetLastError();
}

}  // namespace fdtd_amd
