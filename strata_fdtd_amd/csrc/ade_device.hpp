// Device code of one ADE cell update, shared by the one-step fix-up and the
// patch of multi-step passes.
#pragma once

#include "fdtd_common.hpp"

namespace fdtd_amd {

// The fields of a step's input state: the whole grid (origin 0) or a dense box
// of it with its first cell at (oi, oj, ok).
struct FieldView {
    const float* f[4];              // p, vx, vy, vz
    int oi, oj, ok;
    int ny, nz;                     // extents of the storage
    __device__ __forceinline__ int64_t at(int i, int j, int k) const { return lin(i - oi, j - oj, k - ok, ny, nz); }
};

__device__ __forceinline__ int64_t box_cells(const FusedArgs& a) {
    return static_cast<int64_t>(a.box_hi[0] - a.box_lo[0]) * (a.box_hi[1] - a.box_lo[1]) *
           (a.box_hi[2] - a.box_lo[2]);
}

// One recurrence step of pole pl at box cell b (ade.cpp:25-166, 295-401):
// Debye J <- a J + b x, Lorentz J <- a J + b J_prev + d x with J_prev <- J.
__device__ __forceinline__ float ade_recur(const AdePole& pl, float j0, float* jprev, float x) {
    if (!pl.lorentz) return pl.a * j0 + pl.b * x;
    const float j1 = *jprev;
    *jprev = j0;
    return pl.a * j0 + pl.b * j1 + pl.d * x;
}

// The poles of one cell's update: kFewPoles of the table at a time in scalar
// registers, with the cell's own J (and its step before, Lorentz) of each.
constexpr int kFewPoles = 4;
struct CellPoles {
    AdePole po[kFewPoles];
    int row[kFewPoles];             // its J's index in the density J at hand
    float jo[kFewPoles], jp[kFewPoles];
};

// The density poles' J that a step reads: a.J (rows as registered) or the patch's
// own (second; density poles alone, rows in the table's order), after the step's
// update or, fresh, before it.
struct DensityJ {
    const float* J;
    bool second, fresh;
};

__device__ __forceinline__ void fetch_poles(const FusedArgs& a, const DensityJ& d, int q0, CellPoles& cp) {
#pragma unroll
    for (int x = 0; x < kFewPoles; ++x) {
        cp.po[x] = pole_at(a.poles, min(q0 + x, a.n_pole - 1));
        cp.row[x] = d.second ? q0 + x : cp.po[x].slot;
        if (q0 + x >= a.n_pole) cp.po[x].mat = -1;
    }
}

// Whether material m has poles; cp: the first ones.
__device__ __forceinline__ bool has_pole(const FusedArgs& a, const CellPoles& cp, int m) {
    bool any = false;
#pragma unroll
    for (int x = 0; x < kFewPoles; ++x) any |= cp.po[x].mat == m;
    for (int q = kFewPoles; q < a.n_pole; ++q) any |= pole_at(a.poles, q).mat == m;
    return any;
}

// Whether any lane's material m is the pole's (uniform).
__device__ __forceinline__ bool some_lane(const AdePole& po, int m) {
    return __builtin_amdgcn_ballot_w64(po.mat == m) != 0;
}

// The cell's own J of the poles in cp. Where d is fresh, the density poles' J takes
// this step's update from the cell's pressure p0 (Debye only).
template <typename IX>
__device__ __forceinline__ void fetch_own(const FusedArgs& a, const DensityJ& d, IX b, int m, float p0,
                                          CellPoles& cp) {
    const int64_t box_n = box_cells(a);
#pragma unroll
    for (int x = 0; x < kFewPoles; ++x) {
        const AdePole& po = cp.po[x];
        cp.jo[x] = cp.jp[x] = 0.f;
        if (!some_lane(po, m)) continue;
        cp.jo[x] = ldx(gmem(po.target == 0 ? d.J + cp.row[x] * box_n : a.J + po.slot * box_n), b);
        if (po.lorentz) cp.jp[x] = ldx(gmem(a.Jprev + po.slot * box_n), b);
        if (d.fresh && po.target == 0) cp.jo[x] = ade_recur(po, cp.jo[x], nullptr, p0);
    }
}

// The complete update of cell (i, j, k) from the input state S; POLES: its
// material m has some, and the cell is box cell b. out: p before sources, vx, vy,
// vz, damped. Modulus poles are updated in a.J (own cell only). cp: the table's first
// poles on entry; the cell's own J of them on return.
//
// Instructions are what an update costs (a sphere's 267,000 cells are 16 waves a
// CU; 15.2 us where predicated loads took 16.7), so loads are not predicated but read the cell itself where there is no
// neighbour, offsets are 32-bit, the poles' parameters are in scalar registers
// (four at a time) and poles of other materials are passed over by the wave. The
// table has the Debye poles before the Lorentz ones of each target, so one walk
// adds each face's corrections in ade.cpp:240-401's order.
template <bool NU, bool POLES, typename IX>
__device__ __forceinline__ void ade_cell(const FusedArgs& a, const FieldView& S, const DensityJ& d, int i, int j,
                                         int k, int m, IX b, CellPoles& cp, float out[4]) {
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const IX st[3] = {static_cast<IX>(S.ny) * static_cast<IX>(S.nz), static_cast<IX>(S.nz), 1};
    const IX gs[3] = {static_cast<IX>(ny) * static_cast<IX>(nz), static_cast<IX>(nz), 1};
    const IX c = lidx<IX>(i - S.oi, j - S.oj, k - S.ok, S.ny, S.nz), g = lidx<IX>(i, j, k, ny, nz);
    const int pos[3] = {i, j, k}, dim[3] = {nx, ny, nz};
    const GMEM uint8_t* FL = gmem(a.flags);
    const GMEM float* P = gmem(S.f[0]);
    const float p0 = ldx(P, c);
    const uint32_t f = ldx(FL, g);
    float ph[3], pl[3], vh[3], vl[3], dec[3];
    uint32_t fl[3];
    bool up[3], dn[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        up[x] = pos[x] + 1 < dim[x];
        dn[x] = pos[x] > 0;
        const GMEM float* V = gmem(S.f[1 + x]);
        ph[x] = ldx(P, up[x] ? static_cast<IX>(c + st[x]) : c);
        const IX below = dn[x] ? static_cast<IX>(c - st[x]) : c;
        pl[x] = ldx(P, below);
        vh[x] = ldx(V, c);
        vl[x] = ldx(V, below);
        fl[x] = ldx(FL, dn[x] ? static_cast<IX>(g - gs[x]) : g);
        dec[x] = ldx(gmem(a.dec[x]), static_cast<IX>(pos[x]));
    }
    const int64_t box_n = POLES ? box_cells(a) : 0;
    IX bh[3], bl[3];
    bool mh[3], ml[3];
    if constexpr (POLES) {
        const IX bz = static_cast<IX>(a.box_hi[2] - a.box_lo[2]);
        const IX bs[3] = {static_cast<IX>(a.box_hi[1] - a.box_lo[1]) * bz, bz, 1};
        const GMEM uint8_t* MAT = gmem(a.material);
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            mh[x] = pos[x] + 1 < a.box_hi[x];
            ml[x] = pos[x] > a.box_lo[x];
            bh[x] = mh[x] ? static_cast<IX>(b + bs[x]) : b;
            bl[x] = ml[x] ? static_cast<IX>(b - bs[x]) : b;
            const int above = ldx(MAT, mh[x] ? static_cast<IX>(g + gs[x]) : g);
            const int under = ldx(MAT, ml[x] ? static_cast<IX>(g - gs[x]) : g);
            mh[x] &= above == m;
            ml[x] &= under == m;
        }
        fetch_own(a, d, b, m, p0, cp);
    }
    float hi[3], lo[3];  // v' of the faces above and below, per axis
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        const float ch = NU ? a.cv * (up[x] ? a.ifc[x][pos[x]] : 1.f) : a.cv;
        const float cl = NU ? a.cv * (dn[x] ? a.ifc[x][pos[x] - 1] : 1.f) : a.cv;
        hi[x] = vh[x] + ch * (ph[x] - p0);
        lo[x] = vl[x] + cl * (p0 - pl[x]);
    }
    if constexpr (POLES)
        for (int q0 = 0; q0 < a.n_pole; q0 += kFewPoles) {
            if (q0) {
                fetch_poles(a, d, q0, cp);
                fetch_own(a, d, b, m, p0, cp);
            }
#pragma unroll
            for (int q = 0; q < kFewPoles; ++q) {
                const AdePole& po = cp.po[q];
                if (po.target != 0 || !some_lane(po, m)) continue;
                const GMEM float* Jq = gmem(d.J + cp.row[q] * box_n);
                float jh[3], jl[3];
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    jh[x] = ldx(Jq, bh[x]);
                    jl[x] = ldx(Jq, bl[x]);
                }
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    if (d.fresh) {
                        jh[x] = ade_recur(po, jh[x], nullptr, ph[x]);
                        jl[x] = ade_recur(po, jl[x], nullptr, pl[x]);
                    }
                    const float h = hi[x] + po.corr * (jh[x] - cp.jo[q]), l = lo[x] + po.corr * (cp.jo[q] - jl[x]);
                    hi[x] = mh[x] & (po.mat == m) ? h : hi[x];
                    lo[x] = ml[x] & (po.mat == m) ? l : lo[x];
                }
            }
        }
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        const uint32_t open = FDTD_FLAG_OPEN_X << x;
        hi[x] = up[x] ? ((f & open) ? hi[x] : 0.f) : vh[x];  // last face: neither updated nor masked
        lo[x] = dn[x] & ((fl[x] & open) != 0) ? lo[x] : 0.f;
    }
    const float dvx = hi[0] - lo[0], dvy = hi[1] - lo[1], dvz = hi[2] - lo[2];
    const float icx = NU ? a.icl[0][i] : 1.f, icy = NU ? a.icl[1][j] : 1.f, icz = NU ? a.icl[2][k] : 1.f;
    float pnew;
    if (NU) pnew = p0 + a.cp * (((icx * dvx) + (icy * dvy)) + (icz * dvz));
    else pnew = p0 + a.cp * ((dvx + dvy) + dvz);
    if constexpr (POLES) {
        // modulus poles: source is the native divergence of v'
        const float ix = NU ? icx : a.ade_inv_dx, iy = NU ? icy : a.ade_inv_dx, iz = NU ? icz : a.ade_inv_dx;
        float dA = dvx * ix;
        dA += dvy * iy;
        dA += dvz * iz;
        for (int q0 = 0; q0 < a.n_pole; q0 += kFewPoles) {
            if (a.n_pole > kFewPoles) {
                fetch_poles(a, d, q0, cp);
                fetch_own(a, d, b, m, p0, cp);
            }
#pragma unroll
            for (int q = 0; q < kFewPoles; ++q) {
                const AdePole& po = cp.po[q];
                if (po.target != 1 || po.mat != m) continue;
                float h = cp.jp[q];
                const float jn = ade_recur(po, cp.jo[q], po.lorentz ? &h : nullptr, dA);
                if (po.lorentz) stx(gmem(a.Jprev + po.slot * box_n), b, h);
                stx(gmem(a.J + po.slot * box_n), b, jn);
                pnew += po.corr * jn;
            }
        }
    }
    if (!(f & FDTD_FLAG_AIR)) pnew = 0.f;
    out[0] = ((pnew * dec[0]) * dec[1]) * dec[2];
    out[1] = hi[0] * dec[0];
    out[2] = hi[1] * dec[1];
    out[3] = hi[2] * dec[2];
}

// The density poles' update of the step after, at box cell b with pressure x: from
// the J that ade_cell left in cp (read from d) into `to`, the other of a.J and the
// patch's own.
template <typename IX>
__device__ __forceinline__ void ade_density_next(const FusedArgs& a, const DensityJ& d, IX b, int m, float p0, float x,
                                                 CellPoles& cp, float* to) {
    const int64_t box_n = box_cells(a);
    for (int q0 = 0; q0 < a.n_pole; q0 += kFewPoles) {
        if (a.n_pole > kFewPoles) {
            fetch_poles(a, d, q0, cp);
            fetch_own(a, d, b, m, p0, cp);
        }
#pragma unroll
        for (int q = 0; q < kFewPoles; ++q) {
            const AdePole& po = cp.po[q];
            if (po.target != 0 || po.mat != m) continue;
            float h = cp.jp[q];
            stx(gmem(to + (d.second ? po.slot : q0 + q) * box_n), b, ade_recur(po, cp.jo[q], po.lorentz ? &h : nullptr, x));
            if (po.lorentz) stx(gmem(a.Jprev + po.slot * box_n), b, h);
        }
    }
}

// The step's sweep sources at air cell (i, j, k), in list order.
__device__ __forceinline__ float ade_sources(const FusedArgs& a, int i, int j, int k, int64_t s, float ps) {
    for (int q = 0; q < a.n_src; ++q) {
        const int kind = a.src_kind[q], si = a.src_i[q], sj = a.src_j[q], sk = a.src_k[q];
        const bool point = (si == i) & (sj == j) & (sk == k);
        const bool plane = sj == (si == 0 ? i : (si == 1 ? j : k));
        if (kind == 0 ? point : plane) ps = static_cast<float>(static_cast<double>(ps) + a.wave[q * a.wave_len + s]);
    }
    return ps;
}

// Gather g (0 p, 1..3 velocities) of microphone m: the weighted sum of its 8 corners
// in the corner order of core/solver.py:962-1003 (acc = 0, then acc += w * f). The
// reference sums in float32 when its weights are Python floats (numpy rounds the
// weight to float32 and multiplies in float32) and in float64 when they are numpy
// float64 scalars; mic_f64 selects which. at(flat grid index): the corner's value.
template <typename At>
__device__ __forceinline__ double mic_sum(const FusedArgs& a, int m, int g, At at) {
    const int64_t row = static_cast<int64_t>(m) * 4 + g;
    const int32_t* idx = a.mic_idx + row * 8;
    const double* w = a.mic_w + row * 8;
    if (a.mic_f64[row]) {
        double acc = 0.0;
#pragma unroll
        for (int c = 0; c < 8; ++c) acc = acc + w[c] * static_cast<double>(at(idx[c]));
        return acc;
    }
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < 8; ++c) acc = acc + static_cast<float>(w[c]) * at(idx[c]);
    return acc;
}

}  // namespace fdtd_amd
