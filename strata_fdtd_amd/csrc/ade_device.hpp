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

__device__ __forceinline__ int64_t box_index(const FusedArgs& a, int i, int j, int k) {
    const int by = a.box_hi[1] - a.box_lo[1], bz = a.box_hi[2] - a.box_lo[2];
    return ((static_cast<int64_t>(i - a.box_lo[0]) * by) + (j - a.box_lo[1])) * bz + (k - a.box_lo[2]);
}

__device__ __forceinline__ int64_t box_cells(const FusedArgs& a) {
    return static_cast<int64_t>(a.box_hi[0] - a.box_lo[0]) * (a.box_hi[1] - a.box_lo[1]) *
           (a.box_hi[2] - a.box_lo[2]);
}

__device__ __forceinline__ bool has_pole(const FusedArgs& a, int m) {
    bool any = false;
    if (m)
        for (int q = 0; q < a.n_pole; ++q) any |= pole_at(a.poles, q).mat == m;
    return any;
}

// One recurrence step of pole pl at box cell b (ade.cpp:25-166, 295-401):
// Debye J <- a J + b x, Lorentz J <- a J + b J_prev + d x with J_prev <- J.
__device__ __forceinline__ float ade_recur(const AdePole& pl, float j0, float* jprev, float x) {
    if (!pl.lorentz) return pl.a * j0 + pl.b * x;
    const float j1 = *jprev;
    *jprev = j0;
    return pl.a * j0 + pl.b * j1 + pl.d * x;
}

// The complete update of cell (i, j, k) from the input state S, poles of its
// material (m, 0: none) included; out: p before sources, vx, vy, vz, damped. Jd:
// the density poles' J after this step's update; modulus poles are updated in
// a.J (own cell only).
//
// The six faces and the cell's neighbourhood are loaded at once and the pole
// list is walked once for all faces (Debye poles first, then Lorentz, so each
// face adds its corrections in ade.cpp:240-401's order): walked face by face,
// with a pole's parameters and J read in a chain, the fix-up of the 512^3
// enclosure's sphere (267,000 cells, two poles) took 19.3 us.
template <bool NU>
__device__ __forceinline__ void ade_cell(const FusedArgs& a, const FieldView& S, const float* __restrict__ Jd, int i,
                                         int j, int k, int m, float out[4]) {
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int64_t sy = S.nz, sx = static_cast<int64_t>(S.ny) * S.nz;
    const int64_t gy = nz, gx = static_cast<int64_t>(ny) * nz;
    const int64_t c = S.at(i, j, k), g = lin(i, j, k, ny, nz);
    const int pos[3] = {i, j, k}, dim[3] = {nx, ny, nz};
    const int64_t st[3] = {sx, sy, 1}, gs[3] = {gx, gy, 1};
    const float p0 = S.f[0][c];
    const uint32_t f = a.flags[g];
    float ph[3], pl[3], vh[3], vl[3];
    uint32_t fl[3];
    bool mh[3], ml[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        const bool up = pos[x] + 1 < dim[x], dn = pos[x] > 0;
        ph[x] = up ? S.f[0][c + st[x]] : 0.f;
        pl[x] = dn ? S.f[0][c - st[x]] : 0.f;
        vh[x] = S.f[1 + x][c];
        vl[x] = dn ? S.f[1 + x][c - st[x]] : 0.f;
        fl[x] = dn ? a.flags[g - gs[x]] : 0u;
        mh[x] = m && up && a.material[g + gs[x]] == m;
        ml[x] = m && dn && a.material[g - gs[x]] == m;
    }
    float hi[3], lo[3];  // v' of the faces above and below, per axis
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        const float ch = NU ? a.cv * (pos[x] + 1 < dim[x] ? a.ifc[x][pos[x]] : 1.f) : a.cv;
        const float cl = NU ? a.cv * (pos[x] > 0 ? a.ifc[x][pos[x] - 1] : 1.f) : a.cv;
        hi[x] = vh[x] + ch * (ph[x] - p0);
        lo[x] = vl[x] + cl * (p0 - pl[x]);
    }
    int64_t box_n = 0, b = 0;
    if (m) {
        const int by = a.box_hi[1] - a.box_lo[1], bz = a.box_hi[2] - a.box_lo[2];
        const int64_t bs[3] = {static_cast<int64_t>(by) * bz, bz, 1};
        box_n = box_cells(a);
        b = box_index(a, i, j, k);
        for (int pass = 0; pass < 2; ++pass)
            for (int q = 0; q < a.n_pole; ++q) {
                const AdePole po = pole_at(a.poles, q);
                if (po.target != 0 || po.lorentz != pass || po.mat != m) continue;
                const float* __restrict__ Jq = Jd + q * box_n + b;
                const float j0 = Jq[0];
                float jh[3], jl[3];
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    jh[x] = mh[x] ? Jq[bs[x]] : 0.f;
                    jl[x] = ml[x] ? Jq[-bs[x]] : 0.f;
                }
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    if (mh[x]) hi[x] += po.corr * (jh[x] - j0);
                    if (ml[x]) lo[x] += po.corr * (j0 - jl[x]);
                }
            }
    }
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        const uint32_t open = FDTD_FLAG_OPEN_X << x;
        hi[x] = pos[x] + 1 < dim[x] ? ((f & open) ? hi[x] : 0.f) : vh[x];  // last face: neither updated nor masked
        lo[x] = pos[x] > 0 ? ((fl[x] & open) ? lo[x] : 0.f) : 0.f;
    }
    const float dvx = hi[0] - lo[0], dvy = hi[1] - lo[1], dvz = hi[2] - lo[2];
    const float icx = NU ? a.icl[0][i] : 1.f, icy = NU ? a.icl[1][j] : 1.f, icz = NU ? a.icl[2][k] : 1.f;
    float pnew;
    if (NU) pnew = p0 + a.cp * (((icx * dvx) + (icy * dvy)) + (icz * dvz));
    else pnew = p0 + a.cp * ((dvx + dvy) + dvz);
    if (m) {
        // modulus poles: source is the native divergence of v'
        const float ix = NU ? icx : a.ade_inv_dx, iy = NU ? icy : a.ade_inv_dx, iz = NU ? icz : a.ade_inv_dx;
        float dA = dvx * ix;
        dA += dvy * iy;
        dA += dvz * iz;
        for (int pass = 0; pass < 2; ++pass)
            for (int q = 0; q < a.n_pole; ++q) {
                const AdePole po = pole_at(a.poles, q);
                if (po.target != 1 || po.lorentz != pass || po.mat != m) continue;
                float* Jq = a.J + q * box_n + b;
                const float jn = ade_recur(po, *Jq, po.lorentz ? a.Jprev + q * box_n + b : nullptr, dA);
                *Jq = jn;
                pnew += po.corr * jn;
            }
    }
    if (!(f & FDTD_FLAG_AIR)) pnew = 0.f;
    const float dx = a.dec[0][i], dy = a.dec[1][j], dz = a.dec[2][k];
    out[0] = ((pnew * dx) * dy) * dz;
    out[1] = hi[0] * dx;
    out[2] = hi[1] * dy;
    out[3] = hi[2] * dz;
}

// The step's sweep sources at air cell (i, j, k), in list order.
__device__ __forceinline__ float ade_sources(const FusedArgs& a, int i, int j, int k, int64_t s, float ps) {
    for (int q = 0; q < a.n_src; ++q) {
        bool on;
        if (a.src_kind[q] == 0) {
            on = a.src_i[q] == i && a.src_j[q] == j && a.src_k[q] == k;
        } else {
            const int ax = a.src_i[q], id = a.src_j[q];
            on = ax == 0 ? id == i : (ax == 1 ? id == j : id == k);
        }
        if (on) ps = static_cast<float>(static_cast<double>(ps) + a.wave[q * a.wave_len + s]);
    }
    return ps;
}

}  // namespace fdtd_amd
