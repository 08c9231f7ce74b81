// Device code shared by the kernels that take several time steps per pass
// (multi_step.hip, design_pass.hip): 4-cell lanes, LDS phases, window geometry.
#pragma once

#include <climits>

#include "fdtd_common.hpp"

namespace fdtd_amd {

typedef float f4v __attribute__((ext_vector_type(4)));
// rows of grids whose nz is no multiple of 4 start at any cell: 4-byte aligned
// 16-byte accesses and byte-aligned flag words, which global memory takes
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32u __attribute__((aligned(1)));

#if defined(__HIP_DEVICE_COMPILE__)
#define CMEM __attribute__((address_space(4)))
#else
#define CMEM
#endif
// tables no kernel writes while it runs, read at wave-uniform indices
template <typename T>
__device__ __forceinline__ T uni(const T* t, int64_t i) {
    return ((const CMEM T*)t)[i];
}

// v, to the compiler a new value: an LDS entry read at again(v) is read where it
// is used rather than kept in registers between uses.
__device__ __forceinline__ int again(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(v));
#endif
    return v;
}

__device__ __forceinline__ f4v ld4(const GMEM float* base, uint32_t c) {
    return *reinterpret_cast<const GMEM f4u*>(at32(base, c));
}
template <bool NTS>
__device__ __forceinline__ void st4(GMEM float* base, uint32_t c, f4v v) {
    if constexpr (NTS) __builtin_nontemporal_store(v, reinterpret_cast<GMEM f4u*>(at32(base, c)));
    else *reinterpret_cast<GMEM f4u*>(at32(base, c)) = v;
}

// v where bit `bit` of byte e of f is set, else +0 (element by element)
__device__ __forceinline__ f4v keep(f4v v, uint32_t f, int bit) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
        v[e] = __int_as_float(__float_as_int(v[e]) & __builtin_amdgcn_sbfe(static_cast<int>(f), 8 * e + bit, 1));
    return v;
}

__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// flags of four air cells with every face open, and their y bits alone
constexpr uint32_t kOpen = 0x01010101u * (FDTD_FLAG_AIR | FDTD_FLAG_OPEN_X | FDTD_FLAG_OPEN_Y | FDTD_FLAG_OPEN_Z);
constexpr uint32_t kOpenY = 0x01010101u * FDTD_FLAG_OPEN_Y;
constexpr int kMaxLanes = 256;      // lanes of a window row at most
constexpr int kEvery = INT_MAX, kNowhere = INT_MIN;

constexpr int kWaitLoads = 0x0f70;  // s_waitcnt vmcnt(0), the other counters unlimited

// A workgroup's window of a pass and a thread's place in it (k_multi_step's
// geometry): rows w0 .. w0 + rows, lanes of 4 cells from k0, planes [i0, i1) and
// the rows and cells it stores. iu, id, ir, il: the threads above, below, next and
// before, or the entry NT of zeros where there is none.
struct PassWindow {
    int i0, i1, w0, jlo, jhi, k0, klo, khi;
    int row, kl, iu, id, ir, il;
    int j, k, nv, vlast;            // nv: cells to the row's end; vlast: element of the last z face
    uint32_t c0;
    bool in_win, ld, out, jlast;
};
__device__ __forceinline__ PassWindow pass_window(const PassTile& mt, int NT, int tid, int lb, int nx, int ny, int nz) {
    PassWindow w;
    const int nwin = mt.nseg * mt.njt;
    const int chunk = lb / nwin, win = lb - chunk * nwin;
    const int seg = win % mt.nseg, jt = win / mt.nseg;
    constexpr int T = kPassSteps;
    w.i0 = chunk * mt.units;
    w.i1 = min(nx, w.i0 + mt.units);
    w.w0 = jt * (mt.rows - 2 * T);
    w.jlo = jt == 0 ? 0 : w.w0 + T;
    w.jhi = jt == mt.njt - 1 ? ny : w.w0 + mt.rows - T;
    w.k0 = 4 * (seg == 0 ? 0 : seg * mt.ko - 1);
    w.klo = 4 * seg * mt.ko;
    w.khi = seg == mt.nseg - 1 ? nz : 4 * (seg + 1) * mt.ko;
    w.row = tid / mt.kt;
    w.kl = tid - w.row * mt.kt;
    w.in_win = w.row < mt.rows;
    w.iu = w.row + 1 < mt.rows ? tid + mt.kt : tid;
    w.id = (w.row > 0 && w.in_win) ? tid - mt.kt : NT;
    w.ir = tid + 1 < NT ? tid + 1 : tid;
    w.il = w.kl > 0 ? tid - 1 : NT;
    w.j = w.w0 + w.row;
    w.k = w.k0 + 4 * w.kl;
    w.ld = w.in_win && w.j < ny && w.k < nz;
    w.out = w.ld && w.j >= w.jlo && w.j < w.jhi && w.k >= w.klo && w.k < w.khi;
    w.nv = nz - w.k;
    w.vlast = nz - 1 - w.k;
    w.c0 = static_cast<uint32_t>(w.j) * static_cast<uint32_t>(nz) + static_cast<uint32_t>(w.k);
    w.jlast = w.j == ny - 1;
    return w;
}

// The lane's valid cells of an output (nv >= 4: all).
template <bool NTS>
__device__ __forceinline__ void st_lane(GMEM float* base, uint32_t c, f4v v, int nv) {
    if (nv >= 4) {
        st4<NTS>(base, c, v);
    } else {
#pragma unroll
        for (int e = 0; e < 3; ++e)
            if (e < nv) stx(base, c + e, v[e]);
    }
}

}  // namespace fdtd_amd
