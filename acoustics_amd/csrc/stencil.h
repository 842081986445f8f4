// stencil.h -- device arithmetic shared by the step kernels (kernels.hip) and
// the resident kernel (resident.hip): the same function, with its contraction
// written out, gives the same bits in both.
#pragma once

#include "kernels.h"

namespace fdtd {

// Pointers read out of a SceneDev are generic to the compiler, which then
// emits flat memory instructions; those count against both the vector-memory
// and the LDS counters, so every wait becomes a full wait.  Every scene array
// lives in device global memory: casting to the global address space gives
// global_load/global_store with vmcnt-only waits, and read-only tables cast to
// the constant address space are fetched with scalar loads when the index is
// uniform across the wavefront.
#if defined(__HIP_DEVICE_COMPILE__)
#define AS_GLOBAL __attribute__((address_space(1)))
#define AS_CONST __attribute__((address_space(4)))
#else  // the host pass only parses device code
#define AS_GLOBAL
#define AS_CONST
#endif
template <class T>
__device__ __forceinline__ AS_GLOBAL T *gmem(T *p) { return (AS_GLOBAL T *)p; }
template <class T>
__device__ __forceinline__ const AS_GLOBAL T *gmem(const T *p) { return (const AS_GLOBAL T *)p; }
template <class T>
__device__ __forceinline__ const AS_CONST T *cmem(const T *p) { return (const AS_CONST T *)p; }

// ---------------------------------------------------------------------------
// -f h grad_p . cell_n of a rasterised ghost (f = 1 with centre sampling,
// 0.75 with seven samples), grad_p = -rho (a_s n_b + a_v) (MAC_Grid.cpp:
// 1256-1281): k_raster a_s, plus k_vec a_v along the ghost's axis in a
// scene with acceleration noise
__device__ __forceinline__ double raster_accel_term(const SceneDev &S, const GhostDev &gd, long long step)
{
    const AS_GLOBAL double *acc = gmem(S.acc_tab) + amp_row(S, step) * S.n_ch + gd.obj * S.n_cpo;
    double v = gd.k_raster * acc[0];
    if (S.n_cpo > 1) v = fma(gd.k_vec, acc[1 + gd.vaxis], v);
    return v;
}

// The leapfrog update in increment form, p^{n+1} = p^n + ((p^n - p^{n-1}) +
// lam2 sum_q (p_q - p^n)).  A smooth field changes little between steps and
// between neighbours, so every difference here is exact in FP32 (Sterbenz:
// operands within a factor of two) and the only rounding at the scale of p
// itself is the last addition.  Forming 2 p^n - p^{n-1} and the six-neighbour
// sum instead rounds three times at that scale per step, and the rounding
// errors, fed back as velocity, add up along every propagation path: 1.3e-4
// relative L2 at the listeners after 4000 steps at 256^3, against 1e-4 allowed.
__device__ __forceinline__ float leapfrog1(float c, float prev, float xm, float xp, float ym, float yp, float zm, float zp,
                                           float lam2)
{
    const float lap = ((xm - c) + (xp - c)) + ((ym - c) + (yp - c)) + ((zm - c) + (zp - c));
    return c + fmaf(lam2, lap, c - prev);
}

// The same cell in the merged staggered scheme: its increment d^{n+1} = d^n +
// lam2 sum_q (p_q - p^n), where the staggered update's d is f5/h times the
// divergence of the face velocities.
__device__ __forceinline__ float increment1(float c, float d, float xm, float xp, float ym, float yp, float zm, float zp, float lam2)
{
    const float lap = ((xm - c) + (xp - c)) + ((ym - c) + (yp - c)) + ((zm - c) + (zp - c));
    return fmaf(lam2, lap, d);
}

// Face velocity update on one axis for a face whose old value is v, between
// pressures pl (left) and pr (right); inactive faces stay at zero.  The fma
// is explicit: a face is computed by the two cells that share it and both
// must round it the same way.
__device__ __forceinline__ float face_update(bool active, float4 c, float v, float pl, float pr)
{
    return active ? fmaf(c.y, pr - pl, c.x * v) : 0.f;
}

// Split pressure update pDir <- f3 pDir + f5/h (v_R - v_L).
__device__ __forceinline__ float split_update(float4 c, float q, float dv)
{
    return fmaf(c.w, dv, c.z * q);
}

// One transverse axis of the merged update: lap + f5h (f2_R (p_R - p) - f2_L
// (p - p_L)), cL the cell's table entry (its low face and itself), cR the
// high face's.
__device__ __forceinline__ float transverse_add(float lap, float f5h, float f2L, float f2R, float pl, float pc, float pr)
{
    return fmaf(f5h, fmaf(f2R, pr - pc, -(f2L * (pc - pl))), lap);
}

// ---------------------------------------------------------------------------
// One axis of the ghost-aware Laplacian (MAC_Grid::
// pressureFieldLaplacianGhostCell, MAC_Grid.cpp:187-299) at a cell with
// pressure c, neighbours nm / np and ghost values gm / gp where the
// neighbour is solid: the plain 3-point stencil with ghost values (centre
// sampling, 247-266), or the non-uniform one for ghosts 3h/4 away (seven
// samples, 268-286).
__device__ __forceinline__ double ghost_lap_axis(int seven, bool ghm, bool ghp, double gm, double gp, double nm, double np,
                                                 double c)
{
    const double m = ghm ? gm : nm, p = ghp ? gp : np;
    if (!seven || (!ghm && !ghp)) return p + m - 2.0 * c;
    if (ghm && ghp) return (gp + gm - 2.0 * c) / (9.0 / 16.0);
    if (ghp) return (gp + 0.75 * nm - (7.0 / 4.0) * c) / (21.0 / 32.0);
    return (0.75 * np + gm - (7.0 / 4.0) * c) / (21.0 / 32.0);
}

// p^{n+1} = 2 p^n - p^{n-1} + lam2 L(p^n) of an object-adjacent cell, with L
// h^2 its ghost-aware Laplacian.
__device__ __forceinline__ double special_update(double c, double prev, double lap, double lam2)
{
    return fma(lap, lam2, 2.0 * c - prev);
}

// One pressure source's contribution: amplitude a times the three spatial
// factors, added to pn with one rounding.
__device__ __forceinline__ float add_source(float pn, float a, float gx, float gy, float gz)
{
    return fmaf(a * gx * gy, gz, pn);
}

}  // namespace fdtd
