// Compact-kernel stencils of the two CK-MPM sub-grids (mpm_kernel.cuh:91-114):
// base node, fractional offset t and node-0 weight w0 = 1 - t + sin(2 pi t)/(2 pi)
// per axis; node 1 of an axis has weight 1 - w0.
#pragma once
#include <hip/hip_runtime.h>

namespace ckmpm {

constexpr float kInv2Pi = 0.15915494309189535f;

// sin(2 pi t) / (2 pi) for t in [0, 1): with u = t - 1/2, sin(2 pi t) = -sin(2 pi u);
// |u| > 1/4 folds to 1/2 sgn(u) - u (sin(pi - a) = sin a), so x = 2 pi u' lies in
// [-pi/2, pi/2], where the Taylor series of sin x / x through x^10 is within 4e-8
// (the next term, x^12 / 13!).  Result = -u' (1 - z/3! + z^2/5! - ... - z^5/11!), z = x^2.
__device__ __forceinline__ float SinTwoPiFrac(float t) {
    float u = t - 0.5f;
    if (u > 0.25f) u = 0.5f - u;
    else if (u < -0.25f) u = -0.5f - u;
    const float z = 39.47841760435743f * u * u;  // (2 pi u)^2
    float p = -2.505210838544172e-08f;           // -1 / 11!
    p = p * z + 2.755731922398589e-06f;          //  1 / 9!
    p = p * z - 1.984126984126984e-04f;          // -1 / 7!
    p = p * z + 8.333333333333333e-03f;          //  1 / 5!
    p = p * z - 1.666666666666667e-01f;          // -1 / 3!
    p = p * z + 1.0f;
    return -u * p;
}

// Stencil of one sub-grid at an FP32 position (xs = x * invDx): base cell c,
// fractional offset t and node-0 weight w0 per axis.  mpm_algorithm.cuh:1555-1569,
// mpm_kernel.cuh:91-114 (w0 = 1 - t + sin(2 pi t) / (2 pi)).
struct Stencil32 {
    int c[3];
    float t[3];
    float w0[3];
};
template <int g>
__device__ __forceinline__ void MakeStencil(const float (&xs)[3], Stencil32& s) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float shift = g == 0 ? 0.25f : -0.25f;
        const int c = static_cast<int>(floorf(__fadd_rn(xs[a], shift)));
        const float t = __fadd_rn(xs[a] - static_cast<float>(c), shift);
        s.c[a] = c;
        s.t[a] = t;
        s.w0[a] = 1.0f - t + SinTwoPiFrac(t);
    }
}
// Both sub-grid stencils from one sine per axis.  With x/dx < 2^22 every step is exact
// in FP32: grid 1 has t1 = t0 - 1/2 (same base cell) when t0 >= 1/2, else t1 = t0 + 1/2
// (base cell one lower), which equals MakeStencil<1>'s c and t bit for bit; and
// sin(2 pi t1) = -sin(2 pi t0).  With f = min(t0, t1) in [0, 1/2) both sines are
// +-s, s = sin(2 pi f) / (2 pi) >= 0, and f folds to f' = min(f, 1/2 - f) in [0, 1/4],
// where s = f' P((f')^2) with the Taylor series through f'^11 (the terms of SinTwoPiFrac).
//
// sn and diag hold the moments of both grids that G2P and P2G need (MomentInverse): the
// first moment of an axis, w1 - t, is -sn on grid 0 and +sn on grid 1, and the second
// moments w0 t^2 + w1 (1 - t)^2 = t (1 - t) -+ sn (1 - 2 t) of the two grids add up to
// f (1 - 2 f) + 1/4 - s.
//
// LO <= HI: the grid-0 base cell is clamped to [LO, HI].  A particle within rounding of
// such a cell's face, on the far side of it, then has t just below 0 or above 1, where the
// weights continue (t^3 terms apart) those of its own cell's stencil.
template <int LO = 0, int HI = -1>
__device__ __forceinline__ void MakeStencilPair(const float (&xs)[3], Stencil32& s0, Stencil32& s1, float (&sn)[3],
                                                float (&diag)[3]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float fl = floorf(__fadd_rn(xs[a], 0.25f));
        if (LO <= HI) fl = fminf(fmaxf(fl, static_cast<float>(LO)), static_cast<float>(HI));
        const int c = static_cast<int>(fl);
        const float t = __fadd_rn(xs[a] - fl, 0.25f);
        const bool hi = t >= 0.5f;
        const float t1 = t + (hi ? -0.5f : 0.5f);
        const float f = fminf(t, t1);
        const float fp = fminf(f, 0.5f - f);
        const float z = fp * fp;
        float p = -2.4023869803067623f;       // -(2 pi)^10 / 11!
        p = fmaf(p, z, 6.693849041319626f);   //  (2 pi)^8 / 9!
        p = fmaf(p, z, -12.208116743813388f); // -(2 pi)^6 / 7!
        p = fmaf(p, z, 12.987878804533656f);  //  (2 pi)^4 / 5!
        p = fmaf(p, z, -6.579736267392906f);  // -(2 pi)^2 / 3!
        p = fmaf(p, z, 1.0f);
        const float s = fp * p;
        const float sg = hi ? -s : s;
        s0.c[a] = c;
        s0.t[a] = t;
        s0.w0[a] = 1.0f - t + sg;
        s1.c[a] = hi ? c : c - 1;
        s1.t[a] = t1;
        s1.w0[a] = 1.0f - t1 - sg;
        sn[a] = sg;
        diag[a] = fmaf(f, fmaf(-2.0f, f, 1.0f), 0.25f) - s;
    }
}
__device__ __forceinline__ void MakeStencilPair(const float (&xs)[3], Stencil32& s0, Stencil32& s1) {
    float sn[3], diag[3];
    MakeStencilPair(xs, s0, s1, sn, diag);
}

// scale * D^-1 (xx, xy, xz, yy, yz, zz), D the moment matrix of both grids in units of
// dx^2: diag on the diagonal, 2 sn_a sn_b off it (adjugate / determinant; the reciprocal
// is v_rcp_f32, 1 ulp).
__device__ __forceinline__ void MomentInverse(const float (&sn)[3], const float (&diag)[3], float scale, float (&r)[6]) {
    const float h = 2.0f * sn[0];
    const float xy = h * sn[1], xz = h * sn[2], yz = 2.0f * sn[1] * sn[2];
    const float c00 = diag[1] * diag[2] - yz * yz;
    const float c01 = xz * yz - xy * diag[2];
    const float c02 = xy * yz - xz * diag[1];
    const float id = scale * __builtin_amdgcn_rcpf(diag[0] * c00 + xy * c01 + xz * c02);
    r[0] = id * c00;
    r[1] = id * c01;
    r[2] = id * c02;
    r[3] = id * (diag[0] * diag[2] - xz * xz);
    r[4] = id * (xy * xz - diag[0] * yz);
    r[5] = id * (diag[0] * diag[1] - xy * xy);
}
__device__ __forceinline__ float NodeWeight(const Stencil32& s, int dx, int dy, int dz) {
    const float wx = dx ? 1.0f - s.w0[0] : s.w0[0];
    const float wy = dy ? 1.0f - s.w0[1] : s.w0[1];
    const float wz = dz ? 1.0f - s.w0[2] : s.w0[2];
    return wx * wy * wz;
}

}  // namespace ckmpm
