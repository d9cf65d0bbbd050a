// Compact-kernel stencils of the two CK-MPM sub-grids (mpm_kernel.cuh:91-114):
// base node, fractional offset t and node-0 weight w0 = 1 - t + sin(2 pi t)/(2 pi)
// per axis; node 1 of an axis has weight 1 - w0.
#pragma once
#include "common.h"

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

// Slopes d w0 / d t = -1 + cos(2 pi t) of both sub-grids on one axis, from one cosine: the
// grids' offsets differ by 1/2, so their cosines by the sign.  With f = min(t0, t1) in
// [0, 1/2) and f' = min(f, 1/2 - f) in [0, 1/4], cos(2 pi f) = +-cos(2 pi f'), where the
// Taylor series through x^14 is within 7e-11 (the next term, x^16 / 16!, at x = pi / 2).  In
// FP64 but for the terms from x^8 on (9e-4 at most, in FP32 within 1e-10), so the slopes are
// rounded once, by at most 6e-8: in FP32 the rounding of x^2 and of the last steps made it
// 1.9e-7.  (All terms in FP64: 1 to 2 us more in a 30 and a 49 us launch.)
__host__ __device__ __forceinline__ void SlopePair(float t0, float t1, float& d0, float& d1) {
    const float f = fminf(t0, t1), g = 0.5f - f;
    const double fp = fminf(f, g);
    const double z = 39.478417604357434 * (fp * fp);  // (2 pi f')^2
    const float zf = static_cast<float>(z);
    float t = -1.1470745597729725e-11f;               // -1 / 14!
    t = fmaf(t, zf, 2.08767569878681e-09f);           //  1 / 12!
    t = fmaf(t, zf, -2.755731922398589e-07f);         // -1 / 10!
    t = fmaf(t, zf, 2.48015873015873e-05f);           //  1 / 8!
    double e = z * static_cast<double>(t) - 1.388888888888889e-03;  // -1 / 6!
    e = z * e + 4.166666666666666e-02;                //  1 / 4!
    e = z * (z * e - 0.5);                            // cos(2 pi f') - 1
    const bool neg = (g < f) != (t0 >= 0.5f);         // the sign of cos(2 pi t0)
    const float u = static_cast<float>(e), w = static_cast<float>(-2.0 - e);
    d0 = neg ? w : u;
    d1 = neg ? u : w;
}

// scale * D^-1 (xx, xy, xz, yy, yz, zz), D the moment matrix of both grids in units of
// dx^2: diag on the diagonal, 2 sn_a sn_b off it (adjugate / determinant, data_type.cuh:369-387;
// the reciprocal is v_rcp_f32, 1 ulp).
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

// ---------------------------------------------------------------- velocity window
// Velocities in reach of a particle block's own cells 2..5, in LDS: nodes [2,6]^3 of grid 0
// and [1,6]^3 of grid 1 (node coordinates relative to the block's first node, 0..7 over the
// block and its +1 neighbours).  Strides (in entries) of y and x.
constexpr int kV0Y = 5, kV0X = 25, kV1Y = 6, kV1X = 36;
constexpr int kV0Win = 4 * kV0X + 4 * kV0Y + 5;
constexpr int kVWin = kV0Win + 5 * kV1X + 5 * kV1Y + 6;
constexpr int kCoreNodes = 125 + 216;    // nodes in reach of the block's own cells 2..5
constexpr int kCoreColumns = 2 * (25 + 36);  // their z columns, one per block and (x, y)
// Window entry of node (x, y, z) of sub-grid g.
__device__ __forceinline__ int VEntry(int g, int lx, int ly, int lz) {
    return g ? kV0Win + (lx - 1) * kV1X + (ly - 1) * kV1Y + (lz - 1) : (lx - 2) * kV0X + (ly - 2) * kV0Y + (lz - 2);
}
// Core node e of kCoreNodes, grid 1 first.
__device__ __forceinline__ void CoreNode(int e, int& g, int& lx, int& ly, int& lz) {
    const bool g1 = e < 216;
    const int n = g1 ? 6 : 5, q = g1 ? e : e - 216, lo = g1 ? 1 : 2;
    const int qx = g1 ? q / 36 : q / 25, qy = g1 ? q / 6 : q / 5;
    g = g1 ? 1 : 0;
    lx = qx + lo;
    ly = qy - qx * n + lo;
    lz = q - qy * n + lo;
}

// Fills the window from the 2x2x2 halo blocks: a thread takes a z column of 4 nodes of a
// grid block (16-byte loads) and stores the nodes inside the window: z = lo..3 of the block
// at z offset 0, 4..6 of the one above.
template <int THREADS>
__device__ __forceinline__ void StageVelocity(float* sV, const float* V, const uint32_t* sHalo, uint32_t tid) {
    for (int e = tid; e < kCoreColumns; e += THREADS) {
        const bool g1 = e < 72;
        const int col = (g1 ? e : e - 72) >> 1, zb = e & 1, lo = g1 ? 1 : 2;
        const int lx = (g1 ? col / 6 : col / 5) + lo, ly = col - (lx - lo) * (g1 ? 6 : 5) + lo;
        const uint32_t bi = sHalo[((lx >> 2) << 2) | ((ly >> 2) << 1) | zb];
        const float4* src = reinterpret_cast<const float4*>(V + static_cast<size_t>(bi) * kVFloats + (g1 ? 64 : 0) +
                                                            (lx & 3) * 16 + (ly & 3) * 4);
        const int r0 = VEntry(g1 ? 1 : 0, lx, ly, zb ? 4 : lo);
#pragma unroll
        for (int ch = 0; ch < kVChannels; ++ch) {
            const float4 v = bi != kEmpty ? src[32 * ch] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            float* d = sV + ch * kVWin + r0;
            d[0] = zb ? v.x : (g1 ? v.y : v.z);
            d[1] = zb ? v.y : (g1 ? v.z : v.w);
            if (zb || g1) d[2] = zb ? v.z : v.w;
        }
    }
}

// G2P of sub-grid g from the window: v (grid 0 sets it, grid 1 adds) and B in units of dx.
// B = sum_i v_i (x_i - x_p)^T w_i with x_i - x_p = (o - t) dx per axis:
// B_rc = dx (S_rc - vg_r t_c), S_rc = sum over the nodes with o_c = 1 of w v_r.  The weights
// are a tensor product, so vg and S are contracted axis by axis (z, then y, then x): 22
// instructions per channel.
template <int g>
__device__ __forceinline__ void ContractG2P(const float* sV, const Stencil32& sg, float (&v)[3], float (&B)[9]) {
    constexpr int s1 = g ? kV1Y : kV0Y, s2 = g ? kV1X : kV0X, lo = g ? 1 : 2;
    const float* base = sV + (g ? kV0Win : 0) + (sg.c[0] - lo) * s2 + (sg.c[1] - lo) * s1 + (sg.c[2] - lo);
    const float wx0 = sg.w0[0], wy0 = sg.w0[1], wz0 = sg.w0[2];
    const float wx1 = 1.0f - wx0, wy1 = 1.0f - wy0, wz1 = 1.0f - wz0;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const float* vr = base + r * kVWin;
        float T[4], U[4];  // per (x, y) column: sum over z, z-moment
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int off = (q >> 1) * s2 + (q & 1) * s1;
            U[q] = wz1 * vr[off + 1];
            T[q] = fmaf(wz0, vr[off], U[q]);
        }
        float P[2], Q[2], Z[2];  // per x row: sum over y and z, y-moment, z-moment
#pragma unroll
        for (int ox = 0; ox < 2; ++ox) {
            Q[ox] = wy1 * T[ox * 2 + 1];
            P[ox] = fmaf(wy0, T[ox * 2], Q[ox]);
            Z[ox] = fmaf(wy0, U[ox * 2], wy1 * U[ox * 2 + 1]);
        }
        const float S0 = wx1 * P[1];
        const float vg = fmaf(wx0, P[0], S0);
        const float S[3] = {S0, fmaf(wx0, Q[0], wx1 * Q[1]), fmaf(wx0, Z[0], wx1 * Z[1])};
        v[r] = g ? v[r] + vg : vg;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float b = fmaf(-vg, sg.t[c], S[c]);
            B[r * 3 + c] = g ? B[r * 3 + c] + b : b;
        }
    }
}

// G2P of one sub-grid from the halo blocks in global memory, for a stencil outside the
// velocity window: adds to v (sum of both grids) and B (in units of dx).
__device__ __forceinline__ void GatherG2P(int g, const Stencil32& s, const uint32_t* sHalo, const float* V, float (&v)[3],
                                          float (&B)[9]) {
#pragma unroll 1
    for (int o = 0; o < 8; ++o) {
        const int ox = (o >> 2) & 1, oy = (o >> 1) & 1, oz = o & 1;
        const int lx = min(max(s.c[0] + ox, 0), 7), ly = min(max(s.c[1] + oy, 0), 7), lz = min(max(s.c[2] + oz, 0), 7);
        const uint32_t bi = sHalo[((lx >> 2) << 2) | ((ly >> 2) << 1) | (lz >> 2)];
        if (bi == kEmpty) continue;
        const float* src = V + static_cast<size_t>(bi) * kVFloats + g * 64 + (lx & 3) * 16 + (ly & 3) * 4 + (lz & 3);
        const float w = NodeWeight(s, ox, oy, oz);
        const float d[3] = {static_cast<float>(ox) - s.t[0], static_cast<float>(oy) - s.t[1],
                            static_cast<float>(oz) - s.t[2]};
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const float wv = w * src[128 * r];
            v[r] += wv;
#pragma unroll
            for (int c = 0; c < 3; ++c) B[r * 3 + c] = fmaf(wv, d[c], B[r * 3 + c]);
        }
    }
}

}  // namespace ckmpm
