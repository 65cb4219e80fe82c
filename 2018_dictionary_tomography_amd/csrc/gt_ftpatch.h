// gt_ftpatch.h -- culling of the Fourier grid and plane evaluations.
//
// An FT-space atom contributes I exp(-|U^T k|^2 / 2) exp(-i x . k) where
// |U^T k|^2 < 30 (GaussDictCode/bin/FTGaussian3D.py:95-110, 151-164): its
// support is an ellipsoid about k = 0.  ft_patch_min bounds |U^T k|^2 from
// below over a rectangle of (k1, k2) at fixed k0, so that a patch of samples
// the support cannot reach is skipped; ft_box_meets does the same for a box, and
// kp_row_range bounds the rows of a sample plane that an ellipse reaches.
// Host-callable for the brute-force checks in tests/native.
#pragma once

#include <hip/hip_runtime.h>

namespace gt {

struct FtL {  // the staged part of an FtRec (64 bytes)
    float amp, xh[3], xl[3], u[6], iso, pad[2];
};
static_assert(sizeof(FtL) == 64, "FtL must stay 64 bytes");

// Smallest scaled |U^T k|^2 over k0 fixed and (k1, k2) in [a1, b1] x [a2, b2]
// (U upper triangular in the slot order of FtRec.u, or iso: u[0] / r).
__host__ __device__ inline float ft_patch_min(const FtL &r, float k0, float a1, float b1, float a2, float b2)
{
    if (r.iso != 0.0f) {
        const float m1 = (a1 <= 0.0f && b1 >= 0.0f) ? 0.0f : fminf(a1 * a1, b1 * b1);
        const float m2 = (a2 <= 0.0f && b2 >= 0.0f) ? 0.0f : fminf(a2 * a2, b2 * b2);
        return (fmaf(k0, k0, m1) + m2) * (r.u[0] * r.u[0]);
    }
    // v0 = U00 k0, v1 = U01 k0 + U11 k1, v2 = U02 k0 + U12 k1 + U22 k2
    const float u00 = r.u[0], u11 = r.u[1], u22 = r.u[2], u01 = r.u[3], u12 = r.u[4], u02 = r.u[5];
    const float v0 = u00 * k0, al1 = u01 * k0, al2 = u02 * k0;
    if (!(u11 != 0.0f) || !(u22 != 0.0f)) return 0.0f;  // degenerate: keep
    const float k1s = -al1 / u11, k2s = -fmaf(u12, k1s, al2) / u22;
    if (k1s >= a1 && k1s <= b1 && k2s >= a2 && k2s <= b2) return v0 * v0;
    float best = 3.0e38f;
    const float A = fmaf(u11, u11, u12 * u12);
#pragma unroll
    for (int e = 0; e < 2; e++) {
        // edge k1 = c: v1 fixed, v2 = w + U22 k2 minimised over k2
        const float c = e ? b1 : a1;
        const float v1 = fmaf(u11, c, al1), w = fmaf(u12, c, al2);
        const float k2 = fminf(fmaxf(-w / u22, a2), b2);
        const float v2 = fmaf(u22, k2, w);
        best = fminf(best, fmaf(v1, v1, v2 * v2));
        // edge k2 = d: (al1 + U11 k1)^2 + (w2 + U12 k1)^2 minimised over k1
        const float d = e ? b2 : a2;
        const float w2 = fmaf(u22, d, al2);
        const float k1 = fminf(fmaxf(-fmaf(al1, u11, w2 * u12) / A, a1), b1);
        const float p1 = fmaf(u11, k1, al1), p2 = fmaf(u12, k1, w2);
        best = fminf(best, fmaf(p1, p1, p2 * p2));
    }
    return fmaf(v0, v0, best);
}

// Can the support {|U^T k| < rho} (scaled as FtRec.u, upper-triangular form) reach the box of half
// extents x about the centre m?  Tested on the plane through the centre across
// the gradient g = U v of |v|^2 / 2, v = U^T m: the support reaches rho |v| along g,
// the box comes as near as |v|^2 - sum |g_c| x_c (relative slack 1e-3; NaN keeps).
__host__ __device__ inline bool ft_box_meets(const FtL &r, float m0, float m1, float m2, float x0, float x1, float x2,
                                             float rho)
{
    const float v0 = r.u[0] * m0, v1 = fmaf(r.u[1], m1, r.u[3] * m0);
    const float v2 = fmaf(r.u[4], m1, fmaf(r.u[5], m0, r.u[2] * m2));
    const float n2 = fmaf(v0, v0, fmaf(v1, v1, v2 * v2));
    const float g0 = fmaf(r.u[0], v0, fmaf(r.u[3], v1, r.u[5] * v2));
    const float g1 = fmaf(r.u[1], v1, r.u[4] * v2), g2 = r.u[2] * v2;
    const float reach = fmaf(fabsf(g0), x0, fmaf(fabsf(g1), x1, fabsf(g2) * x2));
    return !(n2 * (1.0f - 1e-4f) - reach > rho * (1.0f + 1e-3f) * sqrtf(n2));
}

// A form that the two tests below may not cull by: not strictly concave, or so
// long and slanted an ellipse that its FP32 coefficients do not place it.
// det = 4 q0 q2 - q1^2 is off by at most 8 u q0 q2 = 4.8e-7 q0 q2, so the half-width
// and the extreme point of kp_row_range by det's relative error / 2 (2.4e-4 at
// the limit) and a root whose discriminant cancels by 5.5e-4 of the half-width:
// less than its widening of 1e-3 down to det = 1e-3 q0 q2 (axis ratio 126 at 45
// degrees).  With a limit of 1e-6 rows with samples up to 1e-3 of the peak went
// missing at ratios from 700 on.
__host__ __device__ inline bool kp_thin(float q0, float q1, float q2)
{
    return !(q0 < 0.0f) || !(q2 < 0.0f) || !(4.0f * q0 * q2 - q1 * q1 > 1e-3f * q0 * q2);
}

// The rows [xlo, xhi] that the ellipse {q0 x^2 + q1 x y + q2 y^2 >= cut} (cut <
// 0) has in the band ya <= y <= yb: its convex part in the band spans from the
// least to the largest x, each at the ellipse's own extreme point when that
// lies in the band, else on the nearer band edge.  Widened by a relative 1e-3;
// everything for a thin form; empty (xlo > xhi) when the band misses the
// ellipse.
__host__ __device__ inline void kp_row_range(float q0, float q1, float q2, float cut, float ya, float yb, float &xlo,
                                             float &xhi)
{
    xlo = -3.0e38f;
    xhi = 3.0e38f;
    if (kp_thin(q0, q1, q2)) return;
    const float det = 4.0f * q0 * q2 - q1 * q1;
    const float hw = sqrtf(4.0f * cut * q2 / det);  // half-width in x
    const float ys = -0.5f * q1 / q2 * hw;          // y of the point x = hw (x = -hw: -ys)
    const float yr = fminf(fmaxf(ys, ya), yb), yl = fminf(fmaxf(-ys, ya), yb);
    // q0 x^2 + q1 y x + q2 y^2 - cut = 0 at y = yr (larger root) and y = yl (smaller root)
    const float dr = q1 * yr * q1 * yr - 4.0f * q0 * (q2 * yr * yr - cut);
    const float dl = q1 * yl * q1 * yl - 4.0f * q0 * (q2 * yl * yl - cut);
    const float tol = 1e-3f * hw;
    const float i2 = -0.5f / q0;
    xhi = fmaf(q1, yr, sqrtf(fmaxf(dr, 0.0f))) * i2 + tol;
    xlo = fmaf(q1, yl, -sqrtf(fmaxf(dl, 0.0f))) * i2 - tol;
}

// Pairing of the m coordinates of one axis under k -> -k, by one block: 0 if
// k[m-1-i] = -k[i] for every i, 1 if k[m-i] = -k[i] for every i >= 1 (the order of
// an even-sized FFT's frequencies, whose first one has no partner), else -1.
__device__ inline int ft_pairing(const float *k, int m)
{
    bool p0 = true, p1 = true;
    for (int i = threadIdx.x; i < m; i += blockDim.x) {
        p0 = p0 && k[m - 1 - i] == -k[i];
        p1 = p1 && (i == 0 || k[m - i] == -k[i]);
    }
    const int a = __syncthreads_and(p0), b = __syncthreads_and(p1);
    return a ? 0 : (b ? 1 : -1);
}

}  // namespace gt
