// gt_volume.hip -- volume render of Gaussian atoms (GaussTomo.discretise).
//
// u(y) = sum_atoms I sqrt(30/pi) exp(-30 |U (y - x)|^2) [|U (y - x)|^2 <= 1]
// (__f / __VolProj, GaussDictCode/bin/NewtonBases.py:237-257, 698-711 and
// NewtonBases2D.py:16-34, 259-271).
//
// One FP64 setup thread per atom writes a VolRec: amplitude, centre as a
// float pair, U scaled so that the exponent is exp2(-|U'(y-x)|^2), and the
// index box of the ellipsoid |U(y-x)| <= 1 on each (ascending) coordinate
// vector.  The 3D render gives each wave 4 x 8 x 8 voxels and the list of the
// atoms whose support meets them; the 2D render, and the 3D one of few atoms on
// large grids, give each block a tile or rows, stage the atoms whose box meets it
// in LDS (in atom order), and accumulate 4 voxels per lane (2D with Kahan sums).
#include <algorithm>

#include "gt_common.h"

namespace gt {

struct VolRec {
    float amp;
    float xh[3], xl[3];
    float u[6];  // scaled U slots [u00, u11, u22, u01, u12, u02]
    float pad0[3];
    int lo[3], hi[3];
    int pad1[10];
};
static_assert(sizeof(VolRec) == 128, "VolRec must stay 128 bytes");

constexpr double SQRT_NEG_KAPPA = 6.578818071009935;  // sqrt(30 log2 e)

template <int D> __global__ __launch_bounds__(256) void vol_setup_kernel(gt_atoms A, gt_vol V, VolRec *recs)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= A.n) return;
    constexpr int NR = Dims<D>::NR;
    PairGeom<D> g;
    load_atom<D>(A, j, g);
    VolRec rec;
    rec.amp = (float)(g.I * sqrt(30.0 / 3.14159265358979323846));
    for (int i = 0; i < 3; i++) {
        const double xv = (i < D) ? g.x[i] : 0.0;
        rec.xh[i] = (float)xv;
        rec.xl[i] = (float)(xv - (double)rec.xh[i]);
        rec.pad0[i] = 0.0f;
    }
    for (int k = 0; k < 6; k++) rec.u[k] = 0.0f;
    for (int k = 0; k < NR; k++) rec.u[k] = (float)(SQRT_NEG_KAPPA * g.U[slot_row(D, k)][slot_col(D, k)]);
    for (int k = 0; k < 10; k++) rec.pad1[k] = 0;
    const float *y[3] = {V.y0, V.y1, V.y2};
    const int m[3] = {V.m0, V.m1, V.m2};
    // Half-widths of {|U(y-x)| <= 1}: norms of the rows of U^{-1}, i.e. of the
    // columns of U^{-T}; U is upper triangular.
    double Ui[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    bool ok = V.sorted != 0;
    for (int i = 0; i < D; i++) ok = ok && g.U[i][i] != 0.0;
    if (ok) {
        for (int c = D - 1; c >= 0; c--) {  // back substitution for U Ui = Id
            for (int col = 0; col < D; col++) {
                double s = (c == col) ? 1.0 : 0.0;
                for (int k = c + 1; k < D; k++) s -= g.U[c][k] * Ui[k][col];
                Ui[c][col] = s / g.U[c][c];
            }
        }
    }
    for (int c = 0; c < 3; c++) {
        if (c >= D) {
            rec.lo[c] = 0;
            rec.hi[c] = 0;
            continue;
        }
        if (!ok) {
            rec.lo[c] = 0;
            rec.hi[c] = m[c] - 1;
            continue;
        }
        double hw = 0.0;
        for (int k = 0; k < D; k++) hw += Ui[c][k] * Ui[c][k];
        hw = sqrt(hw);
        const double pad = 1e-5 * hw + 1e-7;
        rec.lo[c] = lower_idx(y[c], m[c], g.x[c] - hw - pad);
        rec.hi[c] = upper_idx(y[c], m[c], g.x[c] + hw + pad);
    }
    recs[j] = rec;
}

__device__ inline void vkahan(float &s, float &c, float v)
{
    const float y = v - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

// Stage the atoms whose box meets [b_lo, b_hi] (3 axes), keeping atom order.
__device__ inline int vol_stage(const VolRec *__restrict__ recs, int base, int N, const int *b_lo, const int *b_hi,
                                VolRec *list, int *wcnt)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = base + (int)threadIdx.x;
    bool hit = false;
    if (j < N) {
        const VolRec &r = recs[j];
        hit = r.lo[0] <= b_hi[0] && r.hi[0] >= b_lo[0] && r.lo[1] <= b_hi[1] && r.hi[1] >= b_lo[1] &&
              r.lo[2] <= b_hi[2] && r.hi[2] >= b_lo[2];
    }
    const unsigned long long m = __ballot(hit);
    if (lane == 0) wcnt[wave] = __popcll(m);
    __syncthreads();
    int off = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        if (w < wave) off += wcnt[w];
        total += wcnt[w];
    }
    if (hit) {
        const int4 *src = reinterpret_cast<const int4 *>(recs + j);
        int4 *dst = reinterpret_cast<int4 *>(list + off + __popcll(m & ((1ull << lane) - 1ull)));
#pragma unroll
        for (int k = 0; k < 8; k++) dst[k] = src[k];
    }
    __syncthreads();
    return total;
}

constexpr int VCHUNK = 128;

// 3D: block = brick of V3_PARTS parts of 4 x 8 x 8 voxels (lane = (j1, j2), 4
// voxels along j0 per lane), V3_GROUPS waves per part that take every
// V3_GROUPS-th record of its list; bricks nearest the volume centre first.  A
// thread tests one record against the parts: index box, then (for ascending
// coordinates) the plane through the part's centre across the exponent's
// gradient g there: the support reaches |v| rho along g (v = U'(yc - x), rho^2 =
// -kappa), the voxels come as near as |v|^2 - sum |g_c| extent_c.  Records are read
// into scalar registers; a voxel's values are added in FP64, the groups' totals
// in group order.
// Bound by VALU issue and by the central bricks, which meet the most atoms: the
// parts' lists are split so that no wave is much longer than the rest.  1000
// atoms on 128^3: 0.22 ms with 4 x 4 x 64 bricks culled by index box, 0.083 now;
// with four values at a time summed in FP32 0.081, then (parts, groups) = (4, 1)
// 0.116, (4, 2) 0.092, (2, 4) 0.095, (1, 4) 0.089 against 0.086.
constexpr int V3_PARTS = 2, V3_GROUPS = 2, V3_WAVES = V3_PARTS * V3_GROUPS, V3_THREADS = 64 * V3_WAVES;
constexpr int V3_N1 = V3_PARTS == 4 ? 2 : 1, V3_N2 = V3_PARTS / V3_N1;  // parts per axis
constexpr int V3_B1 = 8 * V3_N1, V3_B2 = 8 * V3_N2;
constexpr unsigned V3_BLOCKS = 16384;

// SPARSE: a block walks the ranks, its own and every gridDim.x-th after it.
template <bool SPARSE>
__global__ __launch_bounds__(V3_THREADS) void volume3_kernel(const VolRec *__restrict__ recs, int N, gt_vol V,
                                                             float *__restrict__ u, int e0, int e1, int e2)
{
    __shared__ unsigned short wl[V3_PARTS][V3_THREADS];
    __shared__ int cnt[V3_PARTS][V3_WAVES];
    __shared__ int wlen[V3_PARTS];
    __shared__ double red[V3_GROUPS - 1][V3_PARTS][4][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = wave % V3_PARTS, grp = wave / V3_PARTS;
    const int nb0 = (V.m0 + 3) / 4, nb1 = (V.m1 + V3_B1 - 1) / V3_B1, nb2 = (V.m2 + V3_B2 - 1) / V3_B2;
    const int e[3] = {e0, e1, e2};
    unsigned rank = blockIdx.x;
    do {
        int t[3];
        morton_ranks(rank, e, t);
        if (t[0] >= nb0 || t[1] >= nb1 || t[2] >= nb2) continue;  // whole block: no brick of this rank
        const int b0 = centre_out(t[0], nb0) * 4, b1 = centre_out(t[1], nb1) * V3_B1, b2 = centre_out(t[2], nb2) * V3_B2;
        const int j1 = b1 + 8 * (sub / V3_N2) + (lane >> 3), j2 = b2 + 8 * (sub % V3_N2) + (lane & 7);
        const float y1 = V.y1[min(j1, V.m1 - 1)], y2 = V.y2[min(j2, V.m2 - 1)];
        float y0[4];
#pragma unroll
        for (int k = 0; k < 4; k++) y0[k] = V.y0[min(b0 + k, V.m0 - 1)];
        // centre and half extent of the waves' voxels per axis
        float c0, h0, c1[2], h1[2], c2[2], h2[2];
        {
            const float za = V.y0[b0], zb = V.y0[min(b0 + 3, V.m0 - 1)];
            c0 = 0.5f * (za + zb);
            h0 = 0.5f * (zb - za);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float ya = V.y1[min(b1 + 8 * h, V.m1 - 1)], yb = V.y1[min(b1 + 8 * h + 7, V.m1 - 1)];
                const float xa = V.y2[min(b2 + 8 * h, V.m2 - 1)], xb = V.y2[min(b2 + 8 * h + 7, V.m2 - 1)];
                c1[h] = 0.5f * (ya + yb);
                h1[h] = 0.5f * (yb - ya);
                c2[h] = 0.5f * (xa + xb);
                h2[h] = 0.5f * (xb - xa);
            }
        }
        const float kap = (float)KAPPA;
        double s[4] = {0.0, 0.0, 0.0, 0.0};
        for (int base = 0; base < N; base += V3_THREADS) {
            unsigned mask = 0;
            const int j = base + (int)threadIdx.x;
            if (j < N) {
                const float4 *src = reinterpret_cast<const float4 *>(recs + j);
                // amp, xh[0..2] | xl[0..2], u0 | u1..u4 | u5, pad ; lo[3], hi[3]
                const float4 f0 = src[0], f1 = src[1], f2 = src[2], f3 = src[3];
                const int4 bx = reinterpret_cast<const int4 *>(src)[4];
                const int2 by = reinterpret_cast<const int2 *>(src)[10];
                if ((int)(bx.x <= b0 + 3) & (int)(bx.w >= b0) & (int)(bx.y <= b1 + V3_B1 - 1) & (int)(by.x >= b1) &
                    (int)(bx.z <= b2 + V3_B2 - 1) & (int)(by.y >= b2)) {
                    const float d0 = (c0 - f0.y) - f1.x;
#pragma unroll
                    for (int w = 0; w < V3_PARTS; w++) {
                        const int q1 = w / V3_N2, q2 = w % V3_N2, a1 = b1 + 8 * q1, a2 = b2 + 8 * q2;
                        const float d1 = (c1[q1] - f0.z) - f1.y, d2 = (c2[q2] - f0.w) - f1.z;
                        const float v0 = fmaf(f1.w, d0, fmaf(f2.z, d1, f3.x * d2)), v1 = fmaf(f2.x, d1, f2.w * d2);
                        const float v2 = f2.y * d2;
                        const float n2 = fmaf(v0, v0, fmaf(v1, v1, v2 * v2));
                        const float g0 = f1.w * v0, g1 = fmaf(f2.z, v0, f2.x * v1);
                        const float g2 = fmaf(f3.x, v0, fmaf(f2.w, v1, f2.y * v2));
                        const float reach = fmaf(fabsf(g0), h0, fmaf(fabsf(g1), h1[q1], fabsf(g2) * h2[q2]));
                        // NaN keeps the record
                        const bool apart =
                            V.sorted && n2 * (1.0f - 1e-4f) - reach > ((float)SQRT_NEG_KAPPA + 1e-2f) * sqrtf(n2);
                        if (bx.y <= a1 + 7 && by.x >= a1 && bx.z <= a2 + 7 && by.y >= a2 && !apart) mask |= 1u << w;
                    }
                }
            }
            wave_lists<V3_WAVES, V3_PARTS>(mask, wl, cnt, wlen);
            const int len = __builtin_amdgcn_readfirstlane(wlen[sub]);
            for (int q = grp; q < len; q += V3_GROUPS) {
                smem<VolRec> *r = scalar_ptr(recs) + (base + __builtin_amdgcn_readfirstlane((int)wl[sub][q]));
                const float d1 = (y1 - r->xh[1]) - r->xl[1], d2 = (y2 - r->xh[2]) - r->xl[2];
                const float a0 = fmaf(r->u[3], d1, r->u[5] * d2);
                const float v1 = fmaf(r->u[1], d1, r->u[4] * d2), v2 = r->u[2] * d2;
                const float c = -fmaf(v1, v1, v2 * v2);
                const float amp = r->amp, u0 = r->u[0], xh = r->xh[0], xl = r->xl[0];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float v0 = fmaf(u0, (y0[k] - xh) - xl, a0);
                    const float ex = fmaf(-v0, v0, c);
                    // the term is chosen, not its profile: 0 times an infinite amplitude is no 0
                    const float v = amp * __builtin_amdgcn_exp2f(ex);
                    s[k] += (double)(ex >= kap ? v : 0.0f);
                }
            }
            __syncthreads();
        }
        // the groups' totals, in group order
        if (grp > 0)
#pragma unroll
            for (int k = 0; k < 4; k++) red[grp - 1][sub][k][lane] = s[k];
        __syncthreads();
        if (grp > 0) continue;  // (red is written again after the next brick's barriers)
        for (int g = 0; g < V3_GROUPS - 1; g++)
#pragma unroll
            for (int k = 0; k < 4; k++) s[k] += red[g][sub][k][lane];
        if (j1 < V.m1 && j2 < V.m2)
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (b0 + k < V.m0) u[((size_t)(b0 + k) * V.m1 + j1) * V.m2 + j2] = (float)s[k];
    } while (SPARSE && (rank += gridDim.x) < (1u << (e0 + e1 + e2)));
}

// 3D, few atoms: block = brick of 4 (j0, one per wave) x 4 (j1, per lane) x 64 (j2, lane).
__global__ __launch_bounds__(256) void volume3_rows_kernel(const VolRec *__restrict__ recs, int N, gt_vol V,
                                                           float *__restrict__ u)
{
    __shared__ VolRec list[VCHUNK];
    __shared__ int wcnt[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nb2 = (V.m2 + 63) / 64, nb1 = (V.m1 + 3) / 4;
    int b = blockIdx.x;
    const int bb2 = b % nb2;
    b /= nb2;
    const int bb1 = b % nb1;
    const int bb0 = b / nb1;
    const int j0 = bb0 * 4 + wave, j1b = bb1 * 4, j2 = bb2 * 64 + lane;
    const int blo[3] = {bb0 * 4, j1b, bb2 * 64};
    const int bhi[3] = {min(bb0 * 4 + 3, V.m0 - 1), min(j1b + 3, V.m1 - 1), min(bb2 * 64 + 63, V.m2 - 1)};
    const float y0 = V.y0[min(j0, V.m0 - 1)];
    const float y2 = V.y2[min(j2, V.m2 - 1)];
    float y1[4];
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 4; k++) y1[k] = V.y1[min(j1b + k, V.m1 - 1)];
    for (int base = 0; base < N; base += VCHUNK) {
        // stage with the first VCHUNK threads only
        const int total = vol_stage(recs, base, min(N, base + VCHUNK), blo, bhi, list, wcnt);
        for (int e = 0; e < total; e++) {
            const VolRec &r = list[e];
            if (r.lo[0] > j0 || r.hi[0] < j0) continue;
            const float d0 = (y0 - r.xh[0]) - r.xl[0];
            const float d2 = (y2 - r.xh[2]) - r.xl[2];
            const float a0 = fmaf(r.u[0], d0, r.u[5] * d2);
            const float a1 = r.u[4] * d2;
            const float u2 = r.u[2] * d2;
            const float c2 = u2 * u2;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float d1 = (y1[k] - r.xh[1]) - r.xl[1];
                const float u0 = fmaf(r.u[3], d1, a0);
                const float u1 = fmaf(r.u[1], d1, a1);
                const float q = -fmaf(u0, u0, fmaf(u1, u1, c2));
                if (q >= (float)KAPPA) s[k] += (double)(r.amp * __builtin_amdgcn_exp2f(q));
            }
        }
        __syncthreads();
    }
    if (j0 < V.m0 && j2 < V.m2)
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (j1b + k < V.m1) u[((size_t)j0 * V.m1 + j1b + k) * V.m2 + j2] = (float)s[k];
}

// 2D: block tile = 16 rows (j0, 4 per lane, 4 waves) x 64 cols (j1, lane).
__global__ __launch_bounds__(256) void volume2_kernel(const VolRec *__restrict__ recs, int N, gt_vol V,
                                                      float *__restrict__ u)
{
    __shared__ VolRec list[VCHUNK];
    __shared__ int wcnt[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nb1 = (V.m1 + 63) / 64;
    const int bb0 = blockIdx.x / nb1, bb1 = blockIdx.x - bb0 * nb1;
    const int r0 = bb0 * 16 + wave * 4, j1 = bb1 * 64 + lane;
    const int blo[3] = {bb0 * 16, bb1 * 64, 0};
    const int bhi[3] = {min(bb0 * 16 + 15, V.m0 - 1), min(bb1 * 64 + 63, V.m1 - 1), 0};
    const float y1 = V.y1[min(j1, V.m1 - 1)];
    float y0[4], s[4], c[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        y0[k] = V.y0[min(r0 + k, V.m0 - 1)];
        s[k] = 0.0f;
        c[k] = 0.0f;
    }
    for (int base = 0; base < N; base += VCHUNK) {
        const int total = vol_stage(recs, base, min(N, base + VCHUNK), blo, bhi, list, wcnt);
        for (int e = 0; e < total; e++) {
            const VolRec &r = list[e];
            if (r.lo[0] > r0 + 3 || r.hi[0] < r0) continue;
            const float d1 = (y1 - r.xh[1]) - r.xl[1];
            const float u1 = r.u[1] * d1;
            const float c1 = u1 * u1;
            const float a0 = r.u[2] * d1;  // slot 2 of a 2D atom is u01
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float d0 = (y0[k] - r.xh[0]) - r.xl[0];
                const float u0 = fmaf(r.u[0], d0, a0);
                const float q = -fmaf(u0, u0, c1);
                if (q >= (float)KAPPA) vkahan(s[k], c[k], r.amp * __builtin_amdgcn_exp2f(q));
            }
        }
        __syncthreads();
    }
    if (j1 < V.m1)
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (r0 + k < V.m0) u[(size_t)(r0 + k) * V.m1 + j1] = s[k];
}

int launch_fill(float *p, size_t n, float v, hipStream_t st);

static int check_vol(const gt_vol *v, int dim)
{
    GT_CHECK_ARG(v != nullptr, "volume grid is NULL");
    GT_CHECK_ARG(v->dim == dim, "volume.dim (%d) does not match atoms.dim (%d)", v->dim, dim);
    GT_CHECK_ARG(v->m0 >= 1 && v->m1 >= 1 && v->m2 >= 1, "volume sizes must be >= 1");
    GT_CHECK_ARG(v->m0 < (1 << 24) && v->m1 < (1 << 24) && v->m2 < (1 << 24), "volume sizes out of range");
    if (dim == 2) GT_CHECK_ARG(v->m2 == 1, "2D volume needs m2 == 1");
    GT_CHECK_ARG(v->y0 && v->y1 && (dim == 2 || v->y2), "volume coordinate vectors must be non-NULL");
    GT_CHECK_ARG(v->sorted == 0 || v->sorted == 1, "volume.sorted must be 0 or 1");
    return 0;
}

}  // namespace gt

using namespace gt;

extern "C" size_t gt_volume_workspace(const gt_atoms *atoms, const gt_vol *vol)
{
    (void)vol;
    if (!atoms) return 0;
    return align_up((size_t)atoms->n * sizeof(VolRec));
}

extern "C" int gt_volume(const gt_atoms *atoms, const gt_vol *vol, float *u, void *ws, size_t ws_bytes, void *stream)
{
    int rc;
    if ((rc = check_atoms(atoms)) || (rc = check_vol(vol, atoms->dim))) return rc;
    GT_CHECK_ARG(u != nullptr, "gt_volume: u is NULL");
    const size_t need = gt_volume_workspace(atoms, vol);
    if (need > ws_bytes || (need > 0 && ws == nullptr)) {
        set_error("gt_volume: workspace of %zu bytes given, %zu needed", ws_bytes, need);
        return GT_EWORKSPACE;
    }
    GT_CHECK_ARG(((uintptr_t)ws & 127) == 0, "gt_volume: workspace must be 128-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    const size_t nout = (size_t)vol->m0 * vol->m1 * vol->m2;
    if (atoms->n == 0) return launch_fill(u, nout, 0.0f, st);
    gt_vol V = *vol;
    if (atoms->dim == 2) V.y2 = V.y1;  // unused third axis
    VolRec *recs = (VolRec *)ws;
    const unsigned sb = (unsigned)((atoms->n + 255) / 256);
    if (atoms->dim == 3) {
        hipLaunchKernelGGL(vol_setup_kernel<3>, dim3(sb), dim3(256), 0, st, *atoms, V, recs);
        // bricks numbered by Morton index over 2^e0 x 2^e1 x 2^e2 centre-out ranks
        const int e[3] = {ceil_log2((V.m0 + 3) / 4), ceil_log2((V.m1 + V3_B1 - 1) / V3_B1),
                          ceil_log2((V.m2 + V3_B2 - 1) / V3_B2)};
        GT_CHECK_ARG(e[0] + e[1] + e[2] <= 30, "gt_volume: grid too large");
        prof_begin(st, GT_K_VOLUME);
        const unsigned ranks = 1u << (e[0] + e[1] + e[2]);
        const unsigned long long bricks =
            (unsigned long long)((V.m0 + 3) / 4) * ((V.m1 + V3_B1 - 1) / V3_B1) * ((V.m2 + V3_B2 - 1) / V3_B2);
        const bool sparse = 2 * bricks < ranks;  // most ranks are no bricks
        // Few atoms on many bricks: most see none, and rows of 64 voxels are written
        // faster (where there are such rows).  Call times, us, bricks and rows: 256^3
        // voxels, 1 atom 53 and 24, 32 68 and 54, 64 73 and 78; 512^3, 32 450 and 303, 64
        // 482 and 482; sparse ones, with the blocks below, 384^3, 64 219 and 179, 128 309
        // and 303; 320^3, 128 197 and 188; up to 4096 ranks (128^3, 32 atoms) 19 and 18;
        // rows of 4 voxels (512 x 512 x 4, 32 atoms) 24 and 57.
        if (V.m2 >= 64 && ranks > 4096 && atoms->n <= (sparse && ranks > 32768 ? 128 : 64)) {
            const unsigned long long rows = (unsigned long long)((V.m0 + 3) / 4) * ((V.m1 + 3) / 4) * ((V.m2 + 63) / 64);
            GT_CHECK_ARG(rows < (1ull << 31), "gt_volume: grid too large");
            hipLaunchKernelGGL(volume3_rows_kernel, dim3((unsigned)rows), dim3(256), 0, st, recs, atoms->n, V, u);
        } else {
            // sparse ranks are walked by V3_BLOCKS blocks: starting a block for each
            // costs 1 ns (384^3, 64 atoms 259 us, now 219); with bricks for most ranks
            // a block each is 3 to 10% faster, it starts when another ends
            if (sparse)
                hipLaunchKernelGGL(volume3_kernel<true>, dim3(std::min(ranks, V3_BLOCKS)), dim3(V3_THREADS), 0, st, recs,
                                   atoms->n, V, u, e[0], e[1], e[2]);
            else
                hipLaunchKernelGGL(volume3_kernel<false>, dim3(ranks), dim3(V3_THREADS), 0, st, recs, atoms->n, V, u, e[0],
                                   e[1], e[2]);
        }
        prof_end(st, GT_K_VOLUME);
    } else {
        hipLaunchKernelGGL(vol_setup_kernel<2>, dim3(sb), dim3(256), 0, st, *atoms, V, recs);
        const long blocks = (long)((V.m0 + 15) / 16) * ((V.m1 + 63) / 64);
        prof_begin(st, GT_K_VOLUME);
        hipLaunchKernelGGL(volume2_kernel, dim3((unsigned)blocks), dim3(256), 0, st, recs, atoms->n, V, u);
        prof_end(st, GT_K_VOLUME);
    }
    GT_HIP(hipGetLastError());
    return 0;
}
