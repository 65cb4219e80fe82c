// gt_fourier.hip -- analytic Fourier transform of Gaussian atoms on a grid.
//
// out(k) = sum_atoms I exp(-|U^T k|^2 / 2) exp(-i x . k)   if |U^T k|^2 < 30
// with (I, x, r) the FT-space parameters (Fourier_Transform.py:293-333); the
// isotropic form uses |U^T k|^2 := |k|^2 / r^2.  This is __grid_eval_aniso /
// __grid_eval_iso, GaussDictCode/bin/FTGaussian3D.py:95-110, 151-164.
//
// Accuracy: the phase x . k reaches hundreds of radians, where an FP32 phase
// would carry ~1e-5 relative error.  The setup stores x / (2 pi) as an FP32
// pair (xh + xl, ~48 bits) and the kernel forms the phase in turns with an
// exact FMA product xh * k = p + e, reduces p exactly by rint, and evaluates
// the hardware sine and cosine (argument in turns) on the small remainder.
// Per-point complex sums are taken in FP64.
#include "gt_common.h"
#include "gt_ftpatch.h"

namespace gt {

struct FtRec {
    float amp;
    float xh[3], xl[3];  // x / (2 pi) as float pairs
    float u[6];          // U^T k coefficients scaled by sqrt(log2(e) / 2)
    float iso;           // 1: isotropic form, u[0] = sqrt(log2(e)/2) / r
    float pad0[2];
    int lo[3], hi[3];
    int pad1[10];
};
static_assert(sizeof(FtRec) == 128, "FtRec must stay 128 bytes");

constexpr double HALF_LOG2E_SQRT = 0.8493218002880191;  // sqrt(log2(e) / 2)
constexpr double FT_CUT = 30.0;                         // |U^T k|^2 < 30
constexpr double TWO_PI = 6.283185307179586;

__device__ inline FtRec ft_record(const gt_atoms &A, const gt_kgrid &Kg, int j)
{
    FtRec rec;
    rec.amp = A.I[j];
    for (int i = 0; i < 3; i++) {
        const double xv = (double)A.x[(size_t)j * 3 + i] / TWO_PI;
        rec.xh[i] = (float)xv;
        rec.xl[i] = (float)(xv - (double)rec.xh[i]);
    }
    for (int k = 0; k < 6; k++) rec.u[k] = 0.0f;
    rec.pad0[0] = rec.pad0[1] = 0.0f;
    for (int k = 0; k < 10; k++) rec.pad1[k] = 0;
    double hw[3];
    bool ok = Kg.sorted != 0;
    if (A.iso) {
        const double r = A.r[j];
        rec.iso = 1.0f;
        rec.u[0] = (float)(HALF_LOG2E_SQRT / r);
        for (int c = 0; c < 3; c++) hw[c] = fabs(r) * sqrt(FT_CUT);
        ok = ok && r != 0.0;
    } else {
        rec.iso = 0.0f;
        double U[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
        for (int k = 0; k < 6; k++) {
            U[slot_row(3, k)][slot_col(3, k)] = A.r[(size_t)j * 6 + k];
            rec.u[k] = (float)(HALF_LOG2E_SQRT * A.r[(size_t)j * 6 + k]);
        }
        // {k : |U^T k|^2 < 30}: half-width along k_c = sqrt(30) * |column c of U^{-1}|.
        for (int i = 0; i < 3; i++) ok = ok && U[i][i] != 0.0;
        double Ui[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
        if (ok) {
            for (int c = 2; c >= 0; c--)
                for (int col = 0; col < 3; col++) {
                    double s = (c == col) ? 1.0 : 0.0;
                    for (int k = c + 1; k < 3; k++) s -= U[c][k] * Ui[k][col];
                    Ui[c][col] = s / U[c][c];
                }
        }
        for (int c = 0; c < 3; c++) {
            double s = 0.0;
            for (int i = 0; i < 3; i++) s += Ui[i][c] * Ui[i][c];
            hw[c] = sqrt(FT_CUT * s);
        }
    }
    const float *kv[3] = {Kg.k0, Kg.k1, Kg.k2};
    const int m[3] = {Kg.m0, Kg.m1, Kg.m2};
    for (int c = 0; c < 3; c++) {
        if (!ok) {
            rec.lo[c] = 0;
            rec.hi[c] = m[c] - 1;
        } else {
            const double pad = 1e-5 * hw[c] + 1e-7;
            rec.lo[c] = lower_idx(kv[c], m[c], -hw[c] - pad);
            rec.hi[c] = upper_idx(kv[c], m[c], hw[c] + pad);
        }
    }
    // radius of a ball about k = 0 holding the support's box (+inf: no bound)
    rec.pad0[0] = ok ? (float)(sqrt(hw[0] * hw[0] + hw[1] * hw[1] + hw[2] * hw[2]) * (1.0 + 1e-5) + 1e-6)
                     : __builtin_huge_valf();
    return rec;
}

__global__ __launch_bounds__(256) void ft_setup_kernel(gt_atoms A, gt_kgrid Kg, FtRec *recs)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < A.n) recs[j] = ft_record(A, Kg, j);
}

// phase in turns of x . k for one axis: exact product split, integer part dropped
__device__ inline float turns(float xh, float xl, float k, float &err)
{
    const float p = xh * k;
    const float e = fmaf(xh, k, -p);
    err += fmaf(xl, k, e);
    return p - rintf(p);
}

// ---------------------------------------------------------------------------
// Every atom's support {|U^T k|^2 < 30} is an ellipsoid about k = 0 (about 1%
// of a 128^3 grid), so the samples near the origin see nearly every atom and
// most patches of samples see few or none.  With tables (ft_tabulated) atoms are
// evaluated in three kernels: the atoms' records and phase tables
// (ft_atoms_kernel); per cell of many patches the list of the records that reach
// it, and the list of the patches of the cells with any (ft_bin_kernel, which
// also clears the output); those patches (ft_grid_kernel).
// ---------------------------------------------------------------------------
constexpr int FZ_MAX_ATOMS = 16384;  // more: ft_patch_kernel, without the tables' memory
constexpr size_t FZ_MAX_BYTES = (size_t)256 << 20;  // as above; more only up to the output's size

// State of one evaluation: the axes' pairing, the number of listed patches by
// class of their cell's record count (most first) and the next one to be taken.
constexpr int FZ_CLASSES = 8;
struct FzState {
    int pairing[3];
    unsigned next, count[FZ_CLASSES];
};

// Phase tables and records.  Blocks below `tabs`: one wave per FZ_TAB entries of an
// atom's phase table exp(-i x_c k) over the m0 + m1 + m2 grid coordinates, from FP64,
// the first axis' entries times the amplitude (block 0 also finds the axes' pairing).
// Later blocks: one thread per atom, its record (an isotropic atom's form |k|^2 /
// r^2 as the diagonal U = Id / r).
constexpr int FZ_TAB = 512;
__global__ __launch_bounds__(256) void ft_atoms_kernel(gt_atoms A, gt_kgrid Kg, unsigned tabs, FtRec *recs,
                                                       FzState *state, float2 *__restrict__ tab)
{
    if (blockIdx.x >= tabs) {
        const int j = (int)(blockIdx.x - tabs) * 256 + (int)threadIdx.x;
        if (j >= A.n) return;
        FtRec rec = ft_record(A, Kg, j);
        if (A.iso) {
            rec.u[1] = rec.u[2] = rec.u[0];
            rec.iso = 0.0f;
        }
        recs[j] = rec;
        return;
    }
    if (blockIdx.x == 0) {
        const int s0 = ft_pairing(Kg.k0, Kg.m0), s1 = ft_pairing(Kg.k1, Kg.m1), s2 = ft_pairing(Kg.k2, Kg.m2);
        if (threadIdx.x == 0) {
            state->pairing[0] = (s0 >= 0 && s1 >= 0 && s2 >= 0 && Kg.sorted) ? s0 : -1;
            state->pairing[1] = s1;
            state->pairing[2] = s2;
            state->next = 0u;
            for (int c = 0; c < FZ_CLASSES; c++) state->count[c] = 0u;
        }
    }
    const int lane = threadIdx.x & 63;
    const int m = Kg.m0 + Kg.m1 + Kg.m2, parts = (m + FZ_TAB - 1) / FZ_TAB;
    const unsigned w = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int j = (int)(w / (unsigned)parts), first = (int)(w % (unsigned)parts) * FZ_TAB;
    if (j >= A.n) return;
    const double x0 = A.x[(size_t)j * 3], x1 = A.x[(size_t)j * 3 + 1], x2 = A.x[(size_t)j * 3 + 2], amp = A.I[j];
    float2 *tj = tab + (size_t)j * m;
    for (int i = first + lane; i < min(first + FZ_TAB, m); i += 64) {
        const bool f0 = i < Kg.m0, f1 = i < Kg.m0 + Kg.m1;
        const float k = f0 ? Kg.k0[i] : (f1 ? Kg.k1[i - Kg.m0] : Kg.k2[i - Kg.m0 - Kg.m1]);
        const double t = (f0 ? x0 : (f1 ? x1 : x2)) * (double)k / TWO_PI, am = f0 ? amp : 1.0;
        double sn, cs;
        sincospi(2.0 * (t - rint(t)), &sn, &cs);
        tj[i] = make_float2((float)(am * cs), (float)(-am * sn));
    }
}

// Patches of FZ_K0 x 8 x 8 samples; cells of q[0] x q[1] x q[2] patches, at most
// 16 x 8 x 8 of them, numbered by Morton index over 2^e0 x 2^e1 x 2^e2 centre-out
// ranks: those near k = 0, which meet the most atoms, first.
constexpr int FZ_WAVES = 16, FZ_THREADS = 64 * FZ_WAVES, FZ_K0 = 2, FZ_PATCH = 8;
constexpr unsigned FZ_BLOCKS = 512;  // (one per CU is resident at its 75 registers; 256 blocks: 1% slower)
constexpr int FB_THREADS = 512;       // ft_bin_kernel
struct FzCells {
    int nb[3], q[3], nc[3], e[3];  // patches, patches per cell, cells, bits per axis
    unsigned cells;                // 2^(e0 + e1 + e2): slots of the cell numbering
};

// One block per cell.  Its records, in atom order: a thread per record, index
// box, then (for ascending coordinates) ft_box_meets.  Then its patches, if it
// has any records: appended as (first indices, cell) to the list of the cell's
// class (each of room for all patches), so that the long ones are taken first.
// Left out are those that are written with their partners: out(-k) =
// conj(out(k)), so on a grid that pairs k with -k the patches of k0 < 0 whose
// samples all have a partner.
__global__ __launch_bounds__(FB_THREADS) void ft_bin_kernel(const FtRec *__restrict__ recs, int N, gt_kgrid Kg, FzCells F,
                                                     FzState *state, unsigned short *__restrict__ ids,
                                                     int *__restrict__ counts, int4 *__restrict__ list,
                                                     float2 *__restrict__ out, size_t nout)
{
    for (size_t i = (size_t)blockIdx.x * FB_THREADS + threadIdx.x; i < nout; i += (size_t)gridDim.x * FB_THREADS)
        out[i] = make_float2(0.0f, 0.0f);
    const unsigned cell = blockIdx.x;
    if (cell >= F.cells) return;
    int t[3];
    morton_ranks(cell, F.e, t);
    if (t[0] >= F.nc[0] || t[1] >= F.nc[1] || t[2] >= F.nc[2]) return;
    __shared__ int cnt[FB_THREADS / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int pa[3], pb[3], lo[3], hi[3];  // the cell's patches [pa, pb) and samples [lo, hi]
    const int m[3] = {Kg.m0, Kg.m1, Kg.m2}, size[3] = {FZ_K0, FZ_PATCH, FZ_PATCH};
    const float *kv[3] = {Kg.k0, Kg.k1, Kg.k2};
    float mid[3], ext[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        pa[c] = centre_out(t[c], F.nc[c]) * F.q[c];
        pb[c] = min(pa[c] + F.q[c], F.nb[c]);
        lo[c] = pa[c] * size[c];
        hi[c] = min(pb[c] * size[c], m[c]) - 1;
        const float ka = kv[c][lo[c]], kb = kv[c][hi[c]];
        mid[c] = 0.5f * (ka + kb);
        ext[c] = 0.5f * (kb - ka);
    }
    const int s0 = state->pairing[0], s1 = state->pairing[1], s2 = state->pairing[2];
    if (s0 >= 0 && Kg.k0[hi[0]] < 0.0f && lo[0] >= s0 && lo[1] >= s1 && lo[2] >= s2) return;  // all with partners
    const float rho = (float)(sqrt(FT_CUT) * HALF_LOG2E_SQRT);
    unsigned short *mine = ids + (size_t)cell * N;
    int total = 0;
    for (int base = 0; base < N; base += FB_THREADS) {
        const int j = base + (int)threadIdx.x;
        bool hit = false;
        if (j < N) {
            const FtL rec = *reinterpret_cast<const FtL *>(recs + j);
            const int4 bx = reinterpret_cast<const int4 *>(recs + j)[4];   // lo[3], hi[0]
            const int2 by = reinterpret_cast<const int2 *>(recs + j)[10];  // hi[1], hi[2]
            hit = ((int)(bx.x <= hi[0]) & (int)(bx.w >= lo[0]) & (int)(bx.y <= hi[1]) & (int)(by.x >= lo[1]) &
                   (int)(bx.z <= hi[2]) & (int)(by.y >= lo[2])) != 0 &&
                  (!Kg.sorted || ft_box_meets(rec, mid[0], mid[1], mid[2], ext[0], ext[1], ext[2], rho));
        }
        const unsigned long long mk = __ballot(hit);
        if (lane == 0) cnt[wave] = __popcll(mk);
        __syncthreads();
        int off = total;
#pragma unroll
        for (int w = 0; w < FB_THREADS / 64; w++) {
            if (w < wave) off += cnt[w];
            total += cnt[w];
        }
        if (hit) mine[off + __popcll(mk & ((1ull << lane) - 1ull))] = (unsigned short)j;
        __syncthreads();
    }
    if (threadIdx.x == 0) counts[cell] = total;
    if (total == 0) return;
    int cls = 0;
    while (cls < FZ_CLASSES - 1 && total < (1024 >> cls)) cls++;
    const size_t all = (size_t)F.nb[0] * F.nb[1] * F.nb[2];
    int4 *const mylist = list + cls * all;
    const int np = F.q[0] * F.q[1] * F.q[2];
    for (int base = 0; base < np; base += FB_THREADS) {
        const int i = base + (int)threadIdx.x;
        const int p0 = pa[0] + i / (F.q[1] * F.q[2]), p1 = pa[1] + (i / F.q[2]) % F.q[1], p2 = pa[2] + i % F.q[2];
        bool take = i < np && p0 < pb[0] && p1 < pb[1] && p2 < pb[2];
        const int a0 = p0 * FZ_K0, a1 = p1 * FZ_PATCH, a2 = p2 * FZ_PATCH;
        if (take && s0 >= 0 && Kg.k0[min(a0 + FZ_K0 - 1, Kg.m0 - 1)] < 0.0f && a0 >= s0 && a1 >= s1 && a2 >= s2)
            take = false;
        const unsigned long long mk = __ballot(take);
        unsigned at = 0;
        if (lane == 0 && mk) at = atomicAdd(&state->count[cls], (unsigned)__popcll(mk));
        at = (unsigned)__builtin_amdgcn_readfirstlane((int)at);
        if (take) mylist[at + __popcll(mk & ((1ull << lane) - 1ull))] = make_int4(a0, a1, a2, (int)cell);
    }
}

// A staged record: the form's coefficients and the table entries of the patch's k0's.
struct alignas(16) FzTerm {
    float u[6], pad[2];
    float2 a[FZ_K0];
};

// Blocks of FZ_WAVES waves take patches from the list until it is empty; lane l
// holds offset (l / 8, l % 8) at FZ_K0 k0's.  The waves take every FZ_WAVES-th
// record of the patch's records (a thread per record: index box, then
// ft_box_meets), their FP64 sums added in wave order.  A sample's phase is the
// product of three table entries: per record one complex product for the lane's
// (k1, k2) and one per k0; the values are added in FP64.
// Bound by VALU issue on the central patches and by the latency of a patch's
// staging elsewhere: large blocks keep the first short, the cells' lists and a
// patch counter the second.  2000 atoms on 128^3: 0.227 ms (patches of 64
// samples, every block scanning the atoms in radius order) -> 0.072 with four
// values at a time summed in FP32, 0.076 now; with four, (waves, k0's) = (8, 2)
// 0.083, (8, 4) 0.098, (16, 4) 0.086, (16, 1) 0.114; patches in no order 0.105 to
// 0.13.
__global__ __launch_bounds__(FZ_THREADS) void ft_grid_kernel(const FtRec *__restrict__ recs,
                                                             const float2 *__restrict__ tab, int N, gt_kgrid Kg,
                                                             FzState *__restrict__ state,
                                                             const unsigned short *__restrict__ cellids,
                                                             const int *__restrict__ counts,
                                                             const int4 *__restrict__ patches, size_t all,
                                                             float2 *__restrict__ out)
{
    __shared__ FzTerm list[FZ_THREADS];  // also the reduction buffer at the end
    __shared__ unsigned short ids[FZ_THREADS];
    __shared__ int cnt[FZ_WAVES];
    __shared__ unsigned mine;
    static_assert(sizeof(list) >= sizeof(double2) * FZ_WAVES * FZ_K0 * 64, "reduction buffer");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned upto[FZ_CLASSES];  // listed patches of the classes up to c
    upto[0] = state->count[0];
#pragma unroll
    for (int c = 1; c < FZ_CLASSES; c++) upto[c] = upto[c - 1] + state->count[c];
    const unsigned count = upto[FZ_CLASSES - 1];
    const int s0 = state->pairing[0], s1 = state->pairing[1], s2 = state->pairing[2];
    // the first patch is the block's own number, the next ones from the counter
    for (unsigned at = blockIdx.x; at < count;) {
        unsigned nextat = 0;
        if (threadIdx.x == 0) nextat = gridDim.x + atomicAdd(&state->next, 1u);
        const int4 *slot = patches + at;
#pragma unroll
        for (int c = 1; c < FZ_CLASSES; c++)
            if (at >= upto[c - 1]) slot = patches + (c * all + (at - upto[c - 1]));
        const int4 pt = *slot;
        const int a0 = pt.x, a1 = pt.y, a2 = pt.z, nc = counts[pt.w];
        const unsigned short *cids = cellids + (size_t)pt.w * N;
        const int z0 = min(a0 + FZ_K0 - 1, Kg.m0 - 1);
        const int z1 = min(a1 + FZ_PATCH - 1, Kg.m1 - 1), z2 = min(a2 + FZ_PATCH - 1, Kg.m2 - 1);
        const int i1 = min(a1 + (lane >> 3), Kg.m1 - 1), i2 = min(a2 + (lane & 7), Kg.m2 - 1);
        float k0[FZ_K0];
#pragma unroll
        for (int z = 0; z < FZ_K0; z++) k0[z] = Kg.k0[min(a0 + z, Kg.m0 - 1)];
        const float k1 = Kg.k1[i1], k2 = Kg.k2[i2];
        const float c1a = Kg.k1[a1], c1b = Kg.k1[z1], c2a = Kg.k2[a2], c2b = Kg.k2[z2];
        const bool exact = Kg.sorted != 0;
        const float cut = (float)(FT_CUT * HALF_LOG2E_SQRT * HALF_LOG2E_SQRT);
        // centre and half extents of the patch
        const float m0 = 0.5f * (k0[0] + k0[FZ_K0 - 1]), x0 = 0.5f * (k0[FZ_K0 - 1] - k0[0]);
        const float m1 = 0.5f * (c1a + c1b), x1 = 0.5f * (c1b - c1a), m2 = 0.5f * (c2a + c2b), x2 = 0.5f * (c2b - c2a);
        const int m = Kg.m0 + Kg.m1 + Kg.m2;
        const float2 *tab1 = tab + Kg.m0 + i1, *tab2 = tab + Kg.m0 + Kg.m1 + i2;
        double sr[FZ_K0], si[FZ_K0];
#pragma unroll
        for (int z = 0; z < FZ_K0; z++) sr[z] = si[z] = 0.0;
        for (int base = 0; base < nc; base += FZ_THREADS) {
            bool hit = false;
            int j = 0;
            FtL rec;
            if (base + (int)threadIdx.x < nc) {
                j = cids[base + threadIdx.x];
                rec = *reinterpret_cast<const FtL *>(recs + j);
                const int4 bx = reinterpret_cast<const int4 *>(recs + j)[4];   // lo[3], hi[0]
                const int2 by = reinterpret_cast<const int2 *>(recs + j)[10];  // hi[1], hi[2]
                if ((int)(bx.x <= z0) & (int)(bx.w >= a0) & (int)(bx.y <= z1) & (int)(by.x >= a1) & (int)(bx.z <= z2) &
                    (int)(by.y >= a2))
                    hit = !exact || ft_box_meets(rec, m0, m1, m2, x0, x1, x2, sqrtf(cut));
            }
            const unsigned long long mk = __ballot(hit);
            if (lane == 0) cnt[wave] = __popcll(mk);
            __syncthreads();
            int off = 0, len = 0;
#pragma unroll
            for (int w = 0; w < FZ_WAVES; w++) {
                const int c = cnt[w];
                if (w < wave) off += c;
                len += c;
            }
            len = __builtin_amdgcn_readfirstlane(len);
            if (hit) {
                const int pos = off + __popcll(mk & ((1ull << lane) - 1ull));
                const float2 *ta = tab + (size_t)j * m + a0;
                FzTerm f;
#pragma unroll
                for (int i = 0; i < 6; i++) f.u[i] = rec.u[i];
                f.pad[0] = f.pad[1] = 0.0f;
#pragma unroll
                for (int z = 0; z < FZ_K0; z++) f.a[z] = ta[min(z, z0 - a0)];
                list[pos] = f;
                ids[pos] = (unsigned short)j;
            }
            __syncthreads();
            // the lane's table entries of the next record are loaded while one is summed
            auto entries = [&](int q, float2 &b, float2 &c) {
                const size_t o = (size_t)__builtin_amdgcn_readfirstlane((int)ids[min(q, len - 1)]) * m;
                b = tab1[o];
                c = tab2[o];
            };
            auto sum = [&](int q, const float2 &b, const float2 &c) {
                const FzTerm f = list[q];
                const float pr = fmaf(b.x, c.x, -b.y * c.y), pi = fmaf(b.x, c.y, b.y * c.x);
                const float v1 = f.u[1] * k1, v2 = fmaf(f.u[4], k1, f.u[2] * k2);
#pragma unroll
                for (int z = 0; z < FZ_K0; z++) {
                    const float w0 = f.u[0] * k0[z], w1 = fmaf(f.u[3], k0[z], v1), w2 = fmaf(f.u[5], k0[z], v2);
                    const float nq = fmaf(w0, w0, fmaf(w1, w1, w2 * w2));
                    if (!(nq < cut)) continue;  // (0 times an infinite amplitude is no 0)
                    const float E = __builtin_amdgcn_exp2f(-nq);
                    sr[z] += (double)(E * fmaf(f.a[z].x, pr, -f.a[z].y * pi));
                    si[z] += (double)(E * fmaf(f.a[z].x, pi, f.a[z].y * pr));
                }
            };
            if (wave < len) {
                float2 b, c, bn, cn;
                entries(wave, b, c);
                for (int q = wave;;) {
                    entries(q + FZ_WAVES, bn, cn);
                    sum(q, b, c);
                    if ((q += FZ_WAVES) >= len) break;
                    entries(q + FZ_WAVES, b, c);
                    sum(q, bn, cn);
                    if ((q += FZ_WAVES) >= len) break;
                }
            }
            __syncthreads();
        }
        double2 (*red)[FZ_K0][64] = reinterpret_cast<double2 (*)[FZ_K0][64]>(list);
#pragma unroll
        for (int z = 0; z < FZ_K0; z++) red[wave][z][lane] = make_double2(sr[z], si[z]);
        __syncthreads();
        // wave z adds the waves' sums for k0 z, in wave order, and writes them
        static_assert(FZ_WAVES >= FZ_K0, "a wave per k0");
        const int i0 = a0 + wave;
        if (wave < FZ_K0 && i0 < Kg.m0 && a1 + (lane >> 3) < Kg.m1 && a2 + (lane & 7) < Kg.m2) {
            double tr = 0.0, ti = 0.0;
            for (int w = 0; w < FZ_WAVES; w++) {
                const double2 v = red[w][wave][lane];
                tr += v.x;
                ti += v.y;
            }
            const float2 v = make_float2((float)tr, (float)ti);
            const float kz = Kg.k0[i0];
            const bool partner = s0 >= 0 && i0 >= s0 && i1 >= s1 && i2 >= s2;
            if (!partner || kz >= 0.0f) out[((size_t)i0 * Kg.m1 + i1) * Kg.m2 + i2] = v;
            if (partner && kz > 0.0f) {
                const int n0 = s0 ? Kg.m0 - i0 : Kg.m0 - 1 - i0, n1 = s1 ? Kg.m1 - i1 : Kg.m1 - 1 - i1;
                const int n2 = s2 ? Kg.m2 - i2 : Kg.m2 - 1 - i2;
                out[((size_t)n0 * Kg.m1 + n1) * Kg.m2 + n2] = make_float2(v.x, -v.y);
            }
        }
        if (threadIdx.x == 0) mine = nextat;
        __syncthreads();  // `mine` is written, the buffers are read
        at = mine;
        __syncthreads();
    }
}

// One wave per atom j: its rank = the atoms of larger radius, or of equal
// radius and smaller index; the record is copied to that position.
__global__ __launch_bounds__(256) void ft_rank_kernel(const FtRec *__restrict__ recs, int N, FtRec *__restrict__ sorted)
{
    const int lane = threadIdx.x & 63;
    const int j = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (j >= N) return;
    const float rj = recs[j].pad0[0];
    int rank = 0;
    for (int i = lane; i < N; i += 64) {
        const float ri = recs[i].pad0[0];
        rank += (ri > rj || (ri == rj && i < j)) ? 1 : 0;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) rank += __shfl_xor(rank, o);
    // eight lanes copy the 128-byte record, 16 bytes each
    if (lane < 8)
        reinterpret_cast<int4 *>(sorted + rank)[lane] = reinterpret_cast<const int4 *>(recs + j)[lane];
}

// Without tables (ft_tabulated, or no room for them): the records of at most
// FZ_MAX_ATOMS atoms are put in order of decreasing radius of a ball about k = 0
// holding the support, so that a patch at distance d from the origin only looks at
// the leading records of radius >= d; more are taken in atom order.  One block of 4
// waves per 8 x 8 (k1, k2) patch at one k0; lane l holds the sample at offset (l / 8, l % 8).  Staging (a thread per
// record, records of radius >= the patch's distance from the origin only):
// the record's index box against the patch and, for an ascending grid, the
// least |U^T k|^2 over the patch against the cutoff (ft_patch_min, with a
// relative slack of 1e-4 so that no sample the FP32 test takes is lost);
// records that meet the patch go to LDS in record order.  Wave w evaluates
// the staged records w, w + 4, ... (branch-free: a sample outside the support
// adds an exact zero) summing in FP64, and the 4 partial sums are added in
// wave order: every sample's sum has an order fixed by the record order.
constexpr int FP_THREADS = 256, FP_WAVES = 4, FP_CHUNK = 256, FP_PATCH = 8;

// FINE: the phase in FP64 (of ranked, so at most FZ_MAX_ATOMS records), as
// accurate as the tables; the others' is a sum of FP32 pairs through the hardware
// sine and cosine.
template <bool FINE>
__global__ __launch_bounds__(FP_THREADS) void ft_patch_kernel(const FtRec *__restrict__ recs, int N, gt_kgrid Kg,
                                                              float2 *__restrict__ out, int e0, int e1, int e2,
                                                              int by_radius)
{
    __shared__ FtL list[FP_CHUNK];  // also the reduction buffer at the end
    __shared__ int wcnt[FP_WAVES];
    static_assert(sizeof(list) >= (size_t)FP_WAVES * 64 * sizeof(double2), "reduction buffer");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nb1 = (Kg.m1 + FP_PATCH - 1) / FP_PATCH, nb2 = (Kg.m2 + FP_PATCH - 1) / FP_PATCH;
    const int e[3] = {e0, e1, e2};
    int t[3];
    morton_ranks(blockIdx.x, e, t);
    if (t[0] >= Kg.m0 || t[1] >= nb1 || t[2] >= nb2) return;  // whole block: no patch of this rank
    const int i0 = centre_out(t[0], Kg.m0);
    const int a1 = centre_out(t[1], nb1) * FP_PATCH, a2 = centre_out(t[2], nb2) * FP_PATCH;
    const int z1 = min(a1 + FP_PATCH - 1, Kg.m1 - 1), z2 = min(a2 + FP_PATCH - 1, Kg.m2 - 1);
    const int i1 = a1 + (lane >> 3), i2 = a2 + (lane & 7);
    const float k0 = Kg.k0[i0], k1 = Kg.k1[min(i1, Kg.m1 - 1)], k2 = Kg.k2[min(i2, Kg.m2 - 1)];
    const float c1a = Kg.k1[a1], c1b = Kg.k1[z1], c2a = Kg.k2[a2], c2b = Kg.k2[z2];
    const bool exact = Kg.sorted != 0;
    // distance from k = 0 to the patch (its samples lie in the coordinate box)
    const float g1 = (c1a <= 0.0f && c1b >= 0.0f) ? 0.0f : fminf(fabsf(c1a), fabsf(c1b));
    const float g2 = (c2a <= 0.0f && c2b >= 0.0f) ? 0.0f : fminf(fabsf(c2a), fabsf(c2b));
    const float dmin = exact ? sqrtf(fmaf(k0, k0, fmaf(g1, g1, g2 * g2))) : 0.0f;
    const float cut = (float)(FT_CUT * HALF_LOG2E_SQRT * HALF_LOG2E_SQRT);
    const float cut_keep = cut * (1.0f + 1e-4f);
    double sr = 0.0, si = 0.0;
    for (int base = 0; base < N; base += FP_CHUNK) {
        // records in radius order: this and every later one fall short of the patch
        if (by_radius && recs[base].pad0[0] < dmin) break;
        const int j = base + (int)threadIdx.x;
        bool hit = false;
        if (j < N) {
            const FtL &rec = *reinterpret_cast<const FtL *>(recs + j);
            const int *bx = reinterpret_cast<const int *>(recs + j) + 16;  // lo[3], hi[3]
            hit = rec.pad[0] >= dmin && bx[0] <= i0 && bx[3] >= i0 && bx[1] <= z1 && bx[4] >= a1 && bx[2] <= z2 &&
                  bx[5] >= a2 && (!exact || ft_patch_min(rec, k0, c1a, c1b, c2a, c2b) < cut_keep);
        }
        const unsigned long long m = __ballot(hit);
        if (lane == 0) wcnt[wave] = __popcll(m);
        __syncthreads();
        int off = 0, total = 0;
#pragma unroll
        for (int w = 0; w < FP_WAVES; w++) {
            if (w < wave) off += wcnt[w];
            total += wcnt[w];
        }
        if (hit) {
            FtL rec = *reinterpret_cast<const FtL *>(recs + j);
            if (FINE) {  // the position as doubles, in the place of its float pairs
                const double x[3] = {(double)rec.xh[0] + (double)rec.xl[0], (double)rec.xh[1] + (double)rec.xl[1],
                                     (double)rec.xh[2] + (double)rec.xl[2]};
                __builtin_memcpy(&rec.xh[0], x, sizeof x);
            }
            list[off + __popcll(m & ((1ull << lane) - 1ull))] = rec;
        }
        __syncthreads();
        for (int q = wave; q < total; q += FP_WAVES) {
            const FtL &r = list[q];
            float nq;
            if (r.iso != 0.0f) {
                nq = fmaf(k1, k1, fmaf(k0, k0, k2 * k2)) * (r.u[0] * r.u[0]);
            } else {
                const float v0 = r.u[0] * k0;
                const float v1 = fmaf(r.u[1], k1, r.u[3] * k0);
                const float v2 = fmaf(r.u[4], k1, fmaf(r.u[5], k0, r.u[2] * k2));
                nq = fmaf(v0, v0, fmaf(v1, v1, v2 * v2));
            }
            float sn, cs;
            if (FINE) {
                double x[3];
                __builtin_memcpy(x, &r.xh[0], sizeof x);
                const double t = fma(x[0], (double)k0, fma(x[1], (double)k1, x[2] * (double)k2));
                ft_sincos_fine(t, sn, cs);
            } else {
                float err = 0.0f;
                const float t01 = turns(r.xh[0], r.xl[0], k0, err) + turns(r.xh[1], r.xl[1], k1, err);
                const float tt = (t01 + turns(r.xh[2], r.xl[2], k2, err)) + err;
                ft_sincos_turns(tt, sn, cs);
            }
            const float a = nq < cut ? r.amp * __builtin_amdgcn_exp2f(-nq) : 0.0f;
            sr += (double)(a * cs);
            si += (double)(-a * sn);
        }
        __syncthreads();
    }
    double2 *red = reinterpret_cast<double2 *>(list);  // [wave][lane]
    red[wave * 64 + lane] = make_double2(sr, si);
    __syncthreads();
    if (wave == 0 && i1 < Kg.m1 && i2 < Kg.m2) {
        double tr = 0.0, ti = 0.0;
        for (int w = 0; w < FP_WAVES; w++) {
            const double2 v = red[w * 64 + lane];
            tr += v.x;
            ti += v.y;
        }
        out[((size_t)i0 * Kg.m1 + i1) * Kg.m2 + i2] = make_float2((float)tr, (float)ti);
    }
}

__global__ void cfill_kernel(float2 *p, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = make_float2(0.0f, 0.0f);
}

}  // namespace gt

using namespace gt;

// Workspace: the records; with tables also the state, the cells' record lists,
// the patch lists and the phase tables.
static FzCells ft_cells(const gt_kgrid *g)
{
    FzCells F;
    const int m[3] = {g->m0, g->m1, g->m2}, size[3] = {FZ_K0, FZ_PATCH, FZ_PATCH}, most[3] = {16, 8, 8};
    int bits = 0;
    for (int c = 0; c < 3; c++) {
        F.nb[c] = (m[c] + size[c] - 1) / size[c];
        F.q[c] = (F.nb[c] + most[c] - 1) / most[c];
        F.nc[c] = (F.nb[c] + F.q[c] - 1) / F.q[c];
        F.e[c] = ceil_log2(F.nc[c]);
        bits += F.e[c];
    }
    F.cells = 1u << bits;
    return F;
}
struct FtLayout {
    size_t state, ids, counts, list, tab, total;
};
static FtLayout ft_layout(const gt_atoms *a, const gt_kgrid *g, const FzCells &F)
{
    FtLayout l;
    const size_t n = (size_t)a->n, m = (size_t)g->m0 + g->m1 + g->m2;
    l.state = align_up(n * sizeof(FtRec));
    l.ids = l.state + align_up(sizeof(FzState));
    l.counts = l.ids + align_up(F.cells * n * sizeof(unsigned short));
    l.list = l.counts + align_up(F.cells * sizeof(int));
    l.tab = l.list + align_up((size_t)FZ_CLASSES * F.nb[0] * F.nb[1] * F.nb[2] * sizeof(int4));
    l.total = l.tab + align_up(n * m * sizeof(float2));
    return l;
}

// Without tables: the records and, where they are ranked, their copy in radius order.
static size_t ft_least(const gt_atoms *a)
{
    const size_t one = align_up((size_t)a->n * sizeof(FtRec));
    return a->n <= FZ_MAX_ATOMS ? 2 * one : one;
}

// Are the atoms evaluated with tables?  These grow with atoms x (m0 + m1 + m2)
// and with the number of patches, so a long thin grid of many atoms would take
// hundreds of times its output (16384 atoms on 2^20 x 1 x 1 samples: 137 GB of
// tables for 8 MB).  And few atoms on a small grid are evaluated sooner without: the
// patch kernel costs 2.1 ns per block of 1 x 8 x 8 samples and hardly anything per
// atom until some 128 fill a chunk of records, the tables' kernels 10 us for their
// cells and patches.  Call times with and without tables, us: 64^3 samples, 16 atoms
// 28 and 20, 64 33 and 23, 256 44 and 45; 48^3, 64 atoms 31 and 20, 256 36 and 44;
// 16^3, 128 atoms 18 and 20; 8 x 8 x 4096 (long tables), 64 atoms 27 and 20, 256 34
// and 30, 512 42 and 51; beyond 4096 blocks: 80^3, 16 atoms 30 and 67, 256 x 256 x
// 4, 16 atoms 24 and 30.
static int ft_bits(const gt_kgrid *g, int *e)
{
    e[0] = ceil_log2(g->m0);
    e[1] = ceil_log2((g->m1 + FP_PATCH - 1) / FP_PATCH);
    e[2] = ceil_log2((g->m2 + FP_PATCH - 1) / FP_PATCH);
    return e[0] + e[1] + e[2];
}
static bool ft_tabulated(const gt_atoms *a, const gt_kgrid *g)
{
    if (a->n > FZ_MAX_ATOMS) return false;
    int e[3];
    const int bits = ft_bits(g, e);
    if (bits <= 12 && a->n <= 128 + (1 << bits) / 64 + (g->m0 + g->m1 + g->m2) / 32) return false;
    const size_t out = (size_t)g->m0 * g->m1 * g->m2 * sizeof(float2);
    return ft_layout(a, g, ft_cells(g)).total <= std::max(FZ_MAX_BYTES, out);
}

extern "C" size_t gt_ft_workspace(const gt_atoms *atoms, const gt_kgrid *grid)
{
    if (!atoms || atoms->n <= 0) return 0;
    const bool ok = grid && grid->m0 >= 1 && grid->m1 >= 1 && grid->m2 >= 1;
    if (!ok || !ft_tabulated(atoms, grid)) return ft_least(atoms);
    return ft_layout(atoms, grid, ft_cells(grid)).total;
}

extern "C" int gt_ft_eval(const gt_atoms *atoms, const gt_kgrid *grid, float *out, void *ws, size_t ws_bytes,
                          void *stream)
{
    int rc;
    if ((rc = check_atoms(atoms))) return rc;
    GT_CHECK_ARG(atoms->dim == 3, "gt_ft_eval: only 3D atoms are supported, got dim %d", atoms->dim);
    GT_CHECK_ARG(grid != nullptr && grid->dim == 3, "gt_ft_eval: grid must be a 3D separable grid");
    GT_CHECK_ARG(grid->m0 >= 1 && grid->m1 >= 1 && grid->m2 >= 1, "gt_ft_eval: grid sizes must be >= 1");
    GT_CHECK_ARG(grid->m0 < (1 << 24) && grid->m1 < (1 << 24) && grid->m2 < (1 << 24), "gt_ft_eval: grid too large");
    GT_CHECK_ARG(grid->k0 && grid->k1 && grid->k2, "gt_ft_eval: grid vectors must be non-NULL");
    GT_CHECK_ARG(out != nullptr, "gt_ft_eval: out is NULL");
    // (a workspace that holds no tables is enough for the kernel without them)
    const size_t tables = atoms->n > 0 && ft_tabulated(atoms, grid) ? gt_ft_workspace(atoms, grid) : 0;
    const bool tabulated = tables > 0 && tables <= ws_bytes;
    const size_t need = atoms->n <= 0 ? 0 : (tables > 0 ? std::min(tables, ft_least(atoms)) : ft_least(atoms));
    if (need > ws_bytes || (need > 0 && ws == nullptr)) {
        set_error("gt_ft_eval: workspace of %zu bytes given, %zu needed", ws_bytes, need);
        return GT_EWORKSPACE;
    }
    GT_CHECK_ARG(((uintptr_t)ws & 127) == 0, "gt_ft_eval: workspace must be 128-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    const size_t nout = (size_t)grid->m0 * grid->m1 * grid->m2;
    if (atoms->n == 0) {
        hipLaunchKernelGGL(cfill_kernel, dim3((unsigned)std::min<size_t>((nout + 255) / 256, 65535)), dim3(256), 0,
                           st, (float2 *)out, nout);
        GT_HIP(hipGetLastError());
        return 0;
    }
    FtRec *recs = (FtRec *)ws;
    const unsigned sb = (unsigned)((atoms->n + 255) / 256);
    // patches of 1 x 8 x 8 samples, numbered by Morton index over 2^e0 x 2^e1 x 2^e2 centre-out ranks
    int e[3];
    GT_CHECK_ARG(ft_bits(grid, e) <= 30, "gt_ft_eval: grid too large");
    if (tabulated) {
        const FzCells F = ft_cells(grid);
        const FtLayout l = ft_layout(atoms, grid, F);
        char *w = (char *)ws;
        FzState *state = (FzState *)(w + l.state);
        unsigned short *ids = (unsigned short *)(w + l.ids);
        int *counts = (int *)(w + l.counts);
        int4 *list = (int4 *)(w + l.list);
        float2 *tab = (float2 *)(w + l.tab);
        const size_t patches = (size_t)F.nb[0] * F.nb[1] * F.nb[2];
        const size_t axes = (size_t)grid->m0 + grid->m1 + grid->m2;
        const unsigned tabs = (unsigned)((atoms->n * ((axes + FZ_TAB - 1) / FZ_TAB) + 3) / 4);
        hipLaunchKernelGGL(ft_atoms_kernel, dim3(tabs + sb), dim3(256), 0, st, *atoms, *grid, tabs, recs, state, tab);
        prof_begin(st, GT_K_FT);
        hipLaunchKernelGGL(ft_bin_kernel, dim3(std::max(F.cells, 1024u)), dim3(FB_THREADS), 0, st, recs, atoms->n, *grid, F,
                           state, ids, counts, list, (float2 *)out, nout);
        hipLaunchKernelGGL(ft_grid_kernel, dim3((unsigned)std::min<size_t>(patches, FZ_BLOCKS)), dim3(FZ_THREADS), 0,
                           st, recs, tab, atoms->n, *grid, state, ids, counts, list, patches, (float2 *)out);
        prof_end(st, GT_K_FT);
        GT_HIP(hipGetLastError());
        return 0;
    }
    hipLaunchKernelGGL(ft_setup_kernel, dim3(sb), dim3(256), 0, st, *atoms, *grid, recs);
    const FtRec *order = recs;
    if (atoms->n <= FZ_MAX_ATOMS) {
        FtRec *sorted = (FtRec *)((char *)ws + align_up((size_t)atoms->n * sizeof(FtRec)));
        hipLaunchKernelGGL(ft_rank_kernel, dim3((unsigned)((atoms->n + 3) / 4)), dim3(256), 0, st, recs, atoms->n,
                           sorted);
        order = sorted;
    }
    const unsigned blocks = 1u << (e[0] + e[1] + e[2]);
    prof_begin(st, GT_K_FT);
    if (order != recs)
        hipLaunchKernelGGL(ft_patch_kernel<true>, dim3(blocks), dim3(FP_THREADS), 0, st, order, atoms->n, *grid,
                           (float2 *)out, e[0], e[1], e[2], 1);
    else
        hipLaunchKernelGGL(ft_patch_kernel<false>, dim3(blocks), dim3(FP_THREADS), 0, st, order, atoms->n, *grid,
                           (float2 *)out, e[0], e[1], e[2], 0);
    prof_end(st, GT_K_FT);
    GT_HIP(hipGetLastError());
    return 0;
}
