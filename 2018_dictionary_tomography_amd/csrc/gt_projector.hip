// gt_projector.hip -- forward projection and per-atom derivatives on CDNA4.
//
// Pipeline (all stream-ordered, no host synchronisation):
//   setup    one thread per (atom, angle): FP64 detector Gaussian -> PairRec
//   forward  one block per (angle, 8x64 pixel tile), centre tiles first:
//            stages the angle's records that touch the tile in LDS; each of
//            4 waves owns an 8x16 rectangle (2 pixels per lane) and walks
//            the records whose support meets it; FP64 pixel sums of FP32
//            values taken four records at a time
//   moments  one wave, and one block, per (atom, angle): FP32 separable
//            pixel moments over the rows of each column chunk that the
//            support can reach, LDS-transposed wave reduction, no atomics
//   finish   one wave per atom, one lane per angle: FP64 moment -> (f, g, H)
//            contraction (gt_pair.h), FP64 wave reduction over angles
//
// Reference counterparts: __RadProj_3D/_2p5D (NewtonBases.py:729-756),
// __RadProj (NewtonBases2D.py:284-296), __L2derivs_RadProj_aniso_3D and
// __derivs_RadProj_aniso_3D (NewtonBases.py:792-870, 993-1069) and their 2D
// versions (NewtonBases2D.py:329-401, 444-515).
#include <algorithm>

#include "gt_pixel.h"

namespace gt {

constexpr int TILE_ROWS = 8, TILE_COLS = 64;
constexpr int CHUNK = 256;
constexpr int MOM_STRIDE = 32;  // floats per (atom, angle) moment record
constexpr int MOM_TROWS = 512;  // rows of a moments wave's row table
constexpr int MOM_WAVES = 1;    // waves (pairs) per moments block
constexpr int MODE_LINEAR = GT_MODE_LINEAR, MODE_L2 = GT_MODE_L2, MODE_RESID = GT_MODE_RESID;

__device__ inline void kahan_add(float &s, float &c, float v)
{
    const float y = v - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

// ---------------------------------------------------------------------------
// setup
// ---------------------------------------------------------------------------
template <int D> __global__ __launch_bounds__(256) void setup_kernel(gt_atoms A, gt_geom G, PairRec *recs)
{
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long total = (long)A.n * G.nA;
    if (idx >= total) return;
    const int a = (int)(idx / A.n), j = (int)(idx - (long)a * A.n);
    PairGeom<D> g;
    load_atom<D>(A, j, g);
    load_angle<D>(G, a, g);
    const float *det[2] = {G.p0, G.p1};
    const int nd[2] = {G.n0, G.n1};
    PairRec rec;
    pair_setup<D>(g, det, nd, G.sorted, rec);
    recs[idx] = rec;
}

// Deterministic block-wide compaction of the records that touch a box
// [r_lo, r_hi] x [c_lo, c_hi]; returns the list length.  The list keeps atom
// order, so the per-pixel summation order does not depend on timing.
template <int NW>
__device__ inline int stage_chunk(const PairRec *__restrict__ ra, int base, int N, int r_lo, int r_hi, int c_lo,
                                  int c_hi, PairRec *list, int *wcnt)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = base + (int)threadIdx.x;
    bool hit = false;
    int4 v0 = make_int4(0, 0, 0, 0), v1 = v0, v2 = v0, v3 = v0;
    if (j < N) {
        const int4 *src = reinterpret_cast<const int4 *>(ra + j);
        v0 = src[0];
        v1 = src[1];
        v2 = src[2];
        v3 = src[3];
        // v3 = (lo[0], lo[1], hi[0], hi[1])
        hit = v3.x <= r_hi && v3.z >= r_lo && v3.y <= c_hi && v3.w >= c_lo;
    }
    const unsigned long long m = __ballot(hit);
    if (lane == 0) wcnt[wave] = __popcll(m);
    __syncthreads();
    int off = 0, total = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        if (w < wave) off += wcnt[w];
        total += wcnt[w];
    }
    if (hit) {
        int4 *dst = reinterpret_cast<int4 *>(list + off + __popcll(m & ((1ull << lane) - 1ull)));
        dst[0] = v0;
        dst[1] = v1;
        dst[2] = v2;
        dst[3] = v3;
    }
    __syncthreads();
    return total;
}

// ---------------------------------------------------------------------------
// forward, 2D detectors (3D and 2.5D geometries)
// ---------------------------------------------------------------------------
// Block tile TILE_ROWS x TILE_COLS = 8 x 64 pixels, F3_WAVES = 4 waves; wave
// w owns the 8 x 16 rectangle rows 8 (w / 4) .. +7, columns 16 (w % 4) ..
// +15, and lane l column l % 16 of it, rows l / 16 and l / 16 + 4 (2 pixels
// per lane).  Staging keeps the records that reach a rectangle in LDS and, for
// every wave, the list of those that reach its own (in atom order, so each
// pixel's summation order is fixed).  (8 x 64 tiles of 4 waves measured 138 us
// against 155 us for 16 x 64 tiles of 8 waves: twice the blocks, so the
// centre-first dispatch balances finer.)
//
// Vector issue and LDS bandwidth bound it together (80% of the LDS cycles and
// one vector instruction per cycle and CU).  A wave takes four records at a
// time: lane (u, k) works out what record u's exponent takes from column k and
// row k % 8 of the rectangle, once for the 8 rows and 16 columns that share it,
// and the pixels read the two from LDS: 15 vector instructions and 12 LDS
// cycles per record and wave against 23 and 17 with each lane working on the
// records (three 16-byte broadcast reads each) by itself.  The record itself
// comes as one word per lane and is passed around its row of 16 lanes.  5000
// atoms, 90 x 256^2: 2.02 -> 1.76 ms; 1000, 61 x 128^2: 98.8 -> 88.8 us; 300,
// 45 x 96 x 83: 26.0 -> 22.4 us.  (Records through scalar loads: 102 us of the
// second, their waits are shared with LDS.)
constexpr int F3_WAVES = 4, F3_CHUNK = F3_WAVES * 64;
static_assert(TILE_ROWS == 8 * ((F3_WAVES + 3) / 4) && TILE_COLS == 16 * (F3_WAVES < 4 ? F3_WAVES : 4),
              "the tile is the union of the waves' 8 x 16 rectangles");
// first and last detector coordinate of each row group / column group of the
// waves' rectangles (held in registers: indexed only by unrolled constants)
constexpr int F3_RX = 2 * ((F3_WAVES + 3) / 4), F3_CY = 2 * (F3_WAVES < 4 ? F3_WAVES : 4);

// The tiles at the detector centre carry several times the records of those
// at its edges, and the grid holds more blocks than fit on the device at once:
// blocks are numbered centre tiles first (centre_out / morton_ranks), all
// angles of one tile together (block b: angle b % nA, tile rank b / nA), so
// the heavy tiles start first and the light ones fill the tail.

__device__ inline void stage_rects(const PairRec *__restrict__ ra, int base, int N, int row0, int col0, PairRec *list,
                                   unsigned short (*wl)[F3_CHUNK], int (*cnt)[F3_WAVES], int *wlen, bool exact,
                                   const float (&rx)[F3_RX], const float (&cy)[F3_CY])
{
    const int j = base + (int)threadIdx.x;
    unsigned mask = 0;
    if (j < N) {
        const int4 *src = reinterpret_cast<const int4 *>(ra + j);
        const int4 v0 = src[0], v1 = src[1], v2 = src[2], v3 = src[3];
        // v3 = (lo[0], lo[1], hi[0], hi[1])
        // f0 = (alpha, c_hi0, c_hi1, c_lo0), f1 = (c_lo1, q0, q1, q2), f2 = (q3, q4, q5, pad)
        const float4 f0 = *reinterpret_cast<const float4 *>(&v0), f1 = *reinterpret_cast<const float4 *>(&v1);
        const float4 f2 = *reinterpret_cast<const float4 *>(&v2);
#pragma unroll
        for (int w = 0; w < F3_WAVES; w++) {
            const int r = row0 + 8 * (w >> 2), c = col0 + 16 * (w & 3);
            if (v3.x <= r + 7 && v3.z >= r && v3.y <= c + 15 && v3.w >= c &&
                (!exact || support_meets_rect(f1, f2, (rx[2 * (w >> 2)] - f0.y) - f0.w,
                                           (rx[2 * (w >> 2) + 1] - f0.y) - f0.w, (cy[2 * (w & 3)] - f0.z) - f1.x,
                                           (cy[2 * (w & 3) + 1] - f0.z) - f1.x)))
                mask |= 1u << w;
        }
        if (mask) {
            float4 *dst = reinterpret_cast<float4 *>(list + threadIdx.x);
            dst[0] = f0;
            dst[1] = f1;
            dst[2] = f2;
        }
    }
    wave_lists<F3_WAVES, F3_WAVES>(mask, wl, cnt, wlen);
}

// A group of four records as the pixels read it: per column (the terms linear
// and constant in the row, q0, alpha), per row the offset from the centre.  No
// cut-off test: every record in a wave's list reaches its rectangle, and the
// values at pixels of the rectangle outside the support are below e^-30 of the
// record's peak.
struct F3Tab {
    float4 c[4][16];
    float r[4][8];  // rows 0, 4, 1, 5, ...: a lane's two side by side
};

// (at most 64 VGPRs: eight waves per SIMD)
__global__ __launch_bounds__(F3_WAVES * 64) __attribute__((amdgpu_waves_per_eu(8))) void forward3_kernel(
    const PairRec *__restrict__ recs, int N, int nA, int n0, int n1, const float *__restrict__ p0,
    const float *__restrict__ p1, float *__restrict__ R, const float *__restrict__ sub, int e0, int e1, int sorted,
    double *__restrict__ part)
{
    __shared__ PairRec list[F3_CHUNK];  // (their first 48 bytes)
    __shared__ unsigned short wl[F3_WAVES][F3_CHUNK];
    __shared__ int cnt[F3_WAVES][F3_WAVES];
    __shared__ int wlen[F3_WAVES];
    __shared__ F3Tab tab[F3_WAVES];
    const int tilesR = (n0 + TILE_ROWS - 1) / TILE_ROWS, tilesC = (n1 + TILE_COLS - 1) / TILE_COLS;
    const int a = (int)(blockIdx.x % (unsigned)nA);
    int t[2];
    morton_ranks2(blockIdx.x / (unsigned)nA, e0, e1, t);
    if (t[0] >= tilesR || t[1] >= tilesC) return;  // whole block: no tile of this rank
    const int row0 = centre_out(t[0], tilesR) * TILE_ROWS, col0 = centre_out(t[1], tilesC) * TILE_COLS;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr0 = row0 + 8 * (wave >> 2), wc0 = col0 + 16 * (wave & 3);
    const int i1 = wc0 + (lane & 15);
    const int rA = wr0 + (lane >> 4), rB = rA + 4;
    const float pc = p1[min(i1, n1 - 1)];
    const float pr8 = p0[min(wr0 + (lane & 7), n0 - 1)];
    const int u16 = lane >> 4;
    double sA = 0.0, sB = 0.0;
    // detector coordinates bounding each wave rectangle (first and last
    // row / column), for the exact cull of an ascending detector
    float rx[F3_RX], cy[F3_CY];
#pragma unroll
    for (int w = 0; w < (F3_WAVES + 3) / 4; w++) {
        rx[2 * w] = p0[min(row0 + 8 * w, n0 - 1)];
        rx[2 * w + 1] = p0[min(row0 + 8 * w + 7, n0 - 1)];
    }
#pragma unroll
    for (int w = 0; w < (F3_WAVES < 4 ? F3_WAVES : 4); w++) {
        cy[2 * w] = p1[min(col0 + 16 * w, n1 - 1)];
        cy[2 * w + 1] = p1[min(col0 + 16 * w + 15, n1 - 1)];
    }
    const PairRec *ra = recs + (size_t)a * N;
    for (int base = 0; base < N; base += F3_CHUNK) {
        stage_rects(ra, base, N, row0, col0, list, wl, cnt, wlen, sorted != 0, rx, cy);
        const int len = wlen[wave];
        const unsigned short *wlw = wl[wave];
        if (len > 0) {
            // lane (u, k): record u of the group at column k and row k % 8
            F3Tab &T = tab[wave];
            float vA[4], vB[4];
            const float *lf = reinterpret_cast<const float *>(list) + (lane & 15);
            float w = lf[16 * wlw[min(u16, len - 1)]];
            int nidx = wlw[min(4 + u16, len - 1)];
            const auto group = [&](int e) {
                // words of a record: 0 alpha, 1-2 c_hi, 3-4 c_lo, 5-10 q
                const float dp1 = (pc - row_bcast<2>(w)) - row_bcast<4>(w);
                T.c[u16][lane & 15] =
                    make_float4(fmaf(row_bcast<6>(w), dp1, row_bcast<8>(w)),
                                fmaf(fmaf(row_bcast<7>(w), dp1, row_bcast<9>(w)), dp1, row_bcast<10>(w)),
                                row_bcast<5>(w), row_bcast<0>(w));
                T.r[u16][2 * (lane & 3) + ((lane >> 2) & 1)] = (pr8 - row_bcast<1>(w)) - row_bcast<3>(w);
                wave_sync();
                float4 c[4];
                float2 d[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    c[u] = T.c[u][lane & 15];
                    d[u] = *reinterpret_cast<const float2 *>(&T.r[u][2 * u16]);
                }
                w = lf[16 * nidx];
                nidx = wlw[min(e + 8 + u16, len - 1)];
                wave_sync();
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    vA[u] = c[u].w * __builtin_amdgcn_exp2f(fmaf(fmaf(c[u].z, d[u].x, c[u].x), d[u].x, c[u].y));
                    vB[u] = c[u].w * __builtin_amdgcn_exp2f(fmaf(fmaf(c[u].z, d[u].y, c[u].x), d[u].y, c[u].y));
                }
            };
            int e = 0;
            // the four values of a pixel are summed in FP32 in list order and
            // that sum is added to the pixel's FP64 total: an error of at most
            // 3u times the sum of the four magnitudes, for one conversion and
            // one FP64 add per four records
            for (; e + 4 <= len; e += 4) {
                group(e);
                sA += (double)(((vA[0] + vA[1]) + vA[2]) + vA[3]);
                sB += (double)(((vB[0] + vB[1]) + vB[2]) + vB[3]);
            }
            if (e < len) {
                group(e);
#pragma unroll
                for (int u = 0; u < 3; u++)
                    if (e + u < len) {
                        sA += (double)vA[u];
                        sB += (double)vB[u];
                    }
            }
        }
        __syncthreads();
    }
    // R = projection, or projection - sub (the residual) when sub is given
    float vA = 0.0f, vB = 0.0f;
    if (i1 < n1) {
        const size_t oA = ((size_t)a * n0 + rA) * n1 + i1, oB = ((size_t)a * n0 + rB) * n1 + i1;
        if (rA < n0) R[oA] = vA = sub ? (float)sA - sub[oA] : (float)sA;
        if (rB < n0) R[oB] = vB = sub ? (float)sB - sub[oB] : (float)sB;
    }
    if (!part) return;
    // sum of squares of the wave's rectangle, for the l2 value of the residual
    const double q = wave_sum_f64((double)vA * vA + (double)vB * vB);
    if (lane == 0)
        part[(((size_t)a * tilesR + row0 / TILE_ROWS) * tilesC + col0 / TILE_COLS) * F3_WAVES + wave] = q;
}

// ---------------------------------------------------------------------------
// forward, 1D detectors (2D geometry)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void forward2_kernel(const PairRec *__restrict__ recs, int N, int n0,
                                                       const float *__restrict__ p0, float *__restrict__ R,
                                                       const float *__restrict__ sub, double *__restrict__ part)
{
    __shared__ PairRec list[CHUNK];
    __shared__ int wcnt[4];
    const int a = blockIdx.y;
    const int row0 = blockIdx.x * 256;
    const int i0 = row0 + (int)threadIdx.x;
    const int wave = threadIdx.x >> 6;
    const int w0 = row0 + wave * 64, w1 = w0 + 63;
    const int thi = min(row0 + 255, n0 - 1);
    const float pr = p0[min(i0, n0 - 1)];
    float s = 0.0f, c = 0.0f;
    const PairRec *ra = recs + (size_t)a * N;
    const float kap = (float)KAPPA;
    for (int base = 0; base < N; base += CHUNK) {
        const int total = stage_chunk<4>(ra, base, N, row0, thi, 0, 0, list, wcnt);
        // four records at a time: their values first, then the compensated sum
        // takes them in list order (a few waves per CU: one at a time, every
        // record's LDS reads and exponential were waited for: 50 atoms, 180 angles
        // 12.0 us, now 10.4)
        for (int e = 0; e < total; e += 4) {
            float v[4];
            bool in[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const PairRec &q = list[min(e + u, total - 1)];
                const float dp0 = (pr - q.c_hi[0]) - q.c_lo[0];
                const float qq = fmaf(fmaf(q.q[0], dp0, q.q[3]), dp0, q.q[5]);
                in[u] = e + u < total && !(q.lo[0] > w1 || q.hi[0] < w0) && qq >= kap;
                v[u] = q.alpha * __builtin_amdgcn_exp2f(qq);
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (in[u]) kahan_add(s, c, v[u]);
        }
        __syncthreads();
    }
    float v = 0.0f;
    if (i0 < n0) R[(size_t)a * n0 + i0] = v = sub ? s - sub[(size_t)a * n0 + i0] : s;
    if (!part) return;
    const double q2 = wave_sum_f64((double)v * v);
    if ((threadIdx.x & 63) == 0) part[((size_t)a * gridDim.x + blockIdx.x) * 4 + wave] = q2;
}

// ---------------------------------------------------------------------------
// moments
// ---------------------------------------------------------------------------
// f = 1/2 sum of the forward's n partial sums of squares, in a fixed order.  With
// a moments grid to follow, one wave of it adds PART_CHUNK of them in place and
// one block of the finish grid the n / PART_CHUNK results; without, one block of
// half_sum_kernel adds up to HALF_SUM_MAX itself (46080 of 5000 atoms' 90 x
// 256^2: 8 us) and more after a launch that folds the chunks.  16 loads in
// flight per lane.
constexpr int PART_CHUNK = 1024, HALF_SUM_MAX = 65536;
__device__ inline void chunk_sum(double *__restrict__ part, size_t n, size_t chunk, int lane)
{
    double *p = part + chunk * PART_CHUNK;
    const int m = (int)(n - chunk * PART_CHUNK < PART_CHUNK ? n - chunk * PART_CHUNK : PART_CHUNK);
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) v[u] = p[std::min(lane + 64 * u, m - 1)];
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < 16; u++) s[u & 3] += lane + 64 * u < m ? v[u] : 0.0;
    const double t = wave_sum_f64((s[0] + s[1]) + (s[2] + s[3]));
    if (lane == 0) p[0] = t;  // read by this wave only, before
}
// L2 mode: the sums of C^2 per angle (the value of the pixels outside every
// footprint), SQ_CHUNK pixels by a wave of the moments grid each; the finish adds
// an angle's sq_chunks().  37 atoms, 41 x 101 x 75: 70.2 -> 66.5 us a call
// with the host copy, by a launch and 5.4 us less.
constexpr int SQ_CHUNK = 4096;
__host__ __device__ inline int sq_chunks(long per) { return (int)((per + SQ_CHUNK - 1) / SQ_CHUNK); }
__device__ inline void sumsq_chunk(const float *__restrict__ C, long per, size_t k, double *__restrict__ out, int lane)
{
    const int nch = sq_chunks(per);
    const long a = (long)(k / nch), b = (long)(k % nch) * SQ_CHUNK;
    const float *c = C + a * per + b;
    const int m = (int)(per - b < SQ_CHUNK ? per - b : SQ_CHUNK);
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i = lane; i < m; i += 64 * 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = c[std::min(i + 64 * u, m - 1)];
#pragma unroll
        for (int u = 0; u < 8; u++) s[u & 3] += i + 64 * u < m ? (double)v[u] * (double)v[u] : 0.0;
    }
    const double t = wave_sum_f64((s[0] + s[1]) + (s[2] + s[3]));
    if (lane == 0) out[k] = t;
}
template <int NTHR>
__device__ inline void half_sum(const double *__restrict__ sums, size_t n, size_t stride, double *__restrict__ f,
                                double *red)
{
    double s = 0.0;
    size_t i = threadIdx.x;
    for (; i + 15 * NTHR < n; i += 16 * NTHR) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = sums[(i + u * NTHR) * stride];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] += v[u + 8];
        s += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    if (i < n) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = sums[std::min(i + u * NTHR, n - 1) * stride];
#pragma unroll
        for (int u = 0; u < 16; u++) s += i + u * NTHR < n ? v[u] : 0.0;
    }
    const double t = wave_sum_f64(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = 0.0;
        for (int w = 0; w < NTHR / 64; w++) v += red[w];
        f[0] = 0.5 * v;
    }
}
__global__ __launch_bounds__(64) void chunk_sum_kernel(double *__restrict__ part, size_t n)
{
    chunk_sum(part, n, blockIdx.x, threadIdx.x);
}
__global__ __launch_bounds__(1024) void half_sum_kernel(const double *__restrict__ sums, size_t n, size_t stride,
                                                        double *__restrict__ f)
{
    __shared__ double red[16];
    half_sum<1024>(sums, n, stride, f, red);
}

// Layout of one moment record (32 floats): [0, NM) sum w1 mono, [15, 15+NM)
// sum E^2 mono, [30] sum_fp (alpha E - C)^2, [31] sum_fp C^2 (L2 mode).  Order 1
// takes the degrees up to 2 of the first only (the rest is zero): a gradient
// needs 6 of the 30 moments (3 of 10 on a 1D detector).  5000 atoms, 90 x 256^2,
// linear mode: 2.08 -> 1.58 ms, the last 0.12 of it from 64 registers instead of
// 86 (eight waves per SIMD; order 2's reduction slab allows five).
template <int K, int MODE, int ORDER>
__global__ __launch_bounds__(64 * MOM_WAVES, ORDER == 1 ? 8 : 1) void moments_kernel(const PairRec *__restrict__ recs, int N, int nA,
                                                                 int n0, int n1, const float *__restrict__ p0,
                                                                 const float *__restrict__ p1,
                                                                 const float *__restrict__ C, float *__restrict__ mom,
                                                                 double *__restrict__ part, size_t nparts)
{
    constexpr int NV = ORDER == 2 ? MOM_STRIDE : 8, DEG = ORDER == 2 ? 4 : 2;  // values summed, highest degree
    using Row = typename RowPow<DEG>::type;
    // the reduction slab of a wave doubles as its row table while it walks
    // its pair (order 2: 8 KiB of the 8.25 KiB slab; order 1: 4 KiB)
    constexpr size_t SLAB = std::max(64 * (NV + 1) * sizeof(float), MOM_TROWS * sizeof(Row));
    __shared__ alignas(16) char slab[MOM_WAVES][SLAB];
    // the wave index is uniform: scalar pair index, record and slab base
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long pair = (long)blockIdx.x * MOM_WAVES + wave;
    const bool valid = pair < (long)N * nA;
    if (!valid) {  // the waves past the pairs: f's partial sums
        const size_t k = (size_t)(pair - (long)N * nA);
        if (MODE == MODE_L2) {
            if (k < nparts) sumsq_chunk(C, (long)n0 * n1, k, part, lane);
        } else if (k * PART_CHUNK < nparts) {
            chunk_sum(part, nparts, k, lane);
        }
        return;
    }
    float acc[MOM_STRIDE];
#pragma unroll
    for (int v = 0; v < MOM_STRIDE; v++) acc[v] = 0.0f;
    const PairRec rec = recs[pair];
    const int a = (int)(pair / N);
    if (K == 2)
        pair_moments_rows<MODE, 4, MOM_TROWS, DEG>(rec, p0, p1, C + (size_t)a * n0 * n1, n1, lane, acc,
                                                   reinterpret_cast<Row *>(slab[wave]));
    else
        pair_moments<K, MODE, DEG>(rec, p0, p1, C + (size_t)a * n0 * n1, n1, lane, acc);
    // each wave reduces its own slab: no block barrier, so a wave whose pair
    // is done does not wait for the others of its block
    float (*red)[NV + 1] = reinterpret_cast<float (*)[NV + 1]>(slab[wave]);
#pragma unroll
    for (int v = 0; v < NV; v++) red[lane][v] = acc[ORDER == 2 || v < 6 ? v : 24 + v];
    wave_sync();
    // (the same order of additions for both orders: equal gradients)
    const int col = lane & 31, half = lane >> 5;
    const int v = ORDER == 2 || col < 6 ? col : col - 24;  // its value's slot (order 1: 0..5, 30, 31)
    float s = 0.0f;
    if (v >= 0 && v < NV && (ORDER == 2 || col < 6 || col >= 30))
        for (int i = 0; i < 32; i++) s += red[half * 32 + i][v];
    s += __shfl_xor(s, 32);
    if (half == 0) mom[pair * MOM_STRIDE + col] = s;
}

// FP64 sum of C^2 per angle.
__global__ __launch_bounds__(256) void sumsq_kernel(const float *__restrict__ C, long per, double *__restrict__ out)
{
    __shared__ double red[256];
    const int a = blockIdx.x;
    double s = 0.0;
    for (long i = threadIdx.x; i < per; i += 256) {
        const double v = C[(size_t)a * per + i];
        s += v * v;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[a] = red[0];
}

// ---------------------------------------------------------------------------
// finish
// ---------------------------------------------------------------------------
// With part given, one block more, the first: f from the forward's partial sums.
// One kernel for both orders, so that the gradient is formed by the same
// instructions and an order-1 call returns the bits of an order-2 one.
// W waves per atom: with more than 64 angles a lane of one wave would contract
// several pairs one after the other.
template <int D, int MODE, int W>
__global__ __launch_bounds__(64 * W) void finish_kernel(gt_atoms A, gt_geom G, const PairRec *__restrict__ recs,
                                                    const float *__restrict__ mom, const double *__restrict__ sumC2,
                                                    int want_hess, double *__restrict__ fo, double *__restrict__ go,
                                                    double *__restrict__ Ho, const double *__restrict__ part,
                                                    size_t nparts, double *__restrict__ ftotal)
{
    using Dm = Dims<D>;
    constexpr int P = Dm::P, NM = Dm::NM, NH = P * (P + 1) / 2, NV = 1 + P + NH;
    // row of lane l: [F, grad (P), upper Hessian by rows (NH)]; the lane
    // accumulates its pairs' Hessian entries there directly (a P x P array
    // per lane in registers would spill)
    __shared__ double red[64 * W][NV + 1];
    const int j = (int)blockIdx.x - (part ? 1 : 0), lane = threadIdx.x;
    const int N = A.n;
    if (j < 0) {
        half_sum<64 * W>(part, (nparts + PART_CHUNK - 1) / PART_CHUNK, PART_CHUNK, ftotal, &red[0][0]);
        return;
    }
    double grad[P], F = 0.0;
    for (int i = 0; i < P; i++) grad[i] = 0.0;
    double *row = red[lane];
    for (int k = 0; k < NV; k++) row[k] = 0.0;
    PairGeom<D> g;
    load_atom<D>(A, j, g);
    for (int a = lane; a < G.nA; a += 64 * W) {
        const size_t pi = (size_t)a * N + j;
        const PairRec rec = recs[pi];
        const float *m = mom + pi * MOM_STRIDE;
        if (MODE == MODE_L2 && fo) {
            const int nch = sq_chunks((long)G.n0 * G.n1);
            double c2 = 0.0;
            for (int c = 0; c < nch; c++) c2 += sumC2[(size_t)a * nch + c];
            F += 0.5 * (c2 - (double)m[31] + (double)m[30]);
        }
        const bool empty = rec.lo[0] > rec.hi[0] || (D == 3 && rec.lo[1] > rec.hi[1]);
        if (empty) continue;
        load_angle<D>(G, a, g);
        double S1[NM], S2[NM];
        for (int k = 0; k < NM; k++) {
            S1[k] = m[k];
            S2[k] = m[15 + k];
        }
        if (MODE == MODE_LINEAR) {
            double t[3], s = 0.0;
            matvec_upper<D>(g.U, g.T, t);
            for (int i = 0; i < D; i++) s += t[i] * t[i];
            F += g.I / sqrt(s) * S1[0];
        }
        const double pstar[2] = {(double)rec.c_hi[0] + (double)rec.c_lo[0],
                                 (double)rec.c_hi[1] + (double)rec.c_lo[1]};
        pair_finish_to<D>(g, pstar, S1, S2, MODE != MODE_LINEAR, want_hess, grad, HessUpper<P>{row + 1 + P});
    }
    row[0] = F;
    for (int i = 0; i < P; i++) row[1 + i] = grad[i];
    __syncthreads();
    // columns added 64 rows per wave, then over the waves
    const int row0 = lane & ~63;
    for (int col = lane & 63; col < NV; col += 64) {
        double s = 0.0;
        for (int i = 0; i < 64; i++) s += red[row0 + i][col];
        red[row0][col] = s;  // the rows after it, of this column, are no longer read
    }
    __syncthreads();
    if (W > 1) {
        if (lane >= 64) return;
        for (int col = lane; col < NV; col += 64)
#pragma unroll
            for (int w = 1; w < W; w++) red[0][col] += red[64 * w][col];
        wave_sync();
    }
    const double *v = red[0];
    if (!A.iso) {
        // the lanes write the gradient and the full Hessian, one entry each
        if (lane == 0 && fo) fo[j] = v[0];
        if (lane < P) go[(size_t)j * P + lane] = v[1 + lane];
        if (Ho && want_hess)
            for (int e = lane; e < P * P; e += 64) {
                const int i = e / P, l = e - (e / P) * P;
                const int lo = i < l ? i : l, hi = i < l ? l : i;
                Ho[(size_t)j * P * P + e] = v[1 + P + lo * P - lo * (lo - 1) / 2 + (hi - lo)];
            }
        return;
    }
    if (lane != 0) return;
    if (fo) fo[j] = v[0];
    {
        // U = rho * Id: d r_k / d rho = 1 for the D diagonal slots.
        constexpr int PI = 2 + D;
        double Hf[P][P];
        {
            int k = 1 + P;
            for (int i = 0; i < P; i++)
                for (int l = i; l < P; l++) {
                    Hf[i][l] = v[k];
                    Hf[l][i] = v[k];
                    k++;
                }
        }
        double gi[PI], Hi[PI][PI];
        double E[P][PI];
        for (int i = 0; i < P; i++)
            for (int l = 0; l < PI; l++) E[i][l] = 0.0;
        for (int i = 0; i <= D; i++) E[i][i] = 1.0;
        for (int k = 0; k < D; k++) E[1 + D + k][1 + D] = 1.0;
        for (int l = 0; l < PI; l++) {
            double s = 0.0;
            for (int i = 0; i < P; i++) s += E[i][l] * v[1 + i];
            gi[l] = s;
        }
        for (int l = 0; l < PI; l++) go[(size_t)j * PI + l] = gi[l];
        if (Ho && want_hess) {
            for (int l = 0; l < PI; l++)
                for (int m2 = 0; m2 < PI; m2++) {
                    double s = 0.0;
                    for (int i = 0; i < P; i++)
                        for (int k = 0; k < P; k++) s += E[i][l] * Hf[i][k] * E[k][m2];
                    Hi[l][m2] = s;
                }
            for (int l = 0; l < PI; l++)
                for (int m2 = 0; m2 < PI; m2++) Ho[((size_t)j * PI + l) * PI + m2] = Hi[l][m2];
        }
    }
}

__global__ void fill_kernel(float *__restrict__ p, size_t n, float v)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static inline size_t rec_bytes(const gt_atoms *A, const gt_geom *G)
{
    return align_up((size_t)A->n * G->nA * sizeof(PairRec));
}
static inline size_t mom_bytes(const gt_atoms *A, const gt_geom *G)
{
    return align_up((size_t)A->n * G->nA * MOM_STRIDE * sizeof(float));
}

int launch_setup(const gt_atoms *A, const gt_geom *G, PairRec *recs, hipStream_t st)
{
    const long total = (long)A->n * G->nA;
    if (total == 0) return 0;
    const unsigned blocks = (unsigned)((total + 255) / 256);
    if (G->dim == 3)
        launch_timed(GT_K_SETUP, setup_kernel<3>, dim3(blocks), dim3(256), 0, st, *A, *G, recs);
    else
        launch_timed(GT_K_SETUP, setup_kernel<2>, dim3(blocks), dim3(256), 0, st, *A, *G, recs);
    GT_HIP(hipGetLastError());
    return 0;
}

int launch_fill(float *p, size_t n, float v, hipStream_t st)
{
    if (n == 0) return 0;
    const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 65535);
    hipLaunchKernelGGL(fill_kernel, dim3(blocks), dim3(256), 0, st, p, n, v);
    GT_HIP(hipGetLastError());
    return 0;
}

// Forward projection from precomputed records (used by the fitters too).
__global__ void negate_kernel(float *__restrict__ R, const float *__restrict__ sub, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        R[i] = 0.0f - sub[i];
}

// Forward projection from precomputed records (used by the fitters too);
// with sub != NULL the result is the residual projection - sub.
// part (with n > 0): receives the forward_parts() sums of squares, one per wave.
static size_t forward_parts(const gt_geom *G)
{
    if (G->dim == 3)
        return (size_t)F3_WAVES * G->nA * ((G->n0 + TILE_ROWS - 1) / TILE_ROWS) * ((G->n1 + TILE_COLS - 1) / TILE_COLS);
    return (size_t)4 * G->nA * ((G->n0 + 255) / 256);
}
int launch_forward(const gt_atoms *A, const gt_geom *G, const PairRec *recs, float *R, hipStream_t st,
                   const float *sub, double *part)
{
    const size_t nout = (size_t)G->nA * G->n0 * G->n1;
    if (A->n == 0) {
        if (!sub) return launch_fill(R, nout, 0.0f, st);
        if (nout == 0) return 0;
        hipLaunchKernelGGL(negate_kernel, dim3((unsigned)std::min<size_t>((nout + 255) / 256, 65535)), dim3(256), 0,
                           st, R, sub, nout);
        GT_HIP(hipGetLastError());
        return 0;
    }
    if (G->dim == 3) {
        const int e0 = ceil_log2((G->n0 + TILE_ROWS - 1) / TILE_ROWS), e1 = ceil_log2((G->n1 + TILE_COLS - 1) / TILE_COLS);
        const unsigned long long blocks = (unsigned long long)G->nA << (e0 + e1);
        GT_CHECK_ARG(blocks < (1ull << 31), "forward: too many detector tiles (%d x %d, %d angles)", G->n0, G->n1,
                     G->nA);
        launch_timed(GT_K_FORWARD, forward3_kernel, dim3((unsigned)blocks), dim3(F3_WAVES * 64), 0, st, recs, A->n,
                     G->nA, G->n0, G->n1, G->p0, G->p1, R, sub, e0, e1, G->sorted, part);
    } else {
        const int tiles = (G->n0 + 255) / 256;
        launch_timed(GT_K_FORWARD, forward2_kernel, dim3(tiles, G->nA), dim3(256), 0, st, recs, A->n, G->n0, G->p0, R,
                     sub, part);
    }
    GT_HIP(hipGetLastError());
    return 0;
}

template <int D, int MODE, int ORDER>
static void launch_deriv_kernels(const gt_atoms *A, const gt_geom *G, const PairRec *recs, float *mom,
                                 double *sumC2, const float *C, double *f, double *g, double *H,
                                 double *part, double *ftotal, hipStream_t st)
{
    constexpr int K = D - 1;
    const long pairs = (long)A->n * G->nA;
    // sums beside the moments: a sweep's f from the forward's, an L2 call's C^2
    const size_t nparts = part ? forward_parts(G) : 0;
    const size_t nsq = MODE == MODE_L2 && f ? (size_t)G->nA * sq_chunks((long)G->n0 * G->n1) : 0;
    const size_t waves = (size_t)pairs + (nparts + PART_CHUNK - 1) / PART_CHUNK + nsq;
    launch_timed(GT_K_MOMENTS, moments_kernel<K, MODE, ORDER>, dim3((unsigned)((waves + MOM_WAVES - 1) / MOM_WAVES)),
                 dim3(64 * MOM_WAVES), 0, st, recs,
                 A->n, G->nA, G->n0, G->n1, G->p0, G->p1, C, mom, MODE == MODE_L2 ? sumC2 : part,
                 MODE == MODE_L2 ? nsq : nparts);
    // (1D detectors: 180 angles 11.5 us on one wave, 7.2 on four; a 3D atom's
    // rows take 34 KB per wave, four waves' more than the 64 KB of a static slab)
    if (D == 2 && G->nA > 64)
        launch_timed(GT_K_FINISH, finish_kernel<D, MODE, D == 2 ? 4 : 1>, dim3(A->n + (part ? 1 : 0)), dim3(D == 2 ? 256 : 64), 0,
                     st, *A, *G, recs, mom, sumC2, ORDER == 2 ? 1 : 0, f, g, H, part, nparts, ftotal);
    else
        launch_timed(GT_K_FINISH, finish_kernel<D, MODE, 1>, dim3(A->n + (part ? 1 : 0)), dim3(64), 0, st, *A, *G, recs,
                     mom, sumC2, ORDER == 2 ? 1 : 0, f, g, H, part, nparts, ftotal);
}

// part, ftotal (residual mode): the forward's partial sums and where f goes.
int launch_derivs(const gt_atoms *A, const gt_geom *G, const PairRec *recs, float *mom, double *sumC2,
                  const float *C, int mode, int want_hess, double *f, double *g, double *H, hipStream_t st,
                  double *part = nullptr, double *ftotal = nullptr)
{
    if (A->n == 0) return 0;
    GT_CHECK_ARG((long)A->n * G->nA / 4 < (1L << 31), "too many (atom, angle) pairs for one launch");
    const int D = G->dim;
    if (mode == MODE_RESID) f = nullptr;
#define GT_DISPATCH(DD, MM)                                                                               \
    if (D == DD && mode == MM) {                                                                          \
        if (want_hess)                                                                                    \
            launch_deriv_kernels<DD, MM, 2>(A, G, recs, mom, sumC2, C, f, g, H, part, ftotal, st);        \
        else                                                                                              \
            launch_deriv_kernels<DD, MM, 1>(A, G, recs, mom, sumC2, C, f, g, nullptr, part, ftotal, st);  \
    }
    GT_DISPATCH(3, MODE_LINEAR)
    GT_DISPATCH(3, MODE_L2)
    GT_DISPATCH(3, MODE_RESID)
    GT_DISPATCH(2, MODE_LINEAR)
    GT_DISPATCH(2, MODE_L2)
    GT_DISPATCH(2, MODE_RESID)
#undef GT_DISPATCH
    GT_HIP(hipGetLastError());
    return 0;
}

// Residual projection - data in R and, when f is given, f = 1/2 |R|^2: its sums
// of squares per tile go to part (forward_parts() doubles); without room for
// them (part NULL) or without atoms, per angle to sumC2, by a pass of their own.
// total: also add them up; else the moments and finish kernels do (only with
// part and atoms).
static int launch_residual(const gt_atoms *A, const gt_geom *G, const PairRec *recs, const float *data, float *R,
                           double *f, double *part, double *sumC2, bool total, hipStream_t st)
{
    int rc;
    const bool tiles = f && part && A->n > 0;
    if ((rc = launch_forward(A, G, recs, R, st, data, tiles ? part : nullptr))) return rc;
    if (!f) return 0;
    if (tiles) {
        if (total) {
            size_t n = forward_parts(G), stride = 1;
            if (n > HALF_SUM_MAX) {
                const size_t chunks = (n + PART_CHUNK - 1) / PART_CHUNK;
                hipLaunchKernelGGL(chunk_sum_kernel, dim3((unsigned)chunks), dim3(64), 0, st, part, n);
                n = chunks;
                stride = PART_CHUNK;
            }
            hipLaunchKernelGGL(half_sum_kernel, dim3(1), dim3(1024), 0, st, part, n, stride, f);
        }
    } else {
        hipLaunchKernelGGL(sumsq_kernel, dim3(G->nA), dim3(256), 0, st, R, (long)G->n0 * G->n1, sumC2);
        hipLaunchKernelGGL(half_sum_kernel, dim3(1), dim3(1024), 0, st, sumC2, (size_t)G->nA, (size_t)1, f);
    }
    GT_HIP(hipGetLastError());
    return 0;
}

}  // namespace gt

using namespace gt;

extern "C" size_t gt_forward_workspace(const gt_atoms *atoms, const gt_geom *geom)
{
    if (!atoms || !geom) return 0;
    return rec_bytes(atoms, geom);
}

extern "C" int gt_forward(const gt_atoms *atoms, const gt_geom *geom, float *R, void *ws, size_t ws_bytes,
                          void *stream)
{
    int rc;
    if ((rc = check_atoms(atoms)) || (rc = check_geom(geom, atoms->dim))) return rc;
    GT_CHECK_ARG(R != nullptr, "gt_forward: R is NULL");
    const size_t need = gt_forward_workspace(atoms, geom);
    if (need > ws_bytes || (need > 0 && ws == nullptr)) {
        set_error("gt_forward: workspace of %zu bytes given, %zu needed", ws_bytes, need);
        return GT_EWORKSPACE;
    }
    GT_CHECK_ARG(((uintptr_t)ws & 63) == 0, "gt_forward: workspace must be 64-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    PairRec *recs = (PairRec *)ws;
    if ((rc = launch_setup(atoms, geom, recs, st))) return rc;
    return launch_forward(atoms, geom, recs, R, st, nullptr, nullptr);
}

static size_t ang_bytes(const gt_geom *G) { return align_up((size_t)G->nA * sizeof(double)); }
static size_t part_bytes(const gt_geom *G) { return align_up(forward_parts(G) * sizeof(double)); }
static size_t derivs_bytes(const gt_atoms *A, const gt_geom *G) { return rec_bytes(A, G) + mom_bytes(A, G) + ang_bytes(G); }

extern "C" size_t gt_derivs_workspace(const gt_atoms *atoms, const gt_geom *geom, int mode)
{
    if (!atoms || !geom) return 0;
    if (mode == GT_MODE_RESID) return derivs_bytes(atoms, geom) + part_bytes(geom);
    // (L2: the sums of C^2 in place of one word per angle)
    const size_t sq = align_up((size_t)geom->nA * sq_chunks((long)geom->n0 * geom->n1) * sizeof(double));
    return rec_bytes(atoms, geom) + mom_bytes(atoms, geom) + (mode == GT_MODE_L2 ? sq : ang_bytes(geom));
}

extern "C" int gt_derivs(const gt_atoms *atoms, const gt_geom *geom, const float *C, int mode, int order, double *f,
                         double *g, double *H, void *ws, size_t ws_bytes, void *stream)
{
    int rc;
    if ((rc = check_atoms(atoms)) || (rc = check_geom(geom, atoms->dim))) return rc;
    GT_CHECK_ARG(mode == GT_MODE_LINEAR || mode == GT_MODE_L2 || mode == GT_MODE_RESID,
                 "gt_derivs: mode must be 0 (linear), 1 (L2) or 2 (residual), got %d", mode);
    GT_CHECK_ARG(order == 1 || order == 2, "gt_derivs: order must be 1 or 2, got %d", order);
    GT_CHECK_ARG(C != nullptr || atoms->n == 0, "gt_derivs: C is NULL");
    GT_CHECK_ARG(g != nullptr || atoms->n == 0, "gt_derivs: g is NULL");
    const size_t need = gt_derivs_workspace(atoms, geom, mode);
    if (need > ws_bytes || (need > 0 && ws == nullptr)) {
        set_error("gt_derivs: workspace of %zu bytes given, %zu needed", ws_bytes, need);
        return GT_EWORKSPACE;
    }
    GT_CHECK_ARG(((uintptr_t)ws & 63) == 0, "gt_derivs: workspace must be 64-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    char *w = (char *)ws;
    PairRec *recs = (PairRec *)w;
    float *mom = (float *)(w + rec_bytes(atoms, geom));
    double *sumC2 = (double *)(w + rec_bytes(atoms, geom) + mom_bytes(atoms, geom));
    if ((rc = launch_setup(atoms, geom, recs, st))) return rc;
    return launch_derivs(atoms, geom, recs, mom, sumC2, C, mode, order > 1, f, g, H, st);
}

namespace gt {
// gt_forward_derivs with a workspace of derivs_bytes() or, with the tile sums of
// f (`tiles`), of gt_derivs_workspace() bytes.
int forward_derivs(const gt_atoms *atoms, const gt_geom *geom, const float *data, int order, float *R, double *f,
                   double *g, double *H, void *ws, bool tiles, hipStream_t st)
{
    int rc;
    char *w = (char *)ws;
    PairRec *recs = (PairRec *)w;
    float *mom = (float *)(w + rec_bytes(atoms, geom));
    double *sumC2 = (double *)(w + rec_bytes(atoms, geom) + mom_bytes(atoms, geom));
    double *part = tiles && f && atoms->n > 0 ? (double *)(w + derivs_bytes(atoms, geom)) : nullptr;
    if ((rc = launch_setup(atoms, geom, recs, st))) return rc;
    if ((rc = launch_residual(atoms, geom, recs, data, R, f, part, sumC2, false, st))) return rc;
    return launch_derivs(atoms, geom, recs, mom, sumC2, R, GT_MODE_RESID, order > 1, nullptr, g, H, st, part, f);
}

int check_forward_derivs(const gt_atoms *atoms, const gt_geom *geom, const float *data, int order, const float *R,
                         const double *g)
{
    int rc;
    if ((rc = check_atoms(atoms)) || (rc = check_geom(geom, atoms->dim))) return rc;
    GT_CHECK_ARG(order == 1 || order == 2, "gt_forward_derivs: order must be 1 or 2, got %d", order);
    GT_CHECK_ARG(data != nullptr, "gt_forward_derivs: data is NULL");
    GT_CHECK_ARG(R != nullptr, "gt_forward_derivs: R is NULL");
    GT_CHECK_ARG(g != nullptr || atoms->n == 0, "gt_forward_derivs: g is NULL");
    GT_CHECK_ARG(R != data, "gt_forward_derivs: R must not alias data");
    return 0;
}

size_t forward_derivs_least(const gt_atoms *atoms, const gt_geom *geom) { return derivs_bytes(atoms, geom); }
}  // namespace gt

extern "C" int gt_forward_derivs(const gt_atoms *atoms, const gt_geom *geom, const float *data, int order, float *R,
                                 double *f, double *g, double *H, void *ws, size_t ws_bytes, void *stream)
{
    int rc;
    if ((rc = check_forward_derivs(atoms, geom, data, order, R, g))) return rc;
    const size_t need = gt_derivs_workspace(atoms, geom, GT_MODE_RESID);
    if (need > ws_bytes || (need > 0 && ws == nullptr)) {
        set_error("gt_forward_derivs: workspace of %zu bytes given, %zu needed", ws_bytes, need);
        return GT_EWORKSPACE;
    }
    GT_CHECK_ARG(((uintptr_t)ws & 63) == 0, "gt_forward_derivs: workspace must be 64-byte aligned");
    return forward_derivs(atoms, geom, data, order, R, f, g, H, ws, true, (hipStream_t)stream);
}

extern "C" size_t gt_residual_workspace(const gt_atoms *atoms, const gt_geom *geom)
{
    if (!atoms || !geom) return 0;
    return rec_bytes(atoms, geom) + std::max(part_bytes(geom), ang_bytes(geom));
}

extern "C" int gt_residual(const gt_atoms *atoms, const gt_geom *geom, const float *data, float *R, double *f, void *ws,
                           size_t ws_bytes, void *stream)
{
    int rc;
    if ((rc = check_atoms(atoms)) || (rc = check_geom(geom, atoms->dim))) return rc;
    GT_CHECK_ARG(data != nullptr, "gt_residual: data is NULL");
    GT_CHECK_ARG(R != nullptr, "gt_residual: R is NULL");
    GT_CHECK_ARG(R != data, "gt_residual: R must not alias data");
    const size_t need = gt_residual_workspace(atoms, geom);
    if (need > ws_bytes || (need > 0 && ws == nullptr)) {
        set_error("gt_residual: workspace of %zu bytes given, %zu needed", ws_bytes, need);
        return GT_EWORKSPACE;
    }
    GT_CHECK_ARG(((uintptr_t)ws & 63) == 0, "gt_residual: workspace must be 64-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    PairRec *recs = (PairRec *)ws;
    double *sums = (double *)((char *)ws + rec_bytes(atoms, geom));
    if ((rc = launch_setup(atoms, geom, recs, st))) return rc;
    return launch_residual(atoms, geom, recs, data, R, f, sums, sums, true, st);
}
