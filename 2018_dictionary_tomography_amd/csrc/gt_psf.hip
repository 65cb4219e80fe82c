// gt_psf.hip -- the point-spread ("single particle") projector: detector
// values integrated over each pixel, volume values integrated over each voxel.
//
// SingleParticleGaussTomo binds GaussDictCode/bin/point_spread_functions.py:
//   RadProj          :371-385   P[a][k] = int_{pixel k} R_a(p) dp
//   L2derivs_RadProj :1077-1115 f = 1/2 sum_k (P_k - C_k)^2, its gradient and Hessian
//   derivs_RadProj   :1314-1350 f = sum_k P_k C_k, its gradient and Hessian
//   VolProj          :168-197   u[v] = int_{voxel v} f(y) dy
// with R the line integral of one atom (exp(-30 m) / |UT|, cut where m > 1)
// and f its volume profile.  A pixel is the square of side |p[1] - p[0]|
// around each detector coordinate (per axis; a voxel likewise).
//
// The reference samples each pixel on an 11 x 11 grid that starts one step
// inside the pixel's lower edge and ends one step beyond its upper edge
// (:436-455, 497-520), returns the atom's total for pixels that contain its
// bounding circle and 0 gradients for them (:1012-1015), and uses the first
// axis' spacing for both axes (:563-566).  Here the pixel integral itself is
// computed: for one (atom, angle) the detector profile is alpha 2^(q(d)) with
// q the record's quadratic form (d = p - p*), and the pixel is intersected with
// the bounding box of the support {m <= 1} and integrated on pieces no longer
// than two marginal standard deviations by Gauss-Legendre rules of 3 to 8
// points sized to the piece (error below about 1e-7 of peak x width), the
// second detector axis in closed form when its interval is long (psf_pixel).
//
// Derivatives use the projector's moment contraction (pair_finish) with the
// point moments replaced by pixel-integrated ones, M_k[mono] = int_k mono(d)
// E(d) dd: the linear terms (gradient, and the residual-weighted second
// derivatives) are sums over pixels of weighted M_k; the Gauss-Newton term
// sum_k dP_k dP_k^T, a product of two pixel integrals, enters through the
// products sum_k M_k[m] M_k[m'] of the degree <= 2 monomials.
//
// Rule GT_PSF_SAMPLED reproduces the reference's own numbers instead
// (__rf2 / __rf3 :413-527, __drf2 / __drf3 :924-1075, __if2 / __if3
// :222-291): per (atom, cell) with n the distance of the (projected) centre
// from the cell centre and R = 1 / min diag U, n + R < s gives the atom's
// total (I (pi/30) / det U, or I sqrt(pi/30) / det U in 2D) with no
// derivative, n - R > s gives 0, and otherwise the integrand (no cut-off) is
// sampled at lo + k (hi - lo) / 10, k = 1..11, per axis on [lo, hi] = the
// cell cut to [-R, R] about the centre, each sample weighted (hi - lo) / 11;
// s is half the first detector axis' spacing for both detector axes and half
// the second volume axis' spacing for every volume axis.  The derivatives are
// those of the integrand at the samples (the same moment contraction, with the
// samples for nodes).
#include "gt_pixel.h"

namespace gt {

// Gauss-Legendre rules of 3, 4, 5, 6 and 8 points on [-1, 1], concatenated
// (offsets 0, 3, 7, 12, 18).
__device__ constexpr float GLX[26] = {
    -0.7745966692414834f, 0.0000000000000000f, 0.7745966692414834f, -0.8611363115940526f, -0.3399810435848563f,
    0.3399810435848563f, 0.8611363115940526f, -0.9061798459386640f, -0.5384693101056831f, 0.0000000000000000f,
    0.5384693101056831f, 0.9061798459386640f, -0.9324695142031521f, -0.6612093864662645f, -0.2386191860831969f,
    0.2386191860831969f, 0.6612093864662645f, 0.9324695142031521f, -0.9602898564975362f, -0.7966664774136267f,
    -0.5255324099163290f, -0.1834346424956498f, 0.1834346424956498f, 0.5255324099163290f, 0.7966664774136267f,
    0.9602898564975362f};
__device__ constexpr float GLW[26] = {
    0.5555555555555557f, 0.8888888888888888f, 0.5555555555555557f, 0.3478548451374537f, 0.6521451548625462f,
    0.6521451548625462f, 0.3478548451374537f, 0.2369268850561894f, 0.4786286704993662f, 0.5688888888888890f,
    0.4786286704993662f, 0.2369268850561894f, 0.1713244923791697f, 0.3607615730481389f, 0.4679139345726914f,
    0.4679139345726914f, 0.3607615730481389f, 0.1713244923791697f, 0.1012285362903767f, 0.2223810344533743f,
    0.3137066458778870f, 0.3626837833783618f, 0.3626837833783618f, 0.3137066458778870f, 0.2223810344533743f,
    0.1012285362903767f};

// Points of the rule for an interval of length `len` over which the
// integrand varies on the scale `sc` (a standard deviation): the error of
// each is below about 1e-7 of (peak x len) wherever the interval sits on a
// Gaussian (3 points to len <= 0.5 sc, 4 to 1.0, 5 to 1.4, 6 to 2.0; 8 beyond).
__device__ inline int psf_rule(float len, float sc, int &off)
{
    const float H = len / sc;
    if (H <= 0.5f) { off = 0; return 3; }
    if (H <= 1.0f) { off = 3; return 4; }
    if (H <= 1.4f) { off = 7; return 5; }
    if (H <= 2.0f) { off = 12; return 6; }
    off = 18;
    return 8;
}

// Conditional standard deviation along an axis whose log2-exponent
// coefficient is qd (< 0): the integrand's scale along that axis.
__device__ inline float psf_csig(float qd) { return qd < 0.0f ? rsqrtf(-1.3862943611198906f * qd) : 3.0e38f; }

constexpr int PSF_MAXPIECES = 8;
constexpr int PSF_MS = 40;  // floats per (atom, angle) moment record: S1[15] | Q[21] | f part | pad

struct alignas(16) PsfRec {
    PairRec r;           // alpha, p*, q, inclusive pixel box of the pixels meeting the support
    float sl[2], sh[2];  // support bounding box in d = p - p*
    float sig[2];        // marginal standard deviation of exp(-30 m) per detector axis
    float s[2];          // pixel half-widths
};
static_assert(sizeof(PsfRec) == 96, "PsfRec must stay 96 bytes");

// Tensor rules on whole cells.  Over a cell the exponent is that of its centre
// plus a linear part l . delta plus the quadratic form of the offset delta
// from the centre, and the last depends on the record and the node only.  So
//   int_cell 2^q = 2^q(centre) sum_nodes W[node] prod_axes 2^(l_k delta_k),
// with W[node] = weights x 2^(form(delta)) tabulated once per record: per
// cell one exponential for the centre and NP (even) or NP - 1 (odd) per axis
// instead of NP^K.  W(delta) = W(-delta), so with the sums and differences
// Xe = X+ + X-, Xo = X+ - X- of a node pair only products with an even number
// of differences remain (half the terms).  Magnitude index m of a rule: NP
// even: the NP / 2 positive nodes; NP odd: the centre node, then the positive
// ones (the centre has Xe = 1, Xo = 0).
template <int NP> struct PsfNodes {
    static constexpr int M = (NP + 1) / 2;
    static constexpr bool ODD = (NP & 1) != 0;
};
template <int NP> __host__ __device__ constexpr double psf_node(int m)
{
    return NP == 3   ? (m == 0 ? 0.0 : 0.7745966692414834)
           : NP == 4 ? (m == 0 ? 0.3399810435848563 : 0.8611363115940526)
           : NP == 5 ? (m == 0 ? 0.0 : (m == 1 ? 0.5384693101056831 : 0.9061798459386640))
                     : (m == 0 ? 0.2386191860831969 : (m == 1 ? 0.6612093864662645 : 0.9324695142031521));
}
template <int NP> __host__ __device__ constexpr double psf_weight(int m)
{
    return NP == 3   ? (m == 0 ? 8.0 / 9.0 : 5.0 / 9.0)
           : NP == 4 ? (m == 0 ? 0.6521451548625461 : 0.3478548451374538)
           : NP == 5 ? (m == 0 ? 0.5688888888888889 : (m == 1 ? 0.4786286704993665 : 0.2369268850561891))
                     : (m == 0 ? 0.4679139345726910 : (m == 1 ? 0.3607615730481386 : 0.1713244923791704));
}

// The points per axis of a whole cell of half-widths s whose axes have the
// marginal and conditional standard deviations sig and cs: the largest of the
// axes' rules (3 to 6), or 0 where a cell needs pieces or 8 points (cells
// wider than two standard deviations: psf_pixel / psf_voxel).
__device__ inline int psf_whole_rule(int K, const float *s, const float *sig, const float *cs)
{
    int np = 0, o;
    for (int k = 0; k < K; k++) {
        if (!(s[k] <= sig[k])) return 0;
        np = max(np, psf_rule(2.0f * s[k], cs[k], o));
    }
    return np <= 6 ? np : 0;
}

// Sums and differences of the node pairs of one axis, t = l x (cell half-width).
template <int NP> __device__ inline void psf_axis(float t, float *e, float *o)
{
#pragma unroll
    for (int m = 0; m < PsfNodes<NP>::M; m++) {
        if (PsfNodes<NP>::ODD && m == 0) {
            e[0] = 1.0f;
            o[0] = 0.0f;
            continue;
        }
        const float a = t * (float)psf_node<NP>(m);
        const float p = __builtin_amdgcn_exp2f(a), n = __builtin_amdgcn_exp2f(-a);
        e[m] = p + n;
        o[m] = p - n;
    }
}

// Exponent of a cell's centre below which the cell holds no support: the
// nodes of a whole cell lie within 3 x 0.85 of its centre in the metric of the
// exponent (|.|^2 = -q), so a cell with a node at q >= kappa has its centre at
// q > -84.
constexpr float PSF_CELL_MIN = -84.0f;

// R = 1 / min diag U (:25-30) and the atom's total I (pi/30) / det U, or
// I sqrt(pi/30) / det U in 2D (:60-65): the constants of the sampled rule.
template <int D> __device__ inline void psf_rule_consts(const PairGeom<D> &g, double &rad, double &total)
{
    double dmin = g.U[0][0], dprod = 1.0;
    for (int i = 0; i < D; i++) {
        dmin = fmin(dmin, g.U[i][i]);
        dprod *= g.U[i][i];
    }
    rad = 1.0 / dmin;
    const double c = 3.14159265358979323846 / 30.0;
    total = g.I * (D == 3 ? c : sqrt(c)) / dprod;
}

// Record of the sampled rule: sl = (R, total), s = (s, s) with s half the
// first detector axis' spacing; pixel box = the pixels within |R| + s of p*
// per axis (every other pixel has n - R > s, or n >= |R| + s > s - R, so the
// rule gives it 0).
template <int D>
__device__ inline void psf_setup_sampled(const PairGeom<D> &g, const float *const *det, const int *nd, float hs0,
                                         PsfRec &R)
{
    constexpr int K = Dims<D>::K;
    pair_setup<D>(g, det, nd, 0, R.r);
    double rad, total;
    psf_rule_consts<D>(g, rad, total);
    const double pstar[2] = {(double)R.r.c_hi[0] + (double)R.r.c_lo[0], (double)R.r.c_hi[1] + (double)R.r.c_lo[1]};
    R.sl[0] = (float)rad;
    R.sl[1] = (float)total;
    for (int k = 0; k < 2; k++) {
        R.sh[k] = 0.0f;
        R.sig[k] = 0.0f;
        R.s[k] = hs0;
        if (k >= K) {
            R.r.lo[k] = 0;
            R.r.hi[k] = 0;
            continue;
        }
        const double reach = fabs(rad) + (double)hs0;
        const double pad = 1e-5 * reach + 1e-7;
        R.r.lo[k] = lower_idx(det[k], nd[k], pstar[k] - reach - pad);
        R.r.hi[k] = upper_idx(det[k], nd[k], pstar[k] + reach + pad);
    }
}

template <int D>
__device__ inline void psf_setup(const PairGeom<D> &g, const float *const *det, const int *nd, const float *hs,
                                 PsfRec &R)
{
    constexpr int K = Dims<D>::K;
    pair_setup<D>(g, det, nd, 0, R.r);
    const double pstar[2] = {(double)R.r.c_hi[0] + (double)R.r.c_lo[0], (double)R.r.c_hi[1] + (double)R.r.c_lo[1]};
    PairAlg<D> a;
    pair_alg<D>(g, pstar, a);
    double off[2] = {0.0, 0.0}, hw[2] = {0.0, 0.0}, sg[2] = {1.0, 1.0};
    bool empty = false;
    if (K == 2) {
        const double A00 = a.B[0][0], A01 = a.B[0][1], A11 = a.B[1][1];
        const double det2 = A00 * A11 - A01 * A01;
        if (!(det2 > 1e-12 * A00 * A11 && A00 > 0.0 && A11 > 0.0)) {
            empty = true;
        } else {
            const double i00 = A11 / det2, i01 = -A01 / det2, i11 = A00 / det2;
            const double b0 = a.B[0][2], b1 = a.B[1][2];
            off[0] = -(i00 * b0 + i01 * b1);
            off[1] = -(i01 * b0 + i11 * b1);
            const double rho2 = 1.0 - a.B[2][2] + (b0 * (i00 * b0 + i01 * b1) + b1 * (i01 * b0 + i11 * b1));
            if (!(rho2 >= 0.0)) empty = true;
            hw[0] = sqrt(fmax(rho2, 0.0) * i00);
            hw[1] = sqrt(fmax(rho2, 0.0) * i11);
            sg[0] = sqrt(i00 / 60.0);
            sg[1] = sqrt(i11 / 60.0);
        }
    } else {
        const double A = a.B[0][0], b = a.B[0][1];
        if (!(A > 0.0)) {
            empty = true;
        } else {
            off[0] = -b / A;
            const double rho2 = 1.0 - a.B[1][1] + b * b / A;
            if (!(rho2 >= 0.0)) empty = true;
            hw[0] = sqrt(fmax(rho2, 0.0) / A);
            sg[0] = sqrt(1.0 / (60.0 * A));
        }
    }
    for (int k = 0; k < 2; k++) {
        R.sl[k] = (float)(off[k] - hw[k]);
        R.sh[k] = (float)(off[k] + hw[k]);
        R.sig[k] = (float)sg[k];
        R.s[k] = (k < K) ? hs[k] : 0.0f;
        if (k >= K) {
            R.r.lo[k] = 0;
            R.r.hi[k] = 0;
            continue;
        }
        if (empty) {
            R.r.lo[k] = 1;
            R.r.hi[k] = 0;
            continue;
        }
        const double pad = 1e-5 * (hw[k] + hs[k]) + 1e-7;
        R.r.lo[k] = lower_idx(det[k], nd[k], pstar[k] + off[k] - hw[k] - hs[k] - pad);
        R.r.hi[k] = upper_idx(det[k], nd[k], pstar[k] + off[k] + hw[k] + hs[k] + pad);
    }
}

// Node table of one (atom, angle) for whole pixels: w[(m0 M + m1) 2 + {0, 1}]
// multiplies Xe Ye and Xo Yo (alpha and the pixel's area included).
struct alignas(16) PsfNode2 {
    int np;        // 3 to 6, or 0: psf_pixel
    float pad;
    float w[18];
};
static_assert(sizeof(PsfNode2) == 80, "PsfNode2 must stay 80 bytes");

template <int NP>
__device__ inline void psf_node_table(const PairRec &r, const float *s, PsfNode2 &T)
{
    constexpr int M = PsfNodes<NP>::M;
    const double q0 = r.q[0], q1 = r.q[1], q2 = r.q[2];
    const double area = (double)r.alpha * s[0] * s[1];
#pragma unroll
    for (int m0 = 0; m0 < M; m0++)
#pragma unroll
        for (int m1 = 0; m1 < M; m1++) {
            const double a = s[0] * psf_node<NP>(m0), b = s[1] * psf_node<NP>(m1);
            const double w = area * psf_weight<NP>(m0) * psf_weight<NP>(m1);
            const bool z = PsfNodes<NP>::ODD && (m0 == 0 || m1 == 0);
            const double d = w * exp2(q0 * a * a + q2 * b * b), c = z ? 1.0 : exp2(q1 * a * b);
            T.w[(m0 * M + m1) * 2] = (float)(z ? d : 0.5 * d * (c + 1.0 / c));
            T.w[(m0 * M + m1) * 2 + 1] = (float)(z ? 0.0 : 0.5 * d * (c - 1.0 / c));
        }
}

__device__ inline void psf_node_record(const PsfRec &R, PsfNode2 &T)
{
    const float cs[2] = {psf_csig(R.r.q[0]), psf_csig(R.r.q[2])};
    T.np = psf_whole_rule(2, R.s, R.sig, cs);
    T.pad = 0.0f;
#pragma unroll
    for (int k = 0; k < 18; k++) T.w[k] = 0.0f;
    switch (T.np) {
    case 3: psf_node_table<3>(R.r, R.s, T); break;
    case 4: psf_node_table<4>(R.r, R.s, T); break;
    case 5: psf_node_table<5>(R.r, R.s, T); break;
    case 6: psf_node_table<6>(R.r, R.s, T); break;
    default: break;
    }
    // an amplitude that is not finite (or whose weights are not) stays within
    // its support's box: psf_pixel
    float t = 0.0f;
#pragma unroll
    for (int k = 0; k < 18; k++) t = fmaf(0.0f, T.w[k], t);
    if (!(t == 0.0f)) T.np = 0;
}

// half width of the cells of an ascending coordinate vector, from its first
// spacing (the reference's assumption of a uniform grid, :533, 563)
__device__ inline float psf_cell_half(const float *v) { return 0.5f * fabsf(v[1] - v[0]); }

template <int D>
__global__ __launch_bounds__(256) void psf_setup_kernel(gt_atoms A, gt_geom G, PsfRec *recs, int rule,
                                                        PsfNode2 *nodes)
{
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)A.n * G.nA) return;
    const int a = (int)(idx / A.n), j = (int)(idx - (long)a * A.n);
    PairGeom<D> g;
    load_atom<D>(A, j, g);
    load_angle<D>(G, a, g);
    const float *det[2] = {G.p0, G.p1};
    const int nd[2] = {G.n0, G.n1};
    const float hs[2] = {psf_cell_half(G.p0), D == 3 ? psf_cell_half(G.p1) : 0.0f};
    PsfRec R;
    if (rule == GT_PSF_SAMPLED)
        psf_setup_sampled<D>(g, det, nd, hs[0], R);
    else
        psf_setup<D>(g, det, nd, hs, R);
    recs[idx] = R;
    if (D == 3 && nodes) {
        PsfNode2 T;
        psf_node_record(R, T);
        nodes[idx] = T;
    }
}

// Pieces and step of the composite rule on [L, U]: pieces of at most 2 sigma.
__device__ inline int psf_pieces(float L, float U, float sig, float &h)
{
    const int n = min(PSF_MAXPIECES, max(1, (int)ceilf((U - L) / (2.0f * sig))));
    h = (U - L) / (float)n;
    return n;
}

// Inner integrals in closed form: G[i] = int_l^h u^i exp(-k u^2) du, i < NJ,
// from erf / erfc (G0) and the recursion
//   G_i = [-u^(i-1) exp(-k u^2) / (2k)]_l^h + (i - 1) / (2k) G_(i-2).
// Used only when sqrt(k) (h - l) >= sqrt(2), where the erf difference is well
// conditioned; erfc of the side away from the peak avoids cancellation in
// the tails.
template <int NJ> __device__ inline void psf_inner(float k, float l, float h, float *G)
{
    const float sk = sqrtf(k);
    const float al = sk * l, ah = sk * h;
    float F;
    if (al >= 0.0f)
        F = erfcf(al) - erfcf(ah);
    else if (ah <= 0.0f)
        F = erfcf(-ah) - erfcf(-al);
    else
        F = erff(ah) - erff(al);
    G[0] = 0.88622692545275801f / sk * F;  // sqrt(pi) / 2
    if (NJ > 1) {
        const float el = expf(-al * al), eh = expf(-ah * ah);
        const float i2k = 0.5f / k;
        G[1] = (el - eh) * i2k;
        if (NJ > 2) G[2] = fmaf(l * el - h * eh, i2k, G[0] * i2k);
        if (NJ > 3) G[3] = fmaf(l * l * el - h * h * eh, i2k, 2.0f * G[1] * i2k);
        if (NJ > 4) G[4] = fmaf(l * l * l * el - h * h * h * eh, i2k, 3.0f * G[2] * i2k);
    }
}

// int t^j exp(-k (t - mu)^2) over the same interval, j < NJ, from the G's (t = mu + u).
template <int NJ> __device__ inline void psf_shift(float mu, const float *G, float *T)
{
    T[0] = G[0];
    if (NJ > 1) T[1] = fmaf(mu, G[0], G[1]);
    if (NJ > 2) T[2] = fmaf(mu, fmaf(mu, G[0], 2.0f * G[1]), G[2]);
    if (NJ > 3) T[3] = fmaf(mu, fmaf(mu, fmaf(mu, G[0], 3.0f * G[1]), 3.0f * G[2]), G[3]);
    if (NJ > 4) T[4] = fmaf(mu, fmaf(mu, fmaf(mu, fmaf(mu, G[0], 4.0f * G[1]), 6.0f * G[2]), 4.0f * G[3]), G[4]);
}

template <int NM> struct PsfDeg {
    static constexpr int NJ = NM == 1 ? 1 : NM <= 3 ? 2 : NM <= 6 ? 3 : NM <= 10 ? 4 : 5;
};

// NP x NP Gauss-Legendre rule on [L0, U0] x [L1, U1] (NP = 3 or 4), moments as psf_pixel.
template <int NP, int NM>
__device__ inline void psf_tensor(const float *q, float L0, float U0, float L1, float U1, float *M)
{
    constexpr float X3[3] = {-0.7745966692414834f, 0.0f, 0.7745966692414834f};
    constexpr float W3[3] = {0.5555555555555557f, 0.8888888888888888f, 0.5555555555555557f};
    constexpr float X4[4] = {-0.8611363115940526f, -0.3399810435848563f, 0.3399810435848563f, 0.8611363115940526f};
    constexpr float W4[4] = {0.3478548451374537f, 0.6521451548625462f, 0.6521451548625462f, 0.3478548451374537f};
    const float kap = (float)KAPPA;
    const float m0 = 0.5f * (L0 + U0), r0 = 0.5f * (U0 - L0);
    const float m1 = 0.5f * (L1 + U1), r1 = 0.5f * (U1 - L1);
    constexpr int NJ = PsfDeg<NM>::NJ;
#pragma unroll
    for (int a = 0; a < NP; a++) {
        const float d0 = fmaf(r0, NP == 3 ? X3[a] : X4[a], m0);
        const float wa = r0 * r1 * (NP == 3 ? W3[a] : W4[a]);
        // B_j = sum over the inner nodes of w d1^j, then M[i, j] += d0^i B_j
        float B[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) B[j] = 0.0f;
#pragma unroll
        for (int b = 0; b < NP; b++) {
            const float d1 = fmaf(r1, NP == 3 ? X3[b] : X4[b], m1);
            const float e = pair_q(q, d0, d1);
            float w = (e >= kap) ? wa * (NP == 3 ? W3[b] : W4[b]) * __builtin_amdgcn_exp2f(e) : 0.0f;
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                B[j] += w;
                w *= d1;
            }
        }
        if (NM == 1) {
            M[0] += B[0];
            continue;
        }
        const float P0[5] = {1.0f, d0, d0 * d0, d0 * d0 * d0, d0 * d0 * d0 * d0};
#pragma unroll
        for (int deg = 0; deg <= 4; deg++)
#pragma unroll
            for (int j = 0; j <= deg; j++) {
                const int m = deg * (deg + 1) / 2 + j;
                if (m < NM) M[m] = fmaf(P0[deg - j], B[j < NJ ? j : 0], M[m]);
            }
    }
}



// Pixel-integrated moments of one (atom, angle) over the pixel centred at
// (pc0, pc1): M[mono] = int mono(d) 2^q(d) dd (NM = 1: the value only).
// The pixel is cut to the support's bounding box.  An axis whose interval
// is longer than two marginal standard deviations is integrated in closed
// form (the profile is a 1D Gaussian along it: the last axis for 2D
// detectors, given the first-axis node); otherwise by composite 8-point
// Gauss-Legendre on pieces of at most 2 sigma.  The closed form integrates
// the untruncated Gaussian, which differs from the profile cut at m > 1 by
// less than exp(-30) of its peak.  The number of points per piece follows
// the piece's length over the integrand's scale along the axis (psf_rule).
template <int K, int NM>
__device__ inline void psf_pixel(const PsfRec &R, float pc0, float pc1, float *M)
{
    // 2D detectors: NM counts monomials in (d0, d1); 1D: powers of d0
    constexpr int NJ = (K == 1) ? NM : PsfDeg<NM>::NJ;
    constexpr float LN2 = 0.69314718055994531f;
#pragma unroll
    for (int m = 0; m < NM; m++) M[m] = 0.0f;
    const float c0 = (pc0 - R.r.c_hi[0]) - R.r.c_lo[0];
    const float L0 = fmaxf(c0 - R.s[0], R.sl[0]), U0 = fminf(c0 + R.s[0], R.sh[0]);
    if (!(L0 < U0)) return;
    float h0;
    const int n0 = psf_pieces(L0, U0, R.sig[0], h0);
    const float *q = R.r.q;
    const float kap = (float)KAPPA;
    if (K == 1) {
        if (n0 > 1) {
            // exponent (natural log) -k (d - mu)^2 + peak
            const float k = -LN2 * q[0];
            const float mu = LN2 * q[3] / (2.0f * k);
            const float peak = fmaf(fmaf(q[0], mu, q[3]), mu, q[5]);
            if (peak < kap) return;
            float G[NJ], T[NJ];
            psf_inner<NJ>(k, L0 - mu, U0 - mu, G);
            psf_shift<NJ>(mu, G, T);
            const float w = __builtin_amdgcn_exp2f(peak);
#pragma unroll
            for (int m = 0; m < NM; m++) M[m] = w * T[m];
            return;
        }
        int o0;
        const int g0 = psf_rule(h0, psf_csig(q[0]), o0);
        for (int i0 = 0; i0 < n0; i0++) {
            const float mid = L0 + h0 * ((float)i0 + 0.5f);
            for (int a = 0; a < g0; a++) {
                const float d = fmaf(0.5f * h0, GLX[o0 + a], mid);
                const float e = fmaf(fmaf(q[0], d, q[3]), d, q[5]);
                if (e >= kap) {
                    float w = 0.5f * h0 * GLW[o0 + a] * __builtin_amdgcn_exp2f(e);
#pragma unroll
                    for (int m = 0; m < NM; m++) {
                        M[m] = fmaf(w, 1.0f, M[m]);
                        w *= d;
                    }
                }
            }
        }
        return;
    }
    const float c1 = (pc1 - R.r.c_hi[1]) - R.r.c_lo[1];
    const float L1 = fmaxf(c1 - R.s[1], R.sl[1]), U1 = fminf(c1 + R.s[1], R.sh[1]);
    if (!(L1 < U1)) return;
    float h1;
    const int n1 = psf_pieces(L1, U1, R.sig[1], h1);
    const bool closed = n1 > 1;
    const float k1 = -LN2 * q[2];
    int o0, o1;
    const int g0 = psf_rule(h0, psf_csig(q[0]), o0);
    const int g1 = psf_rule(h1, psf_csig(q[2]), o1);
    if (!closed && n0 == 1 && g0 <= 4 && g1 <= 4) {
        // the common case of an atom wider than the pixel: one tensor rule,
        // unrolled, so that the lanes of a wave (neighbouring pixels of the
        // same atom) run the same instructions
        if (g0 <= 3 && g1 <= 3)
            psf_tensor<3, NM>(q, L0, U0, L1, U1, M);
        else
            psf_tensor<4, NM>(q, L0, U0, L1, U1, M);
        return;
    }
    for (int i0 = 0; i0 < n0; i0++) {
        const float mid0 = L0 + h0 * ((float)i0 + 0.5f);
        for (int a = 0; a < g0; a++) {
            const float d0 = fmaf(0.5f * h0, GLX[o0 + a], mid0);
            const float wa = 0.5f * h0 * GLW[o0 + a];
            float P0[5] = {1.0f, d0, d0 * d0, d0 * d0 * d0, d0 * d0 * d0 * d0};
            if (closed) {
                // given d0 the profile is exp(-k1 (d1 - mu)^2) 2^peak
                const float mu = LN2 * fmaf(q[1], d0, q[4]) / (2.0f * k1);
                const float peak = pair_q(q, d0, mu);
                if (peak < kap) continue;
                float G[NJ], T[NJ];
                psf_inner<NJ>(k1, L1 - mu, U1 - mu, G);
                psf_shift<NJ>(mu, G, T);
                const float w = wa * __builtin_amdgcn_exp2f(peak);
#pragma unroll
                for (int deg = 0; deg <= 4; deg++)
#pragma unroll
                    for (int j = 0; j <= deg; j++) {
                        const int m = deg * (deg + 1) / 2 + j;
                        if (m < NM) M[m] = fmaf(w * P0[deg - j], T[j < NJ ? j : 0], M[m]);
                    }
                continue;
            }
            for (int i1 = 0; i1 < n1; i1++) {
                const float mid1 = L1 + h1 * ((float)i1 + 0.5f);
                for (int b = 0; b < g1; b++) {
                    const float d1 = fmaf(0.5f * h1, GLX[o1 + b], mid1);
                    const float e = pair_q(q, d0, d1);
                    if (e >= kap) {
                        const float w = wa * (0.5f * h1 * GLW[o1 + b]) * __builtin_amdgcn_exp2f(e);
                        if (NM == 1) {
                            M[0] += w;
                        } else {
                            // monomials by degree: 1 | d0 d1 | d0^2 d0d1 d1^2 | ... (mono2 order)
                            float p1[5] = {1.0f, d1, d1 * d1, d1 * d1 * d1, d1 * d1 * d1 * d1};
#pragma unroll
                            for (int deg = 0; deg <= 4; deg++)
#pragma unroll
                                for (int j = 0; j <= deg; j++) {
                                    const int m = deg * (deg + 1) / 2 + j;
                                    if (m < NM) M[m] = fmaf(w, P0[deg - j] * p1[j], M[m]);
                                }
                        }
                    }
                }
            }
        }
    }
}

// The sampled rule for one (atom, angle) and the pixel centred at (pc0, pc1):
// returns the pixel's value; M[mono] = w sum over the samples of mono(d)
// 2^q(d) (zero for total and zero pixels, whose value has no derivative).
// Offsets d = p - p*: the pixel centre sits at c = pc - p* (the reference's
// <x - y, W> is -c), the samples of an axis at L + k h, k = 1..11, with L =
// max(-R, c - s), h = (min(R, c + s) - L) / 10, each of weight 10 h / 11.
template <int K, int NM>
__device__ inline float psf_pixel_sampled(const PsfRec &R, float pc0, float pc1, float *M)
{
    constexpr int NJ = (K == 1) ? NM : PsfDeg<NM>::NJ;
#pragma unroll
    for (int m = 0; m < NM; m++) M[m] = 0.0f;
    const float c0 = (pc0 - R.r.c_hi[0]) - R.r.c_lo[0];
    const float c1 = (K == 2) ? (pc1 - R.r.c_hi[1]) - R.r.c_lo[1] : 0.0f;
    const float rad = R.sl[0], s = R.s[0];
    const float n = (K == 2) ? sqrtf(fmaf(c0, c0, c1 * c1)) : fabsf(c0);
    if (n + rad < s) return R.sl[1];
    if (n - rad > s) return 0.0f;
    const float *q = R.r.q;
    const float L0 = fmaxf(-rad, c0 - s), h0 = 0.1f * (fminf(rad, c0 + s) - L0);
    float w = (10.0f / 11.0f) * h0;
    if (K == 1) {
#pragma unroll
        for (int k = 1; k <= 11; k++) {
            const float d = fmaf((float)k, h0, L0);
            float e = __builtin_amdgcn_exp2f(fmaf(fmaf(q[0], d, q[3]), d, q[5]));
#pragma unroll
            for (int m = 0; m < NM; m++) {
                M[m] += e;
                e *= d;
            }
        }
    } else {
        const float L1 = fmaxf(-rad, c1 - s), h1 = 0.1f * (fminf(rad, c1 + s) - L1);
        w *= (10.0f / 11.0f) * h1;
#pragma unroll 1
        for (int k = 1; k <= 11; k++) {
            const float d0 = fmaf((float)k, h0, L0);
            // exponent along d1 for this d0: q2 d1^2 + (q1 d0 + q4) d1 + (q0 d0^2 + q3 d0 + q5)
            const float b = fmaf(q[1], d0, q[4]), c = fmaf(fmaf(q[0], d0, q[3]), d0, q[5]);
            float B[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++) B[j] = 0.0f;
#pragma unroll
            for (int l = 1; l <= 11; l++) {
                const float d1 = fmaf((float)l, h1, L1);
                float e = __builtin_amdgcn_exp2f(fmaf(fmaf(q[2], d1, b), d1, c));
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    B[j] += e;
                    e *= d1;
                }
            }
            if (NM == 1) {
                M[0] += B[0];
                continue;
            }
            const float P0[5] = {1.0f, d0, d0 * d0, d0 * d0 * d0, d0 * d0 * d0 * d0};
#pragma unroll
            for (int deg = 0; deg <= 4; deg++)
#pragma unroll
                for (int j = 0; j <= deg; j++) {
                    const int m = deg * (deg + 1) / 2 + j;
                    if (m < NM) M[m] = fmaf(P0[deg - j], B[j < NJ ? j : 0], M[m]);
                }
        }
    }
#pragma unroll
    for (int m = 0; m < NM; m++) M[m] *= w;
    return R.r.alpha * M[0];
}

__device__ inline void psf_kahan(float &s, float &c, float v)
{
    const float y = v - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

constexpr int PSF_CHUNK = 64;

// Stage the records of one angle whose pixel box meets [rlo, rhi] x [clo, chi], in atom order.
__device__ inline int psf_stage(const PsfRec *__restrict__ ra, int base, int N, int rlo, int rhi, int clo, int chi,
                                PsfRec *list, int *wcnt)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = base + (int)threadIdx.x;
    bool hit = false;
    if (threadIdx.x < PSF_CHUNK && j < N) {
        const PsfRec &r = ra[j];
        hit = r.r.lo[0] <= rhi && r.r.hi[0] >= rlo && r.r.lo[1] <= chi && r.r.hi[1] >= clo;
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
    if (hit) list[off + __popcll(m & ((1ull << lane) - 1ull))] = ra[j];
    __syncthreads();
    return total;
}

// The forward of 2D detectors with pixel integrals: block = (angle, 8 x 32
// pixels) of 4 waves, numbered centre tiles first (block b: angle b % nA, tile
// of Morton rank b / nA); waves w and w + 2 own the 8 x 16 pixels of columns 16
// (w % 2) .. + 15, lane l column l % 16, rows l / 16 and l / 16 + 4.  A thread
// tests one record against the rectangles (index box, then the support against
// the rectangle widened by half a pixel, support_meets_rect); the two waves of
// a rectangle walk its list in turns of four records and add their sums.
//
// Vector issue and the evenness of the blocks bound it.  Every exponential of a
// cell is a factor of its column times a factor of its row (PfTab): a wave forms
// those of four records at once, 1.5 exponentials per record, lane and node pair
// instead of 8 (two pixels, two axes, two signs) and a product per pixel.  A
// pixel's values are added in FP64.  1000 atoms, 61 x 128^2: 1.59 ms with a form per
// node, 0.45 with the node weights tabulated (8 x 64 pixels per block), 0.39 with
// the factors tabulated, 0.35 with 8 x 32 pixels, 0.32 with two waves per rectangle
// (four: 0.40); 0.86 vector instructions per cycle and CU, exponentials at half
// rate among them, and the LDS busy 26% of the cycles.
constexpr int PF_RECTS = 2, PF_GROUPS = 2, PF_WAVES = PF_RECTS * PF_GROUPS;
constexpr int PF_CHUNK = PF_WAVES * 64, PF_ROWS = 8, PF_COLS = 16 * PF_RECTS;

// A group of four records as the pixels of a wave's rectangle read it.  Along
// a row of pixels a record's exponents at the nodes, t_k x_i, are linear in the
// column, along a column in the row, so every factor 2^(t_k x_i) is one of the
// column (at the rectangle's fifth row) times one of the row.
struct PfTab {
    float4 cn[4][3][16];  // node pair i, column: 2^(t0 x), 2^(-t0 x), 2^(t1 x), 2^(-t1 x)
    float4 rn[4][3][8];   // the rows' factors of the same
    float2 c[4][16];      // the centre's exponent: its terms linear and constant in the row
    float2 r[4][4];       // the offsets of rows r and r + 4
};

template <int NP>
__device__ inline float psf_pixel_nodes(smem<float> *w, const float4 (&cn)[NP / 2], const float4 (&rn)[NP / 2])
{
    constexpr int M = PsfNodes<NP>::M, ODD = PsfNodes<NP>::ODD;
    float Xe[M], Xo[M], Ye[M], Yo[M];
#pragma unroll
    for (int i = 0; i < NP / 2; i++) {
        const float x = cn[i].y * rn[i].y, y = cn[i].w * rn[i].w;
        Xe[i + ODD] = fmaf(cn[i].x, rn[i].x, x);
        Xo[i + ODD] = fmaf(cn[i].x, rn[i].x, -x);
        Ye[i + ODD] = fmaf(cn[i].z, rn[i].z, y);
        Yo[i + ODD] = fmaf(cn[i].z, rn[i].z, -y);
    }
    float s = 0.0f;
#pragma unroll
    for (int m0 = 0; m0 < M; m0++) {
        float a = 0.0f, b = 0.0f;
#pragma unroll
        for (int m1 = 0; m1 < M; m1++) {
            const bool z = ODD && (m0 == 0 || m1 == 0);
            if (ODD && m1 == 0)
                a = w[m0 * M * 2];
            else
                a = fmaf(w[(m0 * M + m1) * 2], Ye[m1], a);
            if (!z) b = fmaf(w[(m0 * M + m1) * 2 + 1], Yo[m1], b);
        }
        if (ODD && m0 == 0)
            s += a;
        else
            s = fmaf(Xe[m0], a, fmaf(Xo[m0], b, s));
    }
    return s;
}

// Record u of the group: its integrals over a lane's two pixels.
template <int NP>
__device__ inline void psf_two_pixels(const PfTab &T, int u, float q0, smem<float> *w, int lane, float &vA, float &vB)
{
    float4 cn[NP / 2], rn[NP / 2];
    const float2 c = T.c[u][lane & 15], r = T.r[u][lane >> 4];
#pragma unroll
    for (int i = 0; i < NP / 2; i++) {
        cn[i] = T.cn[u][i][lane & 15];
        rn[i] = T.rn[u][i][lane >> 4];
    }
    const float eA = fmaf(fmaf(q0, r.x, c.x), r.x, c.y), eB = fmaf(fmaf(q0, r.y, c.x), r.y, c.y);
    const float nA = psf_pixel_nodes<NP>(w, cn, rn);
#pragma unroll
    for (int i = 0; i < NP / 2; i++) rn[i] = T.rn[u][i][(lane >> 4) + 4];
    const float nB = psf_pixel_nodes<NP>(w, cn, rn);
    vA = eA > PSF_CELL_MIN ? __builtin_amdgcn_exp2f(eA) * nA : 0.0f;
    vB = eB > PSF_CELL_MIN ? __builtin_amdgcn_exp2f(eB) * nB : 0.0f;
}

// (96 VGPRs, five waves per SIMD; six: the same time with 72 bytes of spills)
__global__ __launch_bounds__(PF_WAVES * 64) __attribute__((amdgpu_waves_per_eu(5))) void psf_project_kernel(
    const PsfRec *__restrict__ recs, const PsfNode2 *__restrict__ nodes, int N, int nA, int n0, int n1,
    const float *__restrict__ p0, const float *__restrict__ p1, float *__restrict__ R, int e0, int e1)
{
    __shared__ alignas(16) unsigned short wl[PF_RECTS][PF_CHUNK];  // read four at a time
    __shared__ int cnt[PF_RECTS][PF_WAVES];
    __shared__ int wlen[PF_RECTS];
    __shared__ PfTab tab[PF_WAVES];
    __shared__ double part[PF_WAVES - PF_RECTS][2][64];
    const int tilesR = (n0 + PF_ROWS - 1) / PF_ROWS, tilesC = (n1 + PF_COLS - 1) / PF_COLS;
    const int a = (int)(blockIdx.x % (unsigned)nA);
    int t[2];
    morton_ranks2(blockIdx.x / (unsigned)nA, e0, e1, t);
    if (t[0] >= tilesR || t[1] >= tilesC) return;  // whole block: no tile of this rank
    const int row0 = centre_out(t[0], tilesR) * PF_ROWS, col0 = centre_out(t[1], tilesC) * PF_COLS;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rect = wave % PF_RECTS, grp = wave / PF_RECTS;
    const int i1 = col0 + 16 * rect + (lane & 15), rA = row0 + (lane >> 4), rB = rA + 4;
    const float pc = p1[min(i1, n1 - 1)], prA = p0[min(rA, n0 - 1)], prB = p0[min(rB, n0 - 1)];
    const float s0 = psf_cell_half(p0), s1 = psf_cell_half(p1);
    // the rectangle's rows and columns from its fifth row and ninth column on
    const float pr8 = p0[min(row0 + (lane & 7), n0 - 1)], prc = p0[min(row0 + 4, n0 - 1)];
    const float pcc = p1[min(col0 + 16 * rect + 8, n1 - 1)];
    const bool regular = __all(fabsf(pr8 - prc) <= 17.0f * s0 && fabsf(pc - pcc) <= 33.0f * s1);
    const float xa = p0[row0] - s0, xb = p0[min(row0 + PF_ROWS - 1, n0 - 1)] + s0;
    float cy[2 * PF_RECTS];
#pragma unroll
    for (int w = 0; w < PF_RECTS; w++) {
        cy[2 * w] = p1[min(col0 + 16 * w, n1 - 1)] - s1;
        cy[2 * w + 1] = p1[min(col0 + 16 * w + 15, n1 - 1)] + s1;
    }
    const PsfRec *ra = recs + (size_t)a * N;
    const PsfNode2 *na = nodes + (size_t)a * N;
    double sA = 0.0, sB = 0.0;
    for (int base = 0; base < N; base += PF_CHUNK) {
        unsigned mask = 0;
        const int j = base + (int)threadIdx.x;
        if (j < N) {
            const float4 *src = reinterpret_cast<const float4 *>(ra + j);
            const float4 f0 = src[0], f1 = src[1], f2 = src[2];
            const int4 bx = reinterpret_cast<const int4 *>(ra + j)[3];  // lo[0], lo[1], hi[0], hi[1]
            if (bx.x <= row0 + PF_ROWS - 1 && bx.z >= row0 && bx.y <= col0 + PF_COLS - 1 && bx.w >= col0) {
#pragma unroll
                for (int w = 0; w < PF_RECTS; w++) {
                    const int c = col0 + 16 * w;
                    if (bx.y <= c + 15 && bx.w >= c &&
                        support_meets_rect(f1, f2, (xa - f0.y) - f0.w, (xb - f0.y) - f0.w, (cy[2 * w] - f0.z) - f1.x,
                                           (cy[2 * w + 1] - f0.z) - f1.x))
                        mask |= 1u << w;
                }
            }
        }
        wave_lists<PF_WAVES, PF_RECTS>(mask, wl, cnt, wlen);
        const int len = __builtin_amdgcn_readfirstlane(wlen[rect]);
        bool pieces = !regular;  // records that no rule covers whole
        if (len > 0 && regular) {
            // lane (u, k): record u of the group, column k and row k % 8; the
            // record comes as one word per lane (word(k)) and is passed around
            // its row of 16 lanes, the next group's while this one is used
            PfTab &T = tab[wave];
            const unsigned short *lw = wl[rect];
            const int u16 = lane >> 4;
            const auto word = [&](int e) {
                const int jj = base + (int)lw[min(e + u16, len - 1)];
                const int k = lane & 15;
                // np, c_hi, c_lo, q, half-widths
                const float *src = k == 0 ? reinterpret_cast<const float *>(na + jj)
                                          : reinterpret_cast<const float *>(ra + jj) + (k <= 10 ? k : min(k, 12) + 11);
                return *src;
            };
            float wd = word(4 * grp);
            for (int e = 4 * grp; e < len; e += 4 * PF_GROUPS) {
                const float q0 = row_bcast<5>(wd), q1 = row_bcast<6>(wd), q2 = row_bcast<7>(wd);
                const float h0 = row_bcast<11>(wd), h1 = row_bcast<12>(wd);
                const float d1 = (pc - row_bcast<2>(wd)) - row_bcast<4>(wd);
                const float dc = (prc - row_bcast<1>(wd)) - row_bcast<3>(wd);
                const float row = fmaf(q1, d1, row_bcast<8>(wd)), q4 = row_bcast<9>(wd);
                const int np = __float_as_int(row_bcast<0>(wd));
                const float x0 = np == 3 ? (float)psf_node<3>(1)
                                         : (np == 4 ? (float)psf_node<4>(0)
                                                    : (np == 5 ? (float)psf_node<5>(1) : (float)psf_node<6>(0)));
                const float x1 = np == 4 ? (float)psf_node<4>(1)
                                         : (np == 5 ? (float)psf_node<5>(2) : (float)psf_node<6>(1));
                const float x2 = (float)psf_node<6>(2);
                // column factors: the exponents' slopes along the axes at (fifth row, column)
                const float t0 = fmaf(2.0f * q0, dc, row) * h0, t1 = fmaf(q1, dc, fmaf(2.0f * q2, d1, q4)) * h1;
                // row factors: lanes 0-7 along axis 0, lanes 8-15 along axis 1
                const float tr = (lane & 8 ? q1 * h1 : 2.0f * q0 * h0) * (pr8 - prc);
                wave_sync();
                const bool two = __any(np >= 4), three = __any(np == 6);
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    if (i == 1 ? !two : (i == 2 && !three)) continue;
                    const float x = i == 0 ? x0 : (i == 1 ? x1 : x2);
                    T.cn[u16][i][lane & 15] =
                        make_float4(__builtin_amdgcn_exp2f(t0 * x), __builtin_amdgcn_exp2f(-t0 * x),
                                    __builtin_amdgcn_exp2f(t1 * x), __builtin_amdgcn_exp2f(-t1 * x));
                    reinterpret_cast<float2 *>(&T.rn[u16][i][lane & 7])[(lane >> 3) & 1] =
                        make_float2(__builtin_amdgcn_exp2f(tr * x), __builtin_amdgcn_exp2f(-tr * x));
                }
                T.c[u16][lane & 15] = make_float2(row, fmaf(fmaf(q2, d1, q4), d1, row_bcast<10>(wd)));
                reinterpret_cast<float *>(&T.r[u16][lane & 3])[(lane >> 2) & 1] =
                    (pr8 - row_bcast<1>(wd)) - row_bcast<3>(wd);
                int nps[4], jjs[4];
                float q0s[4];
                const uint2 ids = *reinterpret_cast<const uint2 *>(lw + e);  // (entries past the list: not used)
                const unsigned i0 = __builtin_amdgcn_readfirstlane(ids.x), i1 = __builtin_amdgcn_readfirstlane(ids.y);
                jjs[0] = i0 & 0xffffu, jjs[1] = i0 >> 16, jjs[2] = i1 & 0xffffu, jjs[3] = i1 >> 16;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    nps[u] = __builtin_amdgcn_readlane(__float_as_int(wd), 16 * u);
                    q0s[u] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wd), 16 * u + 5));
                }
                wave_sync();
                wd = word(e + 4 * PF_GROUPS);
#pragma unroll 1
                for (int u = 0; u < 4 && e + u < len; u++) {
                    const int jj = base + (u < 2 ? (u == 0 ? jjs[0] : jjs[1]) : (u == 2 ? jjs[2] : jjs[3]));
                    smem<float> *w = scalar_ptr(na + jj)->w;
                    const int npu = u < 2 ? (u == 0 ? nps[0] : nps[1]) : (u == 2 ? nps[2] : nps[3]);
                    const float q0u = u < 2 ? (u == 0 ? q0s[0] : q0s[1]) : (u == 2 ? q0s[2] : q0s[3]);
                    float vA = 0.0f, vB = 0.0f;
                    switch (npu) {
                    case 3: psf_two_pixels<3>(T, u, q0u, w, lane, vA, vB); break;
                    case 4: psf_two_pixels<4>(T, u, q0u, w, lane, vA, vB); break;
                    case 5: psf_two_pixels<5>(T, u, q0u, w, lane, vA, vB); break;
                    case 6: psf_two_pixels<6>(T, u, q0u, w, lane, vA, vB); break;
                    default: pieces = true;
                    }
                    sA += (double)vA;
                    sB += (double)vB;
                }
            }
        }
        if (pieces)
            for (int k = 0; k < len; k++) {
                if ((k >> 2) % PF_GROUPS != grp) continue;  // (the wave's own fours)
                const int jj = base + __builtin_amdgcn_readfirstlane((int)wl[rect][k]);
                if (regular && scalar_ptr(na + jj)->np != 0) continue;
                smem<PairRec> *r = &scalar_ptr(ra + jj)->r;
                // (chosen by the record's box: 0 times an infinite amplitude is no 0)
                const bool in = i1 >= r->lo[1] && i1 <= r->hi[1];
                float m[1];
                psf_pixel<2, 1>(ra[jj], prA, pc, m);
                sA += (double)(in && rA >= r->lo[0] && rA <= r->hi[0] ? r->alpha * m[0] : 0.0f);
                psf_pixel<2, 1>(ra[jj], prB, pc, m);
                sB += (double)(in && rB >= r->lo[0] && rB <= r->hi[0] ? r->alpha * m[0] : 0.0f);
            }
        __syncthreads();
    }
    // the groups' sums, in group order
    if (grp > 0) {
        part[wave - PF_RECTS][0][lane] = sA;
        part[wave - PF_RECTS][1][lane] = sB;
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int g = 1; g < PF_GROUPS; g++) {
        sA += part[(g - 1) * PF_RECTS + rect][0][lane];
        sB += part[(g - 1) * PF_RECTS + rect][1][lane];
    }
    if (i1 < n1) {
        if (rA < n0) R[((size_t)a * n0 + rA) * n1 + i1] = (float)sA;
        if (rB < n0) R[((size_t)a * n0 + rB) * n1 + i1] = (float)sB;
    }
}

// Forward of few atoms, of the sampled rule and of 1D detectors: block = (angle, 16 x 16
// pixels) for 2D detectors, numbered centre tiles first (block b: angle b % nA, tile of Morton rank b / nA over the
// centre-out tile ranks, 2^e0 x 2^e1), or (angle = blockIdx.y, 256 pixels) for
// 1D ones.
template <int K, int RULE>
__global__ __launch_bounds__(256) void psf_forward_kernel(const PsfRec *__restrict__ recs, int N, int nA, int n0,
                                                          int n1, const float *__restrict__ p0,
                                                          const float *__restrict__ p1, float *__restrict__ R, int e0,
                                                          int e1)
{
    __shared__ PsfRec list[PSF_CHUNK];
    __shared__ int wcnt[4];
    int a = blockIdx.y;
    int i0, i1, rlo, rhi, clo, chi;
    if (K == 2) {
        const int ntr = (n0 + 15) / 16, ntc = (n1 + 15) / 16;
        a = (int)(blockIdx.x % (unsigned)nA);
        const int e[3] = {e0, e1, 0};
        int t[3];
        if (RULE == GT_PSF_SAMPLED)
            morton_ranks_loop(blockIdx.x / (unsigned)nA, e, t);
        else
            morton_ranks2(blockIdx.x / (unsigned)nA, e0, e1, t);
        if (t[0] >= ntr || t[1] >= ntc) return;  // whole block: no tile of this rank
        const int tr = centre_out(t[0], ntr), tcc = centre_out(t[1], ntc);
        i0 = tr * 16 + (int)(threadIdx.x >> 4);
        i1 = tcc * 16 + (int)(threadIdx.x & 15);
        rlo = tr * 16;
        rhi = min(rlo + 15, n0 - 1);
        clo = tcc * 16;
        chi = min(clo + 15, n1 - 1);
    } else {
        i0 = blockIdx.x * 256 + (int)threadIdx.x;
        i1 = 0;
        rlo = blockIdx.x * 256;
        rhi = min(rlo + 255, n0 - 1);
        clo = chi = 0;
    }
    const bool valid = i0 < n0 && i1 < n1;
    const float pc0 = p0[min(i0, n0 - 1)];
    const float pc1 = (K == 2) ? p1[min(i1, n1 - 1)] : 0.0f;
    const PsfRec *ra = recs + (size_t)a * N;
    float s = 0.0f, c = 0.0f;
    for (int base = 0; base < N; base += PSF_CHUNK) {
        const int total = psf_stage(ra, base, N, rlo, rhi, clo, chi, list, wcnt);
        for (int e = 0; e < total; e++) {
            const PsfRec &r = list[e];
            if (!valid || r.r.lo[0] > i0 || r.r.hi[0] < i0 || r.r.lo[1] > i1 || r.r.hi[1] < i1) continue;
            float M[1], v;
            if (RULE == GT_PSF_SAMPLED) {
                v = psf_pixel_sampled<K, 1>(r, pc0, pc1, M);
            } else {
                psf_pixel<K, 1>(r, pc0, pc1, M);
                v = r.r.alpha * M[0];
            }
            psf_kahan(s, c, v);
        }
        __syncthreads();
    }
    if (valid) R[((size_t)a * n0 + i0) * n1 + i1] = s;
}

// Moments: one wave per (atom, angle) pair over the pixels of its box.
template <int K, int MODE, int RULE>
__global__ __launch_bounds__(256) void psf_moments_kernel(const PsfRec *__restrict__ recs, int N, int nA, int n0,
                                                          int n1, const float *__restrict__ p0,
                                                          const float *__restrict__ p1, const float *__restrict__ C,
                                                          int order, float *__restrict__ mom)
{
    constexpr int NM = (K == 2) ? 15 : 5, NL = (K == 2) ? 6 : 3, NQ = NL * (NL + 1) / 2;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long pair = (long)blockIdx.x * 4 + wave;
    if (pair >= (long)N * nA) return;
    const PsfRec R = recs[pair];
    const int a = (int)(pair / N);
    float S1[NM], Q[NQ], fp = 0.0f;
#pragma unroll
    for (int m = 0; m < NM; m++) S1[m] = 0.0f;
#pragma unroll
    for (int m = 0; m < NQ; m++) Q[m] = 0.0f;
    const int rows = R.r.hi[0] - R.r.lo[0] + 1, cols = R.r.hi[1] - R.r.lo[1] + 1;
    const long count = (rows > 0 && cols > 0) ? (long)rows * cols : 0;
    const float *Ca = C + (size_t)a * n0 * n1;
    for (long t = lane; t < count; t += 64) {
        const int i0 = R.r.lo[0] + (int)(t / cols), i1 = R.r.lo[1] + (int)(t % cols);
        float M[NM], P;
        if (RULE == GT_PSF_SAMPLED) {
            P = psf_pixel_sampled<K, NM>(R, p0[i0], (K == 2) ? p1[i1] : 0.0f, M);
        } else {
            psf_pixel<K, NM>(R, p0[i0], (K == 2) ? p1[i1] : 0.0f, M);
            P = R.r.alpha * M[0];
        }
        const float cv = Ca[(size_t)i0 * n1 + i1];
        if (MODE == GT_MODE_L2) {
            const float res = P - cv;
#pragma unroll
            for (int m = 0; m < NM; m++) S1[m] = fmaf(res, M[m], S1[m]);
            fp = fmaf(P, 0.5f * P - cv, fp);
            if (order > 1) {
                int k = 0;
#pragma unroll
                for (int u = 0; u < NL; u++)
#pragma unroll
                    for (int v = u; v < NL; v++) {
                        Q[k] = fmaf(M[u], M[v], Q[k]);
                        k++;
                    }
            }
        } else {
#pragma unroll
            for (int m = 0; m < NM; m++) S1[m] = fmaf(cv, M[m], S1[m]);
            fp = fmaf(P, cv, fp);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
        for (int m = 0; m < NM; m++) S1[m] += __shfl_xor(S1[m], o);
#pragma unroll
        for (int m = 0; m < NQ; m++) Q[m] += __shfl_xor(Q[m], o);
        fp += __shfl_xor(fp, o);
    }
    if (lane == 0) {
        float *out = mom + pair * PSF_MS;
        for (int m = 0; m < NM; m++) out[m] = S1[m];
        for (int m = NM; m < 15; m++) out[m] = 0.0f;
        for (int m = 0; m < NQ; m++) out[15 + m] = Q[m];
        for (int m = NQ; m < 21; m++) out[15 + m] = 0.0f;
        out[36] = fp;
        out[37] = out[38] = out[39] = 0.0f;
    }
}

// FP64 sum of C^2 per angle
__global__ __launch_bounds__(256) void psf_sumsq_kernel(const float *__restrict__ C, long per, double *__restrict__ out)
{
    __shared__ double red[4];
    const int a = blockIdx.x;
    double s = 0.0;
    for (long i = threadIdx.x; i < per; i += 256) {
        const double v = C[(size_t)a * per + i];
        s += v * v;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[a] = red[0] + red[1] + red[2] + red[3];
}

// Contraction and reduction over angles: one workgroup per atom, lane = angle.
template <int D, int MODE>
__global__ __launch_bounds__(64) void psf_finish_kernel(gt_atoms A, gt_geom G, const PsfRec *__restrict__ recs,
                                                        const float *__restrict__ mom,
                                                        const double *__restrict__ sumC2, int want_hess,
                                                        double *__restrict__ fo, double *__restrict__ go,
                                                        double *__restrict__ Ho)
{
    using Dm = Dims<D>;
    constexpr int K = Dm::K, P = Dm::P, NM = Dm::NM, NL = (K == 2) ? 6 : 3, NH = P * (P + 1) / 2, NV = 1 + P + NH;
    // row of lane l: [F, grad (P), upper Hessian by rows (NH)]; the lane
    // accumulates its pairs' Hessian entries there directly (a P x P array
    // per lane in registers would spill)
    __shared__ double red[64][NV + 1];
    const int j = blockIdx.x, lane = threadIdx.x;
    const int N = A.n;
    double grad[P], F = 0.0;
    for (int i = 0; i < P; i++) grad[i] = 0.0;
    double *row = red[lane];
    for (int k = 0; k < NV; k++) row[k] = 0.0;
    PairGeom<D> g;
    load_atom<D>(A, j, g);
    for (int a = lane; a < G.nA; a += 64) {
        const size_t pi = (size_t)a * N + j;
        const PsfRec R = recs[pi];
        const float *m = mom + pi * PSF_MS;
        if (MODE == GT_MODE_L2) F += 0.5 * sumC2[a];
        F += (double)m[36];
        if (R.r.lo[0] > R.r.hi[0] || (K == 2 && R.r.lo[1] > R.r.hi[1])) continue;
        load_angle<D>(G, a, g);
        double S1[NM], Q[NL * NL];
        for (int k = 0; k < NM; k++) S1[k] = m[k];
        {
            int k = 0;
            for (int u = 0; u < NL; u++)
                for (int v = u; v < NL; v++) {
                    Q[u * NL + v] = Q[v * NL + u] = m[15 + k];
                    k++;
                }
        }
        const double pstar[2] = {(double)R.r.c_hi[0] + (double)R.r.c_lo[0], (double)R.r.c_hi[1] + (double)R.r.c_lo[1]};
        pair_finish_to<D>(g, pstar, S1, nullptr, MODE == GT_MODE_L2, want_hess, grad, HessUpper<P>{row + 1 + P},
                          MODE == GT_MODE_L2 ? Q : nullptr);
    }
    row[0] = F;
    for (int i = 0; i < P; i++) row[1 + i] = grad[i];
    __syncthreads();
    for (int col = lane; col < NV; col += 64) {
        double s = 0.0;
        for (int i = 0; i < 64; i++) s += red[i][col];
        red[0][col] = s;
    }
    __syncthreads();
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
    double Hf[P][P];
    {
        int k = 1 + P;
        for (int i = 0; i < P; i++)
            for (int l = i; l < P; l++) {
                Hf[i][l] = Hf[l][i] = v[k];
                k++;
            }
    }
    // U = rho Id: the diagonal slots move together
    constexpr int PI = 2 + D;
    auto src = [](int l, int &b, int &n) {
        if (l <= D) {
            b = l;
            n = 1;
        } else {
            b = 1 + D;
            n = D;
        }
    };
    for (int l = 0; l < PI; l++) {
        int b, n;
        src(l, b, n);
        double s = 0.0;
        for (int u = 0; u < n; u++) s += v[1 + b + u];
        go[(size_t)j * PI + l] = s;
    }
    if (Ho && want_hess)
        for (int l = 0; l < PI; l++)
            for (int m2 = 0; m2 < PI; m2++) {
                int b0, c0, b1, c1;
                src(l, b0, c0);
                src(m2, b1, c1);
                double s = 0.0;
                for (int u = 0; u < c0; u++)
                    for (int w = 0; w < c1; w++) s += Hf[b0 + u][b1 + w];
                Ho[((size_t)j * PI + l) * PI + m2] = s;
            }
}

// ---------------------------------------------------------------------------
// Voxel-integrated volume render
// ---------------------------------------------------------------------------
struct alignas(16) PsfVolRec {
    float amp;           // I sqrt(30 / pi)
    float xh[3], xl[3];  // centre as float pairs
    float u[6];          // U slots scaled by sqrt(30 log2 e): exponent = -|U'(y - x)|^2
    float hw[3];         // support half-widths (rows of U^-1)
    int lo[3], hi[3];    // voxel box of the voxels meeting the support
    float pad[2];
};
static_assert(sizeof(PsfVolRec) == 96, "PsfVolRec must stay 96 bytes");

constexpr double PSF_SQRT_NEG_KAPPA = 6.578818071009935;  // sqrt(30 log2 e)

// Rule GT_PSF_SAMPLED: hw = (R, total, s) with s half the second axis'
// spacing, voxel box = the voxels within |R| + s of x per axis.
template <int D> __device__ inline PsfVolRec psf_vol_record(const gt_atoms &A, const gt_vol &V, int j, int rule)
{
    constexpr int NR = Dims<D>::NR;
    PairGeom<D> g;
    load_atom<D>(A, j, g);
    PsfVolRec R;
    R.amp = (float)(g.I * sqrt(30.0 / 3.14159265358979323846));
    for (int i = 0; i < 3; i++) {
        const double xv = (i < D) ? g.x[i] : 0.0;
        R.xh[i] = (float)xv;
        R.xl[i] = (float)(xv - (double)R.xh[i]);
    }
    for (int k = 0; k < 6; k++) R.u[k] = 0.0f;
    for (int k = 0; k < NR; k++) R.u[k] = (float)(PSF_SQRT_NEG_KAPPA * g.U[slot_row(D, k)][slot_col(D, k)]);
    R.pad[0] = R.pad[1] = 0.0f;
    const float *y[3] = {V.y0, V.y1, V.y2};
    const int m[3] = {V.m0, V.m1, V.m2};
    if (rule == GT_PSF_SAMPLED) {
        double rad, total;
        psf_rule_consts<D>(g, rad, total);
        const float sv = psf_cell_half(V.y1);
        R.hw[0] = (float)rad;
        R.hw[1] = (float)total;
        R.hw[2] = sv;
        for (int c = 0; c < 3; c++) {
            if (c >= D) {
                R.lo[c] = 0;
                R.hi[c] = 0;
                continue;
            }
            const double reach = fabs(rad) + (double)sv;
            const double pad = 1e-5 * reach + 1e-7;
            R.lo[c] = lower_idx(y[c], m[c], g.x[c] - reach - pad);
            R.hi[c] = upper_idx(y[c], m[c], g.x[c] + reach + pad);
        }
        return R;
    }
    const float hv[3] = {psf_cell_half(V.y0), psf_cell_half(V.y1), D == 3 ? psf_cell_half(V.y2) : 0.0f};
    double Ui[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    bool ok = true;
    for (int i = 0; i < D; i++) ok = ok && g.U[i][i] != 0.0;
    if (ok)
        for (int c = D - 1; c >= 0; c--)
            for (int col = 0; col < D; col++) {
                double s = (c == col) ? 1.0 : 0.0;
                for (int k = c + 1; k < D; k++) s -= g.U[c][k] * Ui[k][col];
                Ui[c][col] = s / g.U[c][c];
            }
    for (int c = 0; c < 3; c++) {
        R.hw[c] = 0.0f;
        if (c >= D) {
            R.lo[c] = 0;
            R.hi[c] = 0;
            continue;
        }
        if (!ok) {
            R.lo[c] = 1;
            R.hi[c] = 0;
            continue;
        }
        double hw = 0.0;
        for (int k = 0; k < D; k++) hw += Ui[c][k] * Ui[c][k];
        hw = sqrt(hw);
        R.hw[c] = (float)hw;
        const double pad = 1e-5 * (hw + hv[c]) + 1e-7;
        R.lo[c] = lower_idx(y[c], m[c], g.x[c] - hw - hv[c] - pad);
        R.hi[c] = upper_idx(y[c], m[c], g.x[c] + hw + hv[c] + pad);
    }
    return R;
}

template <int D>
__global__ __launch_bounds__(256) void psf_vol_setup_kernel(gt_atoms A, gt_vol V, PsfVolRec *recs, int rule)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < A.n) recs[j] = psf_vol_record<D>(A, V, j, rule);
}

// exponent of one node: -|U'(y - x)|^2 with y - x from the float pairs
template <int D> __device__ inline float psf_vexp(const PsfVolRec &R, const float *dy)
{
    if (D == 3) {
        const float a0 = fmaf(R.u[0], dy[0], fmaf(R.u[3], dy[1], R.u[5] * dy[2]));
        const float a1 = fmaf(R.u[1], dy[1], R.u[4] * dy[2]);
        const float a2 = R.u[2] * dy[2];
        return -fmaf(a0, a0, fmaf(a1, a1, a2 * a2));
    }
    const float a0 = fmaf(R.u[0], dy[0], R.u[2] * dy[1]);
    const float a1 = R.u[1] * dy[1];
    return -fmaf(a0, a0, a1 * a1);
}

// NP^D tensor Gauss-Legendre rule over the box [L, L + 2r] (NP = 3 or 4).
template <int D, int NP> __device__ inline float psf_vtensor(const PsfVolRec &R, const float *L, const float *r)
{
    constexpr float X3[3] = {-0.7745966692414834f, 0.0f, 0.7745966692414834f};
    constexpr float W3[3] = {0.5555555555555557f, 0.8888888888888888f, 0.5555555555555557f};
    constexpr float X4[4] = {-0.8611363115940526f, -0.3399810435848563f, 0.3399810435848563f, 0.8611363115940526f};
    constexpr float W4[4] = {0.3478548451374537f, 0.6521451548625462f, 0.6521451548625462f, 0.3478548451374537f};
    const float kap = (float)KAPPA;
    float acc = 0.0f, dy[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int a = 0; a < NP; a++) {
        dy[0] = fmaf(r[0], (NP == 3 ? X3[a] : X4[a]) + 1.0f, L[0]);
        const float wa = NP == 3 ? W3[a] : W4[a];
#pragma unroll
        for (int b = 0; b < NP; b++) {
            dy[1] = fmaf(r[1], (NP == 3 ? X3[b] : X4[b]) + 1.0f, L[1]);
            const float wb = wa * (NP == 3 ? W3[b] : W4[b]);
            if (D == 2) {
                const float e = psf_vexp<D>(R, dy);
                acc += (e >= kap) ? wb * __builtin_amdgcn_exp2f(e) : 0.0f;
                continue;
            }
#pragma unroll
            for (int c = 0; c < NP; c++) {
                dy[2] = fmaf(r[2], (NP == 3 ? X3[c] : X4[c]) + 1.0f, L[2]);
                const float e = psf_vexp<D>(R, dy);
                acc += (e >= kap) ? wb * (NP == 3 ? W3[c] : W4[c]) * __builtin_amdgcn_exp2f(e) : 0.0f;
            }
        }
    }
    return acc * r[0] * r[1] * (D == 3 ? r[2] : 1.0f);
}

// voxel integral of one atom: composite Gauss-Legendre over voxel x support
// box, pieces of at most 2 marginal standard deviations, points per piece
// from the piece's length over the profile's scale along the axis
// (psf_rule; the scale is the conditional standard deviation, 1 / sqrt(2 ln2
// |column of U'|^2)).
template <int D> __device__ inline float psf_voxel(const PsfVolRec &R, const float *yc, const float *hv)
{
    float L[3], h[3];
    int n[3] = {1, 1, 1}, g[3] = {1, 1, 1}, o[3] = {0, 0, 0};
    const float cn[3] = {R.u[0] * R.u[0],
                         D == 3 ? fmaf(R.u[3], R.u[3], R.u[1] * R.u[1]) : fmaf(R.u[2], R.u[2], R.u[1] * R.u[1]),
                         D == 3 ? fmaf(R.u[5], R.u[5], fmaf(R.u[4], R.u[4], R.u[2] * R.u[2])) : 0.0f};
    bool one = true;
    int gmax = 0;
    for (int c = 0; c < D; c++) {
        const float dc = (yc[c] - R.xh[c]) - R.xl[c];
        L[c] = fmaxf(dc - hv[c], -R.hw[c]);
        const float U = fminf(dc + hv[c], R.hw[c]);
        if (!(L[c] < U)) return 0.0f;
        n[c] = psf_pieces(L[c], U, R.hw[c] * 0.12909944487358055f, h[c]);  // sigma = hw / sqrt(60)
        g[c] = psf_rule(h[c], psf_csig(-cn[c]), o[c]);
        one = one && n[c] == 1;
        gmax = max(gmax, g[c]);
    }
    if (one && gmax <= 4) {
        const float r[3] = {0.5f * h[0], 0.5f * h[1], 0.5f * h[2]};
        return R.amp * (gmax <= 3 ? psf_vtensor<D, 3>(R, L, r) : psf_vtensor<D, 4>(R, L, r));
    }
    const float kap = (float)KAPPA;
    float acc = 0.0f;
    float dy[3] = {0.0f, 0.0f, 0.0f};
    for (int i0 = 0; i0 < n[0]; i0++)
        for (int a = 0; a < g[0]; a++) {
            dy[0] = fmaf(0.5f * h[0], GLX[o[0] + a], L[0] + h[0] * ((float)i0 + 0.5f));
            const float w0 = 0.5f * h[0] * GLW[o[0] + a];
            for (int i1 = 0; i1 < n[1]; i1++)
                for (int b = 0; b < g[1]; b++) {
                    dy[1] = fmaf(0.5f * h[1], GLX[o[1] + b], L[1] + h[1] * ((float)i1 + 0.5f));
                    const float w1 = w0 * 0.5f * h[1] * GLW[o[1] + b];
                    if (D == 2) {
                        const float e = psf_vexp<D>(R, dy);
                        if (e >= kap) acc = fmaf(w1, __builtin_amdgcn_exp2f(e), acc);
                        continue;
                    }
                    for (int i2 = 0; i2 < n[2]; i2++)
                        for (int c = 0; c < g[2]; c++) {
                            dy[2] = fmaf(0.5f * h[2], GLX[o[2] + c], L[2] + h[2] * ((float)i2 + 0.5f));
                            const float e = psf_vexp<D>(R, dy);
                            if (e >= kap) acc = fmaf(w1 * 0.5f * h[2] * GLW[o[2] + c], __builtin_amdgcn_exp2f(e), acc);
                        }
                }
        }
    return R.amp * acc;
}

// The sampled rule for one atom and the voxel centred at yc: n = |yc - x|,
// n + R < s gives the atom's total, n - R > s gives 0, otherwise amp times
// the samples' sum of exp(-30 |U d|^2) at d = L + k h per axis (k = 1..11, L =
// max(-R, c - s), h = (min(R, c + s) - L) / 10, c = yc - x), each of weight
// prod 10 h / 11.
template <int D> __device__ inline float psf_voxel_sampled(const PsfVolRec &R, const float *yc)
{
    float c[3] = {0.0f, 0.0f, 0.0f}, L[3] = {0.0f, 0.0f, 0.0f}, h[3] = {0.0f, 0.0f, 0.0f};
    float n2 = 0.0f;
    for (int i = 0; i < D; i++) {
        c[i] = (yc[i] - R.xh[i]) - R.xl[i];
        n2 = fmaf(c[i], c[i], n2);
    }
    const float rad = R.hw[0], s = R.hw[2], n = sqrtf(n2);
    if (n + rad < s) return R.hw[1];
    if (n - rad > s) return 0.0f;
    float w = R.amp;
    for (int i = 0; i < D; i++) {
        L[i] = fmaxf(-rad, c[i] - s);
        h[i] = 0.1f * (fminf(rad, c[i] + s) - L[i]);
        w *= (10.0f / 11.0f) * h[i];
    }
    float acc = 0.0f, dy[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int a = 1; a <= 11; a++) {
        dy[0] = fmaf((float)a, h[0], L[0]);
        if (D == 2) {
#pragma unroll
            for (int b = 1; b <= 11; b++) {
                dy[1] = fmaf((float)b, h[1], L[1]);
                acc += __builtin_amdgcn_exp2f(psf_vexp<D>(R, dy));
            }
            continue;
        }
#pragma unroll 1
        for (int b = 1; b <= 11; b++) {
            dy[1] = fmaf((float)b, h[1], L[1]);
#pragma unroll
            for (int k = 1; k <= 11; k++) {
                dy[2] = fmaf((float)k, h[2], L[2]);
                acc += __builtin_amdgcn_exp2f(psf_vexp<D>(R, dy));
            }
        }
    }
    return w * acc;
}

// Node table of one 3D atom for whole voxels: w[((m0 M + m1) M + m2) 4 + k], k =
// 0..3, multiplies Xe Ye Ze, Xe Yo Zo, Xo Ye Zo and Xo Yo Ze (amplitude and
// the voxel's volume included).
struct alignas(16) PsfNode3 {
    int np;  // 3 to 6, or 0: psf_voxel
    float pad[3];
    float w[108];
};
static_assert(sizeof(PsfNode3) == 448, "PsfNode3 must stay 448 bytes");

// Entry idx (m0, m1, m2) of the table: the weights of the node and of its
// reflections in the second, third and first axis, combined.  False if it is
// not finite.
template <int NP>
__device__ inline bool psf_node_entry(const PsfVolRec &R, const float *hv, int idx, float *w)
{
    constexpr int M = PsfNodes<NP>::M;
    if (idx >= M * M * M) return true;
    const int mi[3] = {idx / (M * M), (idx / M) % M, idx % M};
    double d[3], f = (double)R.amp;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        double x = psf_node<NP>(0), wt = psf_weight<NP>(0);
#pragma unroll
        for (int m = 1; m < M; m++)
            if (mi[c] == m) {
                x = psf_node<NP>(m);
                wt = psf_weight<NP>(m);
            }
        d[c] = hv[c] * x;
        f *= hv[c] * wt;
    }
    // signs (+++), (++-), (+-+), (-++)
    double W[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const double d0 = k == 3 ? -d[0] : d[0], d1 = k == 2 ? -d[1] : d[1], d2 = k == 1 ? -d[2] : d[2];
        const double a0 = R.u[0] * d0 + R.u[3] * d1 + R.u[5] * d2, a1 = R.u[1] * d1 + R.u[4] * d2, a2 = R.u[2] * d2;
        W[k] = 0.25 * f * exp2(-(a0 * a0 + a1 * a1 + a2 * a2));
    }
    const float v[4] = {(float)(W[0] + W[1] + W[2] + W[3]), (float)(W[0] - W[1] - W[2] + W[3]),
                        (float)(W[0] - W[1] + W[2] - W[3]), (float)(W[0] + W[1] - W[2] - W[3])};
#pragma unroll
    for (int k = 0; k < 4; k++) w[idx * 4 + k] = v[k];
    return isfinite(v[0]) && isfinite(v[1]) && isfinite(v[2]) && isfinite(v[3]);
}

// |column c of U'|^2: the curvature of the exponent along axis c
__device__ inline void psf_col_norms(const PsfVolRec &R, float *cn)
{
    cn[0] = R.u[0] * R.u[0];
    cn[1] = fmaf(R.u[3], R.u[3], R.u[1] * R.u[1]);
    cn[2] = fmaf(R.u[5], R.u[5], fmaf(R.u[4], R.u[4], R.u[2] * R.u[2]));
}

// Record and node table of one atom per wave: lane 0 the record, the lanes one
// table entry each.
__global__ __launch_bounds__(64) void psf_voxel_setup_kernel(gt_atoms A, gt_vol V, PsfVolRec *recs, PsfNode3 *nodes)
{
    __shared__ PsfVolRec R;
    const int j = blockIdx.x, lane = threadIdx.x;
    if (lane == 0) {
        R = psf_vol_record<3>(A, V, j, GT_PSF_EXACT);
        recs[j] = R;
    }
    wave_sync();
    const float hv[3] = {psf_cell_half(V.y0), psf_cell_half(V.y1), psf_cell_half(V.y2)};
    float cn[3], sig[3], cs[3];
    psf_col_norms(R, cn);
    for (int c = 0; c < 3; c++) {
        sig[c] = R.hw[c] * 0.12909944487358055f;  // hw / sqrt(60)
        cs[c] = psf_csig(-cn[c]);
    }
    const int np = psf_whole_rule(3, hv, sig, cs);
    PsfNode3 &T = nodes[j];
    bool finite = true;
    switch (np) {
    case 3: finite = psf_node_entry<3>(R, hv, lane, T.w); break;
    case 4: finite = psf_node_entry<4>(R, hv, lane, T.w); break;
    case 5: finite = psf_node_entry<5>(R, hv, lane, T.w); break;
    case 6: finite = psf_node_entry<6>(R, hv, lane, T.w); break;
    default: break;
    }
    // an amplitude that is not finite (or whose weights are not) stays within
    // its support's box: psf_voxel
    finite = __all(finite);
    if (lane == 0) T.np = finite ? np : 0;
}

template <int NP> __device__ inline float psf_voxel_nodes(smem<float> *w, float t0, float t1, float t2)
{
    constexpr int M = PsfNodes<NP>::M;
    constexpr bool ODD = PsfNodes<NP>::ODD;
    float Xe[M], Xo[M], Ye[M], Yo[M], Ze[M], Zo[M];
    psf_axis<NP>(t0, Xe, Xo);
    psf_axis<NP>(t1, Ye, Yo);
    psf_axis<NP>(t2, Ze, Zo);
    float s = 0.0f;
#pragma unroll
    for (int m0 = 0; m0 < M; m0++) {
        float se = 0.0f, so = 0.0f;
#pragma unroll
        for (int m1 = 0; m1 < M; m1++) {
            float a = 0.0f, b = 0.0f, c = 0.0f, d = 0.0f;
#pragma unroll
            for (int m2 = 0; m2 < M; m2++) {
                smem<float> *q = w + ((m0 * M + m1) * M + m2) * 4;
                const bool z0 = ODD && m0 == 0, z1 = ODD && m1 == 0, z2 = ODD && m2 == 0;
                if (z2)
                    a = q[0];
                else
                    a = fmaf(q[0], Ze[m2], a);
                if (!z1 && !z2) b = fmaf(q[1], Zo[m2], b);
                if (!z0 && !z2) c = fmaf(q[2], Zo[m2], c);
                if (!z0 && !z1) {
                    if (z2)
                        d = q[3];
                    else
                        d = fmaf(q[3], Ze[m2], d);
                }
            }
            if (ODD && m1 == 0) {
                se += a;
                so += c;
            } else {
                se = fmaf(Ye[m1], a, fmaf(Yo[m1], b, se));
                so = fmaf(Ye[m1], c, fmaf(Yo[m1], d, so));
            }
        }
        if (ODD && m0 == 0)
            s += se;
        else
            s = fmaf(Xe[m0], se, fmaf(Xo[m0], so, s));
    }
    return s;
}

// The 3D render with voxel integrals.  Block = brick of 4 x 4 x 8 voxels, two
// cubes of 4 x 4 x 4 (lane = voxel), PX_GROUPS waves per cube that take every
// PX_GROUPS-th record of the cube's list; bricks nearest the volume centre
// first.  A thread tests one record against the cubes: index box, then
// the plane through the cube's centre across the exponent's gradient g there
// (the support reaches |v| rho along it, v = U'(yc - x), rho^2 = -kappa; the
// cube comes as near as |v|^2 - sum |g_c| extent_c).  Records and node tables are
// read into scalar registers; a voxel's values are added in FP64, the groups'
// totals in group order.  Bound by VALU
// issue: a voxel costs 7 to 19 exponentials instead of 27 to 216, and the cube
// test drops what the boxes of slanted ellipsoids keep; 1000 atoms on 64^3:
// 1.75 -> 0.165 ms with bricks of 4 x 8 x 8 and 16 waves, 0.146 with 8 waves,
// 0.124 with bricks of 4 x 4 x 8 and 4 waves per cube (8 per cube: 0.163):
// smaller blocks leave less to the last ones.
constexpr int PX_GROUPS = 4, PX_ROW = 1, PX_CUBES = 2 * PX_ROW, PX_WAVES = PX_GROUPS * PX_CUBES, PX_THREADS = 64 * PX_WAVES;

template <int NP>
__device__ inline float psf_cell_value(smem<float> *w, const float *g, const float *hv, float e)
{
    const float n = psf_voxel_nodes<NP>(w, -2.0f * g[0] * hv[0], -2.0f * g[1] * hv[1], -2.0f * g[2] * hv[2]);
    return e > PSF_CELL_MIN ? __builtin_amdgcn_exp2f(e) * n : 0.0f;
}

__global__ __launch_bounds__(PX_THREADS) __attribute__((amdgpu_waves_per_eu(5))) void psf_voxels_kernel(
    const PsfVolRec *__restrict__ recs, const PsfNode3 *__restrict__ nodes, int N, gt_vol V, float *__restrict__ u,
    int e0, int e1, int e2)
{
    __shared__ alignas(8) unsigned short wl[PX_CUBES][PX_THREADS];
    __shared__ int cnt[PX_CUBES][PX_WAVES];
    __shared__ int wlen[PX_CUBES];
    __shared__ double red[PX_THREADS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cube = wave & (PX_CUBES - 1), grp = wave / PX_CUBES;
    const int nb0 = (V.m0 + 3) / 4, nb1 = (V.m1 + 4 * PX_ROW - 1) / (4 * PX_ROW), nb2 = (V.m2 + 7) / 8;
    const int e[3] = {e0, e1, e2};
    int tb[3];
    morton_ranks(blockIdx.x, e, tb);
    if (tb[0] >= nb0 || tb[1] >= nb1 || tb[2] >= nb2) return;  // whole block
    const int b0 = centre_out(tb[0], nb0) * 4, b1 = centre_out(tb[1], nb1) * 4 * PX_ROW, b2 = centre_out(tb[2], nb2) * 8;
    const int i0 = b0 + (lane >> 4), i1 = b1 + 4 * (cube >> 1) + ((lane >> 2) & 3), i2 = b2 + 4 * (cube & 1) + (lane & 3);
    const bool valid = i0 < V.m0 && i1 < V.m1 && i2 < V.m2;
    const float yc[3] = {V.y0[min(i0, V.m0 - 1)], V.y1[min(i1, V.m1 - 1)], V.y2[min(i2, V.m2 - 1)]};
    const float hv[3] = {psf_cell_half(V.y0), psf_cell_half(V.y1), psf_cell_half(V.y2)};
    // centre and half extent (voxels included) of the brick's cubes per axis
    float cc[3][2], ce[3][2];
    {
        const float *y[3] = {V.y0, V.y1, V.y2};
        const int b[3] = {b0, b1, b2}, m[3] = {V.m0, V.m1, V.m2};
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
            for (int h = 0; h < (c == 0 ? 1 : (c == 1 ? PX_ROW : 2)); h++) {
                const float ya = y[c][min(b[c] + 4 * h, m[c] - 1)], yb = y[c][min(b[c] + 4 * h + 3, m[c] - 1)];
                cc[c][h] = 0.5f * (ya + yb);
                ce[c][h] = 0.5f * (yb - ya) + hv[c];
            }
    }
    double s = 0.0;
    for (int base = 0; base < N; base += PX_THREADS) {
        unsigned mask = 0;
        const int j = base + (int)threadIdx.x;
        if (j < N) {
            const PsfVolRec r = recs[j];
            if ((int)(r.lo[0] <= b0 + 3) & (int)(r.hi[0] >= b0) & (int)(r.lo[1] <= b1 + 4 * PX_ROW - 1) & (int)(r.hi[1] >= b1) &
                (int)(r.lo[2] <= b2 + 7) & (int)(r.hi[2] >= b2)) {
                const float d0 = (cc[0][0] - r.xh[0]) - r.xl[0];
#pragma unroll
                for (int c = 0; c < PX_CUBES; c++) {
                    const int h1 = c >> 1, h2 = c & 1, c1 = b1 + 4 * h1, c2 = b2 + 4 * h2;
                    const float d1 = (cc[1][h1] - r.xh[1]) - r.xl[1], d2 = (cc[2][h2] - r.xh[2]) - r.xl[2];
                    const float v0 = fmaf(r.u[0], d0, fmaf(r.u[3], d1, r.u[5] * d2));
                    const float v1 = fmaf(r.u[1], d1, r.u[4] * d2), v2 = r.u[2] * d2;
                    const float n2 = fmaf(v0, v0, fmaf(v1, v1, v2 * v2));
                    const float g0 = r.u[0] * v0, g1 = fmaf(r.u[3], v0, r.u[1] * v1);
                    const float g2 = fmaf(r.u[5], v0, fmaf(r.u[4], v1, r.u[2] * v2));
                    const float reach = fmaf(fabsf(g0), ce[0][0], fmaf(fabsf(g1), ce[1][h1], fabsf(g2) * ce[2][h2]));
                    // NaN keeps the record
                    const bool apart = n2 * (1.0f - 1e-4f) - reach > ((float)PSF_SQRT_NEG_KAPPA + 1e-2f) * sqrtf(n2);
                    if (r.lo[1] <= c1 + 3 && r.hi[1] >= c1 && r.lo[2] <= c2 + 3 && r.hi[2] >= c2 && !apart)
                        mask |= 1u << c;
                }
            }
        }
        wave_lists<PX_WAVES, PX_CUBES>(mask, wl, cnt, wlen);
        const int len = __builtin_amdgcn_readfirstlane(wlen[cube]);
        bool pieces = false;  // records that no rule covers whole
        for (int k = grp; k < len; k += PX_GROUPS) {
            const int jj = base + __builtin_amdgcn_readfirstlane((int)wl[cube][k]);
            smem<PsfVolRec> *r = scalar_ptr(recs) + jj;
            smem<PsfNode3> *nd = scalar_ptr(nodes) + jj;
            smem<float> *w = nd->w;
            const float u0 = r->u[0], u1 = r->u[1], u2 = r->u[2], u3 = r->u[3], u4 = r->u[4], u5 = r->u[5];
            const float d0 = (yc[0] - r->xh[0]) - r->xl[0], d1 = (yc[1] - r->xh[1]) - r->xl[1],
                        d2 = (yc[2] - r->xh[2]) - r->xl[2];
            const float v0 = fmaf(u0, d0, fmaf(u3, d1, u5 * d2)), v1 = fmaf(u1, d1, u4 * d2), v2 = u2 * d2;
            const float g[3] = {u0 * v0, fmaf(u3, v0, u1 * v1), fmaf(u5, v0, fmaf(u4, v1, u2 * v2))};
            const float ex = -fmaf(v0, v0, fmaf(v1, v1, v2 * v2));
            float v;
            switch (nd->np) {
            case 3: v = psf_cell_value<3>(w, g, hv, ex); break;
            case 4: v = psf_cell_value<4>(w, g, hv, ex); break;
            case 5: v = psf_cell_value<5>(w, g, hv, ex); break;
            case 6: v = psf_cell_value<6>(w, g, hv, ex); break;
            default: v = 0.0f, pieces = true;
            }
            s += (double)v;
        }
        if (pieces)
            for (int k = grp; k < len; k += PX_GROUPS) {
                const int jj = base + __builtin_amdgcn_readfirstlane((int)wl[cube][k]);
                if (scalar_ptr(nodes + jj)->np == 0) s += (double)psf_voxel<3>(recs[jj], yc, hv);
            }
        __syncthreads();
    }
    red[threadIdx.x] = s;
    __syncthreads();
    if (grp == 0 && valid) {
        double t = 0.0;
        for (int g = 0; g < PX_GROUPS; g++) t += red[(g * PX_CUBES + cube) * 64 + lane];
        u[((size_t)i0 * V.m1 + i1) * V.m2 + i2] = (float)t;
    }
}

// The other renders (sampled rule, 2D):
// Block = brick of 4 x 8 x 8 voxels (3D) or 16 x 16 (2D), thread = voxel,
// PV_GROUPS groups of 256 threads on the same brick: group g takes every
// PV_GROUPS-th staged record, and the groups' compensated sums are added in
// group order at the end (deterministic).  Blocks are numbered bricks nearest
// the volume centre first (Morton order over centre-out brick ranks): the
// central bricks meet most atoms, and with several times the blocks that fit
// at once the light outer bricks fill the tail.
constexpr int PV_GROUPS = 4, PV_THREADS = PV_GROUPS * 256, PV_CHUNK = 256;

template <int D, int RULE>
__global__ __launch_bounds__(PV_THREADS) void psf_volume_kernel(const PsfVolRec *__restrict__ recs, int N, gt_vol V,
                                                                float *__restrict__ u, int e0, int e1, int e2)
{
    __shared__ PsfVolRec list[PV_CHUNK];
    __shared__ int wcnt[PV_CHUNK / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int grp = threadIdx.x >> 8, t = threadIdx.x & 255;
    const int B0 = (D == 3) ? 4 : 16, B1 = (D == 3) ? 8 : 16, B2 = (D == 3) ? 8 : 1;
    const int nb0 = (V.m0 + B0 - 1) / B0, nb1 = (V.m1 + B1 - 1) / B1, nb2 = (V.m2 + B2 - 1) / B2;
    const int e[3] = {e0, e1, e2};
    int tb[3];
    morton_ranks_loop(blockIdx.x, e, tb);
    if (tb[0] >= nb0 || tb[1] >= nb1 || tb[2] >= nb2) return;  // whole block
    const int bb0 = centre_out(tb[0], nb0), bb1 = centre_out(tb[1], nb1), bb2 = centre_out(tb[2], nb2);
    const int i0 = bb0 * B0 + t / (B1 * B2), i1 = bb1 * B1 + (t / B2) % B1, i2 = bb2 * B2 + t % B2;
    const int blo[3] = {bb0 * B0, bb1 * B1, bb2 * B2};
    const int bhi[3] = {min(blo[0] + B0 - 1, V.m0 - 1), min(blo[1] + B1 - 1, V.m1 - 1), min(blo[2] + B2 - 1, V.m2 - 1)};
    const bool valid = i0 < V.m0 && i1 < V.m1 && i2 < V.m2;
    const float yc[3] = {V.y0[min(i0, V.m0 - 1)], V.y1[min(i1, V.m1 - 1)], (D == 3) ? V.y2[min(i2, V.m2 - 1)] : 0.0f};
    const float hv[3] = {psf_cell_half(V.y0), psf_cell_half(V.y1), D == 3 ? psf_cell_half(V.y2) : 0.0f};
    float s = 0.0f, c = 0.0f;
    for (int base = 0; base < N; base += PV_CHUNK) {
        // stage the chunk's records that meet the brick (waves 0..3 scan, atom order kept)
        const int j = base + (int)threadIdx.x;
        bool hit = false;
        if (threadIdx.x < PV_CHUNK && j < N) {
            const PsfVolRec &r = recs[j];
            hit = r.lo[0] <= bhi[0] && r.hi[0] >= blo[0] && r.lo[1] <= bhi[1] && r.hi[1] >= blo[1] &&
                  r.lo[2] <= bhi[2] && r.hi[2] >= blo[2];
        }
        const unsigned long long msk = __ballot(hit);
        if (wave < PV_CHUNK / 64 && lane == 0) wcnt[wave] = __popcll(msk);
        __syncthreads();
        int off = 0, total = 0;
#pragma unroll
        for (int w = 0; w < PV_CHUNK / 64; w++) {
            if (w < wave) off += wcnt[w];
            total += wcnt[w];
        }
        if (hit) list[off + __popcll(msk & ((1ull << lane) - 1ull))] = recs[j];
        __syncthreads();
        for (int e = grp; e < total; e += PV_GROUPS) {
            const PsfVolRec &r = list[e];
            if (!valid || r.lo[0] > i0 || r.hi[0] < i0 || r.lo[1] > i1 || r.hi[1] < i1 || r.lo[2] > i2 ||
                r.hi[2] < i2)
                continue;
            psf_kahan(s, c, RULE == GT_PSF_SAMPLED ? psf_voxel_sampled<D>(r, yc) : psf_voxel<D>(r, yc, hv));
        }
        __syncthreads();
    }
    // groups' sums (value minus compensation), added in group order
    float *red = reinterpret_cast<float *>(list);
    static_assert(sizeof(list) >= PV_THREADS * sizeof(float), "reduction buffer");
    red[threadIdx.x] = s - c;
    __syncthreads();
    if (grp == 0 && valid) {
        float ts = 0.0f, tc = 0.0f;
        for (int g = 0; g < PV_GROUPS; g++) psf_kahan(ts, tc, red[g * 256 + t]);
        u[((size_t)i0 * V.m1 + i1) * V.m2 + i2] = ts;
    }
}

__global__ void psf_fill_kernel(float *__restrict__ p, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0.0f;
}

}  // namespace gt

using namespace gt;

static size_t psf_rec_bytes(const gt_atoms *a, const gt_geom *g) { return align_up((size_t)a->n * g->nA * sizeof(PsfRec)); }

// node tables of the 2D-detector forward
static size_t psf_node_bytes(const gt_atoms *a, const gt_geom *g)
{
    return a->dim == 3 ? align_up((size_t)a->n * g->nA * sizeof(PsfNode2)) : 0;
}

extern "C" size_t gt_psf_forward_workspace(const gt_atoms *atoms, const gt_geom *geom)
{
    if (!atoms || !geom) return 0;
    return psf_rec_bytes(atoms, geom) + psf_node_bytes(atoms, geom);
}

static int psf_prepare(const gt_atoms *atoms, const gt_geom *geom, int rule, void *ws, size_t ws_bytes, size_t need,
                       hipStream_t st, const char *who, PsfNode2 *nodes = nullptr)
{
    int rc;
    if ((rc = check_atoms(atoms)) || (rc = check_geom(geom, atoms->dim))) return rc;
    GT_CHECK_ARG(rule == GT_PSF_EXACT || rule == GT_PSF_SAMPLED,
                 "%s: rule must be %d (pixel integral) or %d (the reference's samples), got %d", who, GT_PSF_EXACT,
                 GT_PSF_SAMPLED, rule);
    GT_CHECK_ARG(geom->sorted == 1, "%s: the detector coordinates must ascend (uniform pixels)", who);
    if (need > ws_bytes || (need > 0 && ws == nullptr)) {
        set_error("%s: workspace of %zu bytes given, %zu needed", who, ws_bytes, need);
        return GT_EWORKSPACE;
    }
    GT_CHECK_ARG(((uintptr_t)ws & 63) == 0, "%s: workspace must be 64-byte aligned", who);
    GT_CHECK_ARG(geom->n0 >= 2 && (atoms->dim == 2 || geom->n1 >= 2),
                 "%s: pixel integration needs at least two detector coordinates per axis", who);
    if (atoms->n == 0) return 0;
    PsfRec *recs = (PsfRec *)ws;
    const long pairs = (long)atoms->n * geom->nA;
    const dim3 grid((unsigned)((pairs + 255) / 256));
    if (atoms->dim == 3)
        hipLaunchKernelGGL(psf_setup_kernel<3>, grid, dim3(256), 0, st, *atoms, *geom, recs, rule, nodes);
    else
        hipLaunchKernelGGL(psf_setup_kernel<2>, grid, dim3(256), 0, st, *atoms, *geom, recs, rule,
                           (PsfNode2 *)nullptr);
    GT_HIP(hipGetLastError());
    return 0;
}

extern "C" int gt_psf_forward_rule(const gt_atoms *atoms, const gt_geom *geom, int rule, float *R, void *ws,
                                   size_t ws_bytes, void *stream)
{
    int rc;
    hipStream_t st = (hipStream_t)stream;
    if (!atoms || !geom) {
        set_error("gt_psf_forward: atoms or geometry is NULL");
        return GT_EINVAL;
    }
    // Few atoms (the host-driven fitters project one at a time): most tiles meet none,
    // and psf_project_kernel's cost a fixed time more. 60 angles, us, it and
    // psf_forward_kernel: 512^2 pixels, 1 atom 119 and 73, 4 147 and 103, 6 170 and 153, 8
    // 169 and 168, 16 200 and 324; 256^2, 1 38 and 26, 6 53 and 50, 8 53 and 55.
    const bool whole = atoms->dim == 3 && rule == GT_PSF_EXACT && atoms->n > 6;
    PsfNode2 *nodes = whole ? (PsfNode2 *)((char *)ws + psf_rec_bytes(atoms, geom)) : nullptr;
    if ((rc = psf_prepare(atoms, geom, rule, ws, ws_bytes, gt_psf_forward_workspace(atoms, geom), st,
                          "gt_psf_forward", nodes)))
        return rc;
    GT_CHECK_ARG(R != nullptr, "gt_psf_forward: R is NULL");
    const int n1 = atoms->dim == 3 ? geom->n1 : 1;
    if (atoms->n == 0) {
        const size_t n = (size_t)geom->nA * geom->n0 * n1;
        hipLaunchKernelGGL(psf_fill_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 65535)), dim3(256), 0, st,
                           R, n);
        GT_HIP(hipGetLastError());
        return 0;
    }
    const PsfRec *recs = (const PsfRec *)ws;
    prof_begin(st, GT_K_FORWARD);
    if (whole) {
        const int e0 = ceil_log2((geom->n0 + PF_ROWS - 1) / PF_ROWS), e1 = ceil_log2((n1 + PF_COLS - 1) / PF_COLS);
        GT_CHECK_ARG(((unsigned long long)geom->nA << (e0 + e1)) < (1ull << 31), "gt_psf_forward: too many tiles");
        hipLaunchKernelGGL(psf_project_kernel, dim3((unsigned)((unsigned long long)geom->nA << (e0 + e1))),
                           dim3(PF_WAVES * 64), 0, st, recs, (const PsfNode2 *)nodes, atoms->n, geom->nA, geom->n0, n1,
                           geom->p0, geom->p1, R, e0, e1);
    } else if (atoms->dim == 3) {
        const int e0 = ceil_log2((geom->n0 + 15) / 16), e1 = ceil_log2((n1 + 15) / 16);
        GT_CHECK_ARG(((unsigned long long)geom->nA << (e0 + e1)) < (1ull << 31), "gt_psf_forward: too many tiles");
        const dim3 grid((unsigned)((unsigned long long)geom->nA << (e0 + e1)));
        if (rule == GT_PSF_EXACT)
            hipLaunchKernelGGL((psf_forward_kernel<2, GT_PSF_EXACT>), grid, dim3(256), 0, st, recs, atoms->n, geom->nA,
                               geom->n0, n1, geom->p0, geom->p1, R, e0, e1);
        else
            hipLaunchKernelGGL((psf_forward_kernel<2, GT_PSF_SAMPLED>), grid, dim3(256), 0, st, recs, atoms->n, geom->nA,
                               geom->n0, n1, geom->p0, geom->p1, R, e0, e1);
    } else {
        const dim3 grid((unsigned)((geom->n0 + 255) / 256), (unsigned)geom->nA);
        if (rule == GT_PSF_SAMPLED)
            hipLaunchKernelGGL((psf_forward_kernel<1, GT_PSF_SAMPLED>), grid, dim3(256), 0, st, recs, atoms->n,
                               geom->nA, geom->n0, 1, geom->p0, geom->p0, R, 0, 0);
        else
            hipLaunchKernelGGL((psf_forward_kernel<1, GT_PSF_EXACT>), grid, dim3(256), 0, st, recs, atoms->n, geom->nA,
                               geom->n0, 1, geom->p0, geom->p0, R, 0, 0);
    }
    prof_end(st, GT_K_FORWARD);
    GT_HIP(hipGetLastError());
    return 0;
}

extern "C" int gt_psf_forward(const gt_atoms *atoms, const gt_geom *geom, float *R, void *ws, size_t ws_bytes,
                              void *stream)
{
    return gt_psf_forward_rule(atoms, geom, GT_PSF_EXACT, R, ws, ws_bytes, stream);
}

extern "C" size_t gt_psf_derivs_workspace(const gt_atoms *atoms, const gt_geom *geom)
{
    if (!atoms || !geom) return 0;
    return psf_rec_bytes(atoms, geom) + align_up((size_t)atoms->n * geom->nA * PSF_MS * sizeof(float)) +
           align_up((size_t)geom->nA * sizeof(double));
}

template <int K, int MODE>
static void psf_launch_moments(int rule, dim3 mg, hipStream_t st, const PsfRec *recs, int N, int nA, int n0, int n1,
                               const float *p0, const float *p1, const float *C, int order, float *mom)
{
    if (rule == GT_PSF_SAMPLED)
        hipLaunchKernelGGL((psf_moments_kernel<K, MODE, GT_PSF_SAMPLED>), mg, dim3(256), 0, st, recs, N, nA, n0, n1, p0,
                           p1, C, order, mom);
    else
        hipLaunchKernelGGL((psf_moments_kernel<K, MODE, GT_PSF_EXACT>), mg, dim3(256), 0, st, recs, N, nA, n0, n1, p0,
                           p1, C, order, mom);
}

extern "C" int gt_psf_derivs_rule(const gt_atoms *atoms, const gt_geom *geom, const float *C, int mode, int order,
                                  int rule, double *f, double *g, double *H, void *ws, size_t ws_bytes, void *stream)
{
    int rc;
    hipStream_t st = (hipStream_t)stream;
    if (!atoms || !geom) {
        set_error("gt_psf_derivs: atoms or geometry is NULL");
        return GT_EINVAL;
    }
    GT_CHECK_ARG(mode == GT_MODE_LINEAR || mode == GT_MODE_L2, "gt_psf_derivs: mode must be 0 (linear) or 1 (L2), got %d",
                 mode);
    GT_CHECK_ARG(order == 1 || order == 2, "gt_psf_derivs: order must be 1 or 2, got %d", order);
    GT_CHECK_ARG(C != nullptr || atoms->n == 0, "gt_psf_derivs: C is NULL");
    GT_CHECK_ARG(g != nullptr || atoms->n == 0, "gt_psf_derivs: g is NULL");
    if ((rc = psf_prepare(atoms, geom, rule, ws, ws_bytes, gt_psf_derivs_workspace(atoms, geom), st,
                          "gt_psf_derivs")))
        return rc;
    if (atoms->n == 0) return 0;
    char *w = (char *)ws;
    const PsfRec *recs = (const PsfRec *)w;
    float *mom = (float *)(w + psf_rec_bytes(atoms, geom));
    double *sumC2 = (double *)(w + psf_rec_bytes(atoms, geom) +
                               align_up((size_t)atoms->n * geom->nA * PSF_MS * sizeof(float)));
    const int n1 = atoms->dim == 3 ? geom->n1 : 1;
    const long pairs = (long)atoms->n * geom->nA;
    const dim3 mg((unsigned)((pairs + 3) / 4));
    if (mode == GT_MODE_L2)
        hipLaunchKernelGGL(psf_sumsq_kernel, dim3(geom->nA), dim3(256), 0, st, C, (long)geom->n0 * n1, sumC2);
    prof_begin(st, GT_K_MOMENTS);
    if (atoms->dim == 3) {
        if (mode == GT_MODE_L2)
            psf_launch_moments<2, GT_MODE_L2>(rule, mg, st, recs, atoms->n, geom->nA, geom->n0, n1, geom->p0, geom->p1,
                                              C, order, mom);
        else
            psf_launch_moments<2, GT_MODE_LINEAR>(rule, mg, st, recs, atoms->n, geom->nA, geom->n0, n1, geom->p0,
                                                  geom->p1, C, order, mom);
    } else {
        if (mode == GT_MODE_L2)
            psf_launch_moments<1, GT_MODE_L2>(rule, mg, st, recs, atoms->n, geom->nA, geom->n0, 1, geom->p0, geom->p0,
                                              C, order, mom);
        else
            psf_launch_moments<1, GT_MODE_LINEAR>(rule, mg, st, recs, atoms->n, geom->nA, geom->n0, 1, geom->p0,
                                                  geom->p0, C, order, mom);
    }
    prof_end(st, GT_K_MOMENTS);
    prof_begin(st, GT_K_FINISH);
    const int wh = order > 1;
    if (atoms->dim == 3) {
        if (mode == GT_MODE_L2)
            hipLaunchKernelGGL((psf_finish_kernel<3, GT_MODE_L2>), dim3(atoms->n), dim3(64), 0, st, *atoms, *geom,
                               recs, mom, sumC2, wh, f, g, H);
        else
            hipLaunchKernelGGL((psf_finish_kernel<3, GT_MODE_LINEAR>), dim3(atoms->n), dim3(64), 0, st, *atoms,
                               *geom, recs, mom, sumC2, wh, f, g, H);
    } else {
        if (mode == GT_MODE_L2)
            hipLaunchKernelGGL((psf_finish_kernel<2, GT_MODE_L2>), dim3(atoms->n), dim3(64), 0, st, *atoms, *geom,
                               recs, mom, sumC2, wh, f, g, H);
        else
            hipLaunchKernelGGL((psf_finish_kernel<2, GT_MODE_LINEAR>), dim3(atoms->n), dim3(64), 0, st, *atoms,
                               *geom, recs, mom, sumC2, wh, f, g, H);
    }
    prof_end(st, GT_K_FINISH);
    GT_HIP(hipGetLastError());
    return 0;
}

extern "C" int gt_psf_derivs(const gt_atoms *atoms, const gt_geom *geom, const float *C, int mode, int order,
                             double *f, double *g, double *H, void *ws, size_t ws_bytes, void *stream)
{
    return gt_psf_derivs_rule(atoms, geom, C, mode, order, GT_PSF_EXACT, f, g, H, ws, ws_bytes, stream);
}

extern "C" size_t gt_psf_volume_workspace(const gt_atoms *atoms, const gt_vol *vol)
{
    (void)vol;
    if (!atoms) return 0;
    return align_up((size_t)atoms->n * sizeof(PsfVolRec)) +
           (atoms->dim == 3 ? align_up((size_t)atoms->n * sizeof(PsfNode3)) : 0);
}

extern "C" int gt_psf_volume_rule(const gt_atoms *atoms, const gt_vol *vol, int rule, float *u, void *ws,
                                  size_t ws_bytes, void *stream)
{
    int rc;
    if ((rc = check_atoms(atoms))) return rc;
    GT_CHECK_ARG(rule == GT_PSF_EXACT || rule == GT_PSF_SAMPLED,
                 "gt_psf_volume: rule must be %d (voxel integral) or %d (the reference's samples), got %d",
                 GT_PSF_EXACT, GT_PSF_SAMPLED, rule);
    GT_CHECK_ARG(vol != nullptr && vol->dim == atoms->dim, "gt_psf_volume: volume dimension must match the atoms");
    GT_CHECK_ARG(vol->m0 >= 1 && vol->m1 >= 1 && vol->m2 >= 1, "gt_psf_volume: grid sizes must be >= 1");
    GT_CHECK_ARG(vol->dim == 3 || vol->m2 == 1, "gt_psf_volume: 2D volumes have m2 == 1");
    GT_CHECK_ARG(vol->sorted == 1, "gt_psf_volume: the coordinate vectors must ascend (uniform voxels)");
    GT_CHECK_ARG(vol->y0 && vol->y1 && (vol->dim == 2 || vol->y2), "gt_psf_volume: coordinate vectors missing");
    GT_CHECK_ARG(u != nullptr, "gt_psf_volume: u is NULL");
    const size_t need = gt_psf_volume_workspace(atoms, vol);
    if (need > ws_bytes || (need > 0 && ws == nullptr)) {
        set_error("gt_psf_volume: workspace of %zu bytes given, %zu needed", ws_bytes, need);
        return GT_EWORKSPACE;
    }
    GT_CHECK_ARG(((uintptr_t)ws & 63) == 0, "gt_psf_volume: workspace must be 64-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    GT_CHECK_ARG(vol->m0 >= 2 && vol->m1 >= 2 && (vol->dim == 2 || vol->m2 >= 2),
                 "gt_psf_volume: voxel integration needs at least two coordinates per axis");
    const size_t nout = (size_t)vol->m0 * vol->m1 * vol->m2;
    if (atoms->n == 0) {
        hipLaunchKernelGGL(psf_fill_kernel, dim3((unsigned)std::min<size_t>((nout + 255) / 256, 65535)), dim3(256), 0,
                           st, u, nout);
        GT_HIP(hipGetLastError());
        return 0;
    }
    PsfVolRec *recs = (PsfVolRec *)ws;
    const dim3 sg((unsigned)((atoms->n + 255) / 256));
    // bricks numbered by Morton index over 2^e0 x 2^e1 x 2^e2 centre-out ranks
    int nb[3];
    const bool whole = vol->dim == 3 && rule == GT_PSF_EXACT;
    PsfNode3 *nodes = (PsfNode3 *)((char *)ws + align_up((size_t)atoms->n * sizeof(PsfVolRec)));
    if (whole) {
        hipLaunchKernelGGL(psf_voxel_setup_kernel, dim3((unsigned)atoms->n), dim3(64), 0, st, *atoms, *vol, recs, nodes);
        nb[0] = (vol->m0 + 3) / 4, nb[1] = (vol->m1 + 4 * PX_ROW - 1) / (4 * PX_ROW), nb[2] = (vol->m2 + 7) / 8;
    } else if (vol->dim == 3) {
        hipLaunchKernelGGL(psf_vol_setup_kernel<3>, sg, dim3(256), 0, st, *atoms, *vol, recs, rule);
        nb[0] = (vol->m0 + 3) / 4, nb[1] = (vol->m1 + 7) / 8, nb[2] = (vol->m2 + 7) / 8;
    } else {
        hipLaunchKernelGGL(psf_vol_setup_kernel<2>, sg, dim3(256), 0, st, *atoms, *vol, recs, rule);
        nb[0] = (vol->m0 + 15) / 16, nb[1] = (vol->m1 + 15) / 16, nb[2] = 1;
    }
    const int e[3] = {ceil_log2(nb[0]), ceil_log2(nb[1]), ceil_log2(nb[2])};
    GT_CHECK_ARG(e[0] + e[1] + e[2] <= 30, "gt_psf_volume: grid too large");
    const unsigned blocks = 1u << (e[0] + e[1] + e[2]);
    prof_begin(st, GT_K_VOLUME);
    if (whole) {
        hipLaunchKernelGGL(psf_voxels_kernel, dim3(blocks), dim3(PX_THREADS), 0, st, recs, (const PsfNode3 *)nodes,
                           atoms->n, *vol, u, e[0], e[1], e[2]);
    } else if (vol->dim == 3) {
        hipLaunchKernelGGL((psf_volume_kernel<3, GT_PSF_SAMPLED>), dim3(blocks), dim3(PV_THREADS), 0, st, recs,
                           atoms->n, *vol, u, e[0], e[1], e[2]);
    } else {
        if (rule == GT_PSF_SAMPLED)
            hipLaunchKernelGGL((psf_volume_kernel<2, GT_PSF_SAMPLED>), dim3(blocks), dim3(PV_THREADS), 0, st, recs,
                               atoms->n, *vol, u, e[0], e[1], e[2]);
        else
            hipLaunchKernelGGL((psf_volume_kernel<2, GT_PSF_EXACT>), dim3(blocks), dim3(PV_THREADS), 0, st, recs,
                               atoms->n, *vol, u, e[0], e[1], e[2]);
    }
    prof_end(st, GT_K_VOLUME);
    GT_HIP(hipGetLastError());
    return 0;
}

extern "C" int gt_psf_volume(const gt_atoms *atoms, const gt_vol *vol, float *u, void *ws, size_t ws_bytes,
                             void *stream)
{
    return gt_psf_volume_rule(atoms, vol, GT_PSF_EXACT, u, ws, ws_bytes, stream);
}
