// gt_common.h -- shared host/device helpers of the HIP library.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gausstomo.h"
#include "gt_pair.h"

namespace gt {

// Thread-local last error message (gt_last_error).
void set_error(const char *fmt, ...);

// Optional per-launch event timing (gt_profile_enable / gt_profile_read).
void prof_begin(hipStream_t st, int id);
void prof_end(hipStream_t st, int id);
// The same for a launch timed by its own dispatch: events a, b for
// hipExtLaunchKernelGGL, which records the kernel's start and end in the
// kernel's packet (no packets between launches); false, and both null, when
// the kernel id is not being timed.
bool prof_ext_begin(int id, hipEvent_t *a, hipEvent_t *b);
void prof_ext_end(int id, hipEvent_t a, hipEvent_t b);

template <typename F, typename... Args>
inline void launch_timed(int id, F kernel, dim3 grid, dim3 block, unsigned shmem, hipStream_t st, Args... args)
{
    hipEvent_t a = nullptr, b = nullptr;
    const bool timed = prof_ext_begin(id, &a, &b);
    hipExtLaunchKernelGGL(kernel, grid, block, shmem, st, a, b, 0u, args...);
    if (timed) prof_ext_end(id, a, b);
}

#define GT_CHECK_ARG(cond, ...)          \
    do {                                 \
        if (!(cond)) {                   \
            ::gt::set_error(__VA_ARGS__); \
            return GT_EINVAL;            \
        }                                \
    } while (0)

#define GT_HIP(call)                                                          \
    do {                                                                      \
        hipError_t e_ = (call);                                               \
        if (e_ != hipSuccess) {                                               \
            ::gt::set_error("%s failed: %s", #call, hipGetErrorString(e_));  \
            return GT_EHIP;                                                   \
        }                                                                     \
    } while (0)

constexpr size_t ALIGN = 256;
__host__ __device__ inline size_t align_up(size_t v) { return (v + ALIGN - 1) / ALIGN * ALIGN; }

// Centre-first numbering of tile grids.  Tiles at the centre of a detector,
// volume or k grid meet the most atoms; kernels whose grids hold more blocks
// than fit at once number their blocks so that block b takes the tile whose
// centre-out ranks (t0, t1, t2) have Morton index b (bits dealt to the axes in
// turn while each has bits left; grid of 2^e0 x 2^e1 x 2^e2 ranks).  Ranks
// beyond an axis' tile count are empty blocks.

// t-th index of 0..R-1 from the centre outwards: c, c+1, c-1, c+2, ... with c = (R-1)/2
__device__ inline int centre_out(int t, int R)
{
    const int c = (R - 1) >> 1;
    return (t & 1) ? c + ((t + 1) >> 1) : c - (t >> 1);
}

// Place in a Morton index of bit l of the ranks laid side by side, t[0] | t[1] <<
// e[0] | t[2] << (e[0] + e[1]): the bits dealt before it
__host__ __device__ inline int morton_place(int l, const int *e)
{
    const int d = (l >= e[0]) + (l >= e[0] + e[1]);
    const int b = l - (d > 0 ? e[0] : 0) - (d > 1 ? e[1] : 0);
    const int b0 = b + (d > 0), b1 = b + (d > 1);
    return (b0 < e[0] ? b0 : e[0]) + (b1 < e[1] ? b1 : e[1]) + (b < e[2] ? b : e[2]);
}

// Morton index m -> ranks t[0..2] of a 2^e[0] x 2^e[1] x 2^e[2] grid (at most 31
// bits), by a whole wave: a lane per bit, collected by a ballot.  (A loop over the
// bits is 315 scalar instructions for 21 bits, and a CU has one scalar unit: 2 ns
// for every block of four waves, empty ones included, where the launch itself
// takes less; a 384^3 render of one atom took 546 us.)
__device__ inline void morton_ranks(unsigned m, const int *e, int *t)
{
    const int l = (int)(threadIdx.x & 63u);
    const bool bit = l < e[0] + e[1] + e[2] && ((m >> morton_place(l, e)) & 1u) != 0u;
    const unsigned all = (unsigned)__ballot(bit);
    t[0] = (int)(all & ((1u << e[0]) - 1u));
    t[1] = (int)((all >> e[0]) & ((1u << e[1]) - 1u));
    t[2] = (int)((all >> e[0] >> e[1]) & ((1u << e[2]) - 1u));
}

// The same by a loop over the bits, for kernels whose blocks run for milliseconds: there
// the decode's time is nothing, and the sampled point-spread rule, whose waves it sets
// apart at the start, is faster after it (1000 atoms on 64^3 18.4 against 19.1 ms, on
// 61 x 128^2 pixels 6.21 against 6.29 ms).
__device__ inline void morton_ranks_loop(unsigned m, const int *e, int *t)
{
    t[0] = t[1] = t[2] = 0;
    for (int bit = 0; m != 0u && bit < 31; bit++)
#pragma unroll
        for (int d = 0; d < 3; d++)
            if (bit < e[d]) {
                t[d] |= (int)(m & 1u) << bit;
                m >>= 1;
            }
}

// The even bits of v side by side
__host__ __device__ inline unsigned even_bits(unsigned v)
{
    v &= 0x55555555u;
    v = (v | (v >> 1)) & 0x33333333u;
    v = (v | (v >> 2)) & 0x0f0f0f0fu;
    v = (v | (v >> 4)) & 0x00ff00ffu;
    return (v | (v >> 8)) & 0x0000ffffu;
}

// The same for two axes: bits in turn up to the shorter axis' last, the rest to the
// longer one; some 35 scalar instructions (a lane per bit costs the point-spread
// projection, whose registers are full, 4% of its time).
__host__ __device__ inline void morton_ranks2(unsigned m, int e0, int e1, int *t)
{
    const int c = e0 < e1 ? e0 : e1;
    const unsigned low = m & ((1u << (2 * c)) - 1u), rest = m >> (2 * c) << c;
    t[0] = (int)(even_bits(low) | (e0 > e1 ? rest : 0u));
    t[1] = (int)(even_bits(low >> 1) | (e0 > e1 ? 0u : rest));
}

// smallest e with 2^e >= v (v >= 1)
inline int ceil_log2(long v)
{
    int e = 0;
    while ((1L << e) < v) e++;
    return e;
}

// T in global memory.  Loads and stores through a gmem<T> * are global_*
// instructions (scalar base plus 32-bit offset, counted by the vector-memory
// counter only).  Through a plain pointer the compiler cannot trace to a
// kernel argument (one read from a struct in memory) they would be flat
// ones: 64-bit address arithmetic per access, and counted by the LDS counter
// too, so that every wait for an LDS read also waits for them.
template <typename T> using gmem = __attribute__((address_space(1))) T;

// Raw buffer resource over a read-only array (gfx9 word 3; no bounds beyond
// 32-bit offsets): buffer loads add a per-lane offset, a wave-uniform scalar
// offset and the base in the load itself, so a group of loads whose
// addresses differ by uniform amounts needs one vector offset.
__device__ inline __amdgpu_buffer_rsrc_t buffer_rsrc(const void *base)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, -1, 0x00020000);
}
__device__ inline float buffer_load_f32(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

__device__ inline void buffer_store_f32(__amdgpu_buffer_rsrc_t r, float v, unsigned voff, unsigned soff)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, voff, soff, 0);
}

// A pointer that is the same in every lane, held in scalar registers whatever
// the compiler knows of where it came from: a buffer resource made from one it
// holds per lane costs every load a loop over the lanes' distinct bases.
template <typename T> __device__ inline T *uniform_ptr(T *p)
{
    const unsigned long long v = (unsigned long long)(uintptr_t)p;
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
    return (T *)(uintptr_t)(((unsigned long long)hi << 32) | lo);
}

// Read-only array of an earlier kernel, read at wave-uniform indices through
// the scalar cache: the values land in scalar registers, which cost no LDS
// bandwidth and no vector registers (a wave-uniform index is made with
// readfirstlane).
template <typename T> using smem = __attribute__((address_space(4))) const T;
template <typename T> __device__ inline smem<T> *scalar_ptr(const T *p) { return (smem<T> *)(uintptr_t)p; }

// Per-wave record lists of one staging round, in record order.  Thread t of
// the block holds the NL-bit mask of the lists that record base + t belongs
// to; list w receives the threads t of its members in ascending order (the
// caller adds base).  NW waves, NL lists; wl[w]: NW * 64 entries; cnt: NL x NW;
// wlen[w]: the length of list w.  Two block barriers; the caller puts one
// more before the next round.
template <int NW, int NL>
__device__ inline void wave_lists(unsigned mask, unsigned short (*wl)[NW * 64], int (*cnt)[NW], int *wlen)
{
    const int lane = threadIdx.x & 63, hw = threadIdx.x >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
    unsigned long long mw[NL];
#pragma unroll
    for (int w = 0; w < NL; w++) {
        mw[w] = __ballot((mask >> w) & 1u);
        if (lane == 0) cnt[w][hw] = __popcll(mw[w]);
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NL; w++) {
        int o = 0, t = 0;
#pragma unroll
        for (int h = 0; h < NW; h++) {
            const int c = cnt[w][h];
            if (h < hw) o += c;
            t += c;
        }
        if ((mask >> w) & 1u) wl[w][o + __popcll(mw[w] & below)] = (unsigned short)threadIdx.x;
        if (threadIdx.x == 0) wlen[w] = t;
    }
    __syncthreads();
}

// LDS written by some lanes of a wave, then read by others: order the wave's
// LDS traffic (the lanes of a wave execute together).
__device__ inline void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The value of lane K of each row of 16 lanes, in the whole row
template <int K> __device__ inline float row_bcast(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + K, 0xf, 0xf, true));
}

// sin(2 pi t) and cos(2 pi t) of a phase t in turns, |t| <= 256: the
// hardware sine and cosine, whose argument is in turns (quarter-rate, like
// exp2); measured maximum absolute error 1.25e-7 for |t| <= 1.5 on gfx950.
__device__ inline void ft_sincos_turns(float t, float &sn, float &cs)
{
    sn = __builtin_amdgcn_sinf(t);
    cs = __builtin_amdgcn_cosf(t);
}

// The same by polynomials, t = q / 4 + r with |r| <= 1/8: sin(2 pi r) / r and
// cos(2 pi r) are interpolated in r^2 at the Chebyshev points (4 and 5 terms);
// maximum absolute error 8.2e-8 and 5.8e-8, rms 2e-8.
__device__ inline void ft_sincos_quarter(int q, float r, float &sn, float &cs)
{
    const float z = r * r;
    const float s = r * fmaf(fmaf(fmaf(-75.39643085838416f, z, 81.59244143217468f), z, -41.341662093897966f), z,
                             6.2831852875017855f);
    const float c = fmaf(fmaf(fmaf(fmaf(59.21609823587779f, z, -85.44273312246247f), z, 64.9393151998861f), z,
                              -19.739208647687875f), z, 1.0f);
    const bool odd = (q & 1) != 0;
    const unsigned ss = ((unsigned)q & 2u) << 30, sc = ((unsigned)(q + 1) & 2u) << 30;
    sn = __uint_as_float(__float_as_uint(odd ? c : s) ^ ss);
    cs = __uint_as_float(__float_as_uint(odd ? s : c) ^ sc);
}

// A phase in FP64, of any size.
__device__ inline void ft_sincos_fine(double t, float &sn, float &cs)
{
    const double q = rint(4.0 * t);
    ft_sincos_quarter((int)(q - 4.0 * rint(0.25 * q)), (float)fma(-0.25, q, t), sn, cs);
}

// A phase in FP32, reduced to the nearest quarter turn exactly: about 24
// operations in all, for phases that many samples share.
__device__ inline void ft_sincos_shared(float t, float &sn, float &cs)
{
    const float n = rintf(4.0f * t);
    ft_sincos_quarter((int)n, fmaf(-0.25f, n, t), sn, cs);
}

int check_atoms(const gt_atoms *a);
int check_geom(const gt_geom *g, int dim);

// Atom j into a PairGeom (iso: U = rho * Id).
template <int D> __device__ __host__ inline void load_atom(const gt_atoms &A, int j, PairGeom<D> &g)
{
    constexpr int NR = Dims<D>::NR;
    for (int i = 0; i < 3; i++)
        for (int k = 0; k < 3; k++) g.U[i][k] = 0.0;
    if (A.iso) {
        double rho = A.r[j];
        for (int i = 0; i < D; i++) g.U[i][i] = rho;
    } else {
        // unrolled: constant indices keep U in registers
#pragma unroll
        for (int k = 0; k < NR; k++) g.U[slot_row(D, k)][slot_col(D, k)] = A.r[(size_t)j * NR + k];
    }
    for (int i = 0; i < 3; i++) g.x[i] = (i < D) ? (double)A.x[(size_t)j * D + i] : 0.0;
    g.I = A.I[j];
}

// Orientation a into a PairGeom: T and the detector columns G.
template <int D> __device__ __host__ inline void load_angle(const gt_geom &G, int a, PairGeom<D> &g)
{
    for (int i = 0; i < 3; i++) {
        g.T[i] = 0.0;
        g.G[0][i] = 0.0;
        g.G[1][i] = 0.0;
    }
    const int L = G.lenT;
    // constant indices (a loop to the run-time L would index T and G[0]
    // dynamically and put them in scratch memory)
#pragma unroll
    for (int i = 0; i < 3; i++) {
        if (i < L) {
            g.T[i] = G.T[(size_t)a * L + i];
            g.G[0][i] = G.w0[(size_t)a * L + i];
        }
    }
    if (D == 3) {
        if (L == 3) {
            for (int i = 0; i < 3; i++) g.G[1][i] = G.w1[(size_t)a * 3 + i];
        } else {
            g.G[1][2] = 1.0;  // 2.5D: y = (p0 w0[0], p0 w0[1], p1), NewtonBases.py:684-688
        }
    }
}

// Wave64 helpers.
__device__ inline int lane_id() { return threadIdx.x & 63; }

}  // namespace gt
