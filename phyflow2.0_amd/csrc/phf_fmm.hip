// phf_fmm.hip -- 2-D FMM for the Oseen-smoothed Biot-Savart sum on gfx950.
//
// Replaces the reference's fmm2dInteract (fmm.cpp:88-304) and its CUDA
// pipeline (cudaeval.cu, cudasort.cu).  Computes, for every target z,
//     q(z) = qr + i qi = -sum_j w_j K(|z - z_j|^2) / (z - z_j)
// with the Oseen factor K(r2) = -expm1(-shape r2) scale for r2 < cutoff^2 and
// 1 beyond (fmm.cpp:1166-1179, cudaevalkernels.h:61-71), so the caller's
// velocity is (-qi/2pi, -qr/2pi) exactly as for the reference.
//
// Tree: uniform quad-tree of depth L over the Morton-sorted points
// (phf_tree.hip).  Far-field interactions use the standard 2-D complex
// expansions about box centres, scaled by the box side r:
//   multipole  A_k = sum_j w_j ((z_j - c)/r)^k                   (P2M)
//   local      phi(z) = sum_m B_m ((z - d)/r)^m                  (L2P)
//   M2M        A'_m = sum_{k<=m} C(m,k) 2^-k delta^(m-k) A_k      delta = (c1-c0)/R
//   M2L        B_m = (1/r) (-1)^m u^(m+1) sum_k C(k+m,k) u^k A_k  u = r/(c-d)
//   L2L        B'_m = sum_{j>=m} C(j,m) delta^(j-m) 2^-m B_j
// Near set of a box: boxes within `ws` boxes in x and y, plus every box
// whose gap is below the smoothing cutoff (the expansions represent the
// unsmoothed 1/z kernel, which equals the Oseen kernel only beyond the
// cutoff: the reference's THETACUTOFFCHECK, fmm.cpp:1812-1815).  The
// interaction list of a box is the children of its parent's near set that
// are not in its own near set.  Near pairs at the leaf level are summed
// directly (P2P), fused with the L2P evaluation of the leaf's local
// expansion.
//
// Precision: PHF_PREC_F64 runs every pass in float64.  PHF_PREC_F32C
// stores points as float32 offsets from their leaf centre (formed in
// float64; leaf sides and centre differences are exact in float32 because
// the domain side carries 5 significant bits), runs P2P with compensated
// per-target sums and P2M/M2L/L2P in float32, and keeps the expansions in
// float32; M2M/L2L compute in float64 from and to them.
#include "phf_fmm.hpp"
#include "phf_host.hpp"
#include "phf_fmm_dev.hpp"
#include "phf_p2p_dev.hpp"

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <functional>
#include <memory>
#include <vector>

namespace phf {

__global__ void gather_src_f64(const double *__restrict__ x, const double *__restrict__ y,
                               const double *__restrict__ w, const int32_t *__restrict__ perm,
                               int64_t n, double4 *__restrict__ out)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int32_t j = perm[i];
    out[i] = make_double4(x[j], y[j], w[j], 0.0);
}

__global__ void gather_tgt_f32(const double *__restrict__ x, const double *__restrict__ y,
                               const uint32_t *__restrict__ skeys, int fsh,
                               const int32_t *__restrict__ perm, int64_t n,
                               const double4 *__restrict__ org, double s,
                               float2 *__restrict__ out)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int32_t j = perm[i];
    double cx, cy;
    leaf_center(skeys[i] >> fsh, org->x, org->z, s, cx, cy);
    out[i] = make_float2((float)(x[j] - cx), (float)(y[j] - cy));
}

__global__ void gather_tgt_f64(const double *__restrict__ x, const double *__restrict__ y,
                               const int32_t *__restrict__ perm, int64_t n,
                               double2 *__restrict__ out)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int32_t j = perm[i];
    out[i] = make_double2(x[j], y[j]);
}

// The far field's kernels run beside the near field, whose waves keep the
// vector units busy and which they outlast in small trees: a chain of short
// kernels of few waves each, issued before the near field's (P2M of 1024 leaves
// 54 -> 8 us, M2M 28 -> 9; the evaluation of 65k float64 blobs 246 -> 214 us,
// of 120k float32 ones 179 -> 163; where the near field is the longer, no
// change).
__device__ __forceinline__ void far_priority() { __builtin_amdgcn_s_setprio(3); }

// ---------------------------------------------------------------- P2M ----
// Expansions of four leaves, the children of one box, per workgroup: a wave each,
// or, if none has more than `few` points, all by one wave with sixteen lanes
// each.  A wave takes up to 32 points in two rounds and then spends its time on
// the butterfly, which sixteen lanes have half of; but they are a serial chain of
// a quarter of the points.  The four counts decide, so the sums follow from the
// points alone, and a crowded leaf is not waited for by lanes of small ones.
// float32, order 16, a wave each / by this rule: 300,000 uniform blobs in leaves
// of 18 22.9 / 18.8 us, 1M 31.5 / 28.7; a line at 48 took 9.6 instead of 6.8 us
// for 20,000 float64 blobs.  With one choice for the launch from the mean leaf, a
// thin ring of 20,000 (float64) took 28 us (14 now) or followed its bounding box.
// One leaf with nearly all blobs, float64: 8,628 blobs, order 24, 808 us by
// sixteen lanes, 280 with the table, 202 by a wave.
// inv_s is 1 / s.
template <class T, int NI>
__global__ __launch_bounds__(256) void p2m_kernel(const void *__restrict__ src,
                                                  const int32_t *__restrict__ start, int p1,
                                                  const double4 *__restrict__ org, double s,
                                                  double inv_s,
                                                  typename C2<T>::type *__restrict__ M)
{
    constexpr int32_t few = 32;
    far_priority();
    const int32_t *st = start + 4 * blockIdx.x;
    int32_t s0[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) s0[k] = st[k];
    int32_t most = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) most = max(most, s0[k + 1] - s0[k]);
    const int wv = threadIdx.x >> 6;
    const bool one = most <= few;
    if (one && wv != 0) return;
    const int k = one ? (int)(threadIdx.x >> 4) : wv;
    const uint32_t b = 4 * blockIdx.x + k;
    double cx = 0.0, cy = 0.0;
    if (sizeof(T) == 8) leaf_center(b, org->x, org->z, s, cx, cy);
    typename C2<T>::type *out = M + (int64_t)b * p1;
    const int32_t j0 = k == 0 ? s0[0] : k == 1 ? s0[1] : k == 2 ? s0[2] : s0[3];
    const int32_t j1 = k == 0 ? s0[1] : k == 1 ? s0[2] : k == 2 ? s0[3] : s0[4];
    if (one)
        p2m_leaf<T, NI, 4, false>(src, j0, j1, cx, cy, (T)inv_s, p1, out);
    else
        p2m_leaf<T, NI, 16, false>(src, j0, j1, cx, cy, (T)inv_s, p1, out);
}

// ---------------------------------------------------------- M2M / L2L ----
// Upward pass over up to three levels in one launch: M_m = sum over the four
// children (sum_{k <= m} C(m, k) d^(m-k) rho^k M_k), d the child's centre from
// its parent's and rho = 1/2, both in the parent's side.  d = 2^(-3/2) e^(i
// theta), theta an odd multiple of 45 degrees, so with M'_k = e^(-i theta k)
// M_k the shift is one real matrix for every child of every box,
// S[m][k] = C(m, k) 2^(-3 (m - k) / 2) 2^-k, and its result turns back by
// e^(i theta m): S times the children's real and imaginary parts as columns,
// on v_mfma_f64_16x16x4f64 (lane l holds A[l % 16][4 s + l / 16],
// B[4 s + l / 16][l % 16] and, of the result, row 4 v + l / 16, column
// l % 16; the probe of the layout is the multipole order test).  S stays in
// registers, its zero tiles are left out; eight children are one tile of
// columns, so a wave adds four siblings across its lanes.  One workgroup per
// box of level lev0 takes the levels in turn, in float64 throughout, and keeps
// the boxes between them in LDS.  Empty boxes have zero expansions, so no box
// is skipped.
// (Every level from the finest by complex shifts on the vector units took
// 192 shifts of 6 p1^2 operations for 64 boxes, against 84 of p1^2 matrix
// operations: 262k float64 blobs, order 29, beside the near field 57 us for
// 192 and 45 for 84, and the evaluation 562 -> 515 us, the near field being
// left the vector units; 600k float32 blobs in 16k leaves 431 -> 405.)
struct UpLevels {
    int nlev, lev0, from;
    int64_t off[4];  // coefficient offset (boxes) of each level
    int64_t off_from;
};

typedef double doublex4 __attribute__((ext_vector_type(4)));

// cos and sin of k 45 degrees
__device__ __forceinline__ void eighth_turns(int k, double &c, double &s)
{
    const double h = 0.70710678118654752440;
    const double m = (k & 1) ? h : 1.0;
    const int a = (k + 1) & 7, b = (k - 1) & 7;  // cos > 0 in a = 0..2, sin > 0 in b = 0..2
    c = (k & 3) == 2 ? 0.0 : a < 3 ? m : -m;
    s = (k & 3) == 0 ? 0.0 : b < 3 ? m : -m;
}

// S[m][k] of the shifts, 0 outside 0 <= k <= m < p1
__device__ __forceinline__ double shift_term(const double *__restrict__ pas, int p1, int m, int k)
{
    const int n = m - k;
    if (n < 0 || m >= p1) return 0.0;
    return ldexp(pas[m * p1 + k] * ((n & 1) ? 1.41421356237309504880 : 1.0),
                 -((3 * n + 1) >> 1) - k);
}

// cos and sin of k theta of child q (bit 0: east, bit 1: north)
__device__ __forceinline__ void child_turn(int q, int k, double &c, double &s)
{
    const int turn = (q & 2) ? ((q & 1) ? 1 : 3) : ((q & 1) ? -1 : -3);
    eighth_turns((turn * k) & 7, c, s);
}

template <class T, int MT>
__global__ __launch_bounds__(256) void m2m_kernel(UpLevels u, int p1,
                                                  typename C2<T>::type *__restrict__ M,
                                                  const double *__restrict__ pas)
{
    far_priority();
    constexpr int KS = 4 * MT;
    __shared__ double2 mid[(16 + 4) * 16 * MT];  // the boxes one and two levels up
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int col = lane & 15, kq = lane >> 4, comp = col & 1;
    double a[MT][KS];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int s = 0; s < 4 * (t + 1); ++s) a[t][s] = shift_term(pas, p1, 16 * t + col, 4 * s + kq);
    // e^(i theta kq) of the lane's column, its sine signed for the component
    // that the lane holds; four powers on it turns by 180 degrees
    const int q = (col >> 1) & 3;
    double cs, sn;
    child_turn(q, kq, cs, sn);
    sn = comp ? sn : -sn;
    for (int D = 1; D <= u.nlev; ++D) {
        const int nch = 1 << (2 * (u.nlev - D + 1));  // children in this workgroup
        const int64_t box0 = (int64_t)blockIdx.x << (2 * (u.nlev - D));  // first parent
        const typename C2<T>::type *in = M + (u.off_from + 4 * box0) * p1;
        const double2 *lin = mid + (D == 3 ? 16 * 16 * MT : 0);
        double2 *lout = mid + (D == 2 ? 16 * 16 * MT : 0);
        for (int g = wv; 8 * g < nch; g += 4) {
            const int c = 8 * g + (col >> 1);
            const bool on = c < nch;
            doublex4 acc[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t] = doublex4{0.0, 0.0, 0.0, 0.0};
            double b[KS];
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int k = 4 * s + kq;
                double v = 0.0;
                if (on && k < p1)
                    v = D == 1 ? (double)reinterpret_cast<const T *>(in + (int64_t)c * p1 + k)[comp]
                               : reinterpret_cast<const double *>(lin + c * 16 * MT + k)[comp];
                b[s] = v;
            }
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const double o = __shfl_xor(b[s], 1);
                b[s] = (s & 1) ? -(b[s] * cs) + o * sn : b[s] * cs - o * sn;
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    if (s < 4 * (t + 1))
                        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t][s], b[s], acc[t], 0, 0,
                                                                      0);
            }
            typename C2<T>::type *out = M + (u.off[u.nlev - D] + box0 + (c >> 2)) * p1;
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int m = 16 * t + 4 * v + kq;
                    const double o = __shfl_xor(acc[t][v], 1);
                    double r = (v & 1) ? -(acc[t][v] * cs) - o * sn : acc[t][v] * cs + o * sn;
                    r += __shfl_xor(r, 2);
                    r += __shfl_xor(r, 4);
                    if (on && q == 0 && m < p1) {
                        reinterpret_cast<T *>(out + m)[comp] = (T)r;
                        if (D < u.nlev)
                            reinterpret_cast<double *>(lout + (c >> 2) * 16 * MT + m)[comp] = r;
                    }
                }
        }
        __syncthreads();
    }
}

// Downward pass over up to three levels in one launch: B_m of a child gains
// rho^m sum_{k >= m} C(k, m) d^(k-m) B_k of its parent, m2m_kernel's turns and
// the transpose of its matrix.  One workgroup per box of level lev0 takes the
// levels below it in turn; only the last one's expansions (the next launch's
// parents, or the leaves) are written.  (Each leaf from all its ancestors on
// the vector units: 92 us beside the near field of 262k float64 blobs, order
// 29, against 54, the evaluation 515 -> 477.)
struct DownLevels {
    int nlev, lev0;
    int64_t off[4];  // coefficient offset (boxes) of levels lev0 ..
};

template <class T, int MT>
__global__ __launch_bounds__(256) void l2l_kernel(DownLevels dl, int p1,
                                                  typename C2<T>::type *__restrict__ B,
                                                  const double *__restrict__ pas)
{
    far_priority();
    constexpr int KS = 4 * MT;
    __shared__ double2 mid[(4 + 16) * 16 * MT];  // the boxes one and two levels down
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int col = lane & 15, kq = lane >> 4, comp = col & 1;
    double a[MT][KS];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int s = 4 * t; s < KS; ++s) a[t][s] = shift_term(pas, p1, 4 * s + kq, 16 * t + col);
    const int q = (col >> 1) & 3;
    double cs, sn;
    child_turn(q, kq, cs, sn);
    sn = comp ? sn : -sn;
    for (int D = 1; D <= dl.nlev; ++D) {
        const int nch = 1 << (2 * D);  // children in this workgroup
        const double2 *lin = mid + (D == 3 ? 4 * 16 * MT : 0);
        double2 *lout = mid + (D == 2 ? 4 * 16 * MT : 0);
        for (int g = wv; 8 * g < nch; g += 4) {
            const int c = 8 * g + (col >> 1);
            const bool on = c < nch;
            typename C2<T>::type *out =
                B + (dl.off[D] + ((int64_t)blockIdx.x << (2 * D)) + (on ? c : 0)) * p1;
            double b[KS], own[MT][4];
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int k = 4 * s + kq;
                double v = 0.0;
                if (on && k < p1)
                    v = D == 1 ? (double)reinterpret_cast<const T *>(
                                     B + (dl.off[0] + blockIdx.x) * p1 + k)[comp]
                               : reinterpret_cast<const double *>(lin + (c >> 2) * 16 * MT +
                                                                  k)[comp];
                b[s] = v;
            }
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int m = 16 * t + 4 * v + kq;
                    own[t][v] =
                        on && m < p1 ? (double)reinterpret_cast<const T *>(out + m)[comp] : 0.0;
                }
            doublex4 acc[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const double o = __shfl_xor(b[s], 1);
                b[s] = (s & 1) ? -(b[s] * cs) - o * sn : b[s] * cs + o * sn;
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    if (s >= 4 * t)
                        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t][s], b[s], acc[t], 0, 0,
                                                                      0);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int m = 16 * t + 4 * v + kq;
                    const double o = __shfl_xor(acc[t][v], 1);
                    const double r = own[t][v] + ((v & 1) ? -(acc[t][v] * cs) + o * sn
                                                          : acc[t][v] * cs - o * sn);
                    if (!on || m >= p1) continue;
                    if (D < dl.nlev)
                        reinterpret_cast<double *>(lout + c * 16 * MT + m)[comp] = r;
                    else
                        reinterpret_cast<T *>(out + m)[comp] = (T)r;
                }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- M2L ----
// Levels of one M2L launch: every level >= 2 runs in the same grid (they
// are independent once the upward pass is done), so the short serial link
// chains of the coarse levels overlap with the work of the finest.
constexpr int kM2LMaxLev = 12;
struct M2LLevels {
    int nlev, lev0;
    int64_t blk[kM2LMaxLev + 1];   // first block of each level (grid.x)
    int64_t coff[kM2LMaxLev];      // box offset of the level in the M / B arrays
    int il_base[kM2LMaxLev];       // index of the level's 5 parity offsets
    int il_max[kM2LMaxLev];        // longest interaction list of the level
    int shift[kM2LMaxLev];         // 2 (L - l)
    double inv_r[kM2LMaxLev];      // 1 / box side
};

__device__ __forceinline__ int m2l_level_of(const M2LLevels &lv)
{
    int li = 0;
    while (li + 1 < lv.nlev && (int64_t)blockIdx.x >= lv.blk[li + 1]) ++li;
    return li;
}

// One wave holds G = 64/p1 target boxes of one level; lane (g, m) owns
// coefficient m of box g.  Per link the group forms A'_k = u^k A_k in LDS,
// each lane contracts with its binomial row C(k+m, k) (registers), and
// accumulates (-1)^m u^(m+1) S_m.  Boxes are visited parity-major so the
// groups of a wave mostly share one interaction list.
template <class T, int P1>
__global__ __launch_bounds__(64) void m2l_kernel(
    M2LLevels lv, int p1, const typename C2<T>::type *__restrict__ M,
    typename C2<T>::type *__restrict__ B, const int32_t *__restrict__ start_s,
    const int32_t *__restrict__ start_t, const int2 *__restrict__ il_tau,
    const int32_t *__restrict__ il_offs, const typename C2<T>::type *__restrict__ U, int R,
    const T *__restrict__ binom /* [p1][p1] */)
{
    far_priority();
    using V = typename C2<T>::type;
    __shared__ V Ap[64];
    const int li = m2l_level_of(lv);
    const int l = lv.lev0 + li;
    const V *Ml = M + lv.coff[li] * p1;
    V *Bl = B + lv.coff[li] * p1;
    const int shift = lv.shift[li];
    const int32_t *il_off = il_offs + lv.il_base[li];
    const int il_max = lv.il_max[li];
    const T inv_r = (T)lv.inv_r[li];
    const int lane = threadIdx.x;
    const int G = 64 / p1;
    const int g = lane / p1, m = lane - g * p1;
    const int n = 1 << l, half = n >> 1;
    const int64_t nbox = (int64_t)n * n;
    const int64_t slot = ((int64_t)blockIdx.x - lv.blk[li]) * G + g;
    bool active = g < G && slot < nbox;
    int bx = 0, by = 0, par = 0;
    uint32_t box = 0;
    if (active) {
        const int64_t per = nbox / 4;  // boxes per parity class
        par = (int)(slot / per);
        const int64_t loc = slot - (int64_t)par * per;
        bx = 2 * (int)(loc % half) + (par & 1);
        by = 2 * (int)(loc / half) + (par >> 1);
        box = morton2((uint32_t)bx, (uint32_t)by);
        active = box_count(start_t, box, shift) > 0;
    }
    T crow[P1];
#pragma unroll
    for (int k = 0; k < P1; ++k) crow[k] = (k < p1 && m < p1) ? binom[m * p1 + k] : (T)0;
    const int W2 = 2 * R + 1;
    const int t0 = active ? il_off[par] : 0;
    const int tn = active ? il_off[par + 1] - t0 : 0;
    T ar = 0, ai = 0;
    const T sgn = (m & 1) ? (T)-1 : (T)1;
    for (int t = 0; t < il_max; ++t) {
        bool ok = t < tn;
        int2 o = make_int2(0, 0);
        uint32_t sb = 0;
        if (ok) {
            o = il_tau[t0 + t];
            const int sx = bx + o.x, sy = by + o.y;
            ok = sx >= 0 && sy >= 0 && sx < n && sy < n;
            if (ok) {
                sb = morton2((uint32_t)sx, (uint32_t)sy);
                ok = box_count(start_s, sb, shift) > 0;
            }
        }
        const V *Uo = U + (int64_t)((o.y + R) * W2 + (o.x + R)) * (p1 + 1);
        if (ok) {
            V a = Ml[(int64_t)sb * p1 + m];
            Ap[lane] = cmul(a, Uo[m]);
        }
        __syncthreads();
        if (ok) {
            T sr = 0, si = 0;
            const V *ap = Ap + g * p1;
#pragma unroll
            for (int k = 0; k < P1; ++k) {
                if (k < p1) {
                    V v = ap[k];
                    sr += crow[k] * v.x;
                    si += crow[k] * v.y;
                }
            }
            V um = Uo[m + 1];
            ar += sgn * (um.x * sr - um.y * si);
            ai += sgn * (um.x * si + um.y * sr);
        }
        __syncthreads();
    }
    if (g < G && slot < nbox && m < p1) {
        // boxes without targets get zeros so stale data never leaks into L2L
        Bl[(int64_t)box * p1 + m] = active ? V{ar * inv_r, ai * inv_r} : V{0, 0};
    }
}

// One lane per target box, 64 boxes of one parity class per wave (grid.y =
// parity), so the interaction list, u^k and the binomial rows are uniform
// across the wave and come in as scalar operands.  Each wave produces the
// coefficients m in [MW z, MW z + MW) (grid.z): per link it forms
// A'_k = u^k A_k (all k) and B_m += (-1)^m u^(m+1) sum_k C(k+m, k) A'_k in
// registers, the factorisation and summation order of m2l_kernel, with no
// LDS traffic or barriers; splitting m over waves gives the finest level
// enough waves to hide the load latency.  Requires p1 == P1 (float32).

template <class T, int P1, int MW>
__global__ __launch_bounds__(64) void m2l_box_kernel(
    M2LLevels lv, const typename C2<T>::type *__restrict__ M, typename C2<T>::type *__restrict__ B,
    const int32_t *__restrict__ start_s, const int32_t *__restrict__ start_t,
    const int2 *__restrict__ il_tau, const int32_t *__restrict__ il_offs,
    const typename C2<T>::type *__restrict__ U, int R, const T *__restrict__ binom /* [P1][P1] */)
{
    far_priority();
    using V = typename C2<T>::type;
    const int li = m2l_level_of(lv);
    const int l = lv.lev0 + li;
    const typename C2<T>::type *Ml = M + lv.coff[li] * P1;
    typename C2<T>::type *Bl = B + lv.coff[li] * P1;
    const int32_t *il_off = il_offs + lv.il_base[li];
    const int shift = lv.shift[li];
    const T inv_r = (T)lv.inv_r[li];
    const int lane = threadIdx.x;
    const int par = blockIdx.y;
    const int m0 = blockIdx.z * MW;
    const int n = 1 << l, half = n >> 1;
    const int64_t per = ((int64_t)n * n) / 4;  // boxes per parity class
    const int64_t loc = ((int64_t)blockIdx.x - lv.blk[li]) * 64 + lane;
    const bool in = loc < per;
    int bx = 0, by = 0;
    uint32_t box = 0;
    bool active = false;
    if (in) {
        bx = 2 * (int)(loc % half) + (par & 1);
        by = 2 * (int)(loc / half) + (par >> 1);
        box = morton2((uint32_t)bx, (uint32_t)by);
        active = box_count(start_t, box, shift) > 0;
    }
    T br[MW], bi[MW];
#pragma unroll
    for (int q = 0; q < MW; ++q) br[q] = bi[q] = (T)0;
    const int W2 = 2 * R + 1;
    const int t0 = il_off[par], tn = il_off[par + 1] - t0;
    for (int t = 0; t < tn; ++t) {
        const int2 o = il_tau[t0 + t];
        const int sx = bx + o.x, sy = by + o.y;
        bool ok = active && sx >= 0 && sy >= 0 && sx < n && sy < n;
        uint32_t sb = 0;
        if (ok) {
            sb = morton2((uint32_t)sx, (uint32_t)sy);
            ok = box_count(start_s, sb, shift) > 0;
        }
        if (!ok) continue;
        const V *Uo = U + (int64_t)((o.y + R) * W2 + (o.x + R)) * (P1 + 1);
        const V *A = Ml + (int64_t)sb * P1;
        T apr[P1], api[P1];
#pragma unroll
        for (int k = 0; k < P1; ++k) {
            const V a = A[k], u = Uo[k];
            apr[k] = a.x * u.x - a.y * u.y;
            api[k] = a.x * u.y + a.y * u.x;
        }
#pragma unroll
        for (int q = 0; q < MW; ++q) {
            const int m = m0 + q;
            if (m < P1) {
                T sr = 0, si = 0;
#pragma unroll
                for (int k = 0; k < P1; ++k) {
                    const T c = binom[m * P1 + k];
                    sr += c * apr[k];
                    si += c * api[k];
                }
                const V um = Uo[m + 1];
                const T sgn = (m & 1) ? (T)-1 : (T)1;
                br[q] += sgn * (um.x * sr - um.y * si);
                bi[q] += sgn * (um.x * si + um.y * sr);
            }
        }
    }
    if (in) {
        V *Bb = Bl + (int64_t)box * P1;
#pragma unroll
        for (int q = 0; q < MW; ++q)
            if (m0 + q < P1)  // boxes without targets get zeros (never read stale)
                Bb[m0 + q] = active ? V{br[q] * inv_r, bi[q] * inv_r} : V{(T)0, (T)0};
    }
}

// ------------------------------------------------------ P2P + L2P (leaf) --
// One workgroup of 4 waves per leaf (p2p_leaf): the sources of the leaf's
// near leaves are staged in LDS, every wave sweeps a quarter of them for
// every target, and per-wave TwoSum partials are merged in a fixed order.
// Near offsets [0, ninner) may hold pairs inside the smoothing core; for
// the rest exp(-shape r2) <= 2^-26 for every pair (checked on the host from
// the box gap), so their pairs skip the exponential (bit-identical P).
// Workgroups are dealt round-robin over the 8 XCDs; those of XCD k walk
// the contiguous Morton leaf range [split[k], split[k+1]), which holds an
// eighth of the targets, so the XCDs carry equal work (empty leaves of a
// square domain around an uneven cloud cost nothing) and neighbouring
// leaves share sources in the XCD's L2.
// near set of a single-system leaf: the host-built offset list, offsets
// [0, ninner) first
struct NearList {
    const int2 *near;
    int ninner, bx, by, n;
    float s_f;
    __device__ __forceinline__ bool operator()(int q, uint32_t &sb, float &ox, float &oy,
                                               int &core) const
    {
        const int2 o = near[q];
        const int sx = bx + o.x, sy = by + o.y;
        ox = (float)o.x * s_f;
        oy = (float)o.y * s_f;
        core = q < ninner;
        if (sx < 0 || sy < 0 || sx >= n || sy >= n) return false;
        sb = morton2((uint32_t)sx, (uint32_t)sy);
        return true;
    }
};

// Near-field sums of target leaf b (all threads of the workgroup), written
// in sorted target order: nsum[i] = lam (hi + lo) of both components.
template <int KIND>
__device__ __forceinline__ void p2p_near_leaf_f32s(
    const float4 *__restrict__ src, const int32_t *__restrict__ sp,
    const float2 *__restrict__ tgt, const int32_t *__restrict__ start_t, int Lvl, uint32_t b,
    const int2 *__restrict__ near, int nnear, int ninner, const PairParams &pp, float s_f,
    double2 *__restrict__ nsum, float4 *st, float4 *acc, int q, int P)
{
    const int32_t tl = start_t[b];
    int32_t t0 = tl, t1 = start_t[b + 1];
    if (P > 1) p2p_part(t0, t1, q, P);
    if (t1 <= t0) return;
    const int n = 1 << Lvl;
    const NearList nf{near, ninner, (int)compact_bits(b), (int)compact_bits(b >> 1), n, s_f};
    // scaled coordinates: lam^2 = shape log2(e)
    const float lam = __builtin_sqrtf(-pp.nlog2e_ks_f);
    const int32_t ts = sp[b];
    auto tpos = [&](int32_t i) {
        if (tgt) return tgt[i];
        const float4 r = src[ts + (i - tl)];  // targets are the sources
        return make_float2(r.x, r.y);
    };
    auto out = [&](int32_t i, float ha, float la, float hb, float lb) {
        nsum[i] = make_double2(((double)ha + (double)la) * (double)lam,
                               ((double)hb + (double)lb) * (double)lam);
    };
    p2p_leaf<KIND>(src, sp, st, acc, nnear, nf, t0, t1, tpos, pp, lam, out);
}

template <int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void p2p_near_f32s(
    const float4 *__restrict__ src, const int32_t *__restrict__ sp,
    const float2 *__restrict__ tgt, const int32_t *__restrict__ start_t, int Lvl,
    const int32_t *__restrict__ split, const int2 *__restrict__ near, int nnear, int ninner,
    PairParams pp, float s_f, int P, double2 *__restrict__ nsum)
{
    __shared__ float4 st[P2P_STAGE];
    __shared__ float4 acc[P2P_CHUNKS * 4 * 16];
    const int32_t lo = split[blockIdx.x & 7u];
    const int32_t items = (split[(blockIdx.x & 7u) + 1] - lo) * P;  // P parts of each leaf
    for (int32_t it = (int32_t)(blockIdx.x >> 3); it < items; it += (int32_t)(gridDim.x >> 3)) {
        const int32_t k = P == 1 ? it : it / P;
        p2p_near_leaf_f32s<KIND>(src, sp, tgt, start_t, Lvl, (uint32_t)(lo + k), near, nnear,
                                 ninner, pp, s_f, nsum, st, acc, it - k * P, P);
    }
}

// L2P on the far side (the far field's last kernel, beside the near
// field), one thread per sorted target i with input index o: ffar[o] = the
// local expansion of leaf keys[i] >> fsh at the target (float32 Horner)
// and inv[o] = i, both in input order; targets are the source records (tgt
// null: index bits in .w) or tgt with perm.
__global__ void l2p_far_f32(const float4 *__restrict__ src, const float2 *__restrict__ tgt,
                            const int32_t *__restrict__ perm, const uint32_t *__restrict__ keys,
                            int fsh, int64_t nt, const float2 *__restrict__ Bleaf, int p1,
                            float inv_s, float2 *__restrict__ ffar, int32_t *__restrict__ inv)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nt) return;
    float2 tp;
    int32_t o;
    if (tgt) {
        tp = tgt[i];
        o = perm[i];
    } else {
        const float4 q = src[i];
        tp = make_float2(q.x, q.y);
        o = __float_as_int(q.w);
    }
    double fr, fi;
    l2p_f32(Bleaf + (int64_t)(keys[i] >> fsh) * p1, p1, tp.x * inv_s, tp.y * inv_s, fr, fi);
    ffar[o] = make_float2((float)fr, (float)fi);
    inv[o] = (int32_t)i;
}

// The outputs in input order with the far part: one thread per input index
// o (coalesced writes), its near sums read from sorted position inv[o].
__global__ void out_gather_f32(const int32_t *__restrict__ inv, int64_t nt,
                               const float2 *__restrict__ ffar,
                               const double2 *__restrict__ nsum, double *__restrict__ out_a,
                               double *__restrict__ out_b, int velocity_out)
{
    const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= nt) return;
    const double2 ns = nsum[inv[o]];
    const float2 f = ffar[o];
    const double qr = -(ns.x + (double)f.x);
    const double qi = ns.y - (double)f.y;
    if (velocity_out) {
        // (vx, vy) = (-qi/(2 pi), -qr/(2 pi)) (_induced.py:334-336)
        const double two_pi = 2.0 * 3.141592653589793;
        out_a[o] = -qi / two_pi;
        out_b[o] = -qr / two_pi;
    } else {
        out_a[o] = qr;
        out_b[o] = qi;
    }
}

// The outputs without a far field, one thread per sorted target i: (qr,
// qi) = (-near_a, near_b) to input index perm[i] (perm given) or the source
// record's index bits.
__global__ void out_scatter_f32(const float4 *__restrict__ src, const int32_t *__restrict__ perm,
                                int64_t nt, const double2 *__restrict__ nsum,
                                double *__restrict__ out_a, double *__restrict__ out_b,
                                int velocity_out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nt) return;
    const int32_t o = perm ? perm[i] : __float_as_int(src[i].w);
    const double fr = 0.0, fi = 0.0;
    const double2 ns = nsum[i];
    const double qr = -(ns.x + fr);
    const double qi = ns.y - fi;
    if (velocity_out) {
        // (vx, vy) = (-qi/(2 pi), -qr/(2 pi)) (_induced.py:334-336)
        const double two_pi = 2.0 * 3.141592653589793;
        out_a[o] = -qi / two_pi;
        out_b[o] = -qr / two_pi;
    } else {
        out_a[o] = qr;
        out_b[o] = qi;
    }
}

// float64 near-field sums, one workgroup (4 waves) per target leaf over
// the XCD leaf ranges split by target count, written in sorted target
// order: nsum[i] = (a, b) of target i.  Absolute coordinates and
// pair_f64's operation order.
// Held to 128 VGPRs, four workgroups on a CU (141 unbound, three): 1M blobs,
// 1e-12: the evaluation takes 1520 us against 1563, 120k 289 against 314.
// (That leaves the far field no registers beside four of them; without its
// higher priority it fell so far behind that three were the better.)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void p2p_near_f64s(
    const double4 *__restrict__ src, const int32_t *__restrict__ start_s,
    const double2 *__restrict__ tgt, const int32_t *__restrict__ start_t, int Lvl,
    const int32_t *__restrict__ split, const int2 *__restrict__ near, int nnear, PairParams pp,
    int P, double2 *__restrict__ nsum)
{
    __shared__ double4 st[P2P_STAGE_F64];
    __shared__ double2 acc[P2P_CHUNKS * 4 * 16];
    const int32_t lo = split[blockIdx.x & 7u];
    const int32_t items = (split[(blockIdx.x & 7u) + 1] - lo) * P;  // P parts of each leaf
    const int n = 1 << Lvl;
    for (int32_t it = (int32_t)(blockIdx.x >> 3); it < items; it += (int32_t)(gridDim.x >> 3)) {
        const int32_t k = P == 1 ? it : it / P;
        const uint32_t b = (uint32_t)(lo + k);
        int32_t t0 = start_t[b], t1 = start_t[b + 1];
        if (P > 1) p2p_part(t0, t1, it - k * P, P);
        if (t1 <= t0) continue;
        const NearList nf{near, nnear, (int)compact_bits(b), (int)compact_bits(b >> 1), n, 0.f};
        auto tpos = [&](int32_t i) { return tgt[i]; };
        auto out = [&](int32_t i, double a, double bb) { nsum[i] = make_double2(a, bb); };
        p2p_leaf_f64(src, start_s, st, acc, nnear, nf, t0, t1, tpos, pp, out);
    }
}

// float64 L2P and the output in input order, one thread per sorted target
// i of leaf keys[i] >> fsh: (qr, qi) = (-(a + far_r), b - far_i) with the
// leaf's local expansion at (t - c)/s (Horner).
__global__ void l2p_scatter_f64(const double2 *__restrict__ tgt,
                                const uint32_t *__restrict__ keys, int fsh,
                                const int32_t *__restrict__ perm, int64_t nt,
                                const double4 *__restrict__ org, double s,
                                const double2 *__restrict__ Bleaf, int p1,
                                const double2 *__restrict__ nsum, double *__restrict__ qr,
                                double *__restrict__ qi, int velocity_out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nt) return;
    const double2 tp = tgt[i];
    double fr = 0.0, fi = 0.0;
    if (Bleaf) {
        const uint32_t b = keys[i] >> fsh;
        double cx, cy;
        leaf_center(b, org->x, org->z, s, cx, cy);
        const double inv_s = 1.0 / s;
        const double2 *Bv = Bleaf + (int64_t)b * p1;
        const double zr = (tp.x - cx) * inv_s, zi = (tp.y - cy) * inv_s;
        for (int k = p1 - 1; k >= 0; --k) {
            const double2 c = Bv[k];
            const double nr = fr * zr - fi * zi + c.x;
            const double ni = fr * zi + fi * zr + c.y;
            fr = nr;
            fi = ni;
        }
    }
    const double2 ns = nsum[i];
    const int32_t o = perm[i];
    const double vr = -(ns.x + fr), vi = ns.y - fi;
    if (velocity_out) {
        // (vx, vy) = (-qi/(2 pi), -qr/(2 pi)) (_induced.py:334-336)
        const double two_pi = 2.0 * 3.141592653589793;
        qr[o] = -vi / two_pi;
        qi[o] = -vr / two_pi;
    } else {
        qr[o] = vr;
        qi[o] = vi;
    }
}

// ------------------------------------------------------------ counters --
// Algorithmic work of one evaluation, for roofline accounting: P2P pairs
// (targets of a leaf x sources of its near leaves) and M2L links.
__global__ void count_p2p_pairs(const int32_t *__restrict__ start_s,
                                const int32_t *__restrict__ start_t, int Lvl,
                                const int2 *__restrict__ near, int nnear,
                                unsigned long long *__restrict__ out)
{
    const int64_t nleaf = int64_t(1) << (2 * Lvl);
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nleaf) return;
    const int64_t nt = start_t[b + 1] - start_t[b];
    if (nt == 0) return;
    const int bx = (int)compact_bits((uint32_t)b), by = (int)compact_bits((uint32_t)b >> 1);
    const int n = 1 << Lvl;
    int64_t ns = 0;
    for (int q = 0; q < nnear; ++q) {
        const int sx = bx + near[q].x, sy = by + near[q].y;
        if (sx < 0 || sy < 0 || sx >= n || sy >= n) continue;
        const uint32_t sb = morton2((uint32_t)sx, (uint32_t)sy);
        ns += start_s[sb + 1] - start_s[sb];
    }
    atomicAdd(out, (unsigned long long)(nt * ns));
}

__global__ void count_m2l_links(int l, const int32_t *__restrict__ start_s,
                                const int32_t *__restrict__ start_t, int shift,
                                const int2 *__restrict__ il_tau,
                                const int32_t *__restrict__ il_off,
                                unsigned long long *__restrict__ out)
{
    const int n = 1 << l;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)n * n) return;
    const uint32_t box = (uint32_t)i;
    if (box_count(start_t, box, shift) == 0) return;
    const int bx = (int)compact_bits(box), by = (int)compact_bits(box >> 1);
    const int par = (bx & 1) | ((by & 1) << 1);
    unsigned long long c = 0;
    for (int t = il_off[par]; t < il_off[par + 1]; ++t) {
        const int sx = bx + il_tau[t].x, sy = by + il_tau[t].y;
        if (sx < 0 || sy < 0 || sx >= n || sy >= n) continue;
        if (box_count(start_s, morton2((uint32_t)sx, (uint32_t)sy), shift) > 0) ++c;
    }
    if (c) atomicAdd(out, c);
}

// (qr, qi) -> velocity (vx, vy) = (-qi/(2 pi), -qr/(2 pi)) (_induced.py:334-336)
__global__ void q_to_velocity(const double *__restrict__ qr, const double *__restrict__ qi,
                              int64_t n, double *__restrict__ vx, double *__restrict__ vy)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double two_pi = 2.0 * 3.141592653589793;
    const double a = qr[i], b = qi[i];
    vx[i] = -b / two_pi;
    vy[i] = -a / two_pi;
}

int q_to_velocity_device(Lane *L, const double *qr, const double *qi, int64_t n, double *vx,
                         double *vy)
{
    if (n <= 0) return PHF_OK;
    q_to_velocity<<<div_up(n, 256), 256, 0, L->stream>>>(qr, qi, n, vx, vy);
    PHF_HIP(hipGetLastError());
    return PHF_OK;
}

__global__ void padded_counts(const int32_t *__restrict__ start, int64_t nleaf,
                              uint32_t *__restrict__ cnt)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b > nleaf) return;
    cnt[b] = b < nleaf ? (uint32_t)((start[b + 1] - start[b] + 3) & ~3) : 0u;
}

// Leaf ranges of the 8 XCDs holding equal numbers of targets: split[k]
// (k = 0..8) is the leaf that holds target k ceil(nt/8); without such a target
// the end of the last leaf that has any, so no XCD walks the empty leaves
// behind it (600k blobs in the first 16k of 65k leaves: near field 406 ->
// 337 us).  Every entry has one writer.
__global__ void xcd_leaf_split(const int32_t *__restrict__ start, int64_t nleaf,
                               int32_t *__restrict__ split)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nleaf) return;
    const int64_t nt = start[nleaf];
    const int64_t T = nt > 0 ? (nt + 7) / 8 : 1;
    const int64_t t0 = start[b], t1 = start[b + 1];
    if (t1 == nt && (t0 < nt || (nt == 0 && b == 0)))
        for (int k = 0; k <= 8; ++k)
            if (k == 8 || k * T >= nt) split[k] = nt > 0 ? (int32_t)b + 1 : 0;
    for (int64_t k = (t0 + T - 1) / T; k < 8 && k * T < t1; ++k) split[k] = (int32_t)b;
}

int xcd_split(Lane *L, const int32_t *start, int64_t nleaf, int32_t *split)
{
    xcd_leaf_split<<<div_up(nleaf + 1, 256), 256, 0, L->stream>>>(start, nleaf, split);
    PHF_HIP(hipGetLastError());
    return PHF_OK;
}

__global__ void zero_pads_f32(const int32_t *__restrict__ start, const int32_t *__restrict__ sp,
                              int64_t nleaf, float4 *__restrict__ out)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nleaf) return;
    for (int32_t k = sp[b] + (start[b + 1] - start[b]); k < sp[b + 1]; ++k)
        out[k] = make_float4(0.f, 0.f, 0.f, 0.f);
}

int pad_source_ranges(Lane *L, const int32_t *start, int64_t nleaf, uint32_t *cnt, uint32_t *sp,
                      uint32_t *sums)
{
    padded_counts<<<div_up(nleaf + 1, 256), 256, 0, L->stream>>>(start, nleaf, cnt);
    PHF_HIP(hipGetLastError());
    return device_exclusive_scan_ws(L, cnt, nleaf + 1, sp, sums);
}

int zero_source_pads(Lane *L, const int32_t *start, const int32_t *sp, int64_t nleaf, float4 *src)
{
    if (nleaf > 0) zero_pads_f32<<<div_up(nleaf, 256), 256, 0, L->stream>>>(start, sp, nleaf, src);
    PHF_HIP(hipGetLastError());
    return PHF_OK;
}

// ------------------------------------------------------------- host ------
namespace {

double binom_d(int n, int k)
{
    if (k < 0 || k > n) return 0.0;
    long double r = 1.0L;
    for (int i = 1; i <= k; ++i) r = r * (long double)(n - k + i) / (long double)i;
    return (double)std::llround(r) == (double)r ? (double)r : (double)r;
}

struct Lists {
    std::vector<int2> near_leaf;
    std::vector<std::vector<int2>> il;       // per level: concatenated parities
    std::vector<std::vector<int32_t>> il_off;  // per level: 5 offsets
    int R = 0;
    int il_max_all = 0;
};

std::vector<int2> near_set(double s, double c2, int ws, int Rwin)
{
    std::vector<int2> out;
    for (int dy = -Rwin; dy <= Rwin; ++dy)
        for (int dx = -Rwin; dx <= Rwin; ++dx) {
            if (near_offset(dx, dy, ws, s, c2)) out.push_back(make_int2(dx, dy));
        }
    return out;
}

int near_radius(const std::vector<int2> &v)
{
    int r = 0;
    for (auto &o : v) r = std::max(r, std::max(std::abs(o.x), std::abs(o.y)));
    return r;
}

int near_window(double s, double c2, int ws, int l)
{
    return std::min(std::max(ws, (int)std::ceil(std::sqrt(c2) / s) + 2), 1 << l);
}

Lists make_lists(const Domain &dom, double c2, int ws)
{
    Lists ls;
    const int Lv = dom.L;
    std::vector<std::vector<int2>> nearl(Lv + 1);
    for (int l = 0; l <= Lv; ++l) {
        const double s = dom.D / std::ldexp(1.0, l);
        nearl[l] = near_set(s, c2, ws, near_window(s, c2, ws, l));
    }
    ls.near_leaf = nearl[Lv];
    ls.il.resize(Lv + 1);
    ls.il_off.resize(Lv + 1);
    for (int l = 2; l <= Lv; ++l) {
        auto &lst = ls.il[l];
        auto &off = ls.il_off[l];
        off.push_back(0);
        for (int par = 0; par < 4; ++par) {
            const int px = par & 1, py = par >> 1;
            std::vector<int2> cand;
            for (auto &nu : nearl[l - 1])
                for (int e = 0; e < 4; ++e) {
                    int tx = 2 * nu.x + (e & 1) - px, ty = 2 * nu.y + (e >> 1) - py;
                    bool in_near = false;
                    for (auto &o : nearl[l])
                        if (o.x == tx && o.y == ty) {
                            in_near = true;
                            break;
                        }
                    if (!in_near) cand.push_back(make_int2(tx, ty));
                }
            for (auto &c : cand) {
                ls.R = std::max(ls.R, std::max(std::abs(c.x), std::abs(c.y)));
                lst.push_back(c);
            }
            off.push_back((int32_t)lst.size());
            ls.il_max_all = std::max(ls.il_max_all, (int)cand.size());
        }
    }
    return ls;
}

// Leaf level L (coarsened while the leaf near set reaches beyond 6 boxes,
// for cutoffs large against the box) and the domain side from
// choose_domain_side.
Domain choose_domain(const double4 &hb, int L, double nb, double nt, double cutoff, int ws,
                     double shape_log2, int p1, int chunk, double leaf_side)
{
    const double c2 = cutoff * cutoff;
    for (;;) {
        const double side = choose_domain_side(hb.y - hb.x, hb.w - hb.z, L, nb, nt, cutoff, ws,
                                               shape_log2, p1, chunk, leaf_side);
        const Domain d = make_domain(hb.x, hb.y, hb.z, hb.w, L, side);
        if (L == 0 || near_radius(near_set(d.s, c2, ws, near_window(d.s, c2, ws, L))) <= 6)
            return d;
        --L;
    }
}

// The small host tables of a plan, packed into the lane's pinned staging
// buffer and sent with a single copy.
struct TableBlob {
    std::vector<char> host;
    std::vector<std::pair<size_t, void **>> fix;
    template <class T>
    void add(const std::vector<T> &v, void **d)
    {
        size_t at = (host.size() + 255) & ~size_t(255);
        host.resize(at + std::max<size_t>(sizeof(T) * v.size(), 1));
        if (!v.empty()) std::memcpy(host.data() + at, v.data(), sizeof(T) * v.size());
        fix.push_back({at, d});
    }
    // To dev (at least host.size() bytes) on stream st; wait: the copy is
    // complete on return (launches being recorded into a graph then hold no
    // copy), else it is ordered on st.
    int send(Lane *L, char *dev, hipStream_t st, bool wait)
    {
        if (wait) {
            PHF_HIP(hipMemcpyAsync(dev, host.data(), host.size(), hipMemcpyHostToDevice, st));
            PHF_HIP(hipStreamSynchronize(st));
        } else {
            PHF_TRY(L->pin.ensure(host.size()));
            std::memcpy(L->pin.ptr, host.data(), host.size());
            PHF_HIP(hipMemcpyAsync(dev, L->pin.ptr, host.size(), hipMemcpyHostToDevice, st));
            PHF_TRY(L->pin.mark(st));
        }
        for (auto &f : fix) *f.second = dev + f.first;
        return PHF_OK;
    }
};

}  // namespace

int fmm_order_from_tol(double tol)
{
    // fmm.cpp:538-546 with theta = 0.5 and pot = 1
    int p = (int)std::floor(std::log2(4.0 * tol) / std::log2(0.5) - 1.0) + 1;
    return std::max(p, 2);
}

int fmm_level(int64_t nb, int leaf, int ndirect)
{
    int L;
    if (leaf > 0) {
        double q = (double)std::max<int64_t>(nb, 1) / leaf;
        L = q > 1.0 ? (int)std::lround(std::log(q) / std::log(4.0)) : 0;
    } else {
        // fmm.cpp:553-555
        double v = 0.5 * std::log2(5.0 / 8.0 * (double)nb / std::max(ndirect, 1));
        L = (int)std::ceil(v);
    }
    return std::max(0, std::min(L, 11));
}

// f(integral constant MT) for the tiles of 16 that hold p1 coefficients
template <class F>
static int shift_dispatch(int p1, const F &f)
{
    if (p1 <= 16)
        f(std::integral_constant<int, 1>());
    else if (p1 <= 32)
        f(std::integral_constant<int, 2>());
    else if (p1 <= 41)
        f(std::integral_constant<int, 3>());
    else {
        set_error("expansion order %d too large (max 40)", p1 - 1);
        return PHF_ERR_UNSUPPORTED;
    }
    PHF_HIP(hipGetLastError());
    return PHF_OK;
}


// M2L of every level >= 2 in one launch: the generic coefficient-per-lane
// kernel (G = 64 / p1 boxes per wave) for any order.
template <class T, int P1>
static int launch_m2l(Lane *L, M2LLevels lv, int p1, const void *M, void *B, const int32_t *ss,
                      const int32_t *st, const int2 *il, const int32_t *offs, const void *U, int R,
                      const void *binom)
{
    using V = typename C2<T>::type;
    const int G = 64 / p1;
    int64_t nb = 0;
    lv.blk[0] = 0;
    for (int i = 0; i < lv.nlev; ++i) {
        const int64_t nbox = int64_t(1) << (2 * (lv.lev0 + i));
        lv.blk[i + 1] = lv.blk[i] + (nbox + G - 1) / G;
    }
    nb = lv.blk[lv.nlev];
    m2l_kernel<T, P1><<<(unsigned)nb, 64, 0, L->stream>>>(lv, p1, (const V *)M, (V *)B, ss, st, il,
                                                          offs, (const V *)U, R, (const T *)binom);
    PHF_HIP(hipGetLastError());
    return PHF_OK;
}

template <class T>
static int m2l_dispatch(Lane *L, const M2LLevels &lv, int p1, const void *M, void *B,
                        const int32_t *ss, const int32_t *st, const int2 *il, const int32_t *offs,
                        const void *U, int R, const void *binom)
{
#define PHF_M2L(P) \
    if (p1 <= P) return launch_m2l<T, P>(L, lv, p1, M, B, ss, st, il, offs, U, R, binom);
    PHF_M2L(9)
    PHF_M2L(13)
    PHF_M2L(17)
    PHF_M2L(21)
    PHF_M2L(25)
    PHF_M2L(32)
    PHF_M2L(41)
#undef PHF_M2L
    set_error("expansion order %d too large (max 40)", p1 - 1);
    return PHF_ERR_UNSUPPORTED;
}

// a launch on a stream (recorded with its arguments)
using P2PLaunch = std::function<int(hipStream_t)>;

// How run_fmm_typed hands back its last launches.  With a split, it calls
// mid() after the tree (capture: ends the first recording and begins the
// second), enqueues the far field and returns the near-field launch (sums
// in sorted target order) and the finishing launch (L2P and the output in
// input order) for the caller to issue around the far field.  Without one
// it issues them itself: the far field on the lane's second stream beside
// the near field (fmm_far_fork / fmm_far_done / fmm_far_join), so that the
// near field follows the tree on the lane's stream with no cross-stream
// wait in between.  An empty near launch runs everything in order.
struct FmmPlan;
struct FmmSplit {
    ~FmmSplit();
    std::function<int()> mid;
    P2PLaunch near, finish;
    char **tables_keep = nullptr;  // device tables kept for replays
    std::unique_ptr<FmmPlan> plan;  // and their layout, while recording
    hipStream_t side = nullptr;    // their upload stream while recording
};

static int lane_stream2(Lane *L)
{
    if (!L->stream2) PHF_HIP(hipStreamCreateWithFlags(&L->stream2, hipStreamNonBlocking));
    if (!L->fork_ev) PHF_HIP(hipEventCreateWithFlags(&L->fork_ev, hipEventDisableTiming));
    if (!L->join_ev) PHF_HIP(hipEventCreateWithFlags(&L->join_ev, hipEventDisableTiming));
    return PHF_OK;
}

// Work enqueued on the lane's second stream after fmm_far_fork runs after
// what was enqueued so far on the lane's stream; fmm_far_done marks its
// end, and fmm_far_join makes the lane's stream wait for that mark.
static int fmm_far_fork(Lane *L)
{
    PHF_TRY(lane_stream2(L));
    PHF_HIP(hipEventRecord(L->fork_ev, L->stream));
    PHF_HIP(hipStreamWaitEvent(L->stream2, L->fork_ev, 0));
    return PHF_OK;
}

static int fmm_far_done(Lane *L)
{
    PHF_HIP(hipEventRecord(L->join_ev, L->stream2));
    return PHF_OK;
}

static int fmm_far_join(Lane *L)
{
    PHF_HIP(hipStreamWaitEvent(L->stream, L->join_ev, 0));
    return PHF_OK;
}

// near field on the lane's stream, timed as the P2P stage
static int fmm_near(Lane *L, const P2PLaunch &near, StageTimer &tm)
{
    tm.begin(PHF_STAGE_P2P);
    const int rc = near(L->stream);
    tm.end(PHF_STAGE_P2P);
    return rc;
}

// Tables of one tree shape on the device: near list, interaction lists,
// binomials and powers.  They depend on the order, the precision, the leaf
// level and which box offsets are near at each level (key), not on the points
// or the domain's place and size.  A lane keeps the last kPlans it used, so a
// time step or a call with new points of a like spread neither builds nor
// sends them again (45 us less between the bounding box and the near field of
// 120k blobs).
struct FmmPlan {
    std::vector<uint8_t> key;
    char *dev = nullptr;  // the tables, cap bytes; null: in the arena or a graph's
    size_t cap = 0;
    void *near = nullptr, *pas = nullptr, *bin = nullptr, *U = nullptr, *il = nullptr,
         *iloff = nullptr;
    int nnear = 0, ninner = 0, R = 1;
    std::vector<int> il_base, il_max;
    uint64_t last = 0;
};

FmmSplit::~FmmSplit() = default;

struct FmmPlanCache {
    std::vector<std::unique_ptr<FmmPlan>> v;
    std::unique_ptr<FmmPlan> once;  // of the current call only, in the arena
    uint64_t clock = 0;
};

constexpr size_t kPlans = 6;

// What the tables depend on: near sets are symmetric and shrink with |dy|, so
// the reach in x for every dy >= 0 describes one.
static std::vector<uint8_t> plan_key(const FmmArgs &a, const Domain &dom, int type, bool far,
                                     double shape_log2)
{
    std::vector<uint8_t> k = {(uint8_t)type, (uint8_t)dom.L,      (uint8_t)a.p,
                              (uint8_t)(a.p >> 8), (uint8_t)a.ws, (uint8_t)far};
    const double c2 = a.cutoff * a.cutoff;
    auto reach = [&k](int R, auto in) {
        for (int dy = 0; dy <= R; ++dy) {
            int dx = -1;
            while (dx < R && in(dx + 1, dy)) ++dx;
            if (dx < 0) break;
            k.push_back((uint8_t)(dx + 1));
        }
        k.push_back(0);
    };
    for (int l = far ? 0 : dom.L; l <= dom.L; ++l) {
        const double s = dom.D / std::ldexp(1.0, l);
        reach(near_window(s, c2, a.ws, l),
              [&](int dx, int dy) { return near_offset(dx, dy, a.ws, s, c2); });
    }
    reach(near_window(dom.s, c2, a.ws, dom.L), [&](int dx, int dy) {
        return near_offset(dx, dy, a.ws, dom.s, c2) && near_offset_core(dx, dy, dom.s, shape_log2);
    });
    return k;
}

void fmm_plans_release(Lane *L)
{
    if (!L->fmm_plans) return;
    for (auto &q : L->fmm_plans->v)
        if (q->dev) (void)hipFree(q->dev);
    delete L->fmm_plans;
    L->fmm_plans = nullptr;
}

// The plan of (a, dom): the lane's own, or a new one.  While a graph is being
// recorded (spl) the tables go to the recording instead, which owns them.
template <class T>
static int fmm_plan(Lane *L, const FmmArgs &a, const Domain &dom, const PairParams &pp, bool far,
                    FmmSplit *spl, const FmmPlan **out)
{
    using V = typename C2<T>::type;
    const int Lv = dom.L, p1 = a.p + 1;
    const double shape_log2 = 1.4426950408889634074 * pp.inv_ks;
    if (!L->fmm_plans) L->fmm_plans = new FmmPlanCache;
    FmmPlanCache &c = *L->fmm_plans;
    std::vector<uint8_t> key =
        plan_key(a, dom, (int)sizeof(T), far, shape_log2);
    if (!spl)
        for (auto &q : c.v)
            if (q->key == key) {
                q->last = ++c.clock;
                *out = q.get();
                return PHF_OK;
            }
    std::unique_ptr<FmmPlan> pl(new FmmPlan);
    pl->key = std::move(key);
    const Lists ls = make_lists(dom, a.cutoff * a.cutoff, a.ws);
    // near list at the leaf level, offsets that can hold pairs inside the
    // smoothing core first: for the others the box gap g satisfies
    // shape g^2 log2(e) >= 26 with a 2% margin for float32 rounding of the
    // point offsets, so exp(-shape r2) <= 2^-26 for every pair
    std::vector<int2> near_ord, outer;
    for (const int2 &o : ls.near_leaf)
        (near_offset_core(o.x, o.y, dom.s, shape_log2) ? near_ord : outer).push_back(o);
    pl->ninner = (int)near_ord.size();
    near_ord.insert(near_ord.end(), outer.begin(), outer.end());
    pl->nnear = (int)near_ord.size();
    TableBlob blob;
    blob.add(near_ord, &pl->near);
    pl->il_base.assign(Lv + 1, 0);
    pl->il_max.assign(Lv + 1, 0);
    const int R = pl->R = std::max(ls.R, 1);
    if (far) {
        // Pascal triangle C(m, k) for the multi-level shifts
        std::vector<double> pas((size_t)p1 * p1);
        for (int m = 0; m < p1; ++m)
            for (int k = 0; k < p1; ++k) pas[(size_t)m * p1 + k] = binom_d(m, k);
        blob.add(pas, &pl->pas);
        // M2L: binomial rows C(k+m, k) and powers u^k, u = -1/offset
        std::vector<T> bin((size_t)p1 * p1);
        for (int m = 0; m < p1; ++m)
            for (int k = 0; k < p1; ++k) bin[(size_t)m * p1 + k] = (T)binom_d(k + m, k);
        const int W2 = 2 * R + 1;
        std::vector<V> U((size_t)W2 * W2 * (p1 + 1));
        for (int oy = -R; oy <= R; ++oy)
            for (int ox = -R; ox <= R; ++ox) {
                std::complex<double> u = 0.0;
                if (ox || oy) u = -1.0 / std::complex<double>(ox, oy);
                std::complex<double> pw = 1.0;
                for (int k = 0; k <= p1; ++k) {
                    U[((size_t)(oy + R) * W2 + (ox + R)) * (p1 + 1) + k] =
                        V{(T)pw.real(), (T)pw.imag()};
                    pw *= u;
                }
            }
        blob.add(bin, &pl->bin);
        blob.add(U, &pl->U);
        std::vector<int2> il_all;
        std::vector<int32_t> il_offs;
        for (int l = 2; l <= Lv; ++l) {
            pl->il_base[l] = (int)il_offs.size();
            for (int q = 0; q < 5; ++q) il_offs.push_back((int32_t)il_all.size() + ls.il_off[l][q]);
            for (int q = 0; q < 4; ++q)
                pl->il_max[l] = std::max(pl->il_max[l], ls.il_off[l][q + 1] - ls.il_off[l][q]);
            il_all.insert(il_all.end(), ls.il[l].begin(), ls.il[l].end());
        }
        blob.add(il_all, &pl->il);
        blob.add(il_offs, &pl->iloff);
    }
    const size_t need = blob.host.size();
    if (spl) {
        char *dev;
        PHF_HIP(hipMalloc(&dev, need));
        *spl->tables_keep = dev;
        PHF_TRY(blob.send(L, dev, spl->side, true));
        spl->plan = std::move(pl);
        *out = spl->plan.get();
        return PHF_OK;
    }
    // The least recently used plan makes room, and its buffer serves the new
    // one if it is large enough: the copy below follows, on the lane's stream,
    // every launch that reads it (a call's far field is joined to that stream).
    // So more shapes in turn than are kept cost their tables' transfer, and
    // neither wait for the device nor allocate.
    if (c.v.size() >= kPlans) {
        auto lru = std::min_element(c.v.begin(), c.v.end(), [](const auto &x, const auto &y) {
            return x->last < y->last;
        });
        if ((*lru)->cap < need) {
            PHF_TRY(lane_quiesce(L));
            (void)hipFree((*lru)->dev);
        } else {
            pl->dev = (*lru)->dev;
            pl->cap = (*lru)->cap;
        }
        c.v.erase(lru);
    }
    if (!pl->dev) {
        size_t cap = size_t(64) << 10;
        while (cap < need) cap *= 2;
        if (hipMalloc(&pl->dev, cap) == hipSuccess) {
            pl->cap = cap;
        } else {  // no memory beyond the arena's
            (void)hipGetLastError();
            pl->dev = nullptr;
        }
    }
    if (!pl->dev) {
        char *dev;
        PHF_ALLOC(dev, L->arena, char, need);
        PHF_TRY(blob.send(L, dev, L->stream, false));
        c.once = std::move(pl);
        *out = c.once.get();
        return PHF_OK;
    }
    const int rc = blob.send(L, pl->dev, L->stream, false);
    if (rc != PHF_OK) {
        (void)lane_quiesce(L);
        (void)hipFree(pl->dev);
        return rc;
    }
    pl->last = ++c.clock;
    c.v.push_back(std::move(pl));
    *out = c.v.back().get();
    return PHF_OK;
}

template <class T>
static int run_fmm_typed(Lane *L, const FmmArgs &a, const Domain &dom, const SortedPoints &S,
                         const SortedPoints &Tg, StageTimer &tm, bool *used, FmmInfo *info,
                         FmmSplit *spl, int *nnear_out)
{
    using V = typename C2<T>::type;
    const int Lv = dom.L, p1 = a.p + 1;
    const PairParams pp = make_oseen_params(a.xopt, a.cutoff);

    // sorted point data (the tree stage began in fmm_device)
    void *src, *tgt;
    const int32_t *perm_t = Tg.perm;
    const int32_t *sp = S.start;  // source ranges per leaf
    if (sizeof(T) == 4) {
        // sorted float32 records from build_sorted_payload
        float4 *s4 = S.pay;
        float2 *t2 = nullptr;  // targets == sources: P2P reads the source records
        if (!a.same) {
            PHF_ALLOC(t2, L->arena, float2, (size_t)std::max<int64_t>(a.nt, 1));
            gather_tgt_f32<<<div_up(a.nt, 256), 256, 0, L->stream>>>(
                a.xt, a.yt, Tg.keys, 2 * Tg.fine, Tg.perm, a.nt, dom.org, dom.s, t2);
        }
        src = s4;
        tgt = t2;
    } else {
        double4 *s4;
        PHF_ALLOC(s4, L->arena, double4, (size_t)std::max<int64_t>(a.nb, 1));
        if (a.nb)
            gather_src_f64<<<div_up(a.nb, 256), 256, 0, L->stream>>>(a.xb, a.yb, a.wb, S.perm,
                                                                     a.nb, s4);
        double2 *t2;
        PHF_ALLOC(t2, L->arena, double2, (size_t)std::max<int64_t>(a.nt, 1));
        gather_tgt_f64<<<div_up(a.nt, 256), 256, 0, L->stream>>>(a.xt, a.yt, Tg.perm, a.nt, t2);
        src = s4;
        tgt = t2;
    }
    PHF_HIP(hipGetLastError());

    // the near list (offsets that can hold pairs inside the smoothing core
    // first) and the far field's tables
    const bool far = Lv >= 2 && a.nb > 0;
    std::vector<int64_t> off(Lv + 2, 0);  // level offsets in the coefficient arrays
    for (int l = 0; l <= Lv; ++l) off[l + 1] = off[l] + (int64_t(1) << (2 * l));
    const FmmPlan *pl;
    PHF_TRY(fmm_plan<T>(L, a, dom, pp, far, spl, &pl));
    const int2 *d_near = (const int2 *)pl->near;
    const int nnear = pl->nnear, ninner = pl->ninner;
    const double *d_pas = (const double *)pl->pas;
    const T *d_bin = (const T *)pl->bin;
    const V *d_U = (const V *)pl->U;
    const int2 *d_il = (const int2 *)pl->il;
    const int32_t *d_iloff = (const int32_t *)pl->iloff;
    const std::vector<int> &il_base = pl->il_base, &il_max = pl->il_max;
    const int R = pl->R;
    *nnear_out = nnear;
    V *M = nullptr, *B = nullptr;
    if (far) {
        PHF_ALLOC(M, L->arena, V, (size_t)off[Lv + 1] * p1);
        PHF_ALLOC(B, L->arena, V, (size_t)off[Lv + 1] * p1);
    }
    const uint32_t nleaf = 1u << (2 * Lv);
    if (info && info->want_counts) {
        for (int l = 2; far && l <= Lv; ++l)
            count_m2l_links<<<div_up(int64_t(1) << (2 * l), 256), 256, 0, L->stream>>>(
                l, S.start, Tg.start, 2 * (Lv - l), d_il, d_iloff + il_base[l],
                info->d_counts + 1);
        count_p2p_pairs<<<div_up((int64_t)nleaf, 256), 256, 0, L->stream>>>(
            S.start, Tg.start, Lv, d_near, nnear, info->d_counts);
        PHF_HIP(hipGetLastError());
    }

    // near field and finish: the near field is summed in sorted target
    // order (beside the far field), then the leaf expansions are added and
    // the outputs written in input order
    const int vout = a.velocity_out ? 1 : 0;
    const int P = p2p_parts(dom.occupied, (double)a.nt);
    const uint32_t nl8 = (nleaf * (uint32_t)P + 7) / 8;
    const int32_t *split = Tg.split;  // XCD leaf ranges of the targets
    const int32_t *ts = Tg.start;
    double *qr = a.qr, *qi = a.qi;
    P2PLaunch near, finish, far_tail;
    if (sizeof(T) == 4) {
        const float4 *s4 = (const float4 *)src;
        const float2 *t2 = (const float2 *)tgt;
        const float2 *Bl = far ? (const float2 *)B + off[Lv] * p1 : nullptr;
        const uint32_t *tkeys = Tg.keys;
        const int fsh = 2 * Tg.fine;
        const float s_f = (float)dom.s, inv_s = 1.0f / s_f;
        const int64_t nt = a.nt;
        double2 *nsum;
        PHF_ALLOC(nsum, L->arena, double2, (size_t)std::max<int64_t>(a.nt, 1));
        near = [=](hipStream_t st) {
            if (pp.f32_nocut)
                p2p_near_f32s<PAIR_OSEEN_NOCUT><<<8 * nl8, 256, 0, st>>>(
                    s4, sp, t2, ts, Lv, split, d_near, nnear, ninner, pp, s_f, P, nsum);
            else
                p2p_near_f32s<PAIR_OSEEN><<<8 * nl8, 256, 0, st>>>(
                    s4, sp, t2, ts, Lv, split, d_near, nnear, ninner, pp, s_f, P, nsum);
            PHF_HIP(hipGetLastError());
            return PHF_OK;
        };
        // the far side evaluates the leaf expansions at the targets (after
        // L2L, beside the near field) into input order, with the inverse
        // permutation; the finish then reads the near sums through it and
        // writes the outputs in input order (no scattered writes after the
        // near field)
        if (Bl) {
            float2 *ffar;
            int32_t *inv;
            PHF_ALLOC(ffar, L->arena, float2, (size_t)std::max<int64_t>(a.nt, 1));
            PHF_ALLOC(inv, L->arena, int32_t, (size_t)std::max<int64_t>(a.nt, 1));
            far_tail = [=](hipStream_t st) {
                l2p_far_f32<<<div_up(nt, 256), 256, 0, st>>>(s4, t2, perm_t, tkeys, fsh, nt, Bl,
                                                             p1, inv_s, ffar, inv);
                PHF_HIP(hipGetLastError());
                return PHF_OK;
            };
            finish = [=](hipStream_t st) {
                out_gather_f32<<<div_up(nt, 256), 256, 0, st>>>(inv, nt, ffar, nsum, qr, qi,
                                                                vout);
                PHF_HIP(hipGetLastError());
                return PHF_OK;
            };
        } else {
            finish = [=](hipStream_t st) {
                out_scatter_f32<<<div_up(nt, 256), 256, 0, st>>>(s4, t2 ? perm_t : nullptr, nt,
                                                                 nsum, qr, qi, vout);
                PHF_HIP(hipGetLastError());
                return PHF_OK;
            };
        }
    } else {
        const double4 *s4 = (const double4 *)src;
        const double2 *t2 = (const double2 *)tgt;
        const double2 *Bl = far ? (const double2 *)B + off[Lv] * p1 : nullptr;
        const int32_t *ss = S.start;
        const double4 *org = dom.org;
        const double s = dom.s;
        const uint32_t *tkeys = Tg.keys;
        const int fsh = 2 * Tg.fine;
        const int64_t nt = a.nt;
        double2 *nsum;
        PHF_ALLOC(nsum, L->arena, double2, (size_t)std::max<int64_t>(a.nt, 1));
        near = [=](hipStream_t st) {
            p2p_near_f64s<<<8 * nl8, 256, 0, st>>>(s4, ss, t2, ts, Lv, split, d_near, nnear, pp, P,
                                                   nsum);
            PHF_HIP(hipGetLastError());
            return PHF_OK;
        };
        finish = [=](hipStream_t st) {
            l2p_scatter_f64<<<div_up(nt, 256), 256, 0, st>>>(t2, tkeys, fsh, perm_t, nt, org, s,
                                                             Bl, p1, nsum, qr, qi, vout);
            PHF_HIP(hipGetLastError());
            return PHF_OK;
        };
    }
    tm.end(PHF_STAGE_TREE);
    // without a split: the far field goes to the second stream
    const bool fork = !spl && near;
    int rc = PHF_OK;
    if (spl) {
        rc = spl->mid();
    } else if (fork) {
        // the near field is enqueued first, so that it starts as soon as
        // the tree is done
        rc = fmm_far_fork(L);
        if (rc == PHF_OK) rc = fmm_near(L, near, tm);
        if (rc != PHF_OK) (void)fmm_far_done(L);  // the fork is left balanced
    }
    PHF_TRY(rc);

    // far field (on the lane's stream, or the second stream while the two
    // are swapped); a failure still restores and joins them
    auto far_field = [&]() -> int {
        if (!far) return PHF_OK;
        // P2M
        tm.begin(PHF_STAGE_P2M);
        used[PHF_STAGE_P2M] = true;
        PHF_TRY(p2m_dispatch(p1, [&](auto ni) {
            p2m_kernel<T, decltype(ni)::value><<<nleaf / 4, 256, 0, L->stream>>>(
                src, sp, p1, dom.org, dom.s, 1.0 / dom.s, M + off[Lv] * p1);
        }));
        PHF_HIP(hipGetLastError());
        tm.end(PHF_STAGE_P2M);
        // M2M up to level 2, three levels per launch
        tm.begin(PHF_STAGE_M2M);
        used[PHF_STAGE_M2M] = true;
        for (int from = Lv; from > 2;) {
            UpLevels u{};
            u.nlev = std::min(3, from - 2);
            u.lev0 = from - u.nlev;
            u.from = from;
            u.off_from = off[from];
            for (int i = 0; i < u.nlev; ++i) u.off[i] = off[u.lev0 + i];
            PHF_TRY(shift_dispatch(p1, [&](auto mt) {
                m2m_kernel<T, decltype(mt)::value>
                    <<<1u << (2 * u.lev0), 256, 0, L->stream>>>(u, p1, M, d_pas);
            }));
            from -= u.nlev;
        }
        tm.end(PHF_STAGE_M2M);
        // M2L at every level >= 2 (writes B)
        tm.begin(PHF_STAGE_M2L);
        used[PHF_STAGE_M2L] = true;
        M2LLevels lv{};
        lv.nlev = Lv - 1;
        lv.lev0 = 2;
        for (int l = 2; l <= Lv; ++l) {
            const int i = l - 2;
            lv.coff[i] = off[l];
            lv.il_base[i] = il_base[l];
            lv.il_max[i] = il_max[l];
            lv.shift[i] = 2 * (Lv - l);
            lv.inv_r[i] = 1.0 / (dom.D / std::ldexp(1.0, l));
        }
        if (sizeof(T) == 4 && p1 == 17) {
            // lane-per-box form (float32, order 16)
            constexpr int MW = 4;
            lv.blk[0] = 0;
            for (int i = 0; i < lv.nlev; ++i) {
                const int64_t per = (int64_t(1) << (2 * (i + 2))) / 4;
                lv.blk[i + 1] = lv.blk[i] + (per + 63) / 64;
            }
            const dim3 grid((unsigned)lv.blk[lv.nlev], 4, (17 + MW - 1) / MW);
            m2l_box_kernel<float, 17, MW><<<grid, 64, 0, L->stream>>>(
                lv, (const float2 *)M, (float2 *)B, S.start, Tg.start, d_il, d_iloff,
                (const float2 *)d_U, R, (const float *)d_bin);
            PHF_HIP(hipGetLastError());
        } else {
            PHF_TRY(m2l_dispatch<T>(L, lv, p1, M, B, S.start, Tg.start, d_il, d_iloff, d_U, R,
                                    d_bin));
        }
        tm.end(PHF_STAGE_M2L);
        tm.begin(PHF_STAGE_L2L);
        used[PHF_STAGE_L2L] = true;
        // L2L down to the leaves, three levels per launch, the remainder first
        for (int lev = 2; lev < Lv;) {
            DownLevels dl{};
            dl.nlev = (Lv - lev) % 3 ? (Lv - lev) % 3 : 3;
            dl.lev0 = lev;
            for (int i = 0; i <= dl.nlev; ++i) dl.off[i] = off[lev + i];
            PHF_TRY(shift_dispatch(p1, [&](auto mt) {
                l2l_kernel<T, decltype(mt)::value>
                    <<<1u << (2 * lev), 256, 0, L->stream>>>(dl, p1, B, d_pas);
            }));
            lev += dl.nlev;
        }
        if (far_tail) PHF_TRY(far_tail(L->stream));
        tm.end(PHF_STAGE_L2L);
        return PHF_OK;
    };
    if (fork) std::swap(L->stream, L->stream2);
    rc = far_field();
    if (fork) std::swap(L->stream, L->stream2);
    if (spl) {
        spl->near = near;
        spl->finish = finish;
        return rc;
    }
    if (fork) {
        const int dr = fmm_far_done(L);
        const int jr = dr == PHF_OK ? fmm_far_join(L) : dr;
        PHF_TRY(rc);
        PHF_TRY(jr);
        return finish(L->stream);
    }
    PHF_TRY(rc);
    tm.begin(PHF_STAGE_P2P);
    rc = finish(L->stream);
    tm.end(PHF_STAGE_P2P);
    return rc;
}

// Tree and FMM from the domain on (every launch after the bounding box);
// spl as run_fmm_typed.
static int fmm_enqueue(Lane *L, const FmmArgs &a, const Domain &dom_in, StageTimer &tm,
                       bool *used, FmmInfo *info, FmmSplit *spl, int *nnear)
{
    // points in Morton order inside the leaves too, with the key bits the
    // radix passes leave free: targets that share a wave, and sources taken
    // together, sit close, so that more pair batches skip the smoothing
    // exponential
    const Domain dom = [&] {
        Domain d = dom_in;
        const int kb = 2 * d.L, spare = (kb + 7) / 8 * 8 - kb;
        d.fine = std::min(3, spare / 2);
        return d;
    }();
    SortedPoints S, Tg;
    S.want_split = a.same;
    if (a.prec == PHF_PREC_F32C)
        PHF_TRY(build_sorted_payload(L, dom, a.xb, a.yb, a.wb, a.nb, &S));
    else
        PHF_TRY(build_sorted_points(L, dom, a.xb, a.yb, a.nb, &S));
    if (a.same) {
        Tg = S;
        if (info) {
            info->sorted_pay = S.pay;
            info->sorted_perm = S.pay ? nullptr : S.perm;
            info->sorted_n = a.nb;
        }
    } else {
        // the source build has completed the bounding box at dom.org
        Domain dt = dom;
        dt.parts = nullptr;
        dt.nparts = 0;
        Tg.want_split = true;
        PHF_TRY(build_sorted_points(L, dt, a.xt, a.yt, a.nt, &Tg));
    }
    if (info && info->want_counts) {
        PHF_ALLOC(info->d_counts, L->arena, unsigned long long, 2);
        PHF_HIP(hipMemsetAsync(info->d_counts, 0, 2 * sizeof(unsigned long long), L->stream));
    }
    if (a.prec == PHF_PREC_F32C)
        return run_fmm_typed<float>(L, a, dom, S, Tg, tm, used, info, spl, nnear);
    return run_fmm_typed<double>(L, a, dom, S, Tg, tm, used, info, spl, nnear);
}

// ------------------------------------------------------ captured graphs --
// A lane's recorded FMM launch sequences, in two graphs: bounding box and
// tree, then the far field.  A replay launches the tree graph on the lane's
// stream and then, for float32, the far-field graph on the lane's second
// stream beside the near field, which follows the tree on the lane's stream
// (launched eagerly, so that it is timed on its own), and the finishing
// kernel after both.  An entry is valid
// for the same inputs and outputs (addresses), sizes and parameters and
// the same arena state at the start (its buffers are the same arena
// slices).  A call replays the most recent entry without waiting for the
// bounding box: kernels read the domain corner on the device, and the
// bounding box comes back with the results, so that the caller can check
// that the points kept the recording's leaf level and domain side, from which
// the order of every sum follows (else it evaluates again with a fresh
// recording).
struct FmmGraph {
    FmmArgs a{};
    int L = 0, nnear = 0;
    double D = 0.0;
    Arena::Mark m0, m1;
    hipGraph_t g[2] = {};
    hipGraphExec_t exec[2] = {};
    char *tables = nullptr;     // device tables the graphs' kernels read
    double4 *bb = nullptr;      // the recorded bounding box (arena slot)
    bool bb_host = false;       // the graph also writes it to the pinned copy
    P2PLaunch near, finish;
    uint64_t last = 0;
};

struct FmmGraphCache {
    std::vector<FmmGraph *> v;
    uint64_t clock = 0;
    double4 *hb_host = nullptr;    // pinned copy of the replayed bounding box
};

constexpr size_t kFmmGraphs = 4;

// Destroys a recording and frees its tables; the lane's streams are waited
// for first, so no launch of the recording still reads them.
static void drop_graph(Lane *L, FmmGraph *e)
{
    (void)lane_quiesce(L);
    for (int k = 0; k < 2; ++k) {
        if (e->exec[k]) (void)hipGraphExecDestroy(e->exec[k]);
        if (e->g[k]) (void)hipGraphDestroy(e->g[k]);
    }
    if (e->tables) (void)hipFree(e->tables);
    delete e;
}

void fmm_graphs_release(Lane *L)
{
    (void)lane_quiesce(L);
    if (L->stream2) {
        (void)hipStreamSynchronize(L->stream2);
        (void)hipStreamDestroy(L->stream2);
        L->stream2 = nullptr;
    }
    fmm_plans_release(L);
    if (L->fork_ev) (void)hipEventDestroy(L->fork_ev);
    if (L->join_ev) (void)hipEventDestroy(L->join_ev);
    L->fork_ev = L->join_ev = nullptr;
    if (!L->fmm_graphs) return;
    for (FmmGraph *e : L->fmm_graphs->v) drop_graph(L, e);
    if (L->fmm_graphs->hb_host) (void)hipHostFree(L->fmm_graphs->hb_host);
    delete L->fmm_graphs;
    L->fmm_graphs = nullptr;
}

static bool same_args(const FmmArgs &x, const FmmArgs &y)
{
    return x.xb == y.xb && x.yb == y.yb && x.wb == y.wb && x.nb == y.nb && x.xt == y.xt &&
           x.yt == y.yt && x.nt == y.nt && x.same == y.same && x.xopt == y.xopt &&
           x.cutoff == y.cutoff && x.p == y.p && x.ws == y.ws && x.prec == y.prec &&
           x.Lhint == y.Lhint && x.leaf_side == y.leaf_side && x.qr == y.qr && x.qi == y.qi &&
           x.velocity_out == y.velocity_out;
}

// Record bounding box and tree, then the far field, for (a, dom) from the
// arena's current state.
static int fmm_record(Lane *L, const FmmArgs &a, const Domain &dom0, FmmGraph **out, bool *keep)
{
    FmmGraphCache &c = *L->fmm_graphs;
    // table uploads made while recording go through the lane's second
    // stream, idle then (it carries the far field of launches only)
    PHF_TRY(lane_stream2(L));
    FmmGraph *e = new FmmGraph;
    e->a = a;
    e->L = dom0.L;
    e->D = dom0.D;
    e->m0 = L->arena.mark();
    StageTimer off(L, false);
    bool used[PHF_STAGE_COUNT] = {};
    hipError_t be = hipStreamBeginCapture(L->stream, hipStreamCaptureModeRelaxed);
    if (be != hipSuccess) {
        delete e;
        PHF_HIP(be);
    }
    int part = 0;  // the graph being recorded
    int rc = PHF_OK;
    double4 *bb = L->arena.alloc<double4>(1);
    e->bb = bb;
    if (!bb) rc = PHF_ERR_NOMEM;
    // with sources, the bounding box is completed by the source tree build
    double4 *parts = nullptr;
    int np = 0;
    if (rc == PHF_OK && a.nb > 0)
        rc = device_bbox_parts(L, a.xb, a.yb, a.nb, a.same ? nullptr : a.xt,
                               a.same ? nullptr : a.yt, a.same ? 0 : a.nt, &parts, &np);
    else if (rc == PHF_OK)
        rc = device_bbox(L, a.xb, a.yb, a.nb, a.same ? nullptr : a.xt, a.same ? nullptr : a.yt,
                         a.same ? 0 : a.nt, bb);
    if (rc == PHF_OK) {
        Domain dom = dom0;
        dom.org = bb;
        dom.parts = parts;
        dom.nparts = np;
        // the source tree build also writes the box to the pinned copy
        dom.org_host = parts ? c.hb_host : nullptr;
        e->bb_host = parts != nullptr;
        FmmSplit spl;
        spl.tables_keep = &e->tables;
        spl.side = L->stream2;
        spl.mid = [&]() -> int {
            PHF_HIP(hipStreamEndCapture(L->stream, &e->g[0]));
            part = 1;
            PHF_HIP(hipStreamBeginCapture(L->stream, hipStreamCaptureModeRelaxed));
            part = 2;
            return PHF_OK;
        };
        rc = fmm_enqueue(L, a, dom, off, used, nullptr, &spl, &e->nnear);
        e->near = spl.near;
        e->finish = spl.finish;
        if (rc == PHF_OK && part != 2) {
            set_error("FMM recording did not reach the far field");
            rc = PHF_ERR_DEVICE;
        }
    }
    if (part != 1) {
        hipError_t ce = hipStreamEndCapture(L->stream, &e->g[part == 0 ? 0 : 1]);
        if (rc == PHF_OK && ce != hipSuccess) {
            set_error("HIP error %s ending the FMM graph capture", hipGetErrorName(ce));
            rc = PHF_ERR_DEVICE;
        }
    }
    for (int k = 0; k < 2 && rc == PHF_OK; ++k) {
        hipError_t ie = hipGraphInstantiate(&e->exec[k], e->g[k], nullptr, nullptr, 0);
        if (ie != hipSuccess) {
            set_error("HIP error %s instantiating the FMM graph", hipGetErrorName(ie));
            rc = PHF_ERR_DEVICE;
        }
    }
    if (rc != PHF_OK) {
        drop_graph(L, e);
        return rc;
    }
    e->m1 = L->arena.mark();
    e->last = ++c.clock;
    *out = e;
    // an arena that grew while recording is rebuilt by its next reset: the
    // graph then serves this call only
    *keep = e->m1.nblocks == e->m0.nblocks;
    if (*keep) {
        // one recording per argument set and arena state: the newest
        for (auto it = c.v.begin(); it != c.v.end();)
            if (same_args((*it)->a, a) && (*it)->m0.base0 == e->m0.base0 &&
                (*it)->m0.cur == e->m0.cur && (*it)->m0.top == e->m0.top) {
                drop_graph(L, *it);
                it = c.v.erase(it);
            } else {
                ++it;
            }
        if (c.v.size() >= kFmmGraphs) {
            auto lru = std::min_element(c.v.begin(), c.v.end(), [](FmmGraph *x, FmmGraph *y) {
                return x->last < y->last;
            });
            drop_graph(L, *lru);
            c.v.erase(lru);
        }
        c.v.push_back(e);
    }
    return PHF_OK;
}

// Launch a recorded entry: tree graph, near field beside the far-field
// graph, then the finishing kernel.
static int fmm_replay(Lane *L, FmmGraph *e, StageTimer &tm, int stage0)
{
    hipError_t le = hipGraphLaunch(e->exec[0], L->stream);
    tm.end(PHF_STAGE_TREE);
    if (le != hipSuccess) {
        set_error("HIP error %s launching the FMM tree graph", hipGetErrorName(le));
        return PHF_ERR_DEVICE;
    }
    int rc = PHF_OK;
    if (e->near) {
        // near field first (it starts as soon as the tree is done), then the
        // far-field graph beside it
        PHF_TRY(fmm_far_fork(L));
        const int nr = fmm_near(L, e->near, tm);
        le = hipGraphLaunch(e->exec[1], L->stream2);
        tm.end_on(stage0, L->stream2);
        const int dr = fmm_far_done(L);
        if (le != hipSuccess) {
            set_error("HIP error %s launching the FMM far-field graph", hipGetErrorName(le));
            rc = PHF_ERR_DEVICE;
        }
        const int jr = dr == PHF_OK ? fmm_far_join(L) : dr;
        PHF_TRY(nr);
        PHF_TRY(rc);
        PHF_TRY(jr);
        return e->finish(L->stream);
    }
    le = hipGraphLaunch(e->exec[1], L->stream);
    tm.end(stage0);
    if (le != hipSuccess) {
        set_error("HIP error %s launching the FMM far-field graph", hipGetErrorName(le));
        rc = PHF_ERR_DEVICE;
    }
    PHF_TRY(rc);
    tm.begin(PHF_STAGE_P2P);
    rc = e->finish(L->stream);
    tm.end(PHF_STAGE_P2P);
    return rc;
}

int fmm_device(Lane *L, const FmmArgs &a, StageTimer &tm, bool *used, FmmInfo *info)
{
    if (a.nt == 0) return PHF_OK;
    const bool graph = info && info->graph && !info->want_counts;
    const int stage0 = graph ? PHF_STAGE_TREE_FAR : PHF_STAGE_TREE;
    const double shape_log2 = 1.4426950408889634074 * make_oseen_params(a.xopt, a.cutoff).inv_ks;
    FmmGraph *e = nullptr;
    bool keep = true;
    if (graph) {
        if (!L->fmm_graphs) L->fmm_graphs = new FmmGraphCache;
        FmmGraphCache &c = *L->fmm_graphs;
        if (!c.hb_host) PHF_HIP(hipHostMalloc(&c.hb_host, 256, hipHostMallocCoherent));
        if (!info->no_speculation)
            for (FmmGraph *g : c.v)
                if (same_args(g->a, a) && L->arena.at(g->m0)) e = g;
        if (e) {
            // replay without waiting for the bounding box
            L->arena.jump(e->m0, e->m1);
            e->last = ++c.clock;
            tm.begin(stage0);
        }
    }
    Domain dom{};
    if (!e) {
        // 1. bounding box of sources and targets -> domain
        tm.begin(stage0);
        const Arena::Mark m0 = L->arena.mark();
        double4 *bb;
        PHF_ALLOC(bb, L->arena, double4, 1);
        PHF_TRY(device_bbox(L, a.xb, a.yb, a.nb, a.same ? nullptr : a.xt,
                            a.same ? nullptr : a.yt, a.same ? 0 : a.nt, bb));
        double4 hb;
        PHF_HIP(hipMemcpyAsync(&hb, bb, sizeof(double4), hipMemcpyDeviceToHost, L->stream));
        PHF_HIP(hipStreamSynchronize(L->stream));
        dom = choose_domain(hb, a.Lhint, (double)a.nb, (double)a.nt, a.cutoff, a.ws, shape_log2,
                            a.p + 1, a.prec == PHF_PREC_F32C ? 16 : 64, a.leaf_side);
        dom.org = bb;
        if (graph) {
            // the recording computes the bounding box again in its own slot
            L->arena.jump(L->arena.mark(), m0);
            PHF_TRY(fmm_record(L, a, dom, &e, &keep));
        }
    }
    int nnear = 0;
    if (e) {
        tm.begin(PHF_STAGE_TREE);  // the tree graph
        int rc = fmm_replay(L, e, tm, stage0);
        if (rc == PHF_OK) {
            double4 *hb = L->fmm_graphs->hb_host;
            const hipError_t fe = e->bb_host ? hipSuccess
                                             : hipMemcpyAsync(hb, e->bb, sizeof(double4),
                                                              hipMemcpyDeviceToHost, L->stream);
            if (fe != hipSuccess) {
                set_error("HIP error %s reading the bounding box", hipGetErrorName(fe));
                rc = PHF_ERR_DEVICE;
            }
            const int L0 = e->L;
            const double D0 = e->D;
            info->domain_ok = [hb, a, L0, D0, shape_log2]() {
                const Domain d = choose_domain(*hb, a.Lhint, (double)a.nb, (double)a.nt,
                                               a.cutoff, a.ws, shape_log2, a.p + 1,
                                               a.prec == PHF_PREC_F32C ? 16 : 64, a.leaf_side);
                return d.L == L0 && d.D == D0;
            };
        }
        nnear = e->nnear;
        dom.L = e->L;
        dom.D = e->D;
        if (!keep) {
            // the graphs and their tables must outlive the launches
            const int qr = lane_quiesce(L);
            drop_graph(L, e);
            if (rc == PHF_OK) PHF_TRY(qr);
        }
        PHF_TRY(rc);
        used[PHF_STAGE_TREE_FAR] = used[PHF_STAGE_TREE] = used[PHF_STAGE_P2P] = true;
        info->sorted_pay = nullptr;
        info->sorted_perm = nullptr;
        info->sorted_n = 0;
    } else {
        used[PHF_STAGE_TREE] = used[PHF_STAGE_P2P] = true;
        PHF_TRY(fmm_enqueue(L, a, dom, tm, used, info, nullptr, &nnear));
    }
    if (info) {
        info->L = dom.L;
        info->p = a.p;
        info->nnear = nnear;
        info->D = dom.D;
    }
    return PHF_OK;
}

}  // namespace phf

// ------------------------------------------------------------ C entry ----
using namespace phf;

extern "C" int phf_fmm2d(const double *xb, const double *yb, const double *wb, int64_t nb,
                         const double *xt, const double *yt, int64_t nt, int32_t ndirect,
                         double xopt, double cutoff, double tol, const phf_fmm_opts *opts,
                         double *qr, double *qi)
{
    clear_error();
    PHF_REQUIRE(nb >= 0 && nt >= 0 && nb < (int64_t(1) << 31) && nt < (int64_t(1) << 31),
                "sizes out of range (nb=%lld, nt=%lld)", (long long)nb, (long long)nt);
    PHF_REQUIRE(std::isfinite(xopt) && xopt > 0.0, "xopt must be finite and > 0 (got %g)", xopt);
    PHF_REQUIRE(std::isfinite(cutoff) && cutoff >= 0.0, "cutoff must be finite and >= 0 (got %g)",
                cutoff);
    PHF_REQUIRE(std::isfinite(tol) && tol >= 0.0, "tol must be finite and >= 0 (got %g)", tol);
    phf_fmm_opts o{0, 0, PHF_PREC_F64, 0};
    if (opts) o = *opts;
    PHF_REQUIRE(o.prec == PHF_PREC_F64 || o.prec == PHF_PREC_F32C, "unknown precision %d",
                o.prec);
    PHF_REQUIRE(o.order <= 40, "order must be <= 40 (got %d)", o.order);
    PHF_REQUIRE(o.ws <= 3, "ws must be <= 3 (got %d)", o.ws);
    PHF_TRY(check_host_array(xb, nb, "xBlob"));
    PHF_TRY(check_host_array(yb, nb, "yBlob"));
    PHF_TRY(check_host_array(wb, nb, "wBlob"));
    PHF_TRY(check_host_array(xt, nt, "xTarget"));
    PHF_TRY(check_host_array(yt, nt, "yTarget"));
    PHF_REQUIRE(nt == 0 || (qr && qi), "output arrays are NULL");
    if (nt == 0) return PHF_OK;
    const bool same = (xb == xt && yb == yt && nb == nt);

    LaneGuard g;
    PHF_TRY(g.rc);
    Lane *L = g.lane;
    PHF_TRY(reset_arena(L));
    StageTimer tm(L, timing_enabled());
    bool used[PHF_STAGE_COUNT] = {};
    used[PHF_STAGE_UPLOAD] = used[PHF_STAGE_DOWNLOAD] = used[PHF_STAGE_TOTAL] = true;
    tm.begin(PHF_STAGE_TOTAL);
    tm.begin(PHF_STAGE_UPLOAD);
    double *dxb, *dyb, *dwb, *dxt, *dyt, *dqr, *dqi;
    PHF_TRY(copy_points_in(L, xb, yb, wb, nb, xt, yt, nt, &dxb, &dyb, &dwb, &dxt, &dyt));
    PHF_ALLOC(dqr, L->arena, double, (size_t)nt * 2);
    dqi = dqr + nt;
    tm.end(PHF_STAGE_UPLOAD);
    if (tol == 0.0) {
        // direct sum over all pairs (direct.cpp:1409-1450)
        tm.begin(PHF_STAGE_P2P);
        used[PHF_STAGE_P2P] = true;
        PairParams pp = make_oseen_params(xopt, cutoff);
        PHF_TRY(direct_device(L, PAIR_OSEEN, o.prec, pp, dxb, dyb, dwb, nb, dxt, dyt, nt, dqr,
                              dqi, mostly_far(xb, yb, nb, xt, yt, nt, pp.c2)));
        tm.end(PHF_STAGE_P2P);
    } else {
        FmmArgs a{};
        a.xb = dxb; a.yb = dyb; a.wb = dwb; a.nb = nb;
        a.xt = dxt; a.yt = dyt; a.nt = nt; a.same = same;
        a.xopt = xopt; a.cutoff = cutoff;
        a.p = o.order > 0 ? o.order : fmm_order_from_tol(tol);
        a.ws = o.ws > 0 ? o.ws : 1;
        a.prec = o.prec;
        a.Lhint = fmm_level(nb, o.leaf, ndirect);
        a.qr = dqr;
        a.qi = dqi;
        PHF_TRY(fmm_device(L, a, tm, used, nullptr));
    }
    tm.begin(PHF_STAGE_DOWNLOAD);
    PHF_TRY(copy_out(L, {{qr, dqr, sizeof(double) * nt}, {qi, dqi, sizeof(double) * nt}}));
    tm.end(PHF_STAGE_DOWNLOAD);
    tm.end(PHF_STAGE_TOTAL);
    if (tm.on) PHF_HIP(hipStreamSynchronize(L->stream));
    record_stage_times(L, used);
    return PHF_OK;
}
