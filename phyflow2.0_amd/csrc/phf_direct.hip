// phf_direct.hip -- all-pairs vortex-blob velocity sums on gfx950.
//
// Replaces the reference's direct kernels:
//   * vv2par_kernel (Gaussian, EPS-regularised),
//     src/cpp/blobs/cuda/vv2parGauss_gpu/vv2parGauss_device.cu:41-162
//   * direct_pot1_nomi_oseen_synchronized (fmm2d with tol == 0, Oseen),
//     src/cpp/blobs/c++/fmm2d_py_cpu_gpu/cudaevalkernels.h:61-71, 451-508.
//
// Mapping to CDNA4: one wave64 owns TPL*64 targets held in VGPRs; all
// lanes walk the same source sequence, so each source is fetched once per
// wave with scalar (SMEM) loads and broadcast through SGPR operands: no LDS
// staging and no barriers.  Long source lists are split over a second grid
// dimension; each (target block, source chunk) writes a float64 partial and
// a finishing pass adds the partials in a fixed order, so results do not
// depend on scheduling.
//
// Precision modes
//   F64 : float64 pair arithmetic (w / r2 from the hardware estimate of 1 / r2
//         and its two-term correction).
//   F32C: coordinates differenced in float64 and rounded once, pair
//         arithmetic in float32 (v_exp_f32, v_rcp_f32), sums in blocks of
//         16 terms folded into a TwoSum (hi, lo) accumulator per target.
#include "phf_host.hpp"
#include "phf_ops.hpp"
#include "phf_tree.hpp"

#include <algorithm>
#include <cmath>

namespace phf {

// one source as a kernel uses it, read in place from the x, y, w arrays
struct alignas(32) Src64 {
    double x, y, w, pad;
};
struct alignas(8) Src32c {
    double x, y;
    float w, pad;
};

PairParams make_gauss_params(double ksigmasqr)
{
    PairParams p{};
    p.eps = 1e-12;
    p.inv_ks = 1.0 / ksigmasqr;
    p.c2 = 0.0;
    p.scale = 1.0;
    p.eps_f = (float)p.eps;
    p.nlog2e_ks_f = (float)(-1.4426950408889634074 / ksigmasqr);
    p.c2_f = 0.0f;
    p.scale_f = 1.0f;
    return p;
}

PairParams make_oseen_params(double xopt, double cutoff)
{
    // fmm.cpp:1166-1179 (pot=1, OSEEN, INLINECOMPLEX_DIRECT, cont=true)
    PairParams p{};
    p.eps = 0.0;
    p.c2 = cutoff * cutoff;
    p.inv_ks = 1.2564312086261696770 / (xopt * xopt);
    p.scale = -1.0 / std::expm1(-p.inv_ks * p.c2);
    p.eps_f = 0.0f;
    p.nlog2e_ks_f = (float)(-1.4426950408889634074 * p.inv_ks);
    p.c2_f = (float)p.c2;
    p.scale_f = (float)p.scale;
    p.f32_nocut = (p.scale_f == 1.0f && p.c2 * p.inv_ks * 1.4426950408889634074 > 25.5) ? 1 : 0;
    return p;
}

// ------------------------------------------------------ F32C kernel ------
template <int KIND, int TPL>
__global__ __launch_bounds__(64) void direct_f32c(
    const double *__restrict__ xb, const double *__restrict__ yb, const double *__restrict__ wb,
    int64_t nb, const double *__restrict__ xt,
    const double *__restrict__ yt, int64_t nt, int64_t chunk_len, PairParams pp,
    double2 *__restrict__ part)
{
    const int lane = threadIdx.x;
    const int64_t tbase = (int64_t)blockIdx.x * (kWave * TPL);
    double tx[TPL], ty[TPL];
    float hu[TPL], lu[TPL], hv[TPL], lv[TPL];
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
        int64_t t = tbase + lane + kWave * i;
        tx[i] = t < nt ? xt[t] : 0.0;
        ty[i] = t < nt ? yt[t] : 0.0;
        hu[i] = lu[i] = hv[i] = lv[i] = 0.0f;
    }
    const int64_t j0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t j1 = min(nb, j0 + chunk_len);
    int64_t j = j0;
    for (; j + 16 <= j1; j += 16) {
        float au[TPL], av[TPL];
#pragma unroll
        for (int i = 0; i < TPL; ++i) au[i] = av[i] = 0.0f;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const Src32c s{xb[j + k], yb[j + k], (float)wb[j + k], 0.0f};
#pragma unroll
            for (int i = 0; i < TPL; ++i) {
                float dx = (float)(tx[i] - s.x);
                float dy = (float)(ty[i] - s.y);
                float P = pair_f32<KIND>(dx, dy, s.w, pp);
                au[i] = __builtin_fmaf(P, dx, au[i]);
                av[i] = __builtin_fmaf(P, dy, av[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < TPL; ++i) {
            two_sum_add(hu[i], lu[i], au[i]);
            two_sum_add(hv[i], lv[i], av[i]);
        }
    }
    if (j < j1) {
        float au[TPL], av[TPL];
#pragma unroll
        for (int i = 0; i < TPL; ++i) au[i] = av[i] = 0.0f;
        for (; j < j1; ++j) {
            const Src32c s{xb[j], yb[j], (float)wb[j], 0.0f};
#pragma unroll
            for (int i = 0; i < TPL; ++i) {
                float dx = (float)(tx[i] - s.x);
                float dy = (float)(ty[i] - s.y);
                float P = pair_f32<KIND>(dx, dy, s.w, pp);
                au[i] = __builtin_fmaf(P, dx, au[i]);
                av[i] = __builtin_fmaf(P, dy, av[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < TPL; ++i) {
            two_sum_add(hu[i], lu[i], au[i]);
            two_sum_add(hv[i], lv[i], av[i]);
        }
    }
    double2 *out = part + (int64_t)blockIdx.y * nt;
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
        int64_t t = tbase + lane + kWave * i;
        if (t < nt)
            out[t] = make_double2((double)hu[i] + (double)lu[i], (double)hv[i] + (double)lv[i]);
    }
}

// ------------------------------------------------------- F64 kernel ------
template <int KIND, int TPL>
__global__ __launch_bounds__(64) void direct_f64(
    const double *__restrict__ xb, const double *__restrict__ yb, const double *__restrict__ wb,
    int64_t nb, const double *__restrict__ xt,
    const double *__restrict__ yt, int64_t nt, int64_t chunk_len, PairParams pp,
    double2 *__restrict__ part)
{
    const int lane = threadIdx.x;
    const int64_t tbase = (int64_t)blockIdx.x * (kWave * TPL);
    double tx[TPL], ty[TPL], au[TPL], av[TPL];
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
        int64_t t = tbase + lane + kWave * i;
        tx[i] = t < nt ? xt[t] : 0.0;
        ty[i] = t < nt ? yt[t] : 0.0;
        au[i] = av[i] = 0.0;
    }
    const int64_t j0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t j1 = min(nb, j0 + chunk_len);
    int64_t j = j0;
    for (; j + 8 <= j1; j += 8) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const Src64 s{xb[j + k], yb[j + k], wb[j + k], 0.0};
#pragma unroll
            for (int i = 0; i < TPL; ++i) {
                double dx = tx[i] - s.x;
                double dy = ty[i] - s.y;
                double P = pair_f64<KIND>(dx, dy, s.w, pp);
                au[i] = __builtin_fma(P, dx, au[i]);
                av[i] = __builtin_fma(P, dy, av[i]);
            }
        }
    }
    for (; j < j1; ++j) {
        const Src64 s{xb[j], yb[j], wb[j], 0.0};
#pragma unroll
        for (int i = 0; i < TPL; ++i) {
            double dx = tx[i] - s.x;
            double dy = ty[i] - s.y;
            double P = pair_f64<KIND>(dx, dy, s.w, pp);
            au[i] = __builtin_fma(P, dx, au[i]);
            av[i] = __builtin_fma(P, dy, av[i]);
        }
    }
    double2 *out = part + (int64_t)blockIdx.y * nt;
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
        int64_t t = tbase + lane + kWave * i;
        if (t < nt) out[t] = make_double2(au[i], av[i]);
    }
}

// ------------------------------------- F64 kernel, targets in Morton order --
// The smoothing factor 1 - exp(-r2/ks) costs more than the rest of a pair
// and rounds to 1 beyond r2 = 40 ks (Gaussian) or is 1 beyond the cutoff
// (Oseen), which a wave of scattered targets rarely agrees on.  With the
// targets of a wave close together (perm: target t of the sorted order is
// xt[perm[t]]) most sources are beyond it for all 64: four sources at a time
// are tested and, when no lane is inside, their pairs skip the factor; the
// same P either way.  The partials are in sorted target order.
// Bound by float64 issue: 15 operations and a reciprocal estimate per pair
// beyond it, 36 inside.  20,011 sources, 30,017 targets: 731 us for the call's
// kernels in input order, 430 us sorted (45 us of it the sort); 40,000 x
// 80,000: 3,829 against 1,708 us.
template <int KIND>
__global__ __launch_bounds__(64) void direct_f64_sorted(
    const double *__restrict__ xb, const double *__restrict__ yb, const double *__restrict__ wb,
    int64_t nb, const double *__restrict__ xt, const double *__restrict__ yt,
    const int32_t *__restrict__ perm, int64_t nt, int64_t chunk_len, PairParams pp,
    double2 *__restrict__ part)
{
    const int64_t t = (int64_t)blockIdx.x * kWave + threadIdx.x;
    const int32_t o = perm[t < nt ? t : nt - 1];
    const double tx = xt[o], ty = yt[o];
    // a pair at distance 0 (Oseen) always takes the full form
    const double in2 = KIND == PAIR_GAUSS_EPS ? 40.0 / pp.inv_ks : fmax(pp.c2, 1e-300);
    const double eps = KIND == PAIR_GAUSS_EPS ? pp.eps : 0.0;
    double au = 0.0, av = 0.0;
    const int64_t j0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t j1 = min(nb, j0 + chunk_len);
    int64_t j = j0;
    // the next four sources' scalar loads go out before the current pairs
    double nx[4], ny[4], nw[4];
    const int64_t jl = max(j0, j1 - 4);
    if (j + 4 <= j1)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            nx[k] = xb[j + k];
            ny[k] = yb[j + k];
            nw[k] = wb[j + k];
        }
    for (; j + 4 <= j1; j += 4) {
        double dx[4], dy[4], r2[4], w[4], sx[4], sy[4];
        const int64_t jn = min(j + 4, jl);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            sx[k] = nx[k];
            sy[k] = ny[k];
            w[k] = nw[k];
            nx[k] = xb[jn + k];
            ny[k] = yb[jn + k];
            nw[k] = wb[jn + k];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            dx[k] = tx - sx[k];
            dy[k] = ty - sy[k];
            r2[k] = __builtin_fma(dx[k], dx[k], fma3_f64(dy[k], dy[k], eps));
        }
        const double least = __builtin_fmin(__builtin_fmin(r2[0], r2[1]),
                                            __builtin_fmin(r2[2], r2[3]));
        if (__ballot(least < in2)) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const double P = pair_f64<KIND>(dx[k], dy[k], w[k], pp);
                au = __builtin_fma(P, dx[k], au);
                av = __builtin_fma(P, dy[k], av);
            }
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const double P = div_f64(w[k], r2[k]);
                au = __builtin_fma(P, dx[k], au);
                av = __builtin_fma(P, dy[k], av);
            }
        }
    }
    for (; j < j1; ++j) {
        const double dx = tx - xb[j], dy = ty - yb[j];
        const double P = pair_f64<KIND>(dx, dy, wb[j], pp);
        au = __builtin_fma(P, dx, au);
        av = __builtin_fma(P, dy, av);
    }
    if (t < nt) part[(int64_t)blockIdx.y * nt + t] = make_double2(au, av);
}

// Adds the chunk partials and maps (A, B) = (sum P dx, sum P dy) to the
// reference outputs:
//   Gaussian: vx = inv_2pi * (-B), vy = inv_2pi * A  (vv2parGauss_C_cpu.c:150-151)
//   cutoff:   the same                               (vv2par_C_cpu.c:149-150)
//   Oseen:    qr = -A,  qi = B                       (direct.cpp:1482-1483)
// A workgroup of 4 waves serves 64 targets: wave w adds the w-th quarter of
// the chunks in chunk order (coalesced rows, eight loads in flight), and
// the four quarter sums are added in wave order, so the result is fixed
// for a given chunking.  perm (nullable): partials of target perm[t].
constexpr int FIN_T = 64;  // targets per finishing workgroup
__global__ __launch_bounds__(256) void direct_finish(const double2 *__restrict__ part,
                                                     int nchunk, int64_t nt, int kind,
                                                     const int32_t *__restrict__ perm,
                                                     double *__restrict__ o0,
                                                     double *__restrict__ o1)
{
    __shared__ double2 red[4][FIN_T];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * FIN_T + l;
    const int per = (nchunk + 3) / 4;
    const int c1 = min(nchunk, (w + 1) * per);
    double a = 0.0, b = 0.0;
    if (t < nt) {
        int c = w * per;
        for (; c + 8 <= c1; c += 8) {
            double2 p[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) p[u] = part[(int64_t)(c + u) * nt + t];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                a += p[u].x;
                b += p[u].y;
            }
        }
        for (; c < c1; ++c) {
            const double2 p = part[(int64_t)c * nt + t];
            a += p.x;
            b += p.y;
        }
    }
    red[w][l] = make_double2(a, b);
    __syncthreads();
    if (w != 0 || t >= nt) return;
    a = ((red[0][l].x + red[1][l].x) + red[2][l].x) + red[3][l].x;
    b = ((red[0][l].y + red[1][l].y) + red[2][l].y) + red[3][l].y;
    const int64_t o = perm ? perm[t] : t;
    if (kind == PAIR_GAUSS_EPS || kind == PAIR_CUTOFF) {
        const double inv_2pi = 0.5 / 3.141592653589793;
        o0[o] = inv_2pi * (-b);
        o1[o] = inv_2pi * a;
    } else {
        o0[o] = -a;
        o1[o] = b;
    }
}

// ------------------------------------------------ vorticity (Gaussian) ----
// ww2parGauss_C_cpu.c:133-145:
//   w(t) = (1/pi) sum_m w_m exp(-(|t - z_m|^2 + EPS)/ks) / ks,  EPS = 1e-12
// Same layout as the velocity kernels with one accumulator per target.
template <int TPL, bool CUT>
__global__ __launch_bounds__(64) void vort_f32c(const double *__restrict__ xb,
                                                const double *__restrict__ yb,
                                                const double *__restrict__ wb, int64_t nb,
                                                const double *__restrict__ xt,
                                                const double *__restrict__ yt, int64_t nt,
                                                int64_t chunk_len, PairParams pp,
                                                double *__restrict__ part)
{
    const int lane = threadIdx.x;
    const int64_t tbase = (int64_t)blockIdx.x * (kWave * TPL);
    double tx[TPL], ty[TPL];
    float h[TPL], l[TPL];
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
        const int64_t t = tbase + lane + kWave * i;
        tx[i] = t < nt ? xt[t] : 0.0;
        ty[i] = t < nt ? yt[t] : 0.0;
        h[i] = l[i] = 0.0f;
    }
    const int64_t j0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t j1 = min(nb, j0 + chunk_len);
    for (int64_t j = j0; j < j1; j += 16) {
        const int64_t je = min(j1, j + 16);
        float a[TPL];
#pragma unroll
        for (int i = 0; i < TPL; ++i) a[i] = 0.0f;
        for (int64_t k = j; k < je; ++k) {
            const Src32c s{xb[k], yb[k], (float)wb[k], 0.0f};
#pragma unroll
            for (int i = 0; i < TPL; ++i) {
                const float dx = (float)(tx[i] - s.x), dy = (float)(ty[i] - s.y);
                const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, pp.eps_f));
                const float f = CUT ? __builtin_amdgcn_rsqf(r2) : exp2_f32(r2 * pp.nlog2e_ks_f);
                a[i] = __builtin_fmaf(s.w, f, a[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < TPL; ++i) two_sum_add(h[i], l[i], a[i]);
    }
    double *out = part + (int64_t)blockIdx.y * nt;
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
        const int64_t t = tbase + lane + kWave * i;
        if (t < nt) out[t] = (double)h[i] + (double)l[i];
    }
}

template <int TPL, bool CUT>
__global__ __launch_bounds__(64) void vort_f64(const double *__restrict__ xb,
                                               const double *__restrict__ yb,
                                               const double *__restrict__ wb, int64_t nb,
                                               const double *__restrict__ xt,
                                               const double *__restrict__ yt, int64_t nt,
                                               int64_t chunk_len, PairParams pp,
                                               double *__restrict__ part)
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x;
    const int64_t tbase = (int64_t)blockIdx.x * (kWave * TPL);
    double tx[TPL], ty[TPL], a[TPL];
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
        const int64_t t = tbase + lane + kWave * i;
        tx[i] = t < nt ? xt[t] : 0.0;
        ty[i] = t < nt ? yt[t] : 0.0;
        a[i] = 0.0;
    }
    const int64_t j0 = (int64_t)blockIdx.y * chunk_len;
    const int64_t j1 = min(nb, j0 + chunk_len);
    for (int64_t j = j0; j < j1; ++j) {
        const Src64 s{xb[j], yb[j], wb[j], 0.0};
#pragma unroll
        for (int i = 0; i < TPL; ++i) {
            const double dx = tx[i] - s.x, dy = ty[i] - s.y;
            const double r2 = dx * dx + dy * dy + pp.eps;
            a[i] += CUT ? s.w / sqrt(r2) : s.w * exp_neg_f64(-r2 * pp.inv_ks);
        }
    }
    double *out = part + (int64_t)blockIdx.y * nt;
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
        const int64_t t = tbase + lane + kWave * i;
        if (t < nt) out[t] = a[i];
    }
}

// chunk partials in chunk order, then inv_pi * w / ks (ww2parGauss_C_cpu.c:144)
// or, for the cutoff kernel, inv_2pi * w (ww2par_C_cpu.c:144)
__global__ void vort_finish(const double *__restrict__ part, int nchunk, int64_t nt, double ks,
                            int cut, double *__restrict__ w)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    double a = 0.0;
    int c = 0;
    for (; c + 8 <= nchunk; c += 8) {
        double p[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) p[u] = part[(int64_t)(c + u) * nt + t];
#pragma unroll
        for (int u = 0; u < 8; ++u) a += p[u];
    }
    for (; c < nchunk; ++c) a += part[(int64_t)c * nt + t];
    if (cut) {
        const double inv_2pi = 0.5 / 3.141592653589793;
        w[t] = inv_2pi * a;
    } else {
        const double inv_pi = 1.0 / 3.141592653589793;
        w[t] = inv_pi * a / ks;
    }
}

// ------------------------------------ vorticity of near sources only -----
// A Gaussian term of a source at r2 > kVortCut ks is below 2^-100 |w|, so all
// of them together are below 2^-100 W, W = sum |w|: they cannot change a sum
// of at least 2^-46 W beyond 2^-54 of its value.  Sources and targets are
// sorted in Morton order; a wave of 64 targets takes only the blocks of 64
// sources whose box comes within that radius of its own.  Groups with a target
// whose sum is too small for the argument (outside the flow, cancellation) go
// over the blocks again, out to where a term is 0 in the class's arithmetic.
// A plotting grid that reaches beyond the flow has many of those.
// Whole calls, 100,003 sources and 90,601 targets in float64 / float32: every
// pair 10.0 / 3.2 ms; this way 0.64 / 0.53 ms inside the flow, 0.70 / 0.65 ms
// on a grid twice as wide, 0.40 ms beside it (8.3 and 10.7 ms in either class
// when each small sum took every source).  20,011 sources, 40,401 targets:
// 1.01 / 0.42 ms; 0.36 / 0.26, 0.38 / 0.30, 0.22 ms.
constexpr double kVortCut = 69.4;   // exp(-69.4) < 2^-100
// exp(-746) = 0 in float64; in float32 2^-150 = exp(-103.98) is 0, and r2 is
// within 2^-20 of its value
constexpr double kVortZero64 = 746.0, kVortZero32 = 106.0;
constexpr int kVortBlk = 64;       // sources per block

// Sorted source records of block b (padded with zero circulations at the last
// source), their box {xmin, xmax, ymin, ymax} and sum |w|: one wave each.
__global__ __launch_bounds__(256) void vort_pack(const double *__restrict__ xb,
                                                 const double *__restrict__ yb,
                                                 const double *__restrict__ wb,
                                                 const int32_t *__restrict__ perm, int64_t nb,
                                                 int nblk, double4 *__restrict__ rec,
                                                 double4 *__restrict__ box,
                                                 double *__restrict__ wabs)
{
    const int lane = threadIdx.x & 63;
    const int b = (int)(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (b >= nblk) return;
    const int64_t q = (int64_t)b * kVortBlk + lane;
    const int32_t j = perm[q < nb ? q : nb - 1];
    const double x = xb[j], y = yb[j], w = q < nb ? wb[j] : 0.0;
    rec[q] = make_double4(x, y, w, 0.0);
    double4 bx = make_double4(x, x, y, y);
    double s = fabs(w);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        bx.x = fmin(bx.x, __shfl_xor(bx.x, d));
        bx.y = fmax(bx.y, __shfl_xor(bx.y, d));
        bx.z = fmin(bx.z, __shfl_xor(bx.z, d));
        bx.w = fmax(bx.w, __shfl_xor(bx.w, d));
        s += __shfl_xor(s, d);
    }
    if (lane == 0) {
        box[b] = bx;
        wabs[b] = s;
    }
}

// Sum of a wave's TG targets (lane mod TG) over the blocks b = first (mod step)
// within cut2 of their box; lane / TG takes that part of a block's sources.
// F32: the arithmetic of vort_f32c, 16 terms to a TwoSum.
template <bool F32, int TG>
__device__ __forceinline__ double vort_sum(const double4 *__restrict__ rec,
                                           const double4 *__restrict__ box, int nblk, double tx,
                                           double ty, const PairParams &pp, double cut2, int first,
                                           int step)
{
    constexpr int NS = kVortBlk * TG / kWave;  // sources of a block per lane
    const int lane = threadIdx.x & 63;
    double x0 = tx, x1 = tx, y0 = ty, y1 = ty;
#pragma unroll
    for (int d = TG / 2; d > 0; d >>= 1) {
        x0 = fmin(x0, __shfl_xor(x0, d));
        x1 = fmax(x1, __shfl_xor(x1, d));
        y0 = fmin(y0, __shfl_xor(y0, d));
        y1 = fmax(y1, __shfl_xor(y1, d));
    }
    double a = 0.0;
    float h = 0.f, l = 0.f;
    for (int b0 = first; b0 < nblk; b0 += step * kWave) {
        const int bl = b0 + lane * step;
        bool near = false;
        if (bl < nblk) {
            const double4 bx = box[bl];
            const double gx = fmax(fmax(bx.x - x1, x0 - bx.y), 0.0);
            const double gy = fmax(fmax(bx.z - y1, y0 - bx.w), 0.0);
            near = gx * gx + gy * gy < cut2;
        }
        for (unsigned long long m = __ballot(near); m; m &= m - 1) {
            const int b = b0 + (__ffsll((long long)m) - 1) * step;  // the same in every lane
            const double4 *rb = rec + (int64_t)__builtin_amdgcn_readfirstlane(b) * kVortBlk;
            if (TG < kWave) rb += lane / TG * NS;
            if (F32) {
#pragma unroll 1
                for (int k0 = 0; k0 < NS; k0 += 16) {
                    float s = 0.f;
#pragma unroll
                    for (int k = 0; k < 16; ++k) {
                        const double4 q = rb[k0 + k];
                        const float dx = (float)(tx - q.x), dy = (float)(ty - q.y);
                        const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, pp.eps_f));
                        s = __builtin_fmaf((float)q.z, exp2_f32(r2 * pp.nlog2e_ks_f), s);
                    }
                    two_sum_add(h, l, s);
                }
            } else {
#pragma unroll 1
                for (int k0 = 0; k0 < NS; k0 += 4) {
                    double r2[4], w[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const double4 q = rb[k0 + k];
                        const double dx = tx - q.x, dy = ty - q.y;
                        w[k] = q.z;
                        r2[k] = __builtin_fma(dx, dx, fma3_f64(dy, dy, pp.eps));
                    }
                    const double least = __builtin_fmin(__builtin_fmin(r2[0], r2[1]),
                                                        __builtin_fmin(r2[2], r2[3]));
                    if (__ballot(least < cut2)) {
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            a = __builtin_fma(w[k], exp_neg_f64(-r2[k] * pp.inv_ks), a);
                    }
                }
            }
        }
    }
    return F32 ? (double)h + (double)l : a;
}

// Partial sums of 64 sorted targets over the near blocks b = blockIdx.y (mod
// gridDim.y), so that neighbouring blocks go to different waves.
template <bool F32>
__global__ __launch_bounds__(64) void vort_near(const double4 *__restrict__ rec,
                                                const double4 *__restrict__ box, int nblk,
                                                const double *__restrict__ xt,
                                                const double *__restrict__ yt,
                                                const int32_t *__restrict__ perm, int64_t nt,
                                                PairParams pp, double *__restrict__ part)
{
    const int64_t t = (int64_t)blockIdx.x * kWave + threadIdx.x;
    const int32_t o = perm[t < nt ? t : nt - 1];
    const double a = vort_sum<F32, kWave>(rec, box, nblk, xt[o], yt[o], pp, kVortCut / pp.inv_ks,
                                          (int)blockIdx.y, (int)gridDim.y);
    if (t < nt) part[(int64_t)blockIdx.y * nt + t] = a;
}

// The partials of sorted target t, scaled, to w[perm[t]]; a target whose sum
// is below 2^-46 W sets its bit of its group's need instead.
__global__ __launch_bounds__(256) void vort_near_finish(
    const double *__restrict__ part, int nchunk, int64_t nt, const int32_t *__restrict__ perm,
    const double *__restrict__ wabs, int nblk, double ks, double *__restrict__ w,
    unsigned long long *__restrict__ need)
{
    __shared__ double sh[256];
    double s = 0.0;
    for (int b = threadIdx.x; b < nblk; b += 256) s += wabs[b];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int d = 128; d > 0; d >>= 1) {
        if ((int)threadIdx.x < d) sh[threadIdx.x] += sh[threadIdx.x + d];
        __syncthreads();
    }
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= nt) return;
    double a = 0.0;
    for (int c = 0; c < nchunk; ++c) a += part[(int64_t)c * nt + t];
    const bool ok = fabs(a) >= sh[0] * 0x1p-46;
    const unsigned long long m = __ballot(!ok);
    if ((threadIdx.x & 63) == 0) need[t / kWave] = m;
    const double inv_pi = 1.0 / 3.141592653589793;
    if (ok) w[perm[t]] = inv_pi * a / ks;
}

// The targets in need, over every block that a term can come from: a workgroup
// takes sixteen at a time, its waves in turn over the blocks and added in wave
// order; lanes of targets that are not in need take the place of one that is.
// So a few of them keep many CUs busy: 20,011 sources, 40,401 targets, sigma three
// spacings, a grid half as wide again 876 / 436 us, 644 / 351 so (1,000 / 420 for
// every pair; 64 at a time by sixteen waves before).  Beside a flow, where every
// target is in need and no block near, the box tests are four times as many
// (100,003 sources, 90,601 targets: 373 and 398 us).
constexpr int kRestT = 16, kRestWaves = 8, kRestGrid = 2048;
template <bool F32>
__global__ __launch_bounds__(64 * kRestWaves) void vort_rest(
    const double4 *__restrict__ rec, const double4 *__restrict__ box, int nblk,
    const double *__restrict__ xt, const double *__restrict__ yt, const int32_t *__restrict__ perm,
    int64_t nt, PairParams pp, double ks, double *__restrict__ w,
    const unsigned long long *__restrict__ need)
{
    __shared__ double sh[kRestWaves][kRestT];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, i = lane % kRestT;
    for (int64_t t0 = (int64_t)blockIdx.x * kRestT; t0 < nt; t0 += (int64_t)gridDim.x * kRestT) {
        // (targets beyond nt are not in need)
        const uint32_t m = (uint32_t)(need[t0 / kWave] >> (t0 % kWave)) & ((1u << kRestT) - 1);
        if (m == 0) continue;
        const bool mine = (m >> i) & 1;
        const int32_t o = perm[t0 + (mine ? i : __ffs((int)m) - 1)];
        double a = vort_sum<F32, kRestT>(rec, box, nblk, xt[o], yt[o], pp,
                                         (F32 ? kVortZero32 : kVortZero64) / pp.inv_ks,
                                         __builtin_amdgcn_readfirstlane(wv), kRestWaves);
#pragma unroll
        for (int d = kRestT; d < kWave; d <<= 1) a += __shfl_xor(a, d);
        if (lane < kRestT) sh[wv][lane] = a;
        __syncthreads();
        if ((int)threadIdx.x < kRestT && mine) {
            a = 0.0;
            for (int k = 0; k < kRestWaves; ++k) a += sh[k][i];
            const double inv_pi = 1.0 / 3.141592653589793;
            w[o] = inv_pi * a / ks;
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------- host ------
int upload(Lane *L, const double *host, int64_t n, double **dev)
{
    double *d;
    PHF_ALLOC(d, L->arena, double, (size_t)(n > 0 ? n : 1));
    if (n > 0)
        PHF_HIP(hipMemcpyAsync(d, host, sizeof(double) * n, hipMemcpyHostToDevice, L->stream));
    *dev = d;
    return PHF_OK;
}

int download(Lane *L, const double *dev, int64_t n, double *host)
{
    if (n > 0)
        PHF_HIP(hipMemcpyAsync(host, dev, sizeof(double) * n, hipMemcpyDeviceToHost, L->stream));
    return PHF_OK;
}

// Cell of every target on a 2^B x 2^B grid over the targets' bounding box, in
// Morton order, and its index.
__global__ __launch_bounds__(256) void target_cells(const double *__restrict__ xt,
                                                    const double *__restrict__ yt, int64_t nt,
                                                    const double4 *__restrict__ bb, int B,
                                                    uint32_t *__restrict__ keys,
                                                    int32_t *__restrict__ vals)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nt) return;
    const double4 b = *bb;
    const double ext = fmax(b.y - b.x, b.w - b.z);
    const double scale = ext > 0.0 ? ldexp(1.0, B) / ext : 0.0;
    const double hi = (double)((1u << B) - 1u);
    const double fx = fmin(fmax(floor((xt[i] - b.x) * scale), 0.0), hi);
    const double fy = fmin(fmax(floor((yt[i] - b.z) * scale), 0.0), hi);
    keys[i] = morton2((uint32_t)fx, (uint32_t)fy);
    vals[i] = (int32_t)i;
}

// The points' Morton order on a grid over the box bb (device; a stable sort,
// so a fixed order): perm[t] is the t-th point.  One 8-bit pass of the sort (256
// cells) up to 65,536 points, two (65,536 cells) above: an even spread puts at
// most 256, or 64, points into a cell.  A second pass from 16,384 points on made
// 20,011 x 40,401 vorticity 10 us quicker in its near pass and 30 us slower in
// its sorts.
static int target_order(Lane *L, const double *xt, const double *yt, int64_t nt,
                        const double4 *bb, int32_t **perm)
{
    uint32_t *k0, *k1, *ks;
    int32_t *v0, *v1;
    PHF_ALLOC(k0, L->arena, uint32_t, (size_t)nt);
    PHF_ALLOC(k1, L->arena, uint32_t, (size_t)nt);
    PHF_ALLOC(v0, L->arena, int32_t, (size_t)nt);
    PHF_ALLOC(v1, L->arena, int32_t, (size_t)nt);
    const int B = nt <= 64 * 1024 ? 4 : 8;
    target_cells<<<div_up(nt, 256), 256, 0, L->stream>>>(xt, yt, nt, bb, B, k0, v0);
    PHF_HIP(hipGetLastError());
    return device_radix_sort(L, k0, v0, k1, v1, nt, 2 * B, &ks, perm);
}

// Source chunks of a direct sum over nt targets in groups of 64 * tpl:
// enough chunks that the waves fill the chip in whole rounds, each of at least
// 64 sources (16 in a small sum; a multiple of 16); one chunk once the target groups
// alone fill the chip.  max_chunks caps the count (the partial sums take
// nchunk * nt double2).
static void direct_split(int64_t nt, int tpl, int64_t nb, int64_t *nchunk_out,
                         int64_t *chunk_len_out, int64_t max_chunks = 65535, bool shorten = true)
{
    const int64_t tblock = (int64_t)kWave * tpl;
    const int64_t ngroups = (nt + tblock - 1) / tblock;
    // whole rounds of the 8,192 waves the chip holds: as many chunks as fit
    // into one round, or into the first of up to five that leaves at most 5%
    // of itself empty (18 chunks of 470 groups left a second round of 268
    // waves; 61 chunks of 128 groups, 95% of a round, took 131 us where 64 take
    // 125)
    const int64_t full = 8192;
    // A wave takes its sources one after another, some 180 cycles each in
    // float64, so a call of few waves ends with that chain: down to 16 sources
    // while there are no more than 2048 waves, two per SIMD (400 x 400 float64
    // 12.7 -> 9.8 us, 2025 x 2025 14.9 -> 11.2, 3249 x 3249 float32 16.2 ->
    // 13.4; 4096 waves of 32 sources for 4096 x 4096 float32 took 17.4 against
    // 15.1 us: the partial sums outweigh it).  Not for the vorticity, whose
    // pairs are cheaper and whose finish adds a target's parts in one thread.
    const int64_t fine =
        shorten ? std::max<int64_t>(nb / 64, std::min<int64_t>(nb / 16, 2048 / ngroups)) : nb / 64;
    const int64_t most =
        std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(max_chunks, 65535), fine));
    int64_t nchunk = most;
    if (most * ngroups > full) {
        double best = 0.0;
        for (int64_t r = 1; r <= 5 && best < 0.95; ++r) {
            const int64_t c = std::max<int64_t>(1, std::min<int64_t>(r * full / ngroups, most));
            const double rounds = (double)((c * ngroups + full - 1) / full);
            const double eff = (double)(c * ngroups) / (rounds * full);
            if (eff > best) {
                best = eff;
                nchunk = c;
            }
        }
    }
    int64_t chunk_len = (nb + nchunk - 1) / nchunk;
    chunk_len = std::max<int64_t>(16, (chunk_len + 15) / 16 * 16);
    *nchunk_out = std::max<int64_t>(1, (nb + chunk_len - 1) / chunk_len);
    *chunk_len_out = chunk_len;
}

// Zero partial row for an empty source set (a kernel rather than a memset,
// so the sequence holds only kernel launches).
__global__ __launch_bounds__(256) void zero_part(double2 *__restrict__ part, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) part[i] = make_double2(0.0, 0.0);
}

constexpr int DIRECT_TPL32 = 2, DIRECT_TPL64 = 1;

// Whether a float64 velocity sum sorts its targets (six launches, some 45 us,
// and 0.1 ns a target): from 1e8 pairs, and enough sources that most are
// outside a target's smoothing and a target's saving is more than its sort.
// Call with its kernels, unsorted against sorted: 6.4e7 pairs 91 against 97 us,
// 1.4e8 193 against 149, 6e8 731 against 439; 800 sources x 625,000 targets
// 1,349 against 1,380 us, 1,600 x 312,500 997 against 987, 3,200 x 156,250 835
// against 769; 100 x 1.1M 1,400 against 1,493.  Few targets sort at no cost:
// 250,000 x 2,000 943 against 672 us.
static bool sort_pays(int64_t nb, int64_t nt)
{
    return (double)nb * (double)nt >= 1e8 && nb >= 2048;
}

// Whether the vorticity takes near sources only (a dozen launches, two sorts):
// from 1e8 pairs, in float32, whose pairs cost less, from 4e8, and more where
// the sides are uneven, since either is sorted and few points make no compact
// groups.  Whole calls, every pair against near sources, float64: 1.1e8 pairs
// 257 against 222 us, 8e8 1,045 against 338; 400 sources x 275,000 targets 448
// against 531, 800 x 625,000 1,020 against 959, 220,000 x 500 433 against 488,
// 1M x 500 1,408 against 1,306.  float32: 1.4e8 192 against 215, 8e8 425
// against 285; 1,600 x 312,500 490 against 533, 3,200 x 312,500 626 against
// 574, 1M x 500 1,138 against 1,300, 250,000 x 2,000 586 against 492.
static bool near_pays(int prec, int64_t nb, int64_t nt)
{
    const double pairs = (double)nb * (double)nt;
    if (prec == PHF_PREC_F64)
        return pairs >= 1e8 && pairs * (double)std::min(nb, nt) >= 2.2e11;
    return pairs >= 4e8 && pairs * std::min((double)nb / 3.0, (double)nt) >= 5.4e11;
}

// Whether at least half of the pairs of a sample (32 sources by 32 targets of the
// host arrays, about 2 us) are further apart than r2 = reach2; true without a
// look for sums that never sort.  Kernels as wide as the flow leave the sorted
// passes nothing to skip.  Uniform points, sigma 1 (no pair is far) and 0.03 (a
// quarter is near); every pair, unsorted, against sorted: vorticity, float32,
// 100,000 x 100,000 3,492 against 4,229 and 1,729 us, float64, 5,133 sources x
// 24,469 targets 257 against 316 and 253; velocity, the same, 303 against 333
// and 298.
bool mostly_far(const double *xb, const double *yb, int64_t nb, const double *xt,
                const double *yt, int64_t nt, double reach2)
{
    if ((double)nb * (double)nt < 1e8) return true;
    constexpr int K = 32;
    double x[K], y[K];
    const int64_t kb = std::min<int64_t>(K, nb), kt = std::min<int64_t>(K, nt);
    for (int64_t i = 0; i < kb; ++i) {
        const int64_t j = (2 * i + 1) * (nb / kb) / 2;
        x[i] = xb[j];
        y[i] = yb[j];
    }
    int64_t far = 0;
    for (int64_t k = 0; k < kt; ++k) {
        const int64_t t = (2 * k + 1) * (nt / kt) / 2;
        for (int64_t i = 0; i < kb; ++i) {
            const double dx = xt[t] - x[i], dy = yt[t] - y[i];
            far += dx * dx + dy * dy > reach2;
        }
    }
    return 2 * far >= kb * kt;
}

// Enqueue the pair kernel and the finishing kernel on stream st with the
// partial sums in part (nchunk * nt double2; nchunk, chunk_len from
// direct_split).  perm (float64 only): the targets' Morton order.
template <int KIND>
static int enqueue_direct(hipStream_t st, int prec, const PairParams &pp, const double *xb,
                          const double *yb, const double *wb, int64_t nb, const double *xt,
                          const double *yt, int64_t nt, int64_t nchunk, int64_t chunk_len,
                          double2 *part, double *o0, double *o1, const int32_t *perm = nullptr)
{
    const int tpl = prec == PHF_PREC_F32C ? DIRECT_TPL32 : DIRECT_TPL64;
    const int64_t tblock = (int64_t)kWave * tpl;
    const int64_t ngroups = (nt + tblock - 1) / tblock;
    dim3 grid((unsigned)ngroups, (unsigned)nchunk);
    if (nb == 0) {
        zero_part<<<div_up(nt, 256), 256, 0, st>>>(part, nt);
    } else if (prec == PHF_PREC_F32C) {
        // sources read in place: every lane of a wave reads the same one
        direct_f32c<KIND, DIRECT_TPL32><<<grid, kWave, 0, st>>>(xb, yb, wb, nb, xt, yt, nt,
                                                                chunk_len, pp, part);
    } else if (perm) {
        direct_f64_sorted<KIND><<<grid, kWave, 0, st>>>(xb, yb, wb, nb, xt, yt, perm, nt,
                                                        chunk_len, pp, part);
    } else {
        direct_f64<KIND, DIRECT_TPL64><<<grid, kWave, 0, st>>>(xb, yb, wb, nb, xt, yt, nt,
                                                               chunk_len, pp, part);
    }
    PHF_HIP(hipGetLastError());
    direct_finish<<<div_up(nt, FIN_T), 256, 0, st>>>(
        part, nb == 0 ? 1 : (int)nchunk, nt,
        (KIND == PAIR_GAUSS_EPS || KIND == PAIR_CUTOFF) ? KIND : PAIR_OSEEN, perm, o0, o1);
    PHF_HIP(hipGetLastError());
    return PHF_OK;
}

template <int KIND>
static int launch_direct(Lane *L, int prec, const PairParams &pp, const double *xb,
                         const double *yb, const double *wb, int64_t nb, const double *xt,
                         const double *yt, int64_t nt, double *o0, double *o1, bool far)
{
    const int tpl = prec == PHF_PREC_F32C ? DIRECT_TPL32 : DIRECT_TPL64;
    int64_t nchunk, chunk_len;
    direct_split(nt, tpl, nb, &nchunk, &chunk_len);
    double2 *part;
    PHF_ALLOC(part, L->arena, double2, (size_t)nchunk * (size_t)nt);
    int32_t *perm = nullptr;
    if (prec == PHF_PREC_F64 && KIND != PAIR_CUTOFF && nt < (int64_t(1) << 31) &&
        sort_pays(nb, nt) && far) {
        const int rc = [&]() -> int {
            double4 *bb;
            PHF_ALLOC(bb, L->arena, double4, 1);
            PHF_TRY(device_bbox(L, xt, yt, nt, nullptr, nullptr, 0, bb));
            return target_order(L, xt, yt, nt, bb, &perm);
        }();
        if (rc == PHF_ERR_NOMEM) {  // no room for the sort: the targets as they are
            clear_error();
            perm = nullptr;
        } else {
            PHF_TRY(rc);
        }
    }
    return enqueue_direct<KIND>(L->stream, prec, pp, xb, yb, wb, nb, xt, yt, nt, nchunk,
                                chunk_len, part, o0, o1, perm);
}

static int vorticity_near(Lane *L, int prec, double ks, const PairParams &pp, const double *xb,
                          const double *yb, const double *wb, int64_t nb, const double *xt,
                          const double *yt, int64_t nt, double *w)
{
    const int nblk = (int)div_up(nb, kVortBlk);
    const int64_t ngroups = div_up(nt, kWave);
    // some 8 waves per SIMD, each with at least 8 blocks to look at
    const int nchunk = (int)std::max<int64_t>(
        1, std::min<int64_t>((8192 + ngroups - 1) / ngroups, nblk / 8));
    double4 *bb, *rec, *box;
    double *wabs, *part;
    int32_t *ps, *pt;
    unsigned long long *need;
    PHF_ALLOC(bb, L->arena, double4, 1);
    PHF_ALLOC(rec, L->arena, double4, (size_t)nblk * kVortBlk);
    PHF_ALLOC(box, L->arena, double4, (size_t)nblk);
    PHF_ALLOC(wabs, L->arena, double, (size_t)nblk);
    PHF_ALLOC(part, L->arena, double, (size_t)nchunk * (size_t)nt);
    PHF_ALLOC(need, L->arena, unsigned long long, (size_t)ngroups);
    PHF_TRY(device_bbox(L, xb, yb, nb, xt, yt, nt, bb));
    PHF_TRY(target_order(L, xb, yb, nb, bb, &ps));
    PHF_TRY(target_order(L, xt, yt, nt, bb, &pt));
    vort_pack<<<div_up(nblk, 4), 256, 0, L->stream>>>(xb, yb, wb, ps, nb, nblk, rec, box, wabs);
    const dim3 grid((unsigned)ngroups, (unsigned)nchunk);
    const unsigned rgrid = std::min(div_up(nt, kRestT), (unsigned)kRestGrid);
    const bool f32 = prec == PHF_PREC_F32C;
    if (f32)
        vort_near<true><<<grid, kWave, 0, L->stream>>>(rec, box, nblk, xt, yt, pt, nt, pp, part);
    else
        vort_near<false><<<grid, kWave, 0, L->stream>>>(rec, box, nblk, xt, yt, pt, nt, pp, part);
    vort_near_finish<<<div_up(nt, 256), 256, 0, L->stream>>>(part, nchunk, nt, pt, wabs, nblk, ks,
                                                             w, need);
    if (f32)
        vort_rest<true><<<rgrid, 64 * kRestWaves, 0, L->stream>>>(
            rec, box, nblk, xt, yt, pt, nt, pp, ks, w, need);
    else
        vort_rest<false><<<rgrid, 64 * kRestWaves, 0, L->stream>>>(
            rec, box, nblk, xt, yt, pt, nt, pp, ks, w, need);
    PHF_HIP(hipGetLastError());
    return PHF_OK;
}

int vorticity_device(Lane *L, int prec, double ksigmasqr, const double *xb, const double *yb,
                     const double *wb, int64_t nb, const double *xt, const double *yt, int64_t nt,
                     double *w, bool cutoff, bool far)
{
    if (nt == 0) return PHF_OK;
    PairParams pp = make_gauss_params(ksigmasqr);
    if (cutoff) {  // sigma^2 takes the place of EPS (ww2par_C_cpu.c:140)
        pp.eps = ksigmasqr;
        pp.eps_f = (float)ksigmasqr;
    }
    if (!cutoff && nb < (int64_t(1) << 31) && nt < (int64_t(1) << 31) &&
        near_pays(prec, nb, nt) && far) {
        const Arena::Mark m0 = L->arena.mark();
        const int rc = vorticity_near(L, prec, ksigmasqr, pp, xb, yb, wb, nb, xt, yt, nt, w);
        if (rc != PHF_ERR_NOMEM) return rc;
        // no room for its workspace: every pair
        L->arena.jump(L->arena.mark(), m0);
        clear_error();
    }
    constexpr int TPL32 = 2, TPL64 = 1;
    const int tpl = prec == PHF_PREC_F32C ? TPL32 : TPL64;
    const int64_t tblock = (int64_t)kWave * tpl;
    const int64_t ngroups = (nt + tblock - 1) / tblock;
    int64_t nchunk, chunk_len;
    direct_split(nt, tpl, nb, &nchunk, &chunk_len, 65535, false);
    double *part;
    PHF_ALLOC(part, L->arena, double, (size_t)nchunk * (size_t)nt);
    const dim3 grid((unsigned)ngroups, (unsigned)nchunk);
    if (nb == 0) {
        PHF_HIP(hipMemsetAsync(part, 0, sizeof(double) * nt, L->stream));
    } else if (prec == PHF_PREC_F32C) {
        if (cutoff)
            vort_f32c<TPL32, true><<<grid, kWave, 0, L->stream>>>(xb, yb, wb, nb, xt, yt, nt,
                                                                  chunk_len, pp, part);
        else
            vort_f32c<TPL32, false><<<grid, kWave, 0, L->stream>>>(xb, yb, wb, nb, xt, yt, nt,
                                                                   chunk_len, pp, part);
    } else {
        if (cutoff)
            vort_f64<TPL64, true><<<grid, kWave, 0, L->stream>>>(xb, yb, wb, nb, xt, yt, nt,
                                                                 chunk_len, pp, part);
        else
            vort_f64<TPL64, false><<<grid, kWave, 0, L->stream>>>(xb, yb, wb, nb, xt, yt, nt,
                                                                  chunk_len, pp, part);
    }
    PHF_HIP(hipGetLastError());
    vort_finish<<<div_up(nt, 256), 256, 0, L->stream>>>(part, nb == 0 ? 1 : (int)nchunk, nt,
                                                         ksigmasqr, cutoff ? 1 : 0, w);
    PHF_HIP(hipGetLastError());
    return PHF_OK;
}

int direct_device(Lane *L, int kind, int prec, const PairParams &pp, const double *xb,
                  const double *yb, const double *wb, int64_t nb, const double *xt,
                  const double *yt, int64_t nt, double *o0, double *o1,
                  bool far)
{
    if (nt == 0) return PHF_OK;
    if (kind == PAIR_GAUSS_EPS)
        return launch_direct<PAIR_GAUSS_EPS>(L, prec, pp, xb, yb, wb, nb, xt, yt, nt, o0, o1,
                                             far);
    if (kind == PAIR_CUTOFF)
        return launch_direct<PAIR_CUTOFF>(L, prec, pp, xb, yb, wb, nb, xt, yt, nt, o0, o1,
                                          far);
    if (prec == PHF_PREC_F32C && pp.f32_nocut)
        return launch_direct<PAIR_OSEEN_NOCUT>(L, prec, pp, xb, yb, wb, nb, xt, yt, nt, o0, o1,
                                               far);
    return launch_direct<PAIR_OSEEN>(L, prec, pp, xb, yb, wb, nb, xt, yt, nt, o0, o1,
                                     far);
}

}  // namespace phf

// ------------------------------------------------------------ C entry ----
using namespace phf;

static int vv2par_entry(int kind, const double *xb, const double *yb, const double *wb,
                        int64_t nb, const double *xt, const double *yt, int64_t nt,
                        double ksigmasqr, int32_t prec, double *vx, double *vy);

extern "C" int phf_vv2par_gauss(const double *xb, const double *yb, const double *wb,
                                int64_t nb, const double *xt, const double *yt, int64_t nt,
                                double ksigmasqr, int32_t prec, double *vx, double *vy)
{
    clear_error();
    return vv2par_entry(PAIR_GAUSS_EPS, xb, yb, wb, nb, xt, yt, nt, ksigmasqr, prec, vx, vy);
}

extern "C" int phf_vv2par_cutoff(const double *xb, const double *yb, const double *wb,
                                 int64_t nb, const double *xt, const double *yt, int64_t nt,
                                 double sigmasqr, int32_t prec, double *vx, double *vy)
{
    clear_error();
    return vv2par_entry(PAIR_CUTOFF, xb, yb, wb, nb, xt, yt, nt, sigmasqr, prec, vx, vy);
}

static int vv2par_entry(int kind, const double *xb, const double *yb, const double *wb,
                        int64_t nb, const double *xt, const double *yt, int64_t nt,
                        double ksigmasqr, int32_t prec, double *vx, double *vy)
{
    PHF_REQUIRE(nb >= 0 && nt >= 0, "negative sizes (nb=%lld, nt=%lld)", (long long)nb,
                (long long)nt);
    PHF_REQUIRE(prec == PHF_PREC_F64 || prec == PHF_PREC_F32C, "unknown precision %d", prec);
    PHF_REQUIRE(std::isfinite(ksigmasqr) && ksigmasqr > 0.0,
                "ksigmasqr must be finite and > 0 (got %g)", ksigmasqr);
    PHF_TRY(check_host_array(xb, nb, "xBlob"));
    PHF_TRY(check_host_array(yb, nb, "yBlob"));
    PHF_TRY(check_host_array(wb, nb, "wBlob"));
    PHF_TRY(check_host_array(xt, nt, "xTarget"));
    PHF_TRY(check_host_array(yt, nt, "yTarget"));
    PHF_REQUIRE(nt == 0 || (vx && vy), "output arrays are NULL");
    if (nt == 0) return PHF_OK;

    LaneGuard g;
    PHF_TRY(g.rc);
    Lane *L = g.lane;
    PHF_TRY(reset_arena(L));
    StageTimer tm(L, timing_enabled());
    bool used[PHF_STAGE_COUNT] = {};
    used[PHF_STAGE_UPLOAD] = used[PHF_STAGE_P2P] = used[PHF_STAGE_DOWNLOAD] = true;
    used[PHF_STAGE_TOTAL] = true;

    tm.begin(PHF_STAGE_TOTAL);
    tm.begin(PHF_STAGE_UPLOAD);
    double *dxb, *dyb, *dwb, *dxt, *dyt, *o0, *o1;
    PHF_TRY(copy_points_in(L, xb, yb, wb, nb, xt, yt, nt, &dxb, &dyb, &dwb, &dxt, &dyt));
    PHF_ALLOC(o0, L->arena, double, (size_t)nt * 2);
    o1 = o0 + nt;
    tm.end(PHF_STAGE_UPLOAD);
    tm.begin(PHF_STAGE_P2P);
    PairParams pp = make_gauss_params(ksigmasqr);
    if (kind == PAIR_CUTOFF) {  // r2 = dx^2 + dy^2 + sigma^2 (vv2par_C_cpu.c:144)
        pp.eps = ksigmasqr;
        pp.eps_f = (float)ksigmasqr;
    }
    PHF_TRY(direct_device(L, kind, prec, pp, dxb, dyb, dwb, nb, dxt, dyt, nt, o0, o1,
                          mostly_far(xb, yb, nb, xt, yt, nt, 40.0 * ksigmasqr)));
    tm.end(PHF_STAGE_P2P);
    tm.begin(PHF_STAGE_DOWNLOAD);
    PHF_TRY(copy_out(L, {{vx, o0, sizeof(double) * nt}, {vy, o1, sizeof(double) * nt}}));
    tm.end(PHF_STAGE_DOWNLOAD);
    tm.end(PHF_STAGE_TOTAL);
    if (tm.on) PHF_HIP(hipStreamSynchronize(L->stream));
    record_stage_times(L, used);
    return PHF_OK;
}

static int ww2par_entry(bool cutoff, const double *xb, const double *yb, const double *wb,
                        int64_t nb, const double *xt, const double *yt, int64_t nt,
                        double ksigmasqr, int32_t prec, double *w);

extern "C" int phf_ww2par_gauss(const double *xb, const double *yb, const double *wb,
                                int64_t nb, const double *xt, const double *yt, int64_t nt,
                                double ksigmasqr, int32_t prec, double *w)
{
    clear_error();
    return ww2par_entry(false, xb, yb, wb, nb, xt, yt, nt, ksigmasqr, prec, w);
}

extern "C" int phf_ww2par_cutoff(const double *xb, const double *yb, const double *wb,
                                 int64_t nb, const double *xt, const double *yt, int64_t nt,
                                 double sigmasqr, int32_t prec, double *w)
{
    clear_error();
    return ww2par_entry(true, xb, yb, wb, nb, xt, yt, nt, sigmasqr, prec, w);
}

static int ww2par_entry(bool cutoff, const double *xb, const double *yb, const double *wb,
                        int64_t nb, const double *xt, const double *yt, int64_t nt,
                        double ksigmasqr, int32_t prec, double *w)
{
    PHF_REQUIRE(nb >= 0 && nt >= 0, "negative sizes (nb=%lld, nt=%lld)", (long long)nb,
                (long long)nt);
    PHF_REQUIRE(prec == PHF_PREC_F64 || prec == PHF_PREC_F32C, "unknown precision %d", prec);
    PHF_REQUIRE(std::isfinite(ksigmasqr) && ksigmasqr > 0.0,
                "ksigmasqr must be finite and > 0 (got %g)", ksigmasqr);
    PHF_TRY(check_host_array(xb, nb, "xBlob"));
    PHF_TRY(check_host_array(yb, nb, "yBlob"));
    PHF_TRY(check_host_array(wb, nb, "wBlob"));
    PHF_TRY(check_host_array(xt, nt, "xTarget"));
    PHF_TRY(check_host_array(yt, nt, "yTarget"));
    PHF_REQUIRE(nt == 0 || w, "output array is NULL");
    if (nt == 0) return PHF_OK;
    LaneGuard g;
    PHF_TRY(g.rc);
    Lane *L = g.lane;
    PHF_TRY(reset_arena(L));
    double *dxb, *dyb, *dwb, *dxt, *dyt, *o;
    PHF_TRY(copy_points_in(L, xb, yb, wb, nb, xt, yt, nt, &dxb, &dyb, &dwb, &dxt, &dyt));
    PHF_ALLOC(o, L->arena, double, (size_t)nt);
    PHF_TRY(vorticity_device(L, prec, ksigmasqr, dxb, dyb, dwb, nb, dxt, dyt, nt, o, cutoff,
                             mostly_far(xb, yb, nb, xt, yt, nt, kVortCut * ksigmasqr)));
    return copy_out(L, {{w, o, sizeof(double) * nt}});
}

// ------------------------------------------- allocation-free direct sum ---
// phf_vv2par_gauss_noalloc keeps its partial sums in one file-scope device
// array instead of a workspace from hipMalloc.  Each GPU the library runs
// on holds its own copy until the process ends.  Host code never uses the
// array's name as an address: direct_scratch_setup (called by the library's
// init with the device current) asks the runtime for the device address
// and every launch takes that pointer.
namespace phf {

constexpr int64_t kScratchPart = int64_t(1) << 21;  // double2 entries: 32 MiB
constexpr int kScratchDevices = 64;
static __device__ __align__(256) double2 scratch[kScratchPart];
static double2 *g_scratch[kScratchDevices] = {};

int direct_scratch_setup(int dev)
{
    PHF_REQUIRE(dev >= 0 && dev < kScratchDevices, "device %d out of range", dev);
    if (g_scratch[dev]) return PHF_OK;
    void *p = nullptr;
    PHF_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    PHF_REQUIRE(p != nullptr, "no device address for the direct-sum scratch array");
    g_scratch[dev] = reinterpret_cast<double2 *>(p);
    return PHF_OK;
}

// A kernel argument must lie inside one device (or managed) allocation of
// the current device, so a host pointer fails here instead of faulting the
// GPU.
static int check_device_range(const void *p, int64_t n, const char *name)
{
    if (n == 0) return PHF_OK;
    PHF_REQUIRE(p != nullptr, "%s is NULL but has %lld entries", name, (long long)n);
    hipPointerAttribute_t at{};
    hipError_t e = hipPointerGetAttributes(&at, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        set_error("%s is not device memory (%s)", name, hipGetErrorName(e));
        return PHF_ERR_INVALID;
    }
    PHF_REQUIRE(at.type == hipMemoryTypeDevice || at.type == hipMemoryTypeManaged,
                "%s is not device memory (memory type %d)", name, (int)at.type);
    hipDeviceptr_t base = nullptr;
    size_t bytes = 0;
    e = hipMemGetAddressRange(&base, &bytes, const_cast<void *>(p));
    if (e != hipSuccess) {
        (void)hipGetLastError();
        set_error("%s: allocation range unknown (%s)", name, hipGetErrorName(e));
        return PHF_ERR_INVALID;
    }
    const char *b = reinterpret_cast<const char *>(base);
    const char *q = reinterpret_cast<const char *>(p);
    PHF_REQUIRE(q >= b && (uint64_t)(q - b) + (uint64_t)n * sizeof(double) <= bytes,
                "%s: %lld doubles run past the end of its allocation", name, (long long)n);
    return PHF_OK;
}

}  // namespace phf

extern "C" int phf_vv2par_gauss_noalloc(const double *xb, const double *yb, const double *wb,
                                        int64_t nb, const double *xt, const double *yt,
                                        int64_t nt, double ksigmasqr, int32_t prec, double *vx,
                                        double *vy, void *stream)
{
    clear_error();
    PHF_REQUIRE(nb >= 0 && nt >= 0, "negative sizes (nb=%lld, nt=%lld)", (long long)nb,
                (long long)nt);
    PHF_REQUIRE(nt <= kScratchPart,
                "nt=%lld exceeds the %lld targets the allocation-free scratch holds",
                (long long)nt, (long long)kScratchPart);
    PHF_REQUIRE(nb < (int64_t(1) << 40), "nb out of range (%lld)", (long long)nb);
    PHF_REQUIRE(prec == PHF_PREC_F64 || prec == PHF_PREC_F32C, "unknown precision %d", prec);
    PHF_REQUIRE(std::isfinite(ksigmasqr) && ksigmasqr > 0.0,
                "ksigmasqr must be finite and > 0 (got %g)", ksigmasqr);
    if (nt == 0) return PHF_OK;
    PHF_TRY(Context::get().init());
    const int dev = Context::get().device();
    PHF_HIP(hipSetDevice(dev));
    PHF_REQUIRE(dev >= 0 && dev < kScratchDevices && g_scratch[dev] != nullptr,
                "the direct-sum scratch array of device %d is not set up", dev);
    PHF_TRY(check_device_range(xb, nb, "xBlob"));
    PHF_TRY(check_device_range(yb, nb, "yBlob"));
    PHF_TRY(check_device_range(wb, nb, "wBlob"));
    PHF_TRY(check_device_range(xt, nt, "xTarget"));
    PHF_TRY(check_device_range(yt, nt, "yTarget"));
    PHF_TRY(check_device_range(vx, nt, "vx"));
    PHF_TRY(check_device_range(vy, nt, "vy"));

    const int tpl = prec == PHF_PREC_F32C ? DIRECT_TPL32 : DIRECT_TPL64;
    int64_t nchunk, chunk_len;
    direct_split(nt, tpl, nb, &nchunk, &chunk_len, kScratchPart / nt);
    PHF_REQUIRE(nchunk * nt <= kScratchPart, "partial sums (%lld x %lld) exceed the scratch",
                (long long)nchunk, (long long)nt);
    const PairParams pp = make_gauss_params(ksigmasqr);
    if (stream) {
        // enqueue on the caller's stream; the caller synchronises
        return enqueue_direct<PAIR_GAUSS_EPS>(reinterpret_cast<hipStream_t>(stream), prec, pp,
                                              xb, yb, wb, nb, xt, yt, nt, nchunk, chunk_len,
                                              g_scratch[dev], vx, vy);
    }
    LaneGuard g;
    PHF_TRY(g.rc);
    PHF_TRY(enqueue_direct<PAIR_GAUSS_EPS>(g.lane->stream, prec, pp, xb, yb, wb, nb, xt, yt, nt,
                                           nchunk, chunk_len, g_scratch[dev], vx, vy));
    PHF_HIP(hipStreamSynchronize(g.lane->stream));
    return PHF_OK;
}
