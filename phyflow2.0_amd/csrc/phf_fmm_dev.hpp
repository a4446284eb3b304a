// phf_fmm_dev.hpp -- device helpers shared by the single-system and the
// batched FMM kernels.
#pragma once

#include "phf_device.hpp"
#include "phyflow_amd.h"

#include <type_traits>

namespace phf {

template <class T> struct C2;
template <> struct C2<float> { using type = float2; };
template <> struct C2<double> { using type = double2; };

template <class T> __device__ __forceinline__ typename C2<T>::type cmk(T r, T i)
{
    return typename C2<T>::type{r, i};
}
template <class V> __device__ __forceinline__ V cmul(V a, V b)
{
    return V{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}

// centre of the leaf box with Morton key `key` (side s, origin x0, y0)
__device__ __forceinline__ void leaf_center(uint32_t key, double x0, double y0, double s,
                                            double &cx, double &cy)
{
    uint32_t ix = compact_bits(key), iy = compact_bits(key >> 1);
    cx = x0 + ((double)ix + 0.5) * s;
    cy = y0 + ((double)iy + 0.5) * s;
}

// box counts at level l from leaf offsets (shift = 2 (L - l))
__device__ __forceinline__ int box_count(const int32_t *__restrict__ start, uint32_t b, int shift)
{
    return start[(int64_t)(b + 1) << shift] - start[(int64_t)b << shift];
}

// ----------------------------------------------------------------- P2M --
// Multipole expansion sum_j w_j ((z_j - c) inv_s)^k, k < p1 <= 4 NI, of the
// points [s0, s1) by 4 R lanes of a wave (R = 16 or 4), without LDS.  Lane
// 4 r + q takes the points j = r (mod R) and the powers k = q (mod 4): it forms
// z^q from z and z^2, steps by z^4 through its NI powers and keeps their sums
// in registers; the R lanes of a power are then added by a butterfly.  With MIX
// the sums do not depend on R (which follows from the whole launch in a batch):
// the points fall into sixteen classes j (mod 16) in either case, added in
// index order each and then pairwise in class order, and a lane of R = 4 takes
// four neighbouring classes (its expansions then take up to a third longer).
// Four residues of k balance the products repeated in every lane of a point (2
// squarings, 2 selected) against the butterfly (4 steps of NI).  (With a table of 64 x p1 powers in LDS and each
// column added by one lane, a leaf was a serial chain of 64 LDS reads with
// 64 - p1 lanes idle.)
// Beside the near field of 1M blobs, order 16: 65 us with the table, 19 us so
// and at the far field's wave priority.
// float32 records are relative to the leaf centre; (cx, cy) is the centre
// for float64 ones.
template <class T, int NI, int R, bool MIX>
__device__ __forceinline__ void p2m_leaf(const void *__restrict__ src, int32_t s0, int32_t s1,
                                         double cx, double cy, T inv_s, int p1,
                                         typename C2<T>::type *__restrict__ out)
{
    using V = typename C2<T>::type;
    using Rec = std::conditional_t<sizeof(T) == 4, float4, double4>;
    constexpr int KC = MIX ? 16 / R : 1;    // classes of a lane, KC r ..
    constexpr int STEP = KC == 1 ? R : 16;  // between a class's points
    const int lane = threadIdx.x & (4 * R - 1), q = lane & 3, r = lane >> 2;
    const Rec *rec = reinterpret_cast<const Rec *>(src);
    auto zero = [](V *a) {
#pragma unroll
        for (int i = 0; i < NI; ++i) a[i] = cmk<T>(0, 0);
    };
    auto add = [](V *a, const V *b) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            a[i].x += b[i].x;
            a[i].y += b[i].y;
        }
    };
    auto point = [&](const Rec &pt, V *a) {
        V z;
        if (sizeof(T) == 4)
            z = cmk<T>((T)pt.x * inv_s, (T)pt.y * inv_s);
        else
            z = cmk<T>((T)((pt.x - cx) * inv_s), (T)((pt.y - cy) * inv_s));
        V t = cmk<T>((T)pt.z, 0);
        const V z2 = cmul(z, z), z4 = cmul(z2, z2);
        if (q & 1) t = cmul(t, z);
        if (q & 2) t = cmul(t, z2);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            a[i].x += t.x;
            a[i].y += t.y;
            if (i + 1 < NI) t = cmul(t, z4);
        }
    };
    // the points j, j + STEP, .. of a class; the loads of U points go out together
    auto points = [&](int32_t j0, V *a) {
        constexpr int U = KC == 1 ? 4 : 3;
        for (; j0 < s1; j0 += STEP * U) {
            Rec pt[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int32_t j = j0 + STEP * u;
                pt[u] = rec[j < s1 ? j : s0];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (j0 + STEP * u >= s1) break;
                point(pt[u], a);
            }
        }
    };
    if (__ballot(s1 > s0) == 0) {  // nothing to add up
#pragma unroll
        for (int i = 0; i < NI; ++i)
            if (r == i % R && 4 * i + q < p1) out[4 * i + q] = cmk<T>(0, 0);
        return;
    }
    V acc[NI];
    zero(acc);
    if constexpr (KC == 1) {
        points(s0 + r, acc);
    } else {
        const int32_t j0 = s0 + KC * r;
        Rec first[KC];  // the first point of each class, loaded together
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            const int32_t j = j0 + c;
            first[c] = rec[j < s1 ? j : s1 > s0 ? s0 : 0];
        }
        auto cls = [&](int c, V *a) {
            zero(a);
            if (j0 + c < s1) point(first[c], a);
            points(j0 + c + 16, a);
        };
        V b[NI], c[NI];
        cls(0, acc);
        cls(1, b);
        add(acc, b);
        cls(2, b);
        cls(3, c);
        add(b, c);
        add(acc, b);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
        for (int d = 4; d < 4 * R; d <<= 1) {
            acc[i].x += __shfl_xor(acc[i].x, d);
            acc[i].y += __shfl_xor(acc[i].y, d);
        }
        const int k = 4 * i + q;
        if (r == i % R && k < p1) out[k] = acc[i];
    }
}

// p2m_leaf with MIX for the leaves of a wave, 64 / (4 R) of them; at < 0: none.
// A leaf taken by sixteen lanes is a serial chain of a quarter of its points, so
// the whole wave takes the ones with more than `crowd`, one after another, with
// the same sums.  The full batches that use sixteen lanes have leaves of 64 to
// 128, and their waves four of them to go on with: they take what they took.
template <class T, int NI, int R>
__device__ __forceinline__ void p2m_wave(const void *__restrict__ src, int32_t s0, int32_t s1,
                                         double cx, double cy, T inv_s, int p1,
                                         typename C2<T>::type *__restrict__ M, int64_t at)
{
    if constexpr (R < 16) {
        constexpr int32_t crowd = 256;
        for (uint64_t m = __ballot(s1 - s0 > crowd); m;) {
            const int l = __ffsll((unsigned long long)m) - 1;  // the leaf's first lane
            m &= ~(((1ull << (4 * R)) - 1) << l);
            p2m_leaf<T, NI, 16, true>(src, __shfl(s0, l), __shfl(s1, l), __shfl(cx, l),
                                      __shfl(cy, l), __shfl(inv_s, l), p1,
                                      M + __shfl((long long)at, l));
        }
        if (s1 - s0 > crowd) return;
    }
    if (at >= 0) p2m_leaf<T, NI, R, true>(src, s0, s1, cx, cy, inv_s, p1, M + at);
}

void set_error(const char *fmt, ...) __attribute__((format(printf, 1, 2)));

// Whether a batch's leaves take sixteen lanes rather than a wave: where the mean
// leaf has fewer than 24 points, which a wave takes in little more than one round
// of its 16 points and then spends on the butterfly; and, as a batch has nothing
// beside it, where leaves fill the chip, since sixteen lanes go four times as
// long but with an eighth of the butterfly.  Batches of leaves of 64 float32
// points, order 13: 1,024 leaves 4.8 us by waves, 8.0 by sixteen lanes; 8,192
// leaves 9.0 and 9.8, 16,384 15.4 and 15.0, 131,072 128.6 and 88.1 (108.5 with
// the table).
inline bool p2m_narrow(double points, double leaves)
{
    return points < 24.0 * leaves || leaves >= 12288.0;
}

// f(integral constant NI) for the compiled NI that holds p1 powers
template <class F>
inline int p2m_dispatch(int p1, const F &f)
{
    if (p1 <= 12)
        f(std::integral_constant<int, 3>());
    else if (p1 <= 16)
        f(std::integral_constant<int, 4>());
    else if (p1 <= 20)
        f(std::integral_constant<int, 5>());
    else if (p1 <= 24)
        f(std::integral_constant<int, 6>());
    else if (p1 <= 32)
        f(std::integral_constant<int, 8>());
    else if (p1 <= 44)
        f(std::integral_constant<int, 11>());
    else {
        set_error("expansion order %d too large (max 40)", p1 - 1);
        return PHF_ERR_UNSUPPORTED;
    }
    return PHF_OK;
}

// ------------------------------------------------------ domain choice --
// Shared by the host (single system) and the device (batched systems) so
// that both build the same tree; contraction is off so that both round
// alike.

// side of a square domain covering the extent ext (at least min_side),
// rounded up to 5 significant bits (D / 2^L is then exact)
__host__ __device__ inline double domain_side(double ext, double min_side)
{
#pragma clang fp contract(off)
    double e = ext > min_side ? ext : min_side;
    if (!(e > 0.0)) e = 1.0;
    int k = 0;
    frexp(e, &k);  // e = f 2^k, f in [0.5, 1)
    const double unit = ldexp(1.0, k - 5);
    return ceil(e / unit) * unit;
}

// leaf offset (dx, dy) is near: within ws boxes, or box gap below the cutoff
__host__ __device__ inline bool near_offset(int dx, int dy, int ws, double s, double c2)
{
#pragma clang fp contract(off)
    const int ax = dx < 0 ? -dx : dx, ay = dy < 0 ? -dy : dy;
    if (ax <= ws && ay <= ws) return true;
    const double gx = (double)(ax > 1 ? ax - 1 : 0) * s;
    const double gy = (double)(ay > 1 ? ay - 1 : 0) * s;
    return gx * gx + gy * gy < c2;
}

// near offset whose pairs may lie inside the smoothing core: box gap g with
// shape g^2 log2(e) < 26 (2% margin for float32 rounding of the point
// offsets); beyond it exp(-shape r2) <= 2^-26 for every pair
__host__ __device__ inline bool near_offset_core(int dx, int dy, double s, double shape_log2)
{
#pragma clang fp contract(off)
    const int ax = dx < 0 ? -dx : dx, ay = dy < 0 ? -dy : dy;
    const double gx = (double)(ax > 1 ? ax - 1 : 0) * s * 0.99;
    const double gy = (double)(ay > 1 ? ay - 1 : 0) * s * 0.99;
    return shape_log2 * (gx * gx + gy * gy) < 26.0;
}

// Work estimate of the near field and the leaf-level M2L of a tree with
// leaf level L >= 1 and domain side D over extents (ex, ey), nb sources and
// nt targets spread evenly: near pairs (one inside the smoothing core
// weighs 1.2 for its exponential), lanes left idle by a leaf's partial
// target chunk (half a chunk per leaf), and M2L links at p1^2 pairs each
// (4 |near(L-1)| - |near(L)| per occupied leaf).
__host__ __device__ inline double leaf_work(double ex, double ey, double D, int L, double nb,
                                            double nt, double cutoff, int ws, double shape_log2,
                                            int p1, int chunk)
{
#pragma clang fp contract(off)
    const double c2 = cutoff * cutoff;
    const double s = D / ldexp(1.0, L);
    double wnear = 0.0, nl = 0.0, np = 0.0;
    int R = (int)ceil(cutoff / s) + 2;
    R = R > ws ? R : ws;
    for (int dy = -R; dy <= R; ++dy)
        for (int dx = -R; dx <= R; ++dx)
            if (near_offset(dx, dy, ws, s, c2)) {
                nl += 1.0;
                wnear += near_offset_core(dx, dy, s, shape_log2) ? 1.2 : 1.0;
            }
    const double sp = 2.0 * s;
    int Rp = (int)ceil(cutoff / sp) + 2;
    Rp = Rp > ws ? Rp : ws;
    for (int dy = -Rp; dy <= Rp; ++dy)
        for (int dx = -Rp; dx <= Rp; ++dx)
            if (near_offset(dx, dy, ws, sp, c2)) np += 1.0;
    const double n = ldexp(1.0, L);
    double ox = ceil(ex / s), oy = ceil(ey / s);
    ox = ox < 1.0 ? 1.0 : (ox > n ? n : ox);
    oy = oy < 1.0 ? 1.0 : (oy > n ? n : oy);
    const double occ = ox * oy;
    const double spl = nb / occ, tpl = nt / occ;
    const double idle = tpl > 0.0 ? (tpl + 0.5 * chunk) / tpl : 1.0;
    return nt * spl * wnear * idle + occ * (4.0 * np - nl) * (double)(p1 * p1);
}

// Domain side at leaf level L: the bounding-box side, or one enlarged so
// that leaves are at least the Oseen cutoff wide (the near field is then
// the 3 x 3 block of leaves) when leaf_work rates it cheaper.  leaf_side
// overrides the choice: < 0 the bounding box, > 0 leaves at least
// leaf_side * cutoff wide (an autotuned setting); 0 the cost model.
__host__ __device__ inline double choose_domain_side(double ex, double ey, int L, double nb,
                                                     double nt, double cutoff, int ws,
                                                     double shape_log2, int p1, int chunk,
                                                     double leaf_side = 0.0)
{
#pragma clang fp contract(off)
    const double ext = ex > ey ? ex : ey;
    const double D = domain_side(ext, 0.0);
    if (L < 1 || leaf_side < 0.0) return D;
    if (leaf_side > 0.0)
        return domain_side(ext, leaf_side * cutoff * ldexp(1.0, L) * (1.0 + 1e-12));
    const double Dc = domain_side(ext, cutoff * ldexp(1.0, L) * (1.0 + 1e-12));
    if (!(Dc > D)) return D;
    const double w0 = leaf_work(ex, ey, D, L, nb, nt, cutoff, ws, shape_log2, p1, chunk);
    const double w1 = leaf_work(ex, ey, Dc, L, nb, nt, cutoff, ws, shape_log2, p1, chunk);
    return w1 < w0 ? Dc : D;
}

}  // namespace phf
