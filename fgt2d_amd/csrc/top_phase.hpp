// Device code shared by the kernels that form and evaluate whole cutoff-level
// boxes (kernels2d.hip, kernels3d.hip): the truncated exponentials of a
// point's leaf, and the kernel that finds every point's leaf.
#pragma once

#include <climits>

#include "fgtpw_impl.hpp"

namespace fgtpw {

typedef double d4_top __attribute__((ext_vector_type(4)));

// 1/j!, whole blocks of eight past the longest series
constexpr int TOP_WHOLE = 20;  // terms of a whole exponential's reduced series
struct TopFactorials {
    double v[TOP_RF + 6];
    constexpr TopFactorials() : v()
    {
        double f = 1.0;
        for (int j = 0; j < TOP_RF + 6; ++j) {
            if (j > 0) f *= j;
            v[j] = 1.0 / f;
        }
    }
};
static __constant__ const TopFactorials c_rf = TopFactorials();

// largest of the wavefront's values 0 <= m < 128
__device__ __forceinline__ int wave_max7(int m)
{
    int r = 0;
    bool c = true;
#pragma unroll
    for (int k = 6; k >= 0; --k) {
        const bool b = c && ((m >> k) & 1);
        if (__ballot(b)) {
            r |= 1 << k;
            c = b;
        }
    }
    return r;
}

// e[d][i] = sum_{j<m[i]-d} (i u[i])^j / j!, d < ND (the d-th derivative's
// terms); m[i] < 0: e^{i u[i]} whole, from the series of u less the nearest
// multiple of pi/2 (|u| < 40 here: two fused steps leave it to one rounding,
// and TOP_WHOLE - 2 terms of an argument below pi/4 reach 1e-18) turned back
// by that many quarters.  U ND independent Horner chains at once, the
// factorials in scalar loads of eight, a block ahead of their use.  Where
// every m of the wavefront is the same (points of one level) the terms past m
// get zero coefficients in the first two blocks alone, else every chain masks
// its own (a tile whose points lie in leaves of several levels is common).  A
// chain's sums stay zero until its first term, so both give the same bits.
template <int U, int ND>
__device__ __forceinline__ void top_series(const double (&u_)[U], const int (&m_)[U],
                                           double2 (&e)[ND][U])
{
    double u[U];
    int m[U], turn[U], low = 0;
#pragma unroll
    for (int i = 0; i < U; ++i) {
        u[i] = u_[i];
        m[i] = m_[i];
        turn[i] = 0;
        low = min(low, m[i]);
    }
    const bool whole = __any(low < 0);
    if (__builtin_expect(whole, 0)) {
#pragma unroll
        for (int i = 0; i < U; ++i)
            if (m[i] < 0) {
                const double k = rint(u[i] * 0.6366197723675814);
                u[i] = fma(-k, 6.123233995736766e-17, fma(-k, 1.5707963267948966, u[i]));
                turn[i] = (int)k;
                m[i] = TOP_WHOLE;
            }
    }
    const int m0 = __builtin_amdgcn_readfirstlane(m[0]);
    bool same = true;
    int mm = 0;
#pragma unroll
    for (int i = 0; i < U; ++i) {
        same = same && m[i] == m0;
        mm = max(mm, m[i]);
    }
    double v[U];
#pragma unroll
    for (int i = 0; i < U; ++i) v[i] = -u[i] * u[i];
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < U; ++i) e[d][i] = make_double2(0.0, 0.0);
    const bool uni = __all(same);
    const int mu = uni ? max(m0, 0) : wave_max7(mm);
    int b = max(mu - 1, 0) & ~7;
    double f[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] = c_rf.v[b + t];
    if (uni) {
#pragma unroll 1
        for (int n = 0; n < 2 && b >= 0; ++n, b -= 8) {
            double g[8];
            const int bn = max(b - 8, 0);
#pragma unroll
            for (int t = 0; t < 8; ++t) g[t] = c_rf.v[bn + t];
#pragma unroll
            for (int t = 6; t >= 0; t -= 2)
#pragma unroll
                for (int d = 0; d < ND; ++d) {
                    const double fc = b + t < mu - d ? f[t] : 0.0, fs = b + t + 1 < mu - d ? f[t + 1] : 0.0;
#pragma unroll
                    for (int i = 0; i < U; ++i) {
                        e[d][i].x = e[d][i].x * v[i] + fc;
                        e[d][i].y = e[d][i].y * v[i] + fs;
                    }
                }
#pragma unroll
            for (int t = 0; t < 8; ++t) f[t] = g[t];
        }
#pragma unroll 1
        for (; b >= 0; b -= 8) {
            double g[8];
            const int bn = max(b - 8, 0);
#pragma unroll
            for (int t = 0; t < 8; ++t) g[t] = c_rf.v[bn + t];
#pragma unroll
            for (int t = 6; t >= 0; t -= 2)
#pragma unroll
                for (int d = 0; d < ND; ++d)
#pragma unroll
                    for (int i = 0; i < U; ++i) {
                        e[d][i].x = e[d][i].x * v[i] + f[t];
                        e[d][i].y = e[d][i].y * v[i] + f[t + 1];
                    }
#pragma unroll
            for (int t = 0; t < 8; ++t) f[t] = g[t];
        }
    } else {
#pragma unroll 1
        for (; b >= 0; b -= 8) {
            double g[8];
            const int bn = max(b - 8, 0);
#pragma unroll
            for (int t = 0; t < 8; ++t) g[t] = c_rf.v[bn + t];
#pragma unroll
            for (int t = 6; t >= 0; t -= 2)
#pragma unroll
                for (int d = 0; d < ND; ++d)
#pragma unroll
                    for (int i = 0; i < U; ++i) {
                        e[d][i].x = e[d][i].x * v[i] + (b + t < m[i] - d ? f[t] : 0.0);
                        e[d][i].y = e[d][i].y * v[i] + (b + t + 1 < m[i] - d ? f[t + 1] : 0.0);
                    }
#pragma unroll
            for (int t = 0; t < 8; ++t) f[t] = g[t];
        }
    }
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < U; ++i) e[d][i].y *= u[i];
    if (__builtin_expect(whole, 0)) {
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int i = 0; i < U; ++i) {
                // times i^turn
                const double2 w = e[d][i];
                const double x = (turn[i] & 1) ? -w.y : w.x, y = (turn[i] & 1) ? w.x : w.y;
                e[d][i] = (turn[i] & 2) ? make_double2(-x, -y) : make_double2(x, y);
            }
    }
}

// e times the shift
__device__ __forceinline__ double2 top_shift(const double2 e, const double2 sh)
{
    return make_double2(e.x * sh.x - e.y * sh.y, e.x * sh.y + e.y * sh.x);
}
// m - k terms (the k-th derivative's), whole exponentials staying whole
__device__ __forceinline__ int top_less(int m, int k) { return m < 0 ? m : max(m - k, 0); }

// The leaf rank of every sorted point and the leaves' records: a wavefront
// per leaf.
template <int D>
__global__ __launch_bounds__(256) void k_top_leaves(TopLeafArgs a)
{
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= a.nleaves) return;
    const int b = a.leaf_of_rank[r], l = a.lev[b], d = l - a.ltop;
    if (d < 0) return;  // above the cutoff level: no expansions
    const int s0 = a.ls[r], s1 = a.ls[r + 1], t0 = a.ls2 ? a.ls2[r] : 0, t1 = a.ls2 ? a.ls2[r + 1] : 0;
    for (int i = s0 + lane; i < s1; i += 64) a.pb[i] = r;
    if (a.pb2)
        for (int i = t0 + lane; i < t1; i += 64) a.pb2[i] = r;
    if (lane != 0) return;
    int top = b;
    for (int k = 0; k < d; ++k) top = a.par[top];
    TopRec q;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        q.c[k] = 0;
        q.row[k] = 0;
        if (k >= D) continue;
        q.c[k] = a.cen[D * (long)b + k];
        // the leaf's place among the 2^d boxes of its level along the axis
        const int pos = (int)rint((q.c[k] - a.cen[D * (long)top + k]) * a.ib[l] +
                                  0.5 * ((1 << d) - 1));
        q.row[k] = ((1 << d) - 1 + pos) * a.half;
    }
    // plane-wave route: formation up to fth sources, evaluation below eth points
    const int fth = a.fth[l], eth = a.eth[l], n = s1 - s0;
    q.mf = fth > 0 && (fth == INT_MAX || n <= fth) ? -1 : a.m[l];
    q.me = eth > 0 && (eth == INT_MAX || n + (t1 - t0) < eth) ? -1 : a.m[l];
    a.rec[r] = q;
}

template <int D>
static void top_leaves_launch(const TopLeafArgs& a, hipStream_t s)
{
    if (a.nleaves <= 0) return;
    k_top_leaves<D><<<(a.nleaves + 3) / 4, 256, 0, s>>>(a);
}

}  // namespace fgtpw
