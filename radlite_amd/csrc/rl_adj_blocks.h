// Reverse sweep by independent (block, channel) pairs.
//
// The adjoint of a ray runs backwards: lambda = dL/dI at a segment's end is
// needed before the segment can be reversed.  But over a block of BLK segments
// I -> P I + B, so lambda = lambda_end P: the forward pass keeps, per block and
// channel, I at the block's start and P, and one cheap pass over those
// (k_adj_lambda) gives lambda at every block's end.  From there every pair of a
// block and a channel is on its own.  A channel that does not see the line on a
// block (bounds as in rl_blocks.h, the cut taken so far out that the line's own
// gradients there are below BITS bits of what the block's other channels give)
// passes the dust elements, whose gradient is linear in lambda and lambda I:
// the two sums over those channels are all that the block's dust needs.  The
// pairs that see the line are taken 64 at a time, a lane each.
//
// What bounds it: instruction issue in the element reversals.  The sweep by
// (ray, 64 channels), a segment at a time, stepped every lane through the
// sub-grid points of the few channels at resonance.
// 200 x 100 disk, 100 channels, FP32: reverse sweep 13.1 -> 6.9 ms (pairs 5.7,
// lambda 1.0, bounds 0.2), a fit's step 20.2 -> 11.5 ms with the forward by maps;
// FP64, 32 angles, a step 11.6 -> 5.8 ms; 40 x 24 disk, 24 channels, FP64, a step
// 1.78 -> 0.90.  Half of the lanes of k_adj_pairs have work (SQ counters).
// Held to 128 registers it spills, with more than 168 too few waves are left.
#pragma once
#include "rl_adjoint.h"
#include "rl_blocks.h"
#include "rl_walk.h"

namespace rl {

constexpr int ADJ_WIN = 16;          // blocks of a ray at a time (their sums in LDS)
// rows (nodes) of a batch's lanes held at a time: 25 words a lane, an odd
// stride, so that the 64 rows fall in distinct banks
constexpr int ADJ_ROWS = 5, ADJ_W = ADJ_ROWS * 5;

template <typename T> struct AdjLim;
template <> struct AdjLim<float> { static constexpr float bits = 30.0f, zero = 150.0f; };
template <> struct AdjLim<double> { static constexpr float bits = 60.0f, zero = 1080.0f; };

template <typename T> struct AdjLds {
    T row[64][ADJ_W];
    T iseg[BLK][64];                 // a lane's I before each segment of its block
    double acc[ADJ_WIN * BLK + 1][5];
    int st[ADJ_WIN + 1];             // first pair of each block
};

// dust alone at a node
template <typename T>
__device__ inline FPtT<T> dust_of(const FastRecT<T> &a) {
    return FPtT<T>{a.u, a.sig, a.jdh, a.adh, T(0), T(0)};
}

// the channel velocities [lo, hi] that see the line on the nb blocks of a ray
// of n nodes (lane <-> block; -inf .. inf: every channel), and the blocks' dust
// maps I -> x I + y
template <typename T>
__device__ inline void adj_bounds(int lane, const FastRecT<T> *__restrict__ rec, int n, int nb,
                                  T nu0, float2 *__restrict__ out, double2 *__restrict__ dust) {
    const FastLineT<T> L{nu0, T(0), T(0)};
    const float scale = 0.8325546112f / (float)fabs(nu0);      // sqrt(ln 2)
    for (int j = lane; j < nb; j += 64) {
        float lo = INFINITY, hi = -INFINITY;
        const int k1 = min(j * BLK + BLK, n);
        int k = max(1, j * BLK);
        FastRecT<T> p = rec[k - 1];
        RayMap<T> x;
        for (; k < k1; k++) {
            const FastRecT<T> r = rec[k];
            FastCarryT<T> c;
            int ovs = 0;
            elem_fast<T>(L, x, r.ds, dust_of<T>(p), dust_of<T>(r), r.inv_aa, r.norm, c, ovs);
            // the widest and narrowest profile at node k-1
            const bool two = k > 1;
            const float ia = (float)(two && p.inv_aa < r.inv_aa ? p.inv_aa : r.inv_aa);
            const float ng = (float)(two && p.norm > r.norm ? p.norm : r.norm);
            const float M = fmaxf(fmaxf(blk_ratio(p.jch, p.jdh), blk_ratio(p.dch, p.adh)),
                                  fmaxf(blk_ratio(r.jch, r.jdh), blk_ratio(r.dch, r.adh))) * ng;
            const float most = (float)(fabs(p.jch) + fabs(p.dch) + fabs(r.jch) + fabs(r.dch)) * ng;
            float t = fminf(AdjLim<T>::bits + fmaxf(0.0f, __log2f(M)), AdjLim<T>::zero);
            if (p.dch < T(0) || r.dch < T(0) || !(M >= 0.0f)) t = AdjLim<T>::zero;
            const float z = (sqrtf(t) + 0.01f) * scale / ia;
            lo = fminf(lo, (float)fmin(p.u, r.u) - z);
            hi = fmaxf(hi, (float)fmax(p.u, r.u) + z);
            // never free: the star's intensity, or a line, a velocity or a width that
            // is no number
            if (((int)r.flag & (NF_BLEND | NF_STAR)) || !(most < INFINITY) || !(z < INFINITY) ||
                !blk_sane(p.u, r.u, (float)r.inv_aa, (float)(two ? p.inv_aa : r.inv_aa))) {
                lo = -INFINITY;
                hi = INFINITY;
            }
            p = r;
        }
        out[j] = make_float2(lo, hi);
        dust[j] = make_double2(x.P, x.B);
    }
}

// whether channel velocity v sees the line on a block of bounds b
template <typename T> __device__ inline bool sees(float2 b, T v) {
    return !(b.x > b.y) && !(v < (T)b.x) && !(v > (T)b.y);
}

// the carry at the start of block j of a ray (rec: its first record)
template <typename T>
__device__ inline void block_carry(const FastRecT<T> *__restrict__ rec, int j,
                                   const FastLineT<T> &L, FastCarryT<T> &c) {
    const FastRecT<T> a = rec[max(j * BLK - 1, 0)];
    c.u0 = a.u;
    c.init = 1;
    if (j > 0) {
        T jl0, al0, z_, phi_;
        carried_in<T>(a, L, jl0, al0, z_, phi_);
        carry_start<T>(point_of<T>(a), jl0, al0, c);
        c.init = 0;
    }
}

// the dust gradients of block j (rec: the ray's first record) from s0 = sum
// lambda and s1 = sum lambda I over the channels that do not see the line, into
// the block's rows acc[0 .. BLK] (row m: node j BLK + m - 1).  Called by every
// lane of the wave; lanes without a block pass on = false.
template <typename T>
__device__ inline void block_dust_rev(const FastRecT<T> *__restrict__ rec, int j, int n, bool on,
                                      double s0, double s1, T nu0, double (*acc)[5]) {
    const FastLineT<T> L{nu0, T(0), T(0)};
    const int k0 = max(1, j * BLK);
    const int k1 = on && (s0 != 0.0 || s1 != 0.0) ? min(j * BLK + BLK, n) : k0;   // [k0, k1)
    double pa[BLK], pb[BLK], px[BLK];
    double A = 1.0, B = 0.0;
#pragma unroll 1
    for (int k = k0; k < k1; k++) {
        const FastRecT<T> r = rec[k];
        FastCarryT<T> c;
        RayMap<T> x;
        int ovs = 0;
        pa[k - k0] = A;
        pb[k - k0] = B;
        elem_fast<T>(L, x, r.ds, dust_of<T>(rec[k - 1]), dust_of<T>(r), r.inv_aa, r.norm, c, ovs);
        px[k - k0] = x.P;
        B = B * x.P + x.B;
        A = A * x.P;
    }
    double suf = 1.0;
    PGrad<T> cur, prv;
    pg_zero(cur);
#pragma unroll 1
    for (int k = k1 - 1; k >= k0; k--) {
        const FastRecT<T> r = rec[k];
        T g_h = T(0), g_ln = T(0), gjl0, gal0;
        pg_zero(prv);
        const double l0 = suf * s0, l1 = suf * (pa[k - k0] * s1 + pb[k - k0] * s0);
        elem_rev_sum<T>(L, (T)l1, (T)l0, r.ds, dust_of<T>(rec[k - 1]), dust_of<T>(r), T(0), T(0),
                        r.inv_aa, r.norm, 1, T(0), T(0), T(0), T(0), prv, cur, g_h, g_ln, gjl0,
                        gal0);
        suf *= px[k - k0];
        const int m = k - j * BLK + 1;
        acc[m][0] += (double)cur.jd;
        acc[m][1] += (double)cur.ad;
        cur = prv;
    }
    wave_lds_fence();
    if (k1 > k0) {
        // node k0-1: row 0, the last row of the block before (its rows are in)
        const int m = k0 - j * BLK;
        acc[m][0] += (double)cur.jd;
        acc[m][1] += (double)cur.ad;
    }
    wave_lds_fence();
}

// what a wave knows of its ray
template <typename T> struct AdjRay {
    const FastRecT<T> *rec;          // its first record
    int n, nb, nfr;                  // nodes, blocks, channels
    const float2 *bounds;            // its blocks'
    const T *ckI, *lam;              // [block][channel] I at the start, lambda at the end
    const double *bsum;              // [block][group][2]
    const double *dnu, *velo, *istar;
    T nu0, sf, cai;
};

// the channels cl .. cl + cnt - 1 that see the line on block j
template <typename T>
__device__ inline void block_channels(const AdjRay<T> &y, int j, T v0, T inv, int &cl, int &cnt) {
    const float2 b = y.bounds[j];
    if (b.x > b.y) return;
    channels_in<T>(y.velo, 0, y.nfr, v0, inv, b.x, b.y, cl, cnt);
}

// a batch of pairs, a lane each: lane's block jl of the window that begins at
// block jw, channel ch; on: the lane has a pair.  Blocks first .. last take part,
// the pairs p0 .. pend-1.
template <typename T>
__device__ __forceinline__ void pair_batch(AdjLds<T> &S, const AdjRay<T> &y, int jw, int jl,
                                           int ch, bool on, int first, int last, int p0,
                                           int pend) {
    const int lane = threadIdx.x & 63;
    const int j = jw + jl, kb = j * BLK, n = y.n;
    const FastLineT<T> L{y.nu0, (T)y.dnu[ch], (T)y.velo[ch]};
    const T ist = (T)y.istar[ch];
    const long long slot = (long long)j * y.nfr + ch;
    T I = y.ckI[slot];
    T lam = on ? y.lam[slot] : T(0);
    // I before each of the block's segments, as the forward pass had it
    {
        FastCarryT<T> c;
        block_carry<T>(y.rec, j, L, c);
        int ovs = 0;
#pragma unroll 1
        for (int i = 0; i < BLK; i++) {
            const int k = kb + i;
            S.iseg[i][lane] = I;
            if (k >= 1 && k < n - 1 && i < BLK - 1) {
                const FastRecT<T> r = y.rec[k];
                segment_fast<T>(r, y.rec + k - 1, point_of<T>(r), L, I, ist, y.sf, c, ovs);
            }
        }
    }
    // rows top, top-1, ... (R of them) of the lanes' blocks, summed per block
    auto flush = [&](int top, int R) __attribute__((always_inline)) {
        wave_lds_fence();
        const int per = R * 5, items = (last - first + 1) * per;
        for (int it = lane; it < items; it += 64) {
            const int bl = it / per, q = it - bl * per, b = first + bl;
            const int s = max(S.st[b] - p0, 0), e = min(S.st[b + 1], pend) - p0;
            if (e > s) {
                double sum = 0.0;
                for (int i = s; i < e; i++) sum += (double)S.row[i][q];
                const int r = q / 5;
                S.acc[b * BLK + top - r][q - r * 5] += sum;
            }
        }
        wave_lds_fence();
    };
    T gjl = T(0), gal = T(0), zc, phic;
    PGrad<T> cur, prv;
    pg_zero(cur);
    T isub[33];                      // 33 entries: kept in scratch memory, not registers
    {
        const FastRecT<T> r = y.rec[min(kb + BLK - 1, n - 1)];
        profile_at<T>(L, r.u, r.inv_aa, r.norm, zc, phic);
    }
    int col = 0;
#pragma unroll 1
    for (int m = BLK; m >= 1; m--) {
        // segment k; a lane whose block has no such segment takes another with
        // lambda = 0
        const int k = kb + m - 1;
        const bool has = k >= 1 && k < n;
        const int kc = min(max(k, 1), n - 1);
        const FastRecT<T> r = y.rec[kc];
        const FastRecT<T> a = y.rec[kc - 1];
        T g_lnaa = T(0), g_dls = T(0);
        T jl0c = T(0), al0c = T(0), za = T(0), phia = T(0);
        if (kc > 1) carried_in<T>(a, L, jl0c, al0c, za, phia);
        pg_zero(prv);
        T gj = has ? gjl : T(0), ga = has ? gal : T(0);
        const T li = segment_rev<T>(r, point_of<T>(a), point_of<T>(r), L, S.iseg[m - 1][lane],
                                    has ? lam : T(0), ist, y.sf, kc == 1 ? 1 : 0, jl0c, al0c, zc,
                                    phic, gj, ga, prv, cur, g_lnaa, g_dls, isub);
        if (has) {
            lam = li;
            gjl = gj;
            gal = ga;
            zc = za;
            phic = phia;
        }
        // d lw_mean: phi through inv_aa = 1/(c_aa lw), sub-grid width dls ~ lw
        T *o = S.row[lane] + col * 5;
        o[0] = cur.jd; o[1] = cur.ad; o[2] = cur.jc; o[3] = cur.dc;
        o[4] = (g_dls * r.dls - g_lnaa) * y.cai * r.inv_aa;
        cur = prv;
        if (++col == ADJ_ROWS) {
            flush(m + ADJ_ROWS - 1, ADJ_ROWS);
            col = 0;
        }
    }
    // node kb-1, whose line values under the profile of the segment before the
    // block were carried into it
    {
        const FastRecT<T> a = y.rec[max(kb - 1, 0)];
        const T t1 = (gjl * a.jch + gal * a.dch) * phic;
        T *o = S.row[lane] + col * 5;
        o[0] = cur.jd; o[1] = cur.ad;
        o[2] = cur.jc + gjl * phic;
        o[3] = cur.dc + gal * phic;
        o[4] = -t1 * (T(1) - T(2) * zc * zc) * y.cai * a.inv_aa;
    }
    flush(BLK + 1 - ADJ_ROWS - 1, BLK + 1 - ADJ_ROWS);
}

// forward: the maps of a ray's pairs, packed the same way (one wave), to outP and
// outB [block][channel]
template <typename T>
__device__ __forceinline__ void adj_ray_maps(const AdjRay<T> &y, T *__restrict__ outP,
                                             T *__restrict__ outB) {
    const int lane = threadIdx.x & 63;
    const T v0 = (T)y.velo[0], v1 = (T)y.velo[y.nfr - 1];
    const T inv = y.nfr > 1 ? (T)(y.nfr - 1) / (v1 - v0) : T(0);
    for (int jw = 0; jw < y.nb; jw += 64) {
        const int m = min(64, y.nb - jw);
        int cl = 0, cnt = 0;
        if (lane < m) block_channels<T>(y, jw + lane, v0, inv, cl, cnt);
        int incl = cnt;
        for (int d = 1; d < 64; d <<= 1) {
            const int t = __shfl_up(incl, d);
            if (lane >= d) incl += t;
        }
        const int st = incl - cnt, total = lane_of(incl, m - 1);
#pragma unroll 1
        for (int p0 = 0; p0 < total; p0 += 64) {
            const int p = min(p0 + lane, total - 1);
            int jl = 0;                       // the last block that begins at or before p
            for (int d = 32; d >= 1; d >>= 1) {
                const int t = __shfl(st, min(jl + d, 63));
                if (jl + d < m && t <= p) jl += d;
            }
            const int ch = __shfl(cl, jl) + p - __shfl(st, jl);
            const int j = jw + jl, kb = j * BLK;
            const FastLineT<T> L{y.nu0, (T)y.dnu[ch], (T)y.velo[ch]};
            const T ist = (T)y.istar[ch];
            FastCarryT<T> c;
            block_carry<T>(y.rec, j, L, c);
            RayMap<T> x;
            int ovs = 0;
#pragma unroll 1
            for (int i = 0; i < BLK; i++) {
                const int k = kb + i;
                if (k >= 1 && k < y.n) {
                    const FastRecT<T> r = y.rec[k];
                    segment_fast<T>(r, y.rec + k - 1, point_of<T>(r), L, x, ist, y.sf, c, ovs);
                }
            }
            if (p0 + lane < total) {
                const long long slot = (long long)j * y.nfr + ch;
                outP[slot] = (T)x.P;
                outB[slot] = (T)x.B;
            }
        }
    }
}

// the node gradients of one ray (one wave)
template <typename T>
__device__ __forceinline__ void adj_ray(AdjLds<T> &S, const AdjRay<T> &y, int ngrp,
                                        double *__restrict__ gnode) {
    const int lane = threadIdx.x & 63;
    const T v0 = (T)y.velo[0], v1 = (T)y.velo[y.nfr - 1];
    const T inv = y.nfr > 1 ? (T)(y.nfr - 1) / (v1 - v0) : T(0);
    double *flat = &S.acc[0][0];
    if (lane < 5) flat[lane] = 0.0;
    for (int jw = 0; jw < y.nb; jw += ADJ_WIN) {
        const int m = min(ADJ_WIN, y.nb - jw);
        for (int i = 5 + lane; i < (m * BLK + 1) * 5; i += 64) flat[i] = 0.0;
        int cl = 0, cnt = 0;
        double s0 = 0.0, s1 = 0.0;
        if (lane < m) {
            block_channels<T>(y, jw + lane, v0, inv, cl, cnt);
            const double *s = y.bsum + (long long)(jw + lane) * ngrp * 2;
            for (int g = 0; g < ngrp; g++) {
                s0 += s[2 * g];
                s1 += s[2 * g + 1];
            }
        }
        int incl = cnt;
        for (int d = 1; d <= ADJ_WIN; d <<= 1) {      // lane m too
            const int t = __shfl_up(incl, d);
            if (lane >= d) incl += t;
        }
        const int st = incl - cnt, total = lane_of(incl, m - 1);
        if (lane <= m) S.st[lane] = st;          // lane m: the total (m < 64)
        wave_lds_fence();
        block_dust_rev<T>(y.rec, jw + min(lane, m - 1), y.n, lane < m, s0, s1, y.nu0,
                          S.acc + min(lane, m - 1) * BLK);
#pragma unroll 1
        for (int p0 = 0; p0 < total; p0 += 64) {
            const int pend = min(p0 + 64, total), p = min(p0 + lane, pend - 1);
            int jl = 0;
            for (int b = 1; b < m; b++) jl += p >= lane_of(st, b) ? 1 : 0;
            const int ch = __shfl(cl, jl) + p - __shfl(st, jl);
            pair_batch<T>(S, y, jw, jl, ch, p0 + lane < pend, lane_of(jl, 0),
                          lane_of(jl, pend - 1 - p0), p0, pend);
        }
        // rows 0 .. m BLK - 1 are complete; the last begins the next window
        const bool end = jw + ADJ_WIN >= y.nb;
        const int rows = m * BLK + (end ? 1 : 0), node0 = jw * BLK - 1;
        for (int i = lane; i < rows * 5; i += 64) {
            const int node = node0 + i / 5;
            if (node >= 0 && node < y.n) gnode[(long long)node0 * 5 + i] = flat[i];
        }
        wave_lds_fence();
        if (!end && lane < 5) flat[lane] = flat[m * BLK * 5 + lane];
        wave_lds_fence();
    }
}

}  // namespace rl
