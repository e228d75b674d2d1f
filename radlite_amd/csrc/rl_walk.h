// The wave walk of the formal solution: 64/cw rays x cw channels per wave, the
// rays' records through LDS block by block (rl_blocks.h).
//
// A wave's lanes are on the same block of their rays: one whose line none of
// a ray's lanes can see is one multiply-add, and the others' segments are
// integrated by the lanes that see them.  (A lane that walked its own list of
// blocks would meet the sub-gridded segments at another time than its
// neighbours, and the wave would run through both kinds at every step: 54 ms
// for the 400 x 200 disk's two inclinations, 50 ms without blocks, 26 ms in
// step, 19 ms with the records through LDS.)
// Whether a lane takes a block's map or its segments is the lane's own
// matter, so results do not depend on which lanes share a wave.
//
// Sixteen channels per ray (cw = 16) keep the union of what the lanes see
// small: with T = 1000 K (R/AU)^-1/2 and 200 channels over +-40 km/s the wave
// integrates 19% of its segments (64 channels: 30%, 32: 28%, a lane alone:
// 11%).
//
// The lanes of a ray load 16 block records at a time, one each, and for a
// block that is integrated the records of its nodes, a 16-byte piece each, and
// read them from LDS (broadcasts): three vector loads per lane and block
// instead of two or more per lane and segment.
#pragma once
#include "rl_device.h"
#include "rl_fwd32.h"

namespace rl {

constexpr int WALK_WIN = 16;                // block records held at a time
// waves per SIMD of the FP32 kernels: at 8 (64 registers) 36 values spill, the
// sub-grid path's among them (400 x 200 disk 19.9 against 19.2 ms, 97 x 61
// disk 0.68 against 0.63)
constexpr int FORMAL32_WAVES = 6;

template <typename T> struct WalkLds;
// nodes k0-1 .. k0+BLK-1 of a ray (clamped to the ray): SegHot, SegAux, NodeLine
template <> struct WalkLds<float> {
    static constexpr int N = BLK + 1;
    BlkRec win[4][WALK_WIN];
    float4 st[4][3 * N];
};
// nodes k0-2 .. k0+BLK-1
template <> struct WalkLds<double> {
    static constexpr int N = BLK + 2;
    BlkRec win[4][WALK_WIN];
    NodeRec<double> st[4][N];
};

// LDS written by a wave's lanes is read by its other lanes: LDS operations
// of a wave are performed in order, so only the compiler must keep it
__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the four 16-bit fields of a ballot over rays of 1 << cwl lanes, combined
__device__ inline unsigned fold16(unsigned long long m, int cwl) {
    unsigned r = (unsigned)m;
    if (cwl < 6) r |= (unsigned)(m >> 32);
    if (cwl < 5) r |= r >> 16;
    return r & 0xffffu;
}

// The blocks [j0, j1) of each ray.  free(A, B, overshoots): the lane takes the
// block's map; stage(j): the ray's lanes load block j's nodes into LDS (called
// for the rays that have a block j); integrate(j): the lane integrates it.
// on: the lane has a channel to integrate; blk null: no block is free.
template <typename T, typename Free, typename Stage, typename Integrate>
__device__ __forceinline__ void walk(BlkRec (*win)[WALK_WIN], int cwl,
                                     const BlkRec *__restrict__ blk, int j0, int j1, bool on,
                                     float ulo, float uhi, T uch, const Free &free,
                                     const Stage &stage, const Integrate &integrate) {
    const int lane = threadIdx.x & 63, g = lane >> cwl, li = lane & ((1 << cwl) - 1);
    // the ray's channels
    if (!on) { ulo = INFINITY; uhi = -INFINITY; }
    for (int m = 1; m < (1 << cwl); m <<= 1) {
        ulo = fminf(ulo, __shfl_xor(ulo, m));
        uhi = fmaxf(uhi, __shfl_xor(uhi, m));
    }
    for (int jw = j0; __any(jw < j1); jw += WALK_WIN) {
        const bool act = li < WALK_WIN && jw + li < j1;
        float lo = INFINITY, hi = -INFINITY;          // no block: the identity, free
        double A = 1.0, B = 0.0;
        if (act) {
            lo = -INFINITY;
            hi = INFINITY;
            if (blk) {
                const BlkRec *r = blk + jw + li;
                lo = r->lo; hi = r->hi; A = r->A; B = r->B;
            }
        }
        wave_lds_fence();
        if (li < WALK_WIN) {
            BlkRec *w = &win[g][li];
            w->lo = lo; w->hi = hi; w->A = A; w->B = B;
        }
        const unsigned busy = fold16(__ballot(act && !(uhi < lo || ulo > hi)), cwl);
        const unsigned have = fold16(__ballot(act), cwl);
        const bool over = __any(act && (__float_as_int(lo) & (2 * BLK - 1)) != 0);
        wave_lds_fence();
        const int nw = 32 - __clz((int)have);
        for (int b = 0; b < nw; b++) {
            const BlkRec &w = win[g][b];
            if (!((busy >> b) & 1)) {
                free(w.A, w.B, over ? blk_overshoots(w) : 0);
                continue;
            }
            const bool mine = jw + b < j1;
            if (mine) stage(g, li, jw + b);
            wave_lds_fence();
            if (mine && on) {
                if (blk_free(w, uch)) free(w.A, w.B, blk_overshoots(w));
                else integrate(g, jw + b);
            }
            wave_lds_fence();
        }
    }
}

// FP32: charintline (telescope.F:3889-4312) over the blocks [j0, j1) of a ray
// of n nodes, on split records (rl_fwd32.h)
template <bool AFF>
__device__ __forceinline__ void walk_split(WalkLds<float> &S, int cwl,
                                           const SegHot *__restrict__ hot,
                                           const SegAux *__restrict__ aux,
                                           const NodeLine *__restrict__ line,
                                           const BlkRec *__restrict__ blk, int n, int j0, int j1,
                                           bool on, float uch, Acc32<AFF> &x, float istar,
                                           float sf, bool &ovf, int &maser) {
    constexpr int N = WalkLds<float>::N;
    Car32 c;
    bool fresh = true;
    walk(S.win, cwl, blk, j0, j1, on, uch, uch, uch,
         [&](double A, double B, int over) __attribute__((always_inline)) {
             x.map(A, B);
             ovf = ovf || over != 0;
             fresh = true;
         },
         [&](int g, int li, int j) __attribute__((always_inline)) {
             if (li >= N) return;
             const int k = min(max((j << BLK_LOG) - 1 + li, 0), n - 1);
             S.st[g][li] = reinterpret_cast<const float4 *>(hot)[k];
             S.st[g][N + li] = reinterpret_cast<const float4 *>(aux)[k];
             S.st[g][2 * N + li] = reinterpret_cast<const float4 *>(line)[k];
         },
         [&](int g, int j) __attribute__((always_inline)) {
             const SegHot *sh = reinterpret_cast<const SegHot *>(S.st[g]);
             const SegAux *sa = reinterpret_cast<const SegAux *>(S.st[g] + N);
             const NodeLine *sl = reinterpret_cast<const NodeLine *>(S.st[g] + 2 * N);
             const int k0 = j << BLK_LOG, i1 = min(BLK, n - k0);
             if (fresh) {
                 // the carry of node k0-1 as the end of segment k0-1 (its
                 // profile); the ray's first node under segment 1's
                 const int m = j > 0 ? 0 : 1;
                 const SegHot hp = sh[2 * m];
                 carry32(pt_of(sa[m].u, sl[m]), uch, hp.ag, hp.ng, c);
                 fresh = false;
             }
             for (int i = j > 0 ? 0 : 1; i < i1; i++) {
                 segment32(x, sh + i + 1, sa + i + 1, sl + i + 1, uch, istar, sf, c, ovf, maser);
             }
         });
}

// FP64: the same on whole node records, with the reference's own arithmetic
template <bool AFF>
__device__ __forceinline__ void walk_exact(WalkLds<double> &S, int cwl,
                                           const NodeRec<double> *__restrict__ rec,
                                           const BlkRec *__restrict__ blk, int n, int j0, int j1,
                                           bool on, const LineK<double> &L, Acc<double, AFF> &x,
                                           double istar, double sf, int &ovs, int &maser) {
    constexpr int N = WalkLds<double>::N;
    Carry<double> c;
    c.init = 1; c.phi0 = 0.0; c.srcl0 = 0.0; c.alpl0 = 0.0; c.S0 = 0.0;
    bool fresh = true;
    const float uf = (float)L.uch;
    walk(S.win, cwl, blk, j0, j1, on, nextafterf(uf, -INFINITY), nextafterf(uf, INFINITY), L.uch,
         [&](double A, double B, int over) __attribute__((always_inline)) {
             x.map(A, B);
             ovs += over;
             fresh = true;
         },
         [&](int g, int li, int j) __attribute__((always_inline)) {
             const int k0 = (j << BLK_LOG) - 2;
             for (int p = li; p < 4 * N; p += 1 << cwl) {
                 const int k = min(max(k0 + (p >> 2), 0), n - 1);
                 reinterpret_cast<float4 *>(S.st[g])[p] =
                     reinterpret_cast<const float4 *>(rec)[(size_t)k * 4 + (p & 3)];
             }
         },
         [&](int g, int j) __attribute__((always_inline)) {
             const NodeRec<double> *sr = S.st[g];
             const int k0 = j << BLK_LOG, i1 = min(BLK, n - k0);
             if (fresh && j > 0) carry_of<double>(L, sr[0], sr[1], c);
             fresh = false;
             for (int i = j > 0 ? 0 : 1; i < i1; i++)
                 segment_exact<double>(L, x, sr[i + 1], sr[i + 2], istar, sf, c, ovs, maser);
         });
}

}  // namespace rl
