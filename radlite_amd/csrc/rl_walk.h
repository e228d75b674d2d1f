// The formal solution of one ray, all channels of a chunk, by one wave.
//
// Along a ray a channel sees the line in about a tenth of the blocks
// (rl_blocks.h); in the others every channel takes the block's own map.  So the
// (block, channel) pairs that see the line, a block's channels consecutive, are
// taken 64 at a time, a lane each, as a stream along the ray:
//
//   stage      the nodes of the blocks that the 64 pairs begin, into LDS (the
//              next blocks' loads are in flight while a batch is integrated)
//   integrate  each lane its pair's map I -> P I + B, into LDS
//   compose    a lane per channel: the maps of the blocks now complete, in
//              order, the pair's where there is one, else the block's own
//
// A batch costs about the same full or not: at each of its 8 segments it waits for
// the longest of its lanes' sub-grid loops.  With few channels the blocks that LDS
// holds make up a small part of one, so that where a window of 64 blocks has that
// few pairs they are taken 64 at a time from any number of blocks, each lane from
// its block's nodes in memory.  Formal solution, one inclination, +-30 km/s: 400 x
// 200 disk, 64 angles, 9 channels, FP32, 1.17 -> 0.65 ms, 40 channels 1.20 -> 0.88; FP64
// 2.36 -> 1.16 and 2.47 -> 2.03; 100 x 60 disk, 50 channels, FP64, 0.87 -> 0.83 a call.
//
// What bounds it: instruction issue, then the latency of a batch's steps.
// Lanes that held one (ray, channel) each and met at every block that one of 16
// channels saw had work in 38% of their instructions, and a ray of many blocks
// was one serial chain; packed pairs fill 65% (SQ counters, 400 x 200 disk, 200
// channels, FP32; 0.92 VALU instructions a cycle and compute unit), and their chains
// are a block long.  One launch, 400 x 200 disk, two inclinations, FP32: 19.3 -> 16.1 ms;
// 200 x 100 disk, FP64: 4.8 -> 3.1 ms; 100 x 60 disk, FP64: 0.96 -> 0.40 ms;
// 97 x 61 disk, FP32: 0.62 -> 0.27 ms.  (A wave per eighth of a ray, for
// launches of few rays: 14 of 64 lanes with work, 1.22 ms for the 100 x 60
// disk.  Without the loads in flight ahead of a batch: 19.0 against 16.1 ms.)
//
// A channel's maps are the same whatever else its wave holds, and are applied
// one by one: results do not depend on chunks, batches or the launch.
#pragma once
#include "rl_device.h"
#include "rl_fwd32.h"

namespace rl {

// waves per SIMD that the kernels' registers are held to: FP32 in five, with
// chunks of 128 channels, spilled in the element loop (22.9 against 19.0 ms for
// the 400 x 200 disk); FP64 in two did not spill but waited (3.96 against 3.69
// ms, 200 x 100 disk)
constexpr int FORMAL32_WAVES = 4, FORMAL64_WAVES = 3;

// block records held at a time (a lane each); blocks whose nodes are in LDS, and
// of these, those that one batch of pairs takes
constexpr int RECS = 64, SLOTS = 11, BATCH_BLOCKS = 7;
// a chunk has up to GROUPS groups of 64 channels: a ray's records are read once
// per chunk, and the ring of a chunk's pairs leaves room for the four waves
constexpr int GROUPS = 4;

template <typename T> struct Nodes;
// nodes k0-1 .. k0+BLK-1 of a block (clamped to the ray): SegHot, SegAux, NodeLine
template <> struct Nodes<float> {
    static constexpr int N = BLK + 1, PIECES = 3 * N, AHEAD = 128 / PIECES;
};
// nodes k0-2 .. k0+BLK-1
template <> struct Nodes<double> {
    static constexpr int N = BLK + 2, PIECES = 4 * N, AHEAD = 128 / PIECES;
};

struct Map {
    double P, B;
};

// one wave's share of LDS, for chunks of up to 64 G channels
template <typename T, int G> struct WalkLds {
    static constexpr int RING = 64 * G + 64;           // a chunk's pairs of one block + 64
    Map map[RING];                                     // pair p at p % RING
    float4 st[SLOTS][Nodes<T>::PIECES];
};

// LDS written by a wave's lanes is read by its other lanes: LDS operations
// of a wave are performed in order, so only the compiler must keep it
__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline int lane_of(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ inline double lane_of(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// FP32: the sign of a map's factor (never negative) marks an overshoot
__device__ inline double mark(double P, bool ovf) { return copysign(P, ovf ? -1.0 : 1.0); }
__device__ inline bool marked(double P) { return __double2hiint(P) < 0; }

// the channels of [c0, c1) whose velocity lies in [lo, hi]: their first, cl, and
// number, cnt.  v ascends, or descends for a line of negative rest frequency (v =
// dnu/nu0), or is no number (a passband without end): such a channel is taken.
// v0: v[c0]; inv: channels per velocity (negative descending, 0 for one channel).
template <typename T>
__device__ inline void channels_in(const double *__restrict__ v, int c0, int c1, T v0, T inv,
                                   float lo, float hi, int &cl, int &cnt) {
    const T s = inv < T(0) ? T(-1) : T(1);       // s v ascends
    const T b0 = s * (T)(inv < T(0) ? hi : lo), b1 = s * (T)(inv < T(0) ? lo : hi);
    // the number of channels that come before the bound, from where it would lie
    // if the channels were exactly even
    auto bound = [&](T est, auto before) {
        int c = (int)fmin(fmax(est, (T)c0), (T)c1);
        while (c > c0 && !before(c - 1)) c--;
        while (c < c1 && before(c)) c++;
        return c;
    };
    cl = bound((T)c0 + (s * b0 - v0) * inv, [&](int k) { return s * (T)v[k] < b0; });
    cnt = max(0, bound((T)c0 + (s * b1 - v0) * inv + T(1),
                       [&](int k) { return !(s * (T)v[k] > b1); }) - cl);
}

// the channels of a chunk as a wave holds them
struct Chans {
    const double *velo;
    int c0, c1, ng;             // [c0, c1), groups of 64
};

// The nb blocks of a ray: I[g] the intensity of channel c0 + 64 g + lane; over:
// FP32, bit g set on an overshoot.  stage(j, piece): a piece of block j's
// nodes; before(c): what channel c needs, loaded while the nodes arrive;
// integrate(nodes, j, c, that): the map of block j for channel c; direct(j, c,
// that): the same from the nodes in memory (G = 1); passed(g, n): n overshoots of a
// block's own map.
template <typename T, int G, typename Stage, typename Before, typename Integrate, typename Direct,
          typename Free>
__device__ __forceinline__ void walk(WalkLds<T, G> &S, const BlkRec *__restrict__ blk, int nb,
                                     const Chans &ch, double (&I)[G], unsigned &over,
                                     const Stage &stage, const Before &before,
                                     const Integrate &integrate, const Direct &direct,
                                     const Free &passed) {
    using Pre = decltype(before(0));
    constexpr int RING = WalkLds<T, G>::RING;
    constexpr bool FEW = G == 1;
    const int lane = threadIdx.x & 63;
    const T v0 = (T)ch.velo[ch.c0], v1 = (T)ch.velo[ch.c1 - 1];
    const T inv = ch.c1 - ch.c0 > 1 ? (T)(ch.c1 - 1 - ch.c0) / (v1 - v0) : T(0);
    const unsigned long long upto = (2ull << lane) - 1;
    for (int jw = 0; jw < nb; jw += RECS) {
        const int m = min(RECS, nb - jw);
        // the blocks' records and channel ranges, a lane each
        int cl = ch.c0, cnt = 0, nov = 0;
        double bA = 1.0, bB = 0.0;
        if (lane < m) {
            const BlkRec *r = blk + jw + lane;
            const float lo = r->lo, hi = r->hi;
            bA = r->A;
            bB = r->B;
            nov = __float_as_int(lo) & (2 * BLK - 1);
            if (!(lo > hi))          // (-inf with an overshoot count is NaN)
                channels_in<T>(ch.velo, ch.c0, ch.c1, v0, inv, lo, hi, cl, cnt);
        }
        int incl = cnt;                          // pairs up to and with the lane's block
        for (int d = 1; d < RECS; d <<= 1) {
            const int t = __shfl_up(incl, d);
            if (lane >= d) incl += t;
        }
        const int st = incl - cnt, total = lane_of(incl, m - 1);
        const bool some = cnt > 0, overs = __any(nov != 0);
        // the blocks with pairs that are not in LDS yet, and of these the first
        // `ahead` whose nodes are in registers (slots by rank); none where the
        // pairs of BATCH_BLOCKS blocks do not fill a batch, and there are more
        unsigned long long rest = __ballot(some);
        const int seen = __popcll(rest);
        const bool sparse = FEW && seen > BATCH_BLOCKS && total * BATCH_BLOCKS < 64 * seen;
        if (sparse) rest = 0;
        const int rank = __popcll(rest & (upto >> 1));
        int staged = 0, ahead = 0;
        float4 piece[2];
        auto load = [&]() __attribute__((always_inline)) {
            unsigned long long r = rest;
            int j[Nodes<T>::AHEAD];
            ahead = 0;
#pragma unroll
            for (int k = 0; k < Nodes<T>::AHEAD; k++) {
                j[k] = __ffsll(r) - 1;
                ahead += r != 0;
                r &= r - 1;
            }
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int p = lane + 64 * q, k = p / Nodes<T>::PIECES;
                int jk = j[0];
#pragma unroll
                for (int i = 1; i < Nodes<T>::AHEAD; i++) jk = k == i ? j[i] : jk;
                if (k < ahead) piece[q] = stage(jw + jk, p - k * Nodes<T>::PIECES);
            }
        };
        load();
        for (int p0 = 0, b = 0; b < m;) {
            int pend = total;
            if (sparse && p0 < total) {
                pend = min(p0 + 64, total);
                const int p = min(p0 + lane, pend - 1);
                int j = 0;                       // the last block that begins at or before p
                for (int d = RECS / 2; d >= 1; d >>= 1) {
                    const int t = __shfl(st, min(j + d, 63));
                    if (j + d < m && t <= p) j += d;
                }
                const int c = __shfl(cl, j) + p - __shfl(st, j);
                const Pre pre = before(c);
                wave_lds_fence();
                if (p0 + lane < pend) {
                    const Map q = direct(jw + j, c, pre);
                    int i = p0 % RING + lane;
                    S.map[i >= RING ? i - RING : i] = q;
                }
                wave_lds_fence();
            } else if (p0 < total) {
                // the pairs p0 .. pend-1 of at most BATCH_BLOCKS blocks: the one
                // that holds p0 (lane l0) and those that begin after it
                const int l0 = 63 - __clzll(__ballot(some && st <= p0));
                unsigned long long more = __ballot(some && st > p0 && st < p0 + 64);
                pend = min(p0 + 64, total);
                const int p = p0 + lane, r0 = lane_of(rank, l0);
                int r = r0, r1 = r0, j = l0, c = lane_of(cl, l0) - lane_of(st, l0);
                while (more) {
                    const int l = __ffsll(more) - 1, s = lane_of(st, l);
                    more &= more - 1;
                    if (r1 + 1 - r0 == BATCH_BLOCKS) {
                        pend = s;
                        break;
                    }
                    r1++;
                    const bool in = p >= s;
                    r = in ? r1 : r;
                    j = in ? l : j;
                    c = in ? lane_of(cl, l) - s : c;
                }
                const Pre pre = before(min(c + p, ch.c1 - 1));
                wave_lds_fence();
                while (staged <= r1) {
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        const int p = lane + 64 * q, k = p / Nodes<T>::PIECES;
                        if (k < ahead)
                            S.st[(staged + k) % SLOTS][p - k * Nodes<T>::PIECES] = piece[q];
                    }
                    staged += ahead;
                    for (int k = 0; k < ahead; k++) rest &= rest - 1;
                    load();
                }
                wave_lds_fence();
                if (p < pend) {
                    const Map q = integrate(S.st[r % SLOTS], jw + j, c + p, pre);
                    int i = p0 % RING + lane;
                    S.map[i >= RING ? i - RING : i] = q;
                }
                wave_lds_fence();
            }
            // the blocks complete at pair pend
            const int e = __popcll(__ballot(lane < m && incl <= pend));
            for (; b < e; b++) {
                const int n = lane_of(cnt, b), c = lane_of(cl, b) - ch.c0;
                const double A0 = lane_of(bA, b), B0 = lane_of(bB, b);
                const int s = lane_of(st, b) % RING;
                const int nv = overs ? lane_of(nov, b) : 0;
#pragma unroll
                for (int g = 0; g < G; g++) {
                    if (G > 1 && g >= ch.ng) break;
                    double mP = A0, mB = B0;
                    if (c < 64 * g + 64 && c + n > 64 * g) {     // the group has pairs
                        const int i = 64 * g + lane - c;
                        if ((unsigned)i < (unsigned)n) {
                            const Map q = S.map[s + i >= RING ? s + i - RING : s + i];
                            mP = q.P;
                            mB = q.B;
                            if (sizeof(T) == 4) {
                                over |= marked(mP) ? 1u << g : 0u;
                                mP = fabs(mP);
                            }
                        } else if (nv > 0) {
                            passed(g, nv);
                        }
                    } else if (nv > 0) {
                        passed(g, nv);
                    }
                    I[g] = sizeof(T) == 4 ? __builtin_fma(I[g], mP, mB) : I[g] * mP + mB;
                }
            }
            p0 = pend;
        }
        wave_lds_fence();
    }
}

// FP32: block j of a ray of n nodes for one channel on split records (rl_fwd32.h);
// sh, sa, sl: those of node 8 j - 1
__device__ __forceinline__ Map block_split(const SegHot *sh, const SegAux *sa, const NodeLine *sl,
                                           int j, int n, float uch, const double *istar, float sf,
                                           int &maser) {
    Acc32<true> x{0.0, 1.0};
    Car32 c;
    bool ovf = false;
    // the carry of node k0-1 as the end of segment k0-1 (its profile); the
    // ray's first node under segment 1's
    const int m = j > 0 ? 0 : 1, i1 = min(BLK, n - (j << BLK_LOG));
    const SegHot hp = sh[2 * m];
    carry32(pt_of(sa[m].u, sl[m]), uch, hp.ag, hp.ng, c);
    for (int i = m; i < i1; i++)
        segment32(x, sh + i + 1, sa + i + 1, sl + i + 1, uch, istar, sf, c, ovf, maser);
    return Map{mark(x.P, ovf), x.I};
}

// staged as Nodes<float> holds them
__device__ __forceinline__ Map block_split(const float4 *st, int j, int n, float uch,
                                           const double *istar, float sf, int &maser) {
    constexpr int N = Nodes<float>::N;
    return block_split(reinterpret_cast<const SegHot *>(st),
                       reinterpret_cast<const SegAux *>(st + N),
                       reinterpret_cast<const NodeLine *>(st + 2 * N), j, n, uch, istar, sf, maser);
}

// FP64: the same on whole node records, with the reference's own arithmetic; sr:
// that of node 8 j - 2
__device__ __forceinline__ Map block_exact(const NodeRec<double> *sr, int j, int n,
                                           const LineK<double> &L, const double *istar, double sf,
                                           int &ovs, int &maser) {
    Acc<double, true> x{0.0, 1.0};
    Carry<double> c;
    c.init = 1; c.phi0 = 0.0; c.srcl0 = 0.0; c.alpl0 = 0.0; c.S0 = 0.0;
    const int i1 = min(BLK, n - (j << BLK_LOG));
    if (j > 0) carry_of<double>(L, sr[0], sr[1], c);
    for (int i = j > 0 ? 0 : 1; i < i1; i++)
        segment_exact<double>(L, x, sr[i + 1], sr[i + 2], istar, sf, c, ovs, maser);
    return Map{x.P, x.I};
}

}  // namespace rl
