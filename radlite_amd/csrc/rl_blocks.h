// Line-free blocks of a trajectory.
//
// An element of the formal solution is an affine map of the intensity,
// I -> xp I + q (qdr_src_2, transfer.F:1498-1571).  Where the line's share
// of emissivity and opacity is below half a unit in the last place of the
// dust's at both ends, the element is the dust element bit for bit, the
// same for every such channel.  So the segments of a ray are taken in
// blocks of BLK, and the node pass forms, per item and block, the
// composition of its dust elements (A, B) and the range of channel
// velocities [lo, hi] outside which the line vanishes in that sense on
// all of the block: a channel outside it takes the block as one multiply-add.
//
// Block j of a ray holds the segments k (nodes k-1 -> k) with k / BLK == j
// (k = 0, which ends no segment, is the identity).  Ray r's records start
// at blk_of(first node, r), which needs no offsets of its own: a ray of n
// nodes has ceil(n / BLK) <= floor((b + n) / BLK) - floor(b / BLK) + 1 of them.
#pragma once
#include "rl_device.h"
#include "rl_fwd32.h"

namespace rl {

// the profile argument squared (in units of log 2: e = 2^-z2) from which the
// line cannot be seen: |line| <= M e |dust| with e <= 2^-(bits) / M
//   T = bits + log2 M,  bits = mantissa + 2 (one for half an ulp, one margin)
// at least 16 (z > 4 in units of the width over sqrt(log2 e), 3.3 widths: the
// sub-grid, 3 widths about the resonance, is then out of reach) and at most
// the exponent at which e itself is 0
template <typename T> struct BlkLim;
template <> struct BlkLim<float> { static constexpr float bits = 26.0f, zero = 150.0f; };
template <> struct BlkLim<double> { static constexpr float bits = 56.0f, zero = 1080.0f; };

// sqrt(T) for the largest line-to-dust ratio M of a segment (inverted: the
// line opacity is negative somewhere: only a line that is exactly 0 may be
// left out, so that the maser test sees every other)
template <typename T>
__device__ inline float blk_zcut(float M, bool inverted) {
    float t = BlkLim<T>::bits + __log2f(M);         // M = 0: -inf
    t = fminf(fmaxf(t, 16.0f), BlkLim<T>::zero);    // NaN: 16, but then lo and hi are NaN too
    if (inverted || !(M >= 0.0f)) t = BlkLim<T>::zero;
    return sqrtf(t) + 0.01f;                        // the bounds' own rounding
}

// whether a segment's velocities and the widths of the two segments at its start are
// such that bounds can be given at all (a negative width has them the wrong way round)
template <typename T> __device__ inline bool blk_sane(T u0, T u1, float w0, float w1) {
    return fabs(u0) + fabs(u1) < (T)INFINITY && w0 > 0.0f && w1 > 0.0f;
}

// |x| / |d| as a ratio of line to dust: 0 without line, inf without dust
template <typename T>
__device__ inline float blk_ratio(T x, T d) {
    return x == T(0) ? 0.0f : (float)(fabs(x) / fabs(d));
}

// One wave, lane <-> node k = 64 c + lane: the segments' maps (A, B) and
// bounds composed over each block, written by the block's first lane.  ovf:
// the dust element overshoots; the count of those goes into the low bits of
// lo (1e-6 of it, within the margin of blk_zcut).
__device__ inline void blk_store(int lane, int k, int n, double A, double B, float lo, float hi,
                                 bool ovf, BlkRec *__restrict__ blk) {
    if (!(lo == lo) || !(hi == hi)) { lo = -INFINITY; hi = INFINITY; }
    for (int d = 1; d < BLK; d *= 2) {
        // the later half of the block after the earlier: (A2, B2) o (A, B)
        const double A2 = __shfl_down(A, d), B2 = __shfl_down(B, d);
        B = A2 * B + B2;
        A = A2 * A;
        lo = fminf(lo, __shfl_down(lo, d));
        hi = fmaxf(hi, __shfl_down(hi, d));
    }
    const unsigned long long m = __ballot(ovf);
    if ((lane & (BLK - 1)) == 0 && k < n) {
        if (!(A >= 0.0) || !(B == B)) { lo = -INFINITY; hi = INFINITY; }
        const int nov = __popc((unsigned)(m >> lane) & ((1u << BLK) - 1));
        BlkRec r;
        r.lo = __int_as_float((__float_as_int(lo) & ~(2 * BLK - 1)) | nov);
        r.hi = hi;
        r.A = A;
        r.B = B;
        blk[k >> BLK_LOG] = r;
    }
}

}  // namespace rl
