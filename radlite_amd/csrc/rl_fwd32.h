// Single-precision forward trace on split records: the batched spectrum
// path of the FP32 mode (charintline, telescope.F:3889-4312, with
// clever_integrate_element_linedust line.F:4636-4848,
// integrate_element_linedust line.F:4515-4624, voigt_profile
// line.F:2280-2314 and qdr_src_2 transfer.F:1498-1571).
//
// What a segment needs is split by what it depends on:
//
//   SegHot / SegAux  per trajectory node, independent of the line: built
//                    once per inclination (path length, projected
//                    velocity, the line width's profile scale and
//                    normalisation, the sub-grid length, node flags);
//   NodeLine         per item and node: the node's dust and line
//                    coefficients, scaled (16 bytes).
//
// With e = exp(-z^2) the unnormalised Gaussian profile, the profile of a
// segment with mean width lwav at channel velocity uch (dnu/nu0) is
// phi = (ng/|nu0|) e with z = (uch - u) / (3.33567e-6 lwav), ng =
// 0.56419583546 / (3.33567e-6 lwav): the same quantity voigt_profile forms
// from aa = 3.33567e-6 |nu0| lwav, its 1/|nu0| moved into the line
// coefficients.  The argument is carried pre-multiplied by sqrt(log2 e)
// (ag) so that e is one hardware exp2.
//
// The hot loop reads 32 bytes per segment (SegHot + NodeLine); a segment
// that may be sub-gridded, carries a node flag, or starts the ray takes
// the general path, which also reads SegAux and the start node's record.
#pragma once
#include "rl_device.h"

namespace rl {

struct alignas(16) SegHot {
    float hds;   // ds/2 (0 on a hole chord); sign bit set: the general path
    float ag;    // sqrt(log2 e) / (3.33567e-6 lwav)  [per unit of u]
    float uag;   // u_k * ag
    float ng;    // 0.56419583546 / (3.33567e-6 lwav)
};

// (ds is SegHot's: 2 |hds| is the single-precision ds exactly, the
// halving and doubling being exact in binary)
struct alignas(16) SegAux {
    float u;       // Omega.v/c at node k
    float dls;     // sub-grid line length ds/x (line.F:4733-4738), < 0: never
    float inv_du;  // 1 / (u_k - u_{k-1})
    int flag;      // NF_* bits of node k
};

// one 16-byte load (read field by field, the record took four)
__device__ inline SegAux load_aux(const SegAux *p) {
    const float4 v = *reinterpret_cast<const float4 *>(p);
    SegAux a;
    a.u = v.x;
    a.dls = v.y;
    a.inv_du = v.z;
    a.flag = __float_as_int(v.w);
    return a;
}

// j = |sig| (jdh + jcl ng e), alpha = |sig| (adh + dcl ng e); sig is the
// node's scale (its dust opacity where there is dust, adh = 1); the sign
// bit of sig is set where there is no dust (adh = 0).  jcl and dcl are the
// line coefficients of line.F:4578-4588 over sig |nu0|.
struct alignas(16) NodeLine {
    float sig, jdh, jcl, dcl;
};

constexpr float SQRT_LOG2E = 1.20112240878644977f;

// A block of BLK segments as a channel without the line sees it: outside
// [lo, hi] (dnu/nu0) I <- A I + B; the low bits of lo count its elements that
// overshoot (rl_blocks.h)
constexpr int BLK_LOG = 3, BLK = 1 << BLK_LOG;
struct BlkRec {
    float lo, hi;
    double A, B;
};
__host__ __device__ inline long long blk_of(long long b, int ray) { return (b >> BLK_LOG) + ray; }
__host__ __device__ inline long long blk_count(long long nnodes, int nrays) {
    return (nnodes >> BLK_LOG) + nrays;
}
template <typename T> __device__ inline bool blk_free(const BlkRec &r, T uch) {
    return uch < (T)r.lo || uch > (T)r.hi;
}
__device__ inline int blk_overshoots(const BlkRec &r) {
    return __float_as_int(r.lo) & (2 * BLK - 1);
}

__device__ inline float nl_adh(float sig) { return __float_as_int(sig) < 0 ? 0.0f : 1.0f; }
__device__ inline bool seg_general(float hds) { return __float_as_int(hds) < 0; }
__device__ inline float ex2(float x) { return __builtin_amdgcn_exp2f(x); }

// the values an element needs of its start point, carried from the element
// that ended there: sig*alpha/sig and sig*j/sig (the products the optical
// depth and the bracket add), alpha/sig (its sign picks the source
// functions) and the source function
struct Car32 {
    float sa0 = 0.0f, sj0 = 0.0f, ah0 = 0.0f, S0 = 0.0f;
};

// a point of the general path: scaled values (adh explicit)
struct Pt32 {
    float u, sig, jdh, adh, jcl, dcl;
};

__device__ inline Pt32 pt_of(float u, const NodeLine &q) {
    return Pt32{u, fabsf(q.sig), q.jdh, nl_adh(q.sig), q.jcl, q.dcl};
}

// the carry of a start point p under a segment's profile (ag, ng)
__device__ inline void carry32(const Pt32 &p, float uch, float ag, float ng, Car32 &c) {
    const float z = (uch - p.u) * ag;
    const float e = ex2(-(z * z));
    const float ah = fmaf(p.dcl * ng, e, p.adh);
    const float jh = fmaf(p.jcl * ng, e, p.jdh);
    c.sa0 = p.sig * ah;
    c.sj0 = p.sig * jh;
    c.ah0 = ah;
    c.S0 = ah > 0.0f ? FOps<float>::sdiv(jh, ah) : 0.0f;
}

// One element from the carried start point to an end point with scaled
// values (sg, adh, jdh) and profile-weighted line coefficients jcn = jcl
// ng, dcn = dcl ng at e: the map I <- I + (q - I e0) with e0 = 1 - exp(-dtau),
// q = min(Q, J_max) (qdr_src_2, transfer.F:1498-1571); ovf is set on an
// overshoot (Q > 2 J_max).
__device__ __forceinline__ void elem_map32(float hds, float e, float jcn, float dcn, float sg, float adh,
                                  float jdh, Car32 &c, bool &ovf, float &e0, float &q) {
    const float ah1 = fmaf(dcn, e, adh);
    const float jh1 = fmaf(jcn, e, jdh);
    const float sa1 = sg * ah1, sj1 = sg * jh1;
    const float dtau = (c.sa0 + sa1) * hds;
    const float theomax = (c.sj0 + sj1) * hds;
    float wa, wb, xp, ra;
    qdr_weights_f<float>(dtau, wa, wb, xp, ra, e0);
    // source functions with the fall-backs of transfer.F:1528-1541
    const float q1 = ah1 > 0.0f ? FOps<float>::sdiv(jh1, ah1) : 0.0f;
    const float q0 = c.S0;
    const float s1 = c.ah0 > 0.0f ? q0 : (ah1 > 0.0f ? q1 : 0.0f);
    const float s2 = ah1 > 0.0f ? q1 : (c.ah0 > 0.0f ? q0 : 0.0f);
    q = dtau > 1e-9f ? fmaf(wa, s1, wb * s2) : theomax;   // 1e-9 is REAL*4
    ovf = ovf || (q > 2.0f * theomax);
    q = fminf(q, theomax);
    c.sa0 = sa1;
    c.sj0 = sj1;
    c.ah0 = ah1;
    c.S0 = q1;
}

// What a lane carries along its ray: the intensity, or (AFF) the map I -> P I
// + I' of the part of the ray it has passed.  In double precision (the
// elements' values in single): the elements a channel does not see the line
// in are the same maps for every such channel, taken one by one or composed,
// so that channels on and off the line differ by the line alone and not by
// the rounding of the dust's sum, of which a weak line is a small part.  e0 =
// 1 - exp(-dtau) rather than exp(-dtau): thin elements keep their digits.
template <bool AFF> struct Acc32 {
    double I, P;
    __device__ void step(float e0, float q) {
        I = I + __builtin_fma(-I, (double)e0, (double)q);
        if (AFF) P = __builtin_fma(-P, (double)e0, P);
    }
    __device__ void map(double A, double B) {
        I = __builtin_fma(I, A, B);
        if (AFF) P = P * A;
    }
};

// an element ending at point p of the general path
template <bool AFF>
__device__ __forceinline__ void elem_pt32(Acc32<AFF> &x, float hds, const Pt32 &p, float uch, float ag,
                                 float ng, Car32 &c, bool &ovf, float &e_out) {
    const float z = (uch - p.u) * ag;
    const float e = ex2(-(z * z));
    e_out = e;
    float e0, q;
    elem_map32(hds, e, p.jcl * ng, p.dcl * ng, p.sig, p.adh, p.jdh, c, ovf, e0, q);
    x.step(e0, q);
}

// The general path of segment k (nodes k-1 -> k) up to its last element: node
// flags (hole chord, central-beam star blend, star intensity: the element then
// starts afresh from the start point under its own profile) and the sub-grid of
// clever_integrate_element_linedust (line.F:4706-4800): points s_i = sleft +
// (i-1) lg, i = 1..31, used where 0 < s_i < ds, the quantities interpolated
// linearly in s, the width held at the segment's mean.  Returns ds; sa: the
// last point's s.
template <bool AFF>
__device__ __forceinline__ float seg_general32(Acc32<AFF> &x, const SegHot &h, float u0,
                                      const SegAux &a1, const NodeLine &q0, const NodeLine &q1,
                                      float uch, const double *istar, float sf, Car32 &c,
                                      bool &ovf, float &sa) {
    float ds = 2.0f * fabsf(h.hds);                     // (float)ds, hds = (float)(ds/2)
    const int fl = a1.flag;
    if (fl & NF_RESET) ds = 0.0f;
    if (fl & NF_BLEND) x.map((double)(1.0f - sf), (double)(sf * (float)*istar));
    if (fl & NF_STAR) x.map(0.0, (double)(float)*istar);
    if (fl) carry32(pt_of(u0, q0), uch, h.ag, h.ng, c);
    sa = 0.0f;
    if (a1.dls >= 0.0f) {                                 // 6x > 1 (line.F:4715)
        const float s_c = ds * (uch - u0) * a1.inv_du;
        const float sright = s_c + 3.0f * a1.dls, sleft = s_c - 3.0f * a1.dls;
        if (sright > 0.0f && sleft < ds) {
            const Pt32 p0 = pt_of(u0, q0), p1 = pt_of(a1.u, q1);
            const float lg = (sright - sleft) * (1.0f / 30.0f);
            const float f0 = FOps<float>::fdiv(-sleft, lg), f1 = FOps<float>::fdiv(ds - sleft, lg);
            int i = f0 > 0.0f ? max(1, (int)fminf(f0, 40.0f)) : 1;
            int ihi = f1 < 40.0f ? min(31, (int)fmaxf(f1, -2.0f) + 2) : 31;
            // the bounds are at most two points too wide: cut here, so that a
            // wave's loop is as long as its longest lane's points
            auto at = [&](int i) { return sleft + (float)(i - 1) * lg; };
            i += !(at(i) > 0.0f);
            i += !(at(i) > 0.0f);
            ihi -= !(at(ihi) < ds);
            ihi -= !(at(ihi) < ds);
            // the nodes' scales relative to the larger; where both are below
            // the single-precision range (no optical depth to speak of) the
            // points are weighted equally
            const float sm = fmaxf(p0.sig, p1.sig);
            const float rel0 = sm > 0.0f ? p0.sig / sm : 1.0f;
            const float rel1 = sm > 0.0f ? p1.sig / sm : 1.0f;
            const float inv_ds = FOps<float>::fdiv(1.0f, ds);
            for (; i <= ihi; i++) {
                const float s = at(i);
                if (s > 0.0f && s < ds) {
                    // linear interpolation of the unscaled quantities
                    // (line.F:4775-4790) through relative weights
                    const float e = s * inv_ds, ep = 1.0f - e;
                    float w0 = ep * rel0, w1 = e * rel1;
                    const float W = w0 + w1, iw = FOps<float>::fdiv(1.0f, W);
                    w0 *= iw;
                    w1 *= iw;
                    const Pt32 b{ep * p0.u + e * p1.u, sm * W, w0 * p0.jdh + w1 * p1.jdh,
                                 w0 * p0.adh + w1 * p1.adh, w0 * p0.jcl + w1 * p1.jcl,
                                 w0 * p0.dcl + w1 * p1.dcl};
                    float eb;
                    elem_pt32(x, 0.5f * (s - sa), b, uch, h.ag, h.ng, c, ovf, eb);
                    sa = s;
                }
            }
        }
    }
    return ds;
}

// segment k from the carry (hot, aux, line: at node k; the general path reads
// the node before it as well).  The last (or only) element of every segment is
// one piece of code: in a wave whose lanes hold both kinds of segment it runs
// once.
template <bool AFF>
__device__ __forceinline__ void segment32(Acc32<AFF> &x, const SegHot *hot, const SegAux *aux,
                                          const NodeLine *line, float uch, const double *istar, float sf,
                                          Car32 &c, bool &ovf, int &maser) {
    const SegHot h = *hot;
    const NodeLine q = *line;
    float hds = h.hds, ds = 2.0f * h.hds, z = fmaf(uch, h.ag, -h.uag);
    if (seg_general(h.hds)) {
        const SegAux a = load_aux(aux);
        float sa;
        ds = seg_general32(x, h, aux[-1].u, a, line[-1], q, uch, istar, sf, c, ovf, sa);
        hds = 0.5f * (ds - sa);
        z = (uch - a.u) * h.ag;
    }
    const float e = ex2(-(z * z));
    const float dcn = q.dcl * h.ng, sig = fabsf(q.sig);
    float e0, b;
    elem_map32(hds, e, q.jcl * h.ng, dcn, sig, nl_adh(q.sig), q.jdh, c, ovf, e0, b);
    x.step(e0, b);
    // maser flag (telescope.F:4295-4297): line alpha * ds < -0.01 at the end;
    // the line coefficient is negative only where the populations are inverted (or
    // the width negative)
    if (dcn < 0.0f && sig * (dcn * e) * ds < -0.01f) maser = 1;
}

// charintline (telescope.F:3889-4312) on split records, one lane: one channel
// (uch = dnu/nu0) of one ray of n nodes from the outer boundary intensity I0,
// block by block: a seen block after a line-free one from its own carry, as
// rl_walk.h takes every block, one after a seen one from that one's.
__device__ inline double trace_split(const SegHot *__restrict__ hot, const SegAux *__restrict__ aux,
                                     const NodeLine *__restrict__ line,
                                     const BlkRec *__restrict__ blk, int n, float uch, double I0,
                                     const double *istar, float sf, int &ovs, int &maser) {
    Acc32<false> x{I0, 1.0};
    if (n < 2) return I0;
    Car32 c;
    bool ovf = false, fresh = true;
    for (int k0 = 0; k0 < n; k0 += BLK) {
        const BlkRec r = blk[k0 >> BLK_LOG];
        if (blk_free(r, uch)) {
            x.map(r.A, r.B);
            ovf = ovf || blk_overshoots(r) != 0;
            fresh = true;
            continue;
        }
        for (int k = max(k0, 1); k < min(n, k0 + BLK); k++) {
            if (fresh) {
                // the carry of node k-1 as the end of segment k-1 (its profile);
                // the ray's first node under segment 1's
                const SegHot hp = hot[k > 1 ? k - 1 : 1];
                carry32(pt_of(aux[k - 1].u, line[k - 1]), uch, hp.ag, hp.ng, c);
                fresh = false;
            }
            segment32(x, hot + k, aux + k, line + k, uch, istar, sf, c, ovf, maser);
        }
    }
    ovs += ovf ? 1 : 0;
    return x.I;
}

}  // namespace rl
