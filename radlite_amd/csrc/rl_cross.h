// The crossings of one ray by one wave: trajectory() (rl_traj.h) with its
// sequential merge replaced by ranks.
//
// The merge's two lists, the cone and the sphere crossings, ascend in s, and so
// do the two groups of extra points once each is sorted.  So every entry's
// place in the merge is its index plus the number of entries of the other
// lists that the merge takes before it, which a lane finds by bisection:
//
//   a cone before a sphere where its s is smaller (equal: the sphere first),
//   an extra point before an entry where its s is smaller (equal: the entry),
//   the first group's extra point before the second's on equal s,
//   no extra point after the last entry.
//
// Entries outside the grid drop out (a prefix sum over the ranks).  The test of
// an entry against the one emitted before it, s - sprev > eps r, is made
// against the neighbour: where all pass, that is the same.  A ray for which any
// of this does not hold (cones that are not contiguous, a list out of order, a
// value that is not a number, two crossings within eps) is left to the
// sequential code: its count is set to CROSS_SEQUENTIAL.  Every value is formed
// by the expression that rl_traj.h forms it by, so the records are the same bits.
#pragma once
#include "rl_traj.h"

namespace rl {

constexpr int CROSS_SEQUENTIAL = -1;
constexpr int CROSS_EXTRA = 40;              // LDS entries of extra points (at most 34)

// LDS bytes for slots of nmax entries: the lists (later the entries' radii),
// the merged s and codes, the extra points
inline __host__ __device__ size_t cross_wave_lds(int nmax) {
    return (size_t)nmax * 20 + CROSS_EXTRA * 12 + 64;
}

// entries of the ascending v[0..n) that are < x (or <= x)
__device__ inline int count_below(const double *v, int n, double x, bool equal) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int m = (lo + hi) >> 1;
        if (equal ? v[m] <= x : v[m] < x) lo = m + 1; else hi = m;
    }
    return lo;
}

// v[0..n) ascending and below top, every value a number (the whole wave)
__device__ inline bool ascending(const double *v, int n, double top) {
    bool ok = true;
    for (int i = threadIdx.x; i < n; i += 64)
        ok = ok && v[i] < top && (i == 0 || v[i - 1] <= v[i]);
    return __all(ok);
}

// One wave: the nodes of a ray into cr (slots of nmax), returns their number,
// CROSS_SEQUENTIAL, or minus a stop code in err_code.
__device__ inline int cross_wave(const GridView &g, const double *__restrict__ tan2, double x0,
                                 double z0, double theta0, double costh0, double sinth0,
                                 bool blend, int nmax, double *lds, CrossRec *__restrict__ cr,
                                 int &err_code) {
    const int lane = threadIdx.x;
    const unsigned long long below = (1ull << lane) - 1;
    const double eps = TELESC_EPS, epsplus = 1.0e1 * TELESC_EPS, pi = PICONST;
    const int nr = g.nr;
    Traj t(g, tan2, x0, z0, theta0, costh0, sinth0, nullptr, nullptr, nullptr, 0);
    t.pitheta0 = 0.5 * pi - theta0;
    t.costh02 = costh0 * costh0;
    t.sinth02 = sinth0 * sinth0;
    const double sinth02 = t.sinth02, costh02 = t.costh02;
    t.iyeq = g.ny / 2;
    t.iyend = g.ny;
    err_code = 0;

    // the cones with two roots (telescope.F:2968-3000)
    int first = 0, last = 0, n = 0;
    for (int i0 = 1; i0 <= t.iyeq; i0 += 64) {
        const int iy = i0 + lane;
        bool two = false;
        if (iy <= t.iyeq) {
            const double tanth2 = tan2[iy];
            const double a = tanth2 * costh02 - sinth02;
            const double b = 2.0 * tanth2 * costh0 * z0;
            const double c = tanth2 * z0 * z0 - x0 * x0;
            two = b * b - 4.0 * a * c > 0.0;
        }
        const unsigned long long m = __ballot(two);
        if (m) {
            if (!first) first = i0 + __ffsll(m) - 1;
            last = i0 + 63 - __clzll(m);
            n += __popcll(m);
        }
    }
    if (n > 0 && last - first + 1 != n) return CROSS_SEQUENTIAL;
    t.isnr = n;
    t.iy0 = first;
    t.isdblnr = 0;
    for (int i0 = 1; i0 <= n; i0 += 64) {
        const int is = i0 + lane;
        t.isdblnr += __popcll(__ballot(is <= n && fabs(0.5 * pi - g.TH(first + is - 1)) >
                                                      fabs(t.pitheta0)));
    }
    t.iup = t.pitheta0 > 0.0 ? 1 : 0;
    t.branchA = z0 * t.pitheta0 > 0.0 ? 1 : 0;
    t.ith_amount = 2 * n;

    // the spheres (telescope.F:3241-3290)
    const double bimpact = sqrt(x0 * x0 + z0 * z0 * (1.0 - costh02));
    int ix = 0;
    for (int i0 = 1; i0 <= nr && !ix; i0 += 64) {
        const unsigned long long m = __ballot(i0 + lane <= nr && g.R(min(i0 + lane, nr)) > bimpact);
        if (m) ix = i0 + __ffsll(m) - 1;
    }
    if (!ix) { err_code = E_INPUT; return 0; }
    t.ir_min = bimpact <= g.rstar ? 0 : ix;
    t.bimpact = bimpact;
    t.half = nr + 1 - t.ir_min;
    t.ir_amount = 2 * t.half;
    {   // discriminant sanity (telescope.F:3293-3300)
        const double r = g.R(nr), b = 2.0 * costh0 * z0, c = x0 * x0 + z0 * z0 - r * r;
        if (b * b - 4.0 * c + eps * b * b < 0.0) { err_code = E_INPUT; return 0; }
    }

    // the lists, and behind them the merge
    const int nt = t.ith_amount, ns = t.ir_amount;
    double *th = lds, *rs = lds + nt, *rad = lds, *ms = lds + nmax, *ex = ms + nmax;
    int *mc = reinterpret_cast<int *>(ex + CROSS_EXTRA), *exc = mc + nmax;
    if (nt + ns + CROSS_EXTRA - 6 > nmax) return CROSS_SEQUENTIAL;
    for (int i = lane; i < nt; i += 64) {
        int itheta;
        t.th_entry(i + 1, th[i], itheta);
    }
    for (int i = lane; i < ns; i += 64) {
        double r;
        int irx;
        t.r_entry(i + 1, rs[i], r, irx);
    }
    __syncthreads();
    if (!ascending(th, nt, 1.0e30) || !ascending(rs, ns, 1.0e30)) return CROSS_SEQUENTIAL;

    // extra points (telescope.F:3417-3606), a lane each: the first group by its
    // place in the reference's stable sort
    int n1 = 0, n2 = 0;
    if (bimpact > g.R(1)) {
        const double s3 = 0.0 - z0 * costh0;
        const int isrt = hunt_bisect([&](int i) { return rs[i - 1]; }, ns, s3);
        auto at = [&](int k) { return k > ns ? 1.0e30 : (k < 1 ? 0.0 : rs[k - 1]); };
        const double rZ = at(isrt - 1), rA = at(isrt), rB = at(isrt + 1), rC = at(isrt + 2);
        n1 = 1 + 4 * RAYADPT;
        // in the reference's order: s3, then the intervals (s3, rB), (rA, s3), (rB, rC), (rZ, rA)
        const int q = lane > 0 ? (lane - 1) / RAYADPT : 0, iad = (lane - 1) % RAYADPT + 1;
        const double s1 = q == 0 ? s3 : (q == 1 ? rA : (q == 2 ? rB : rZ));
        const double s2 = q == 0 ? rB : (q == 1 ? s3 : (q == 2 ? rC : rA));
        const double ds = (s2 - s1) / (1.0 + 1.0 * RAYADPT);
        const double s = lane == 0 ? s3 : iad * ds + s1;
        if (lane < n1) ms[lane] = s;
        __syncthreads();
        int place = 0;
        for (int k = 0; k < n1; k++) {
            const double o = ms[k];
            place += o < s || (o == s && k < lane);
        }
        if (lane < n1) {
            ex[place] = s;
            exc[place] = lane == 0 ? (t.ir_min << 1) | 1 : 1 << 1;
        }
    }
    {
        const double s3 = x0 * x0 * costh0 / (z0 * sinth02);
        const double rr = t.thr(s3);
        if (rr > g.R(1) && rr < g.R(nr)) {
            const int ixh = t.hunt_r(rr);
            if (ixh == 0 || ixh == nr) { err_code = E_HUNT; return 0; }
            auto at = [&](int k) { return k > nt ? 1.0e30 : th[k - 1]; };
            const int isrt = nt > 0 ? hunt_bisect([&](int i) { return at(i); }, nt, s3) : 0;
            bool keep = lane == 0;
            double s = s3;
            if (!(isrt - RAYRNPT + 1 < 1 || isrt + RAYRNPT > nt)) {
                const double tZ = at(isrt - 1), tA = at(isrt), tB = at(isrt + 1), tC = at(isrt + 2);
                const double e1[4] = {s3, tA, tB, tZ}, e2[4] = {tB, s3, tC, tA};
                for (int k = 0; k < 4; k++) {
                    if (e2[k] == e1[k]) { err_code = E_EXEQ; return 0; }
                    if (e2[k] < e1[k]) { err_code = E_EXORD; return 0; }
                }
                // ascending: (tZ, tA), (tA, s3), s3, (s3, tB), (tB, tC)
                const bool mid = lane == 2 * RAYADPT;
                const int l = lane - (lane > 2 * RAYADPT ? 1 : 0);
                const int q = l / RAYADPT, iad = l % RAYADPT + 1;
                const double s1 = q == 0 ? tZ : (q == 1 ? tA : (q == 2 ? s3 : tB));
                const double s2 = q == 0 ? tA : (q == 1 ? s3 : (q == 2 ? tB : tC));
                const double ds = (s2 - s1) / (1.0 + 1.0 * RAYADPT);
                if (!mid) s = iad * ds + s1;
                keep = lane <= 4 * RAYADPT;
                if (keep && !mid) {
                    const int ixx = t.hunt_r(t.thr(s));
                    keep = !(ixx == 0 || ixx == nr);                // :3580
                }
            }
            const unsigned long long m = __ballot(keep);
            n2 = __popcll(m);
            if (keep) {
                ex[n1 + __popcll(m & below)] = s;
                exc[n1 + __popcll(m & below)] = 1 << 1;
            }
        }
    }
    __syncthreads();
    // (1e30: past the last sphere, after every entry)
    if (!ascending(ex, n1, 1.0e31) || !ascending(ex + n1, n2, 1.0e31)) return CROSS_SEQUENTIAL;

    // the merge (telescope.F:3610-3677): every entry to its place
    const int nent = nt + ns;
    const double *ex2 = ex + n1;
    for (int i = lane; i < nt; i += 64) {
        const double s = th[i];
        int is, root, itheta;
        t.th_index(i + 1, is, root, itheta);
        const int k = i + count_below(rs, ns, s, true) + count_below(ex, n1, s, false) +
                      count_below(ex2, n2, s, false);
        ms[k] = s;
        mc[k] = 2 | itheta << 5;
    }
    for (int i = lane; i < ns; i += 64) {
        const double s = rs[i];
        const int is = i + 1 <= t.half ? i + 1 : ns - i;
        const int k = i + count_below(th, nt, s, false) + count_below(ex, n1, s, false) +
                      count_below(ex2, n2, s, false);
        ms[k] = s;
        mc[k] = 1 | (nr - is + 1) << 5;
    }
    int nx;
    {
        bool in = false;
        if (lane < n1 + n2) {
            const double s = ex[lane];
            const int e = lane < n1 ? lane + count_below(ex2, n2, s, false)
                                    : lane - n1 + count_below(ex, n1, s, true);
            const int k = count_below(th, nt, s, true) + count_below(rs, ns, s, true);
            const int code = exc[lane];
            in = k < nent;
            if (in) {
                ms[e + k] = s;
                mc[e + k] = 3 | (code & 1) << 2 | ((code >> 1) - 1) << 5;
            }
        }
        nx = __popcll(__ballot(in));
    }
    __syncthreads();

    // what lies on the grid, in order
    const double rmaxt = g.R(nr) * (1.0 - epsplus), rmaxr = g.R(nr) * (1.0 + epsplus);
    const double rmint = g.R(1) * (1.0 + epsplus), rminr = g.R(1) * (1.0 - epsplus);
    int kept = 0;
    for (int i0 = 0; i0 < nent + nx; i0 += 64) {
        const int i = i0 + lane;
        bool in = false;
        double s = 0.0, r = 0.0;
        int code = 0;
        if (i < nent + nx) {
            s = ms[i];
            code = mc[i];
            const int icr = code & 3, idx = code >> 5;
            if (icr == 1) r = idx == 0 ? g.rstar : g.R(idx);
            else r = (code >> 2) & 1 ? bimpact : t.thr(s);
            in = (icr == 1 ? r <= rmaxr && r >= rminr : r <= rmaxt && r >= rmint) &&
                 s >= -1.0e30 && s <= 1.0e30;
        }
        const unsigned long long m = __ballot(in);
        const int k = kept + __popcll(m & below);
        __syncthreads();
        if (in) {
            ms[k] = s;
            mc[k] = code;
            rad[k] = r;
        }
        kept += __popcll(m);
    }
    __syncthreads();
    bool apart = true;
    for (int i = lane; i < kept; i += 64)
        apart = apart && (ms[i] - (i > 0 ? ms[i - 1] : -1.0e30)) > eps * rad[i];
    if (!__all(apart)) return CROSS_SEQUENTIAL;

    // the records: flags and cell guesses as the sequential sink forms them
    int gr = 0, gt = 0, on_prev = 0;
    bool pending = blend;
    for (int i0 = 0; i0 < kept; i0 += 64) {
        const int i = i0 + lane;
        const bool act = i < kept;
        const int code = act ? mc[i] : 0, icr = code & 3, idx = code >> 5;
        const int v = idx + 1 <= 0xFFFF ? idx + 1 : 0;
        const bool on = icr == 1 && idx == 1;
        const unsigned long long m1 = __ballot(icr == 1), m2 = __ballot(icr == 2),
                                 mo = __ballot(on && i > 0);
        const int p1 = 63 - __clzll(m1 & below), p2 = 63 - __clzll(m2 & below);
        const int v1 = __shfl(v, max(p1, 0)), v2 = __shfl(v, max(p2, 0));
        const int a = p1 >= 0 ? v1 : gr, b = p2 >= 0 ? v2 : gt;
        const int on_b = __shfl_up((int)on, 1);
        int flag = 0;
        if (on && i > 0) {
            if (lane == 0 ? on_prev : on_b) flag |= NF_RESET;
            if (pending && mo && lane == __ffsll(mo) - 1) flag |= NF_BLEND;
        }
        if (act && i < nmax) cr[i] = CrossRec{ms[i], code | flag << 3, a | b << 16};
        if (m1) gr = __shfl(v, 63 - __clzll(m1));
        if (m2) gt = __shfl(v, 63 - __clzll(m2));
        if (mo) pending = false;
        on_prev = __shfl((int)on, 63);
    }
    if (kept > nmax) { err_code = E_CAP; return nmax; }
    return kept;
}

}  // namespace rl
