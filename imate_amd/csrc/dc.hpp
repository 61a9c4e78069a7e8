// Divide-and-conquer eigensolve of a symmetric tridiagonal, with only the
// first row of the eigenvector matrix, by the threads of one workgroup.
//
// Cuppen's method (Numer. Math. 36, 1981) with the rank-one updates of
// Bunch, Nielsen & Sorensen (Numer. Math. 31, 1978) and the modified update
// vector of Gu & Eisenstat (SIAM J. Matrix Anal. Appl. 15, 1994): the
// tridiagonal is torn into 2 x 2 blocks, T = diag(T1, T2) + |rho| u u^T with
// u = e_last + sign(rho) e_first at every coupling, and neighbouring blocks
// are merged level by level. A merge needs only the last row of the
// eigenvectors of T1 and the first row of those of T2, so the first and last
// row of every block is all that is carried: O(K^2) work in all, and every
// root of a merge is an independent thread.
//
// The code is written for a group g of threads (g.tid, g.nt, g.sync()), so
// that a group of one thread runs it on the host. A row (a root, a pole) is
// worked on by P neighbouring threads, which take every P-th term of its
// sums and products and combine them with g.sum / g.prod (the same value in
// all P of them). What bounds the solver is the latency of those loops: 20
// rows took 112 us with one thread per root in rolled loops, 41 us with 8
// and four terms in flight.
#pragma once

#include <cfloat>
#include <cmath>

#if defined(__HIP__)
#include <hip/hip_runtime.h>
#define SLQ_DC __device__ __forceinline__
#else
#define SLQ_DC inline
#endif

namespace slq {

// Doubles and ints of work per row of the matrix.
constexpr int kDcDoubles = 11;
constexpr int kDcInts = 1;

// Couplings below this fraction of the norm count as zero: an eigenvalue moves
// by no more than the coupling, and the squares of what is left (of a rotation's
// coupling, of the reciprocal gaps of a merge) stay in range. Kept, one of
// 1e-163 between equal diagonal entries gave a rotation of e / 0.
constexpr double kDcLeast = 0x1p-400;

struct DcWork {
    double *d, *e, *f;                 // diagonal -> eigenvalues, couplings, first row
    double *l, *ds, *zs, *fs, *ls;     // last row; a pair's rows in order
    double *mu, *org;                  // roots org + mu
    double *zh;
    int *cnt;
};

SLQ_DC DcWork dc_carve(double* base, int K)
{
    DcWork w;
    w.d = base;
    w.e = base + K;
    w.f = base + 2 * K;
    w.l = base + 3 * K;
    w.ds = base + 4 * K;
    w.zs = base + 5 * K;
    w.fs = base + 6 * K;
    w.ls = base + 7 * K;
    w.mu = base + 8 * K;
    w.org = base + 9 * K;
    w.zh = base + 10 * K;
    w.cnt = (int*) (base + kDcDoubles * K);
    return w;
}

// 1 / x to about one ulp.
SLQ_DC double dc_rcp(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    r = fma(fma(-x, r, 1.0), r, r);
    return r;
#else
    return 1.0 / x;
#endif
}

// sqrt(x), x >= 0, and 1 / sqrt(x), x > 0, to about one ulp.
SLQ_DC double dc_rsqrt(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double r = __builtin_amdgcn_rsq(x);
    r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
    r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
    return r;
#else
    return 1.0 / sqrt(x);
#endif
}

SLQ_DC double dc_sqrt(double x) { return x > 0.0 ? x * dc_rsqrt(x) : 0.0; }

// Couplings and gaps up to this do not count: two ulps of the pair's norm.
SLQ_DC double dc_tolerance(double low, double high, double rho)
{
    return 2.0 * DBL_EPSILON * fmax(fmax(fabs(low), fabs(high)), rho);
}

// term(k, in) for k = sub, sub + P, ..., four at a time so that their
// latencies overlap; past the end with in = false and the last index (whose
// term must then be neutral).
template <int P, typename F>
SLQ_DC void dc_terms(int sub, int n, const F& term)
{
    for (int k0 = sub; k0 < n; k0 += 4 * P)
    {
#pragma unroll
        for (int u = 0; u < 4; ++u)
        {
            const int k = k0 + u * P;
            term(k < n ? k : n - 1, k < n);
        }
    }
}

// Root j of 1 + rho sum_k z_k^2 / (d_k - x) = 0 over n ascending poles d,
// as x = org + mu with org the closer of the two poles around it; by P
// threads (sub = 0 .. P - 1). The iteration interpolates the sums over the
// poles on either side by one pole each (Li's "middle way", LAPACK Working
// Note 89) inside a bracket that every evaluation shrinks; a step out of the
// bracket is replaced by its midpoint.
template <int P, typename G>
SLQ_DC void dc_root(const G& g, const double* __restrict__ d, const double* __restrict__ z,
                    int n, int j, double rho, int sub, double& org, double& mu)
{
    const bool last = j == n - 1;
    const double dj = d[j];
    double lo, hi, x, base = dj;
    if (last)
    {
        double zz = 0.0;
        dc_terms<P>(sub, n, [&](int k, bool in) { zz += in ? z[k] * z[k] : 0.0; });
        lo = 0.0;
        hi = rho * g.template sum<P>(zz);
        x = 0.5 * hi;
    }
    else
    {
        const double dn = d[j + 1], gap = dn - dj, mid = 0.5 * gap;
        double rest = 0.0;
        dc_terms<P>(sub, n, [&](int k, bool in) {
            const double zk = !in || k == j || k == j + 1 ? 0.0 : z[k];
            rest += zk * zk * dc_rcp((d[k] - dj) - mid);
        });
        rest = g.template sum<P>(rest);
        const double a1 = rho * z[j] * z[j], b1 = rho * z[j + 1] * z[j + 1];
        const double c = 1.0 + rho * rest;
        if (c + (b1 - a1) * dc_rcp(mid) >= 0.0)
        {
            lo = 0.0;
            hi = mid;
            const double a = c * gap + a1 + b1, b = a1 * gap;
            const double s = dc_sqrt(fabs(a * a - 4.0 * b * c));
            x = a >= 0.0 ? 2.0 * b * dc_rcp(a + s) : (a - s) * dc_rcp(2.0 * c);
        }
        else
        {
            base = dn;
            lo = -mid;
            hi = 0.0;
            const double a = -c * gap + a1 + b1, b = b1 * gap;
            const double s = dc_sqrt(fabs(a * a + 4.0 * b * c));
            x = a >= 0.0 ? -2.0 * b * dc_rcp(a + s) : (a - s) * dc_rcp(2.0 * c);
        }
        if (!(x > lo && x < hi)) x = 0.5 * (lo + hi);
    }
    for (int it = 0; it < 60; ++it)
    {
        double psi = 0.0, dpsi = 0.0, phi = 0.0, dphi = 0.0;
        dc_terms<P>(sub, n, [&](int k, bool in) {
            const double zk = in ? z[k] : 0.0, q = zk * dc_rcp((d[k] - base) - x);
            const double t = zk * q, u = q * q;
            const bool left = k <= j;
            psi += left ? t : 0.0;
            dpsi += left ? u : 0.0;
            phi += left ? 0.0 : t;
            dphi += left ? 0.0 : u;
        });
        psi = g.template sum<P>(psi);
        dpsi = g.template sum<P>(dpsi);
        phi = g.template sum<P>(phi);
        dphi = g.template sum<P>(dphi);
        const double v = 1.0 + rho * (psi + phi);
        // psi <= 0 <= phi: the sum of the moduli bounds the rounding of v
        if (fabs(v) <= DBL_EPSILON * (1.0 + rho * (phi - psi))) break;
        if (v < 0.0) lo = x;
        else hi = x;
        dpsi *= rho;
        dphi *= rho;
        const double D0 = (dj - base) - x;
        double eta;
        if (last)
            eta = D0 * v * dc_rcp(v - D0 * dpsi);
        else
        {
            const double D1 = (d[j + 1] - base) - x;
            const double c = v - D0 * dpsi - D1 * dphi;
            const double a = (D0 + D1) * v - D0 * D1 * (dpsi + dphi);
            const double b = D0 * D1 * v;
            const double s = dc_sqrt(fabs(a * a - 4.0 * b * c));
            // the root of c eta^2 - a eta + b of smaller modulus
            const bool neg = a <= 0.0 && c != 0.0;
            eta = (neg ? a - s : 2.0 * b) * dc_rcp(neg ? 2.0 * c : c == 0.0 ? 2.0 * a : a + s);
            if (!(v * eta < 0.0)) eta = -v * dc_rcp(dpsi + dphi);
        }
        double y = x + eta;
        if (!(y > lo && y < hi)) y = 0.5 * (lo + hi);
        if (y == x) break;
        x = y;
    }
    org = base;
    mu = x;
}

// Eigenvalues of the tridiagonal (w.d, w.e[0 .. K - 2]) into w.d and the
// first row of its eigenvectors into w.f, unordered. Every thread of the
// group calls it after the inputs are visible to the group; the outputs are
// visible to the group on return. Non-finite inputs give false (and no
// output), the same for every thread.
template <int P, typename G>
SLQ_DC bool dc_first_row(const G& g, const DcWork& w, int K)
{
    // scale by a power of two (exact) so that squares neither overflow nor
    // underflow; a sum of the moduli is not finite if an entry is not. The
    // terms are scaled down so that finite entries (at most 2 K) do not
    // overflow it, and up again where that would lose them
    auto moduli = [&](double by) {
        double sum = 0.0;
#pragma unroll 4
        for (int i = 0; i < K; ++i)
            sum += by * fabs(w.d[i]) + (i + 1 < K ? by * fabs(w.e[i]) : 0.0);
        return sum;
    };
    double sum = moduli(0x1p-12);
    if (!(sum <= DBL_MAX)) return false;
    int ex = 12;
    if (sum < 0x1p-900)
    {
        sum = moduli(0x1p100);
        ex = -100;
    }
    ex = sum > 0.0 ? ex + ilogb(sum) : 0;
    const int sub = g.tid % P, row0 = g.tid / P, rows = g.nt / P;
    g.sync();
    for (int i = g.tid; i < K; i += g.nt)
    {
        w.ds[i] = ldexp(w.d[i], -ex);
        if (i + 1 < K)
        {
            const double ei = ldexp(w.e[i], -ex);
            w.e[i] = fabs(ei) < kDcLeast ? 0.0 : ei;
        }
    }
    g.sync();
    // 2 x 2 blocks by one Jacobi rotation, torn from their neighbours
    for (int i = 2 * g.tid; i < K; i += 2 * g.nt)
    {
        const double a = w.ds[i] - (i > 0 ? fabs(w.e[i - 1]) : 0.0);
        if (i + 1 == K)
        {
            w.d[i] = a;
            w.f[i] = 1.0;
            w.l[i] = 1.0;
            continue;
        }
        const double b = w.ds[i + 1] - (i + 2 < K ? fabs(w.e[i + 1]) : 0.0), e = w.e[i];
        // t = tan of the angle that annihilates e, |t| <= 1
        const double h = 0.5 * (b - a), r = sqrt(h * h + e * e);
        const double t = e == 0.0 ? 0.0 : e / (h + copysign(r, h));
        const double c = 1.0 / sqrt(1.0 + t * t), sn = t * c;
        w.d[i] = a - t * e;
        w.d[i + 1] = b + t * e;
        w.f[i] = c;
        w.l[i] = -sn;
        w.f[i + 1] = sn;
        w.l[i + 1] = c;
    }
    g.sync();
    for (int s = 2; s < K; s *= 2)
    {
        // rows sorted by their block pair's eigenvalues, with the update
        // vector z and the first and last rows of the pair
        for (int i = row0; i < K; i += rows)
        {
            const int B = i & ~(2 * s - 1), mid = B + s;
            if (mid >= K) continue;
            const int end = B + 2 * s < K ? B + 2 * s : K;
            const double di = w.d[i];
            int pos = 0;
            dc_terms<P>(sub, end - B, [&](int k, bool in) {
                const double dj = w.d[B + k];
                pos += in && (dj < di || (dj == di && B + k < i)) ? 1 : 0;
            });
            pos = B + g.template sum<P>(pos);
            if (sub != 0) continue;
            if (i == B) w.cnt[B] = end - B;
            const bool first = i < mid;
            const double sg = w.e[mid - 1] < 0.0 ? -M_SQRT1_2 : M_SQRT1_2;
            w.ds[pos] = di;
            w.zs[pos] = first ? M_SQRT1_2 * w.l[i] : sg * w.f[i];
            w.fs[pos] = first ? w.f[i] : 0.0;
            w.ls[pos] = first ? 0.0 : w.l[i];
        }
        g.sync();
        // deflation: entries of negligible z, and of two close eigenvalues
        // the one that a rotation can free of z, are final. Most pairs have
        // none, which a test of all neighbours at once finds
        for (int i = g.tid; i < K; i += g.nt)
        {
            const int B = i & ~(2 * s - 1);
            if (B + s >= K) continue;
            const int end = B + 2 * s < K ? B + 2 * s : K, ni = i + 1 < end ? i + 1 : i;
            const double rho = 2.0 * fabs(w.e[B + s - 1]);
            const double tol = dc_tolerance(w.ds[B], w.ds[end - 1], rho);
            const double z = w.zs[i], zn = w.zs[ni], dd = w.ds[ni] - w.ds[i];
            if (rho * fabs(z) <= tol ||
                (ni > i && fabs(dd * z * zn) <= tol * (z * z + zn * zn)))
                w.cnt[B] = -1;
        }
        g.sync();
        // the others one thread per pair, in order; final rows go to the end
        // of the pair's rows
        for (int B = 2 * s * g.tid; B + s < K; B += 2 * s * g.nt)
        {
            if (w.cnt[B] >= 0) continue;
            const int end = B + 2 * s < K ? B + 2 * s : K;
            const double rho = 2.0 * fabs(w.e[B + s - 1]);
            const double tol = dc_tolerance(w.ds[B], w.ds[end - 1], rho);
            int n = 0, out = end - 1;
            bool have = false;
            double pd = 0.0, pz = 0.0, pf = 0.0, pl = 0.0;
            double nd = w.ds[B], nz = w.zs[B], nf = w.fs[B], nl = w.ls[B];
            for (int i = B; i < end; ++i)
            {
                double cd = nd, cz = nz, cf = nf, cl = nl;
                const int ni = i + 1 < end ? i + 1 : i;   // loads ahead of the stores
                nd = w.ds[ni];
                nz = w.zs[ni];
                nf = w.fs[ni];
                nl = w.ls[ni];
                if (rho * fabs(cz) <= tol)
                {
                    w.d[out] = cd;
                    w.f[out] = cf;
                    w.l[out] = cl;
                    --out;
                    continue;
                }
                if (have)
                {
                    const double r2 = pz * pz + cz * cz;
                    if (fabs((cd - pd) * pz * cz) <= tol * r2)
                    {
                        const double tau = sqrt(r2), c = cz / tau, t = -pz / tau;
                        w.d[out] = pd * (c * c) + cd * (t * t);
                        w.f[out] = c * pf + t * cf;
                        w.l[out] = c * pl + t * cl;
                        --out;
                        cd = pd * (t * t) + cd * (c * c);
                        cf = c * cf - t * pf;
                        cl = c * cl - t * pl;
                        cz = tau;
                    }
                    else
                    {
                        w.ds[B + n] = pd;
                        w.zs[B + n] = pz;
                        w.fs[B + n] = pf;
                        w.ls[B + n] = pl;
                        ++n;
                    }
                }
                have = true;
                pd = cd;
                pz = cz;
                pf = cf;
                pl = cl;
            }
            if (have)
            {
                w.ds[B + n] = pd;
                w.zs[B + n] = pz;
                w.fs[B + n] = pf;
                w.ls[B + n] = pl;
                ++n;
            }
            w.cnt[B] = n;
        }
        g.sync();
        for (int i = row0; i < K; i += rows)
        {
            const int B = i & ~(2 * s - 1), j = i - B;
            if (B + s >= K || j >= w.cnt[B]) continue;
            double org, mu;
            dc_root<P>(g, w.ds + B, w.zs + B, w.cnt[B], j, 2.0 * fabs(w.e[B + s - 1]), sub, org,
                    mu);
            w.org[i] = org;
            w.mu[i] = mu;
        }
        g.sync();
        // the update vector whose exact eigenvalues are the computed roots
        for (int i = row0; i < K; i += rows)
        {
            const int B = i & ~(2 * s - 1), k = i - B;
            if (B + s >= K || k >= w.cnt[B]) continue;
            const int n = w.cnt[B];
            const double dk = w.ds[i];
            double p = 1.0;
            dc_terms<P>(sub, n, [&](int j, bool in) {
                const double num = (w.org[B + j] - dk) + w.mu[B + j];
                const double den = w.ds[B + (j < k ? j : j + 1 < n ? j + 1 : j)] - dk;
                const double f = j < n - 1 ? num * dc_rcp(den) : num;
                p *= in ? f : 1.0;
            });
            p = g.template prod<P>(p);
            w.zh[i] = copysign(dc_sqrt(fabs(p)), w.zs[i]);
        }
        g.sync();
        for (int i = row0; i < K; i += rows)
        {
            const int B = i & ~(2 * s - 1);
            if (B + s >= K || i - B >= w.cnt[B]) continue;
            const int n = w.cnt[B];
            const double base = w.org[i], mu = w.mu[i];
            double nn = 0.0, sf = 0.0, sl = 0.0;
            dc_terms<P>(sub, n, [&](int j, bool in) {
                const int k = B + j;
                const double v = in ? w.zh[k] * dc_rcp((w.ds[k] - base) - mu) : 0.0;
                nn = fma(v, v, nn);
                sf = fma(w.fs[k], v, sf);
                sl = fma(w.ls[k], v, sl);
            });
            nn = g.template sum<P>(nn);
            sf = g.template sum<P>(sf);
            sl = g.template sum<P>(sl);
            const double r = dc_rsqrt(nn);
            w.d[i] = base + mu;
            w.f[i] = sf * r;
            w.l[i] = sl * r;
        }
        g.sync();
    }
    for (int i = g.tid; i < K; i += g.nt) w.d[i] = ldexp(w.d[i], ex);
    g.sync();
    return true;
}

}  // namespace slq
