// Host build of the tridiagonal eigensolvers and quadrature (one thread), for
// test_tridiagonal_cpu.py.
#include <cstdint>
#include <vector>

#include "dc.hpp"
#include "ql.hpp"

namespace {

struct OneThread {
    int tid = 0, nt = 1;
    void sync() const {}
    template <int P, typename T>
    T sum(T x) const
    {
        return x;
    }
    template <int P>
    double prod(double x) const
    {
        return x;
    }
};

}  // namespace

// Divide-and-conquer: eigenvalues and first row of the eigenvectors; 1 if
// solved.
extern "C" int divide_and_conquer(const double* d, const double* e, int K, double* theta,
                                  double* first)
{
    std::vector<double> work((size_t) K * (slq::kDcDoubles + 1) + 1);
    const slq::DcWork w = slq::dc_carve(work.data(), K);
    for (int i = 0; i < K; ++i)
    {
        w.d[i] = d[i];
        w.e[i] = i + 1 < K ? e[i] : 0.0;
    }
    if (!slq::dc_first_row<1>(OneThread{}, w, K)) return 0;
    for (int i = 0; i < K; ++i)
    {
        theta[i] = w.d[i];
        first[i] = w.f[i];
    }
    return 1;
}

// The host path's quadrature of one tridiagonal (gram: bidiagonal).
extern "C" double quadrature(const double* alpha, const double* beta, int m, int gram, int func,
                             double coefficient)
{
    slq::QuadArgs a = {};
    double out = 0.0;
    std::vector<double> work((size_t) 6 * m);
    a.m = m;
    a.gram = gram;
    a.func = func;
    a.fp[0] = coefficient;
    a.exponent = 1.0;
    a.n = 1.0;
    slq::quadrature_one(a, alpha, beta, 1, 0, work.data(), work.data() + 2 * m,
                        work.data() + 4 * m, 1, &out, nullptr, nullptr);
    return out;
}
