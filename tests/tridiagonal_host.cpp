// Host build of the tridiagonal eigensolvers (one thread), for
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
