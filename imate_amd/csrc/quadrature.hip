// Gauss quadrature of the Krylov recurrences on the device, in FP64.
//
// Reference: after each Lanczos run imate calls LAPACK ?stev('V') on the
// tridiagonal T (alpha diagonal, beta off-diagonal), takes the eigenvalues
// theta_i and the first component tau_i of each eigenvector, and forms
// n * sum_i tau_i^2 f(theta_i^p) (imate/_c_trace_estimator/c_trace_estimator.cpp:
// 545-621, diagonalization.cpp:88-118). For Golub-Kahn it calls ?bdsdc on the
// upper bidiagonal B and uses theta = sigma^2 with tau the first component of
// each right singular vector (c_trace_estimator.cpp:505-535,
// diagonalization.cpp:189-231). With B = I the Ritz values of A + t_j I are
// the Ritz values of A + t_0 I shifted by t_j - t_0 (c_trace_estimator.cpp:
// 564-594, c_affine_matrix_function.cpp get_eigenvalue).
//
// Here a workgroup owns one probe and solves its tridiagonal by
// divide-and-conquer (dc.hpp), carrying only the first and last rows of the
// eigenvectors of each block. The bidiagonal case is solved as the 2k x 2k
// Golub-Kahan tridiagonal with zero diagonal and off-diagonal (alpha_0,
// beta_0, alpha_1, ..., alpha_{k-1}), whose eigenvalues are +-sigma_i; the
// eigenvectors of +sigma_i and -sigma_i are (v_0, +-u_0, v_1, +-u_1, ...) /
// sqrt(2), so tau_i^2 is the sum of both z_0^2, the i-th largest eigenvalue
// taken with the i-th smallest: for a zero singular value, whose two
// eigenvectors are any pair of that plane, only the sum is the weight
// (twice one of them was up to 0.3 off). Matrices past kDcMaxRows
// rows (their work arrays would not fit the LDS) run the implicit QL of
// ql.hpp, the host path's solver, one probe per workgroup.
//
// What bounds it: latency. One probe's QL is a serial chain of about
// 0.65 m^2 plane rotations of some hundred dependent FP64 operations each
// (measured 266 us at m = 20, 525 at 30, 1840 at 60, the same for one probe
// or 64), while divide-and-conquer is log2(m) merges whose roots are
// independent threads: 41, 54 and 77 us. The matrix function at the
// nodes is spread over the threads too: by node for a few inquiries, by
// inquiry for many (256 inquiries at m = 30 took 2.9 ms in one thread per
// probe).

#include <cfloat>
#include <cmath>

#include "slq_internal.hpp"
#include "ql.hpp"
#include "dc.hpp"
#include "lanes.hpp"

namespace slq {

namespace {

// Rows up to which the divide-and-conquer work arrays are taken: 92 bytes a
// row, 92 KB of the CU's 160 KB of LDS.
constexpr int kDcMaxRows = 1024;
// Inquiries up to which the threads share the nodes of one inquiry.
constexpr int kFewInquiries = 8;

struct Workgroup {
    int tid, nt;
    __device__ __forceinline__ void sync() const { __syncthreads(); }
    template <int P, typename T>
    __device__ __forceinline__ T sum(T x) const
    {
        return lanes_sum<P>(x);
    }
    template <int P>
    __device__ __forceinline__ double prod(double x) const
    {
        return lanes_product<P>(x);
    }
};

template <int NT, int P>
__global__ __launch_bounds__(NT) void quadrature_dc_kernel(QuadArgs a)
{
    extern __shared__ double sh[];
    const int p = blockIdx.x;
    const Workgroup g{(int) threadIdx.x, NT};
    const int k = a.sizes[p] > 0 ? a.sizes[p] : a.m;
    const int K = a.gram ? 2 * k : k;
    const DcWork w = dc_carve(sh, K);
    const double* al = a.alpha + p;
    const double* be = a.beta + p;
    for (int i = g.tid; i < k; i += NT)
    {
        const double ai = al[(int64_t) i * kBlock];
        const double bi = i < k - 1 ? be[(int64_t) i * kBlock] : 0.0;
        if (a.gram)
        {
            w.d[2 * i] = 0.0;
            w.d[2 * i + 1] = 0.0;
            w.e[2 * i] = ai;
            w.e[2 * i + 1] = bi;
        }
        else
        {
            w.d[i] = ai;
            w.e[i] = bi;
        }
    }
    g.sync();
    const bool ok = dc_first_row<P>(g, w, K);
    // nodes and weights in order: ascending, or the k largest singular
    // values descending
    double* th = w.ds;
    double* tau = w.zs;
    if (ok)
        for (int i = g.tid; i < K; i += NT)
        {
            const double di = w.d[i];
            int r = 0;
            for (int j = 0; j < K; ++j)
            {
                const double dj = w.d[j];
                r += ((a.gram ? dj > di : dj < di) || (dj == di && j < i)) ? 1 : 0;
            }
            if (r < k) th[r] = a.gram ? di * di : di;
            // with gram -sigma's behind +sigma's
            tau[r < k ? r : k + (K - 1 - r)] = w.f[i];
        }
    g.sync();
    if (ok && a.gram)
    {
        for (int i = g.tid; i < k; i += NT) tau[i] = pair_weight(tau[i], tau[k + i]);
        g.sync();
    }
    if (a.theta_out)
        for (int i = g.tid; i < a.m; i += NT)
        {
            a.theta_out[(size_t) p * a.m + i] = ok && i < k ? th[i] : (i < k ? NAN : 0.0);
            a.tau_out[(size_t) p * a.m + i] = ok && i < k ? tau[i] : (i < k ? NAN : 0.0);
        }
    const int jn = a.shift ? a.q : 1;
    const double t0 = a.shift ? a.params[0] : 0.0;
    double* out = a.samples + (size_t) p * a.q_stride;
    auto term = [&](int i, double tj) {
        return node_term(a, a.shift ? (th[i] - t0) + tj : th[i], tau[i]);
    };
    if (jn > kFewInquiries)
    {
        for (int j = g.tid; j < jn; j += NT)
        {
            const double tj = a.params[j];
            double sum = 0.0;
            if (ok)
                for (int i = 0; i < k; ++i) sum += term(i, tj);
            out[j] = ok ? a.n * sum : NAN;
        }
        return;
    }
    for (int j = 0; j < jn; ++j)
    {
        const double tj = a.shift ? a.params[j] : 0.0;
        double sum = 0.0;
        if (ok)
            for (int i = g.tid; i < k; i += NT) sum += term(i, tj);
        for (int s = 1; s < kWave; s <<= 1) sum += __shfl_xor(sum, s);
        if (NT > kWave)
        {
            double* red = w.fs;
            if (g.tid % kWave == 0) red[g.tid / kWave] = sum;
            g.sync();
            sum = 0.0;
            for (int v = 0; v < NT / kWave; ++v) sum += red[v];
            g.sync();
        }
        if (g.tid == 0) out[a.shift ? j : a.j_out] = ok ? a.n * sum : NAN;
    }
}

// One probe per workgroup and thread, for matrices past kDcMaxRows rows.
__global__ __launch_bounds__(64) void quadrature_ql_kernel(QuadArgs a)
{
    extern __shared__ double sh[];
    const int p = blockIdx.x;
    const int K2 = a.gram ? 2 * a.m : a.m;
    quadrature_one(a, a.alpha + p, a.beta + p, kBlock, a.sizes[p], sh, sh + K2,
                   sh + (size_t) 2 * K2, 1, a.samples + (size_t) p * a.q_stride,
                   a.theta_out ? a.theta_out + (size_t) p * a.m : nullptr,
                   a.tau_out ? a.tau_out + (size_t) p * a.m : nullptr);
}

}  // namespace

int run_quadrature(hipStream_t s, const double* alpha, const double* beta,
                   const int32_t* sizes, int count, int m, int gram, int func,
                   const double* func_params, double exponent, double n,
                   const double* params_dev, int q,
                   int shift, int j_out, int q_stride, double* samples_dev,
                   double* theta_dev, double* tau_dev)
{
    QuadArgs a;
    a.alpha = alpha;
    a.beta = beta;
    a.sizes = sizes;
    a.count = count;
    a.m = m;
    a.gram = gram;
    a.func = func;
    for (int i = 0; i < 4; ++i) a.fp[i] = func_params ? func_params[i] : 0.0;
    a.exponent = exponent;
    a.n = n;
    a.params = params_dev;
    a.q = q;
    a.shift = shift;
    a.j_out = j_out;
    a.q_stride = q_stride;
    a.samples = samples_dev;
    a.theta_out = theta_dev;
    a.tau_out = tau_dev;
    const int K2 = gram ? 2 * m : m;
    if (K2 <= kDcMaxRows)
    {
        const size_t lds = (size_t) K2 * (kDcDoubles * sizeof(double) + kDcInts * sizeof(int));
        // 8 threads a row while 512 threads (256 up to 32 rows, for cheaper
        // barriers: 41 against 45 us at m = 20, 54 against 62 at 30) cover
        // them, then fewer: 77 us at 60 rows and 166 at 120 (gram, m = 60)
        // against 81 and 216 with 256 threads
        auto kern = quadrature_dc_kernel<512, 1>;
        if (K2 <= 32) kern = quadrature_dc_kernel<256, 8>;
        else if (K2 <= 64) kern = quadrature_dc_kernel<512, 8>;
        else if (K2 <= 128) kern = quadrature_dc_kernel<512, 4>;
        const int nt = K2 <= 32 ? 256 : 512;
        if (lds > 64 * 1024)
            SLQ_CHECK(hipFuncSetAttribute((const void*) kern,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds));
        hipLaunchKernelGGL(kern, dim3(count), dim3(nt), lds, s, a);
        SLQ_CHECK(hipGetLastError());
        return SLQ_OK;
    }
    const size_t lds = sizeof(double) * 3 * (size_t) K2;
    if (lds > 160 * 1024)
    {
        set_error("lanczos_degree %d too large for the device eigensolver", m);
        return SLQ_E_ARG;
    }
    if (lds > 64 * 1024)
        SLQ_CHECK(hipFuncSetAttribute((const void*) quadrature_ql_kernel,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds));
    hipLaunchKernelGGL(quadrature_ql_kernel, dim3(count), dim3(1), lds, s, a);
    SLQ_CHECK(hipGetLastError());
    return SLQ_OK;
}

}  // namespace slq
