// Lanczos on a small matrix in one launch: a workgroup per probe, the
// recurrence's two vectors in its LDS for all m steps.
//
// The reference recurrence is that of krylov.hip (lanczos_ring;
// imate/_c_trace_estimator/c_lanczos_tridiagonalization.cpp:117-235), with
// the vectors unnormalised and scaled where they are read. A step multiplies
// by the CSR rows (L neighbouring lanes per row, operand entries gathered
// from LDS), sums alpha over the workgroup, updates and sums the norm: two
// workgroup barriers and no launch, where the block kernels take four
// launches of at least 4-5 us a step whatever the size. All arithmetic on
// vectors is FP64, also for FP32 matrices and for the mixed-precision form,
// which reads the FP64 values of an FP64 matrix.
//
// What bounds it: every workgroup reads the whole matrix from its XCD's L2
// every step, at the rate its vector loads issue (a wavefront's load takes
// 4 to 8 clocks of the CU's address unit): loads are unconditional and as
// few as the row lengths allow. logdet with degree 20 and default samples at
// n = 50 took 381 us with the block kernels, 142 us with this one (33 us of
// it); an FP32 matrix of 1003 rows and 30 a row 855 and 650 us (0.23 ms).

#include <cstdlib>

#include "slq_internal.hpp"
#include "lanes.hpp"

namespace slq {

namespace {

constexpr int kRows = 4;   // rows a lane has in flight

struct ResidentArgs {
    const int64_t* indptr;
    const int32_t* indices;
    const void* vals;
    int64_t n;
    int nnz;
    double t;               // identity shift (0: none)
    int shift;
    int m;
    double s0;              // 1 / |probe|
    double tol_sqrt_n;
    const void* X0;         // [n][64]
    double* alpha;          // [m][64]
    double* beta;           // [m][64]
    int32_t* sizes;         // [64]
};

// Sum of x over the workgroup, the same in every thread. `red` holds one
// value per wavefront and is free again after the caller's next barrier but
// one, so calls alternate between two of them.
template <int NT>
__device__ __forceinline__ double group_sum(double x, double* red)
{
    x = lanes_sum<64>(x);
    const int wave = threadIdx.x / kWave;
    if (threadIdx.x % kWave == 0) red[wave] = x;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < NT / kWave; ++w) s += red[w];
    return s;
}

// L lanes per row, each with E entries of it in flight.
template <typename V, typename X, int NT, int L, int E>
__global__ __launch_bounds__(NT) void resident_lanczos_kernel(ResidentArgs a)
{
    extern __shared__ double sh[];
    const int n = (int) a.n;
    double* x = sh;                 // v_j / s: the gathered vector
    double* y = sh + n;             // v_{j-1} / s', then w, then the residual
    double* red = sh + 2 * n;       // two sets of per-wavefront sums
    int* rp = (int*) (red + 2 * (NT / kWave));   // row pointers
    const int p = blockIdx.x;
    const int tid = threadIdx.x;
    const V* __restrict__ vals = (const V*) a.vals;
    const int32_t* __restrict__ indices = a.indices;
    const X* __restrict__ X0 = (const X*) a.X0;
    for (int i = tid; i < n; i += NT)
    {
        x[i] = (double) X0[(int64_t) i * kBlock + p];
        y[i] = 0.0;
    }
    for (int i = tid; i <= n; i += NT) rp[i] = (int) a.indptr[i];
    __syncthreads();
    const int sub = tid % L;
    double s = a.s0, s_prev = 0.0, beta = 0.0;
    int size = 0;
    int j = 0;
    for (; j < a.m && size == 0; ++j)
    {
        // w = (A + tI) v_j - beta_{j-1} v_{j-1}, alpha_j = v_j . (A + tI) v_j
        double dot = 0.0;
        for (int r0 = tid / L; r0 < n; r0 += kRows * (NT / L))
        {
            int beg[kRows], len[kRows], c[kRows][E];
            V v[kRows][E];
#pragma unroll
            for (int u = 0; u < kRows; ++u)
            {
                const int row = r0 + u * (NT / L);
                beg[u] = row < n ? rp[row] : 0;
                len[u] = row < n ? rp[row + 1] - beg[u] : 0;
            }
#pragma unroll
            for (int u = 0; u < kRows; ++u)
#pragma unroll
                for (int i = 0; i < E; ++i)
                {
                    // past the row's end its last entry (or the matrix's)
                    // with value zero: no load is conditional
                    const int k = i * L + sub;
                    const unsigned int at = min(beg[u] + min(k, max(len[u] - 1, 0)), a.nnz - 1);
                    c[u][i] = indices[at];
                    const V w = vals[at];
                    v[u][i] = k < len[u] ? w : V(0);
                }
#pragma unroll
            for (int u = 0; u < kRows; ++u)
            {
                const int row = r0 + u * (NT / L);
                double acc = 0.0;
#pragma unroll
                for (int i = 0; i < E; ++i)
                    acc = fma((double) v[u][i], s * x[c[u][i]], acc);
                for (int k = E * L + sub; k < len[u]; k += L)
                    acc = fma((double) vals[beg[u] + k], s * x[indices[beg[u] + k]], acc);
                acc = lanes_sum<L>(acc);
                if (row < n && sub == 0)
                {
                    const double vr = s * x[row];
                    if (a.shift) acc = acc + a.t * vr;
                    dot += vr * acc;
                    y[row] = acc - beta * (s_prev * y[row]);
                }
            }
        }
        const double alpha = group_sum<NT>(dot, red);
        // r = w - alpha_j v_j, beta_j = |r|
        double nn = 0.0;
        for (int i = tid; i < n; i += NT)
        {
            const double r = y[i] - alpha * (s * x[i]);
            y[i] = r;
            nn += r * r;
        }
        const double b = sqrt(group_sum<NT>(nn, red + NT / kWave));
        if (tid == 0)
        {
            a.alpha[(int64_t) j * kBlock + p] = alpha;
            a.beta[(int64_t) j * kBlock + p] = b;
        }
        if (b < a.tol_sqrt_n) size = j + 1;
        s_prev = s;
        s = 1.0 / b;
        beta = b;
        double* z = x;
        x = y;
        y = z;
    }
    // steps past a breakdown hold nothing
    for (int i = j + tid; i < a.m; i += NT)
    {
        a.alpha[(int64_t) i * kBlock + p] = 0.0;
        a.beta[(int64_t) i * kBlock + p] = 0.0;
    }
    if (tid == 0) a.sizes[p] = size;
}

template <int NT>
size_t lds_bytes(int64_t n)
{
    return sizeof(double) * (2 * (size_t) n + 2 * (NT / kWave)) + sizeof(int) * ((size_t) n + 1);
}

template <typename V, typename X, int NT, int L, int E>
int launch(const ResidentArgs& a, hipStream_t s)
{
    const size_t lds = lds_bytes<NT>(a.n);
    auto kern = resident_lanczos_kernel<V, X, NT, L, E>;
    if (lds > 64 * 1024)
        SLQ_CHECK(hipFuncSetAttribute((const void*) kern,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds));
    hipLaunchKernelGGL(kern, dim3(kBlock), dim3(NT), lds, s, a);
    SLQ_CHECK(hipGetLastError());
    return SLQ_OK;
}

// Lanes per row and entries per lane that cover a row of ordinary length
// (the mean and 1.2 deviations of a Poisson count).
struct Shape {
    int lanes, entries;
};

Shape shape_of(const DevCSR& c)
{
    const double avg = (double) c.nnz / (double) c.nrows;
    const double want = avg + 1.2 * std::sqrt(avg);
    if (want <= 4) return {4, 1};
    if (want <= 8) return {4, 2};
    if (want <= 16) return {4, 4};
    if (want <= 32) return {8, 4};
    if (want <= 64) return {16, 4};
    return {32, 4};
}

template <typename V, typename X, int NT>
int launch_sized(const ResidentArgs& a, Shape sh, hipStream_t s)
{
    if (sh.entries == 1) return launch<V, X, NT, 4, 1>(a, s);
    if (sh.entries == 2) return launch<V, X, NT, 4, 2>(a, s);
    if (sh.lanes == 4) return launch<V, X, NT, 4, 4>(a, s);
    if (sh.lanes == 8) return launch<V, X, NT, 8, 4>(a, s);
    if (sh.lanes == 16) return launch<V, X, NT, 16, 4>(a, s);
    return launch<V, X, NT, 32, 4>(a, s);
}

// 256 threads for the smallest matrices (cheaper barriers), else 1024.
template <typename V, typename X>
int launch_any(const ResidentArgs& a, Shape sh, hipStream_t s)
{
    return a.n <= 128 ? launch_sized<V, X, 256>(a, sh, s) : launch_sized<V, X, 1024>(a, sh, s);
}

}  // namespace

// Small enough for the resident kernel: a step takes about 1.5 us + 0.57 us
// per unit of `cost`, where a round of rows costs one unit and one for every
// entry a lane has in flight, and a row longer than its lanes' entries one
// for every further trip. The block kernels take 14 to 27 us a step at these
// sizes; up to 30 units the resident kernel was 1.16 to 3.2 times as fast in
// whole calls (n = 50 to 7000, 3 to 75 entries a row), at 40 units 0.9 to 1.1
// times. Launch settings given for the handle, profiling and SLQ_TILE_ROWS
// ask for the block kernels.
constexpr int64_t kMostCost = 30;

bool resident_fits(const slq_op* op, int gram, int ortho)
{
    const MatrixStore& A = *op->A;
    const DevCSR& c = A.csr;
    if (gram || ortho != 0 || A.dense || op->kind == OP_AFFINE_B || op->user_launch ||
        op->prof.enabled || c.nnz == 0 || lds_bytes<1024>(c.nrows) > 150 * 1024 ||
        std::getenv("SLQ_TILE_ROWS"))
        return false;
    const Shape sh = shape_of(c);
    const int64_t rows = kRows * (1024 / sh.lanes);
    const int64_t rounds = (c.nrows + rows - 1) / rows;
    const int64_t tail = c.max_row - sh.lanes * sh.entries;
    const int64_t cost =
        rounds * (1 + sh.entries) + (tail > 0 ? (tail + sh.lanes - 1) / sh.lanes : 0);
    return cost <= kMostCost;
}

int run_resident(const RecurrenceArgs& ra)
{
    const slq_op* op = ra.op;
    const DevCSR& c = op->A->csr;
    ResidentArgs a;
    a.indptr = c.indptr;
    a.indices = c.indices;
    a.vals = c.data;
    a.n = c.nrows;
    a.nnz = (int) c.nnz;
    a.t = ra.t;
    a.shift = op->kind == OP_AFFINE_I ? 1 : 0;
    a.m = ra.m;
    a.s0 = 1.0 / std::sqrt((double) c.nrows);
    a.tol_sqrt_n = ra.tol * std::sqrt((double) c.nrows);
    a.X0 = ra.X0;
    a.alpha = ra.alpha;
    a.beta = ra.beta;
    a.sizes = ra.sizes;
    const Shape sh = shape_of(c);
    if (c.dtype == SLQ_F32) return launch_any<float, float>(a, sh, op->stream);
    if (ra.precision == SLQ_PREC_MIXED) return launch_any<double, float>(a, sh, op->stream);
    return launch_any<double, double>(a, sh, op->stream);
}

}  // namespace slq
