// Row tiles (DevTiles) of CSR matrices built on the device.
//
// The union of the columns of a tile's R rows is found without sorting: an
// entry opens a slab if its column is in none of the tile's earlier rows,
// and a column's slab is the number of such opening entries with a smaller
// column, summed over the rows. Rows are sorted, so both are binary
// searches of one row's column in the others, one lane per entry, in the
// L1 cache (a tile's columns are a few KB). For A + tB the tile has the R
// rows of A and the R rows of B, and the slab of a column is the same sum
// over all of them.
//
// What bounds it: the latency of the searches (R rows x log2 row length L1
// loads per entry), one wavefront to a row, so matrices of a few long rows
// stay on the host (TileShape). The host sort and scatter that this replaces
// (build_tiles, still used for rows that are unsorted or repeat a column and
// for matrices of a few thousand entries) took about 27 ns per entry, 34 of
// the 36 ms of a logdet of a new 20011-row matrix of 1 M entries; here
// 0.19 ms (0.26 ms with one search after the other and four wavefronts a
// tile; 1003 rows of 30 entries: 0.050 against 0.097 ms).

#include <algorithm>
#include <climits>

#include "slq_internal.hpp"

namespace slq {

namespace {

// Flags of tile_count_kernel.
constexpr int kBadColumn = 1;   // column out of range
constexpr int kDescending = 2;  // columns of a row not ascending
constexpr int kRepeated = 4;    // a row repeats a column
constexpr int kLongRow = 8;     // not done: a long row

constexpr int32_t kOpens = INT32_MIN;   // flag bit of `pre`: the entry opens a slab

// One CSR matrix of a tile: pre[k] counts the opening entries before entry
// k in its row (with kOpens when k opens one itself), rowcnt[r] those of row r.
struct RowSet {
    const int64_t* indptr;
    const int32_t* indices;
    int32_t* pre;
    int32_t* rowcnt;
};

// Positions of column c in kAtOnce neighbouring rows [beg, end) of a set:
// the first whose column is not less. `top` is the largest power of two up to
// the longest of the rows. The searches take the same steps side by side
// (probes past a row's end read its last entry, or the set's first, and do
// not count), so that their loads are in flight together.
constexpr int kAtOnce = 4;

__device__ __forceinline__ void search(const int32_t* __restrict__ indices,
                                       const int64_t (&beg)[kAtOnce],
                                       const int64_t (&end)[kAtOnce], int64_t top, int32_t c,
                                       int64_t (&pos)[kAtOnce])
{
#pragma unroll
    for (int q = 0; q < kAtOnce; ++q) pos[q] = beg[q];
    for (int64_t st = top; st > 0; st >>= 1)
    {
        int32_t v[kAtOnce];
#pragma unroll
        for (int q = 0; q < kAtOnce; ++q)
        {
            const int64_t at = (pos[q] + st < end[q] ? pos[q] + st : end[q]) - 1;
            v[q] = indices[at > 0 ? at : 0];
        }
#pragma unroll
        for (int q = 0; q < kAtOnce; ++q)
            if (pos[q] + st <= end[q] && v[q] < c) pos[q] += st;
    }
}

// Largest power of two up to the longest row of tile t in the set (0: all
// empty).
template <int R>
__device__ __forceinline__ int64_t tile_top(const RowSet& s, int64_t nrows, int64_t t)
{
    int64_t longest = 0;
    for (int r = 0; r < R && t * R + r < nrows; ++r)
    {
        const int64_t len = s.indptr[t * R + r + 1] - s.indptr[t * R + r];
        longest = len > longest ? len : longest;
    }
    return longest > 0 ? (int64_t) 1 << (63 - __builtin_clzll((uint64_t) longest)) : 0;
}

// Bounds of the rows first .. first + kAtOnce - 1 of tile t (empty past the
// last row).
template <int R>
__device__ __forceinline__ void row_bounds(const RowSet& s, int64_t nrows, int64_t t, int first,
                                           int64_t (&beg)[kAtOnce], int64_t (&end)[kAtOnce])
{
#pragma unroll
    for (int q = 0; q < kAtOnce; ++q)
    {
        const int64_t row = t * R + first + q;
        beg[q] = row < nrows ? s.indptr[row] : 0;
        end[q] = row < nrows ? s.indptr[row + 1] : 0;
    }
}

constexpr int kTileThreads = 512;
constexpr int kTileWaves = kTileThreads / kWave;

// One workgroup per tile, a wavefront per row: opening entries, their number
// per tile (tile_cnt), what is wrong with the columns (status[0]) and the
// entries of the second set that the first has too (overlap).
template <int R>
__global__ __launch_bounds__(kTileThreads) void tile_count_kernel(
    int64_t nrows, int64_t ncols, int64_t ntiles, RowSet s0, RowSet s1, int nsets,
    const TileShape* __restrict__ shape, int32_t* __restrict__ tile_cnt,
    int* __restrict__ status, unsigned long long* __restrict__ overlap)
{
    if (shape && shape->long_row())
    {
        if (blockIdx.x == 0 && threadIdx.x == 0) *status = kLongRow;
        return;
    }
    __shared__ int cnt[kTileWaves];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int bad = 0;
    unsigned long long both = 0;
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x)
    {
        int mine = 0;
        const int64_t top0 = tile_top<R>(s0, nrows, t);
        const int64_t top1 = nsets > 1 ? tile_top<R>(s1, nrows, t) : 0;
        for (int l = wave; l < nsets * R; l += kTileWaves)
        {
            const int64_t row = t * R + l % R;
            if (row >= nrows) continue;
            const RowSet& s = l < R ? s0 : s1;
            const int64_t beg = s.indptr[row], end = s.indptr[row + 1];
            int run = 0;
            for (int64_t base = beg; base < end; base += kWave)
            {
                const int64_t k = base + lane;
                const bool in = k < end;
                const int32_t c = in ? s.indices[k] : 0;
                if (in)
                {
                    if (c < 0 || c >= ncols) bad |= kBadColumn;
                    if (k > beg)
                    {
                        const int32_t p = s.indices[k - 1];
                        bad |= p > c ? kDescending : p == c ? kRepeated : 0;
                    }
                }
                bool found = !in;
                // the rows before this one, and for the second set all of
                // the first (the same row there tells the overlap)
                for (int set = 0; set < (l < R ? 1 : 2); ++set)
                {
                    const RowSet& q = set == 0 ? s0 : s1;
                    const int64_t top = set == 0 ? top0 : top1;
                    const int rows = l < R || set == 1 ? l % R : R;
                    for (int o = 0; o < rows; o += kAtOnce)
                    {
                        int64_t ob[kAtOnce], oe[kAtOnce], pos[kAtOnce];
                        row_bounds<R>(q, nrows, t, o, ob, oe);
                        search(q.indices, ob, oe, top, c, pos);
#pragma unroll
                        for (int u = 0; u < kAtOnce; ++u)
                        {
                            const bool hit = in && o + u < rows && pos[u] < oe[u] &&
                                             q.indices[pos[u]] == c;
                            if (l >= R && set == 0 && o + u == l - R && hit) ++both;
                            found = found || hit;
                        }
                    }
                }
                const uint64_t opens = __ballot(!found);
                if (in)
                    s.pre[k] = (run + __popcll(opens & (((uint64_t) 1 << lane) - 1))) |
                               (found ? 0 : kOpens);
                run += __popcll(opens);
            }
            if (lane == 0) s.rowcnt[row] = run;
            mine += run;
        }
        if (lane == 0) cnt[wave] = mine;
        __syncthreads();
        if (threadIdx.x == 0)
        {
            int sum = 0;
            for (int w = 0; w < kTileWaves; ++w) sum += cnt[w];
            tile_cnt[t] = sum;
        }
        __syncthreads();
    }
    if (bad) atomicOr(status, bad);
    if (both) atomicAdd(overlap, both);
}

// The tiles' columns, and of every entry its value (`vals`, with `data`)
// and its position in the set's value array (`src0`, `src1`).
template <int R, typename T>
__global__ __launch_bounds__(kTileThreads) void tile_fill_kernel(
    int64_t nrows, int64_t ntiles, RowSet s0, RowSet s1, int nsets,
    const int64_t* __restrict__ tptr, const int32_t* __restrict__ tile_cnt,
    const T* __restrict__ data, int32_t* __restrict__ cols, T* __restrict__ vals,
    int32_t* __restrict__ src0, int32_t* __restrict__ src1)
{
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x)
    {
        const int64_t first = tptr[t], last = tptr[t + 1];
        const int cnt = tile_cnt[t];
        const int64_t top0 = tile_top<R>(s0, nrows, t);
        const int64_t top1 = nsets > 1 ? tile_top<R>(s1, nrows, t) : 0;
        for (int l = wave; l < nsets * R; l += kTileWaves)
        {
            const int64_t row = t * R + l % R;
            if (row >= nrows) continue;
            const RowSet& s = l < R ? s0 : s1;
            const int64_t beg = s.indptr[row], end = s.indptr[row + 1];
            for (int64_t base = beg; base < end; base += kWave)
            {
                const int64_t k = base + lane;
                const bool in = k < end;
                const int32_t c = in ? s.indices[k] : 0;
                const int32_t own = in ? s.pre[k] : 0;
                int64_t slab = first + (own & INT32_MAX);
                for (int o = 0; o < nsets * R; o += kAtOnce)
                {
                    const RowSet& q = o < R ? s0 : s1;
                    int64_t ob[kAtOnce], oe[kAtOnce], pos[kAtOnce];
                    row_bounds<R>(q, nrows, t, o % R, ob, oe);
                    search(q.indices, ob, oe, o < R ? top0 : top1, c, pos);
#pragma unroll
                    for (int u = 0; u < kAtOnce; ++u)
                    {
                        const int64_t orow = t * R + o % R + u;
                        if (o + u == l || orow >= nrows) continue;
                        slab += pos[u] < oe[u] ? (q.pre[pos[u]] & INT32_MAX) : q.rowcnt[orow];
                    }
                }
                if (!in) continue;
                const size_t slot = tile_slot(R, slab, l % R);
                if (vals) vals[slot] = data[k];
                (l < R ? src0 : src1)[slot] = (int32_t) k;
                if (own < 0)
                {
                    cols[slab] = c;
                    // padding slabs repeat the tile's last column
                    if (slab == first + cnt - 1)
                        for (int64_t p = slab + 1; p < last; ++p) cols[p] = c;
                }
            }
        }
    }
}

// The shape of one or two patterns (cleared before, with the entries set).
template <int R>
__global__ __launch_bounds__(256) void tile_shape_kernel(int64_t nrows, int64_t ntiles, RowSet s0,
                                                         RowSet s1, int nsets, int64_t nnz,
                                                         TileShape* __restrict__ shape)
{
    const int pad = R == 16 ? 8 : 1;
    long long longest = 0, slabs = 0;
    for (int64_t t = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; t < ntiles;
         t += (int64_t) gridDim.x * blockDim.x)
    {
        long long most = 0;
        for (int64_t r = t * R; r < (t + 1) * R && r < nrows; ++r)
        {
            most = max(most, (long long) (s0.indptr[r + 1] - s0.indptr[r]));
            if (nsets > 1) most = max(most, (long long) (s1.indptr[r + 1] - s1.indptr[r]));
        }
        longest = max(longest, most);
        slabs += (most + pad - 1) / pad * pad;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) shape->nnz = nnz;
    if (longest) atomicMax((unsigned long long*) &shape->longest, (unsigned long long) longest);
    if (slabs) atomicAdd((unsigned long long*) &shape->slabs, (unsigned long long) slabs);
}

struct Temp {
    void* p = nullptr;
    ~Temp()
    {
        if (p) (void) hipFree(p);
    }
};

template <int R>
int device_tiles_r(hipStream_t s, const DevCSR& a, const DevCSR* b, double min_density,
                   DevTiles& out, int32_t** src_a, int32_t** src_b, TileStatus& st)
{
    const int64_t n = a.nrows;
    const int64_t T = (n + R - 1) / R;
    const int nsets = b ? 2 : 1;
    auto up = [](size_t x) { return (x + 255) & ~(size_t) 255; };
    const size_t b_pre = up(sizeof(int32_t) * (size_t) a.nnz);
    const size_t b_pre2 = b ? up(sizeof(int32_t) * (size_t) b->nnz) : 0;
    const size_t b_row = up(sizeof(int32_t) * (size_t) n);
    const size_t b_cnt = up(sizeof(int32_t) * (size_t) T);
    Temp tmp;
    // one allocation: status words, tile counts, row counts, entry ranks
    if (hipMalloc(&tmp.p, 256 + b_cnt + nsets * b_row + b_pre + b_pre2) != hipSuccess)
    {
        (void) hipGetLastError();   // the caller builds on the host instead
        return SLQ_OK;
    }
    char* base = (char*) tmp.p;
    unsigned long long* overlap = (unsigned long long*) base;
    int* status = (int*) (base + 8);
    TileShape* shape = (TileShape*) (base + 16);
    int32_t* cnt = (int32_t*) (base + 256);
    char* p = base + 256 + b_cnt;
    RowSet s0{a.indptr, a.indices, (int32_t*) (p + nsets * b_row), (int32_t*) p};
    RowSet s1 = s0;
    if (b)
        s1 = RowSet{b->indptr, b->indices, (int32_t*) (p + nsets * b_row + b_pre),
                    (int32_t*) (p + b_row)};
    const dim3 grid((unsigned) std::min<int64_t>(T, 1 << 20));
    SLQ_CHECK(hipMemsetAsync(base, 0, 256, s));
    if (!st.rows_known)
        hipLaunchKernelGGL(tile_shape_kernel<R>,
                           dim3((unsigned) std::min<int64_t>((T + 255) / 256, 1024)), dim3(256), 0,
                           s, n, T, s0, s1, nsets, a.nnz + (b ? b->nnz : 0), shape);
    hipLaunchKernelGGL(tile_count_kernel<R>, grid, dim3(kTileThreads), 0, s, n, a.ncols, T, s0,
                       s1, nsets, st.rows_known ? nullptr : (const TileShape*) shape, cnt, status,
                       overlap);
    SLQ_CHECK(hipGetLastError());
    // status, overlap and the tile counts in one copy
    std::vector<char> host(256 + b_cnt);
    SLQ_CHECK(hipMemcpyAsync(host.data(), base, host.size(), hipMemcpyDeviceToHost, s));
    SLQ_CHECK(hipStreamSynchronize(s));
    int flags;
    unsigned long long both;
    std::memcpy(&both, host.data(), sizeof(both));
    std::memcpy(&flags, host.data() + 8, sizeof(flags));
    if (flags & kLongRow)
    {
        TileShape sh;
        std::memcpy(&sh, host.data() + 16, sizeof(sh));
        st.built = sh.none(R, min_density);
        return SLQ_OK;
    }
    st.checked = true;
    st.bad_column = (flags & kBadColumn) != 0;
    st.sorted = (flags & kDescending) == 0;
    st.strict = st.sorted && (flags & kRepeated) == 0;
    if (st.bad_column || !st.strict || !st.want_tiles) return SLQ_OK;
    const int32_t* hc = (const int32_t*) (host.data() + 256);
    std::vector<int64_t> tptr(T + 1, 0);
    for (int64_t t = 0; t < T; ++t)
        tptr[t + 1] = tptr[t] + (R == 16 ? (hc[t] + 7) / 8 * 8 : hc[t]);
    const int64_t U = tptr[T];
    const int64_t nnz = a.nnz + (b ? b->nnz - (int64_t) both : 0);
    st.built = true;
    if (U == 0 || (double) nnz / ((double) U * R) < min_density) return SLQ_OK;
    DevTiles d;
    d.R = R;
    d.ntiles = T;
    d.nslabs = U;
    const size_t vb = a.dtype == SLQ_F64 ? 8 : 4;
    const size_t slots = (size_t) U * R;
    int32_t* sa = nullptr;
    int32_t* sb = nullptr;
    hipError_t e;
    if ((e = hipMalloc(&d.ptr, sizeof(int64_t) * (T + 1))) != hipSuccess ||
        (e = hipMalloc(&d.cols, sizeof(int32_t) * U)) != hipSuccess ||
        (e = hipMalloc(&d.vals, vb * slots)) != hipSuccess ||
        (e = hipMalloc(&sa, sizeof(int32_t) * slots)) != hipSuccess ||
        (b && (e = hipMalloc(&sb, sizeof(int32_t) * slots)) != hipSuccess) ||
        (e = hipMemcpyAsync(d.ptr, tptr.data(), sizeof(int64_t) * (T + 1),
                            hipMemcpyHostToDevice, s)) != hipSuccess ||
        (e = hipMemsetAsync(d.vals, 0, vb * slots, s)) != hipSuccess ||
        (e = hipMemsetAsync(sa, 0xff, sizeof(int32_t) * slots, s)) != hipSuccess ||
        (b && (e = hipMemsetAsync(sb, 0xff, sizeof(int32_t) * slots, s)) != hipSuccess))
    {
        (void) hipStreamSynchronize(s);
        free_tiles(d);
        if (sa) (void) hipFree(sa);
        if (sb) (void) hipFree(sb);
        return hip_status(e, "tile allocation", __FILE__, __LINE__);
    }
    if (a.dtype == SLQ_F64)
        hipLaunchKernelGGL((tile_fill_kernel<R, double>), grid, dim3(kTileThreads), 0, s, n, T,
                           s0, s1, nsets, d.ptr, cnt, (const double*) a.data, d.cols,
                           b ? nullptr : (double*) d.vals, sa, sb);
    else
        hipLaunchKernelGGL((tile_fill_kernel<R, float>), grid, dim3(kTileThreads), 0, s, n, T,
                           s0, s1, nsets, d.ptr, cnt, (const float*) a.data, d.cols,
                           b ? nullptr : (float*) d.vals, sa, sb);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(s);   // before the temporaries go
    if (e != hipSuccess)
    {
        free_tiles(d);
        (void) hipFree(sa);
        if (sb) (void) hipFree(sb);
        return hip_status(e, "tile fill", __FILE__, __LINE__);
    }
    if (b)
    {
        *src_a = sa;
        *src_b = sb;
    }
    else
        d.src = sa;
    out = d;
    return SLQ_OK;
}

}  // namespace

TileShape tile_shape(int64_t nrows, const int64_t* indptr, int R, int64_t& decreasing)
{
    TileShape sh;
    sh.nnz = indptr[nrows];
    decreasing = -1;
    for (int64_t r = 0; r < nrows; ++r)
    {
        const int64_t len = indptr[r + 1] - indptr[r];
        if (len < 0)
        {
            decreasing = r;
            return sh;
        }
        sh.longest = std::max(sh.longest, len);
    }
    if (!sh.long_row()) return sh;
    const int64_t pad = R == 16 ? 8 : 1;
    for (int64_t t = 0; t * R < nrows; ++t)
    {
        int64_t most = 0;
        for (int64_t r = t * R; r < std::min<int64_t>((t + 1) * R, nrows); ++r)
            most = std::max(most, indptr[r + 1] - indptr[r]);
        sh.slabs += (most + pad - 1) / pad * pad;
    }
    return sh;
}

int device_tiles(hipStream_t s, const DevCSR& a, const DevCSR* b, int R, double min_density,
                 DevTiles& out, int32_t** src_a, int32_t** src_b, TileStatus& st)
{
    out = DevTiles();
    if (a.nnz + (b ? b->nnz : 0) > (int64_t) INT32_MAX || a.nnz == 0) return SLQ_OK;
    return R == 8 ? device_tiles_r<8>(s, a, b, min_density, out, src_a, src_b, st)
                  : device_tiles_r<16>(s, a, b, min_density, out, src_a, src_b, st);
}

}  // namespace slq
