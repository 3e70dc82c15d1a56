// Sums over the rows of a matrix (the gradients of biases and of layer_norm's parameters): ordinary float32 additions.
//
// Bound by memory, one read of the matrix.  A work-group of 256 lanes takes up to 64 columns of a range of rows: WIDE lanes with
// 128-bit loads side by side (at most 256 contiguous bytes of a row; as few as cover the matrix) and 256 / WIDE rows at a time,
// eight loads in flight per lane, the lanes of a column added through LDS in a tree.  Where the rows keep a lane busy for more
// than eight such rounds they are cut into ranges of about one round, whose sums go to the workspace and are added by the
// same kernel in a second launch (which costs what eight rounds do: 1000 x 197 5.3 us in one launch, 6.1 in two).  Two
// matrices of one shape can be summed in one launch.
// Rounding: the eight loaded values are added as a tree and the trees' sums in a cascade, kChain at a time on each of
// kLevels levels, so that a value passes through fewer than 64 rounded additions at the sizes of a model's gradients and
// fewer than 100 in any matrix of up to 2^31 values, however long a lane's share of the rows is (many columns leave no
// work-groups to cut the rows for: 4096 rows of 131073 equal values near 1 in one chain per lane were off by 1.5e-5, now by
// less than 4e-6).  The order depends on the two sizes alone: not on a second matrix beside, nor on strides or alignment
// (128-bit loads at any float's address; where a row's last loads would pass its end they start earlier and some columns are
// summed twice alike).
// Measured against torch's sum over dim 0 (which clears a buffer first where it cuts the rows), us: 96 x 128 3.2 (torch 4.2),
// 256 x 64 3.4 (5.0), 4096 x 1024 5.9 (20), 12608 x 768 10.8 (26), 65536 x 1024 twice 93, 4096 x 10000 34 (181), 10^6 x 1
// 5.8 (10.7), 10^6 x 10 14 (22).  With sixteen lanes across whatever the width, cut from 256 rows on and a range's odd rows one by
// one: 256 x 64 5.2, 12608 x 768 12.6 and the last two 35 and 39.  A linear layer of 12608 x 192 -> 768 with its gradients
// 277 -> 266 us with these sums, 4096 x 512 -> 1024 375 -> 361.
#include <algorithm>
#include <cstdint>

#include "../../include/pam_hip_extra.h"
#include "pam_common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kFlight = 8;              // loads in flight per lane: a round
constexpr long kMostGroups = 2048;      // work-groups per matrix of a launch that cuts the rows: eight per compute unit
constexpr long kRoundsAlone = 8;        // rounds of a lane up to which the rows are not cut
constexpr int kChain = 16, kLevels = 4;

struct Sums { const float* in[2]; float* out[2]; long row_stride[2]; };

// VEC: values per lane and load, WIDE: lanes per row.  Work-group (x, y, z): the x-th VEC * WIDE columns, range y of the rows,
// matrix z; the sums of range y go to out[z] + y * n.  n is at least VEC.
template <int VEC, int WIDE>
__global__ __launch_bounds__(kThreads) void column_sums_kernel(Sums s, long rows, long n, long range)
{
    constexpr int kColumns = VEC * WIDE, kDeep = kThreads / WIDE;
    typedef float vec __attribute__((ext_vector_type(VEC)));
    typedef float vec_any __attribute__((ext_vector_type(VEC), aligned(4)));
    __shared__ float part[kDeep][kColumns];
    const int tx = threadIdx.x % WIDE, ty = threadIdx.x / WIDE;
    const long base = (long)blockIdx.x * kColumns, column = min(base + tx * VEC, n - VEC);
    const long first = (long)blockIdx.y * range, last = min(rows, first + range);
    const long stride = s.row_stride[blockIdx.z], step = stride * kDeep;
    const float* at = s.in[blockIdx.z] + column + (first + ty) * stride;
    long left = last - first - ty;                  // rows from the lane's next one to the range's end
    vec level[kLevels] = {}, v[kFlight];
    auto tree = [&]() __attribute__((always_inline)) { return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])); };
    unsigned trees = 0;
    for (; left > (kFlight - 1) * kDeep; left -= kFlight * kDeep) {
#pragma unroll
        for (int u = 0; u < kFlight; ++u, at += step) v[u] = *reinterpret_cast<const vec_any*>(at);
        level[0] += tree();
        ++trees;
        if (trees % kChain == 0) {
            unsigned whole = kChain;
#pragma unroll
            for (int l = 0; l + 1 < kLevels; ++l, whole *= kChain)
                if (trees % whole == 0) { level[l + 1] += level[l]; level[l] = 0.0f; }
        }
    }
    vec total = 0.0f;
    if (left > 0) {                                 // the rest, all in flight too: rows past the end are the first one again and count as zeros
#pragma unroll
        for (int u = 0; u < kFlight; ++u) v[u] = *reinterpret_cast<const vec_any*>(at + (u * kDeep < left ? u * step : 0));
#pragma unroll
        for (int u = 1; u < kFlight; ++u) if (u * kDeep >= left) v[u] = 0.0f;
        total = tree();
    }
#pragma unroll
    for (int l = 0; l < kLevels; ++l) total += level[l];
    union { vec v; float f[VEC]; } sums;
    sums.v = total;
#pragma unroll
    for (int e = 0; e < VEC; ++e)                   // (a lane that starts earlier writes what its neighbour does)
        if (column + e >= base) part[ty][column + e - base] = sums.f[e];
    for (int half = kDeep / 2; half >= 1; half /= 2) {
        __syncthreads();
        for (int i = threadIdx.x; i < half * kColumns; i += kThreads) part[i / kColumns][i % kColumns] += part[i / kColumns + half][i % kColumns];
    }
    __syncthreads();
    if (threadIdx.x < kColumns && base + threadIdx.x < n) s.out[blockIdx.z][(long)blockIdx.y * n + base + threadIdx.x] = part[0][threadIdx.x];
}

// values per load and lanes per row for n columns: the narrowest that covers them, up to 64 columns
struct Lanes { int vec, wide; int columns() const { return vec * wide; } };
Lanes lanes_for(long n)
{
    const int vec = n < 4 ? 1 : 4;
    int wide = 1;
    while (wide < 16 && (long)vec * wide < n) wide *= 2;
    return Lanes{vec, wide};
}

// rows per range and number of ranges
struct Cut { long range, ranges; };
Cut cut_rows(long rows, long n)
{
    const Lanes l = lanes_for(n);
    const long round = (long)kFlight * (kThreads / l.wide), groups = (n + l.columns() - 1) / l.columns();
    if (rows <= kRoundsAlone * round) return Cut{rows, 1};
    const long most = std::max(1L, std::min({(rows + round - 1) / round, kMostGroups / groups, 65535L}));
    const long range = (rows + most - 1) / most;
    return Cut{range, (rows + range - 1) / range};
}

void launch(const Sums& s, int matrices, long rows, long n, const Cut& cut, hipStream_t st)
{
    const Lanes l = lanes_for(n);
    const dim3 grid((unsigned)((n + l.columns() - 1) / l.columns()), (unsigned)cut.ranges, (unsigned)matrices);
#define PAM_COLUMN_SUMS(V, W) if (l.vec == V && l.wide == W) { hipLaunchKernelGGL((column_sums_kernel<V, W>), grid, dim3(kThreads), 0, st, s, rows, n, cut.range); return; }
    PAM_COLUMN_SUMS(4, 16) PAM_COLUMN_SUMS(4, 8) PAM_COLUMN_SUMS(4, 4) PAM_COLUMN_SUMS(4, 2) PAM_COLUMN_SUMS(4, 1)
    PAM_COLUMN_SUMS(1, 4) PAM_COLUMN_SUMS(1, 2) PAM_COLUMN_SUMS(1, 1)
#undef PAM_COLUMN_SUMS
}

}  // namespace

extern "C" {

size_t pam_hip_column_sums_workspace_bytes(long rows, long n, int matrices)
{
    if (rows <= 0 || n <= 0 || matrices < 1 || matrices > 2) return 0;
    const Cut cut = cut_rows(rows, n);
    return cut.ranges > 1 ? (size_t)(cut.ranges * n) * matrices * sizeof(float) : 0;
}

int pam_hip_column_sums(const float* a, long a_row_stride, float* a_sums, const float* b, long b_row_stride, float* b_sums,
                        long rows, long n, void* workspace, size_t workspace_bytes, void* stream)
{
    if (rows < 0 || n < 0 || rows > (1L << 40) || n > (1L << 36)) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "column_sums: size out of range");
    if (n == 0) return PAM_HIP_OK;
    if (!a_sums || (rows > 0 && !a) || (b_sums && rows > 0 && !b)) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "column_sums: null pointer");
    const int matrices = b_sums ? 2 : 1;
    Sums s{{a, b}, {a_sums, b_sums}, {a_row_stride, b_row_stride}};
    const hipStream_t st = (hipStream_t)stream;
    if (rows == 0) { launch(s, matrices, 0, n, Cut{1, 1}, st); return pamhost::check_launch("column_sums"); }
    const Cut cut = cut_rows(rows, n);
    if (cut.ranges > 1) {
        const size_t need = (size_t)(cut.ranges * n) * matrices * sizeof(float);
        if (!workspace || workspace_bytes < need) return pamhost::fail(PAM_HIP_ERR_WORKSPACE, "column_sums: workspace of %zu bytes needed", need);
        float* part = (float*)workspace;
        Sums first = s;
        first.out[0] = part; first.out[1] = part + cut.ranges * n;
        launch(first, matrices, rows, n, cut, st);
        const int rc = pamhost::check_launch("column_sums");
        if (rc != PAM_HIP_OK) return rc;
        s.in[0] = first.out[0]; s.in[1] = first.out[1];
        s.row_stride[0] = s.row_stride[1] = n;
        launch(s, matrices, cut.ranges, n, Cut{cut.ranges, 1}, st);
    } else {
        launch(s, matrices, rows, n, cut, st);
    }
    return pamhost::check_launch("column_sums");
}

}  // extern "C"
