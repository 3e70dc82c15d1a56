// Sums over the rows of a matrix (the gradients of biases and of layer_norm's parameters): ordinary float32 additions.
//
// Bound by memory, one read of the matrix.  A work-group of 256 lanes takes 64 columns of a range of rows: 16 lanes with
// 128-bit loads side by side (256 contiguous bytes of a row) and 16 rows at a time, eight loads in flight per lane, the
// sixteen lanes of a column added through LDS in a tree.  Where one range of rows would leave compute units without work
// the rows are cut into ranges of at least kLeastRows, whose sums go to the workspace and are added by the same kernel in
// a second launch.  Two matrices of one shape can be summed in one launch.
// Rounding: the eight loaded values are added as a tree and the trees' sums in a cascade, kChain at a time on each of
// kLevels levels, so that a value passes through fewer than 64 rounded additions at the sizes of a model's gradients and
// fewer than 100 in any matrix of up to 2^31 values, however long a lane's share of the rows is (many columns leave no
// work-groups to cut the rows for: 4096 rows of 131073 equal values near 1 in one chain per lane were off by 1.5e-5, now by
// less than 4e-6).  The order depends on the two sizes alone: not on a second matrix beside, nor on strides or alignment
// (128-bit loads at any float's address; n that are no multiple of four take one value per load).
// Measured against torch's sum over dim 0 (which also clears a buffer first, 5 us): a linear layer of 12608 x 192 -> 768 with
// its gradients 277 -> 266 us, 4096 x 512 -> 1024 375 -> 361.
#include <algorithm>
#include <cstdint>

#include "../../include/pam_hip_extra.h"
#include "pam_common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kColumns = 64;            // per work-group
constexpr long kLeastRows = 128;        // per range
constexpr long kMostGroups = 2048;      // work-groups per matrix of a launch that cuts the rows: eight per compute unit
constexpr int kChain = 16, kLevels = 4;

struct Sums { const float* in[2]; float* out[2]; long row_stride[2]; };

// VEC: values per lane and load.  Work-group (x, y, z): columns x * 64 ..., range y of the rows, matrix z; the sums of
// range y go to out[z] + y * n.
template <int VEC>
__global__ __launch_bounds__(kThreads) void column_sums_kernel(Sums s, long rows, long n, long range)
{
    constexpr int kWide = kColumns / VEC, kDeep = kThreads / kWide;
    constexpr int kFlight = 8;
    typedef float vec __attribute__((ext_vector_type(VEC)));
    typedef float vec_any __attribute__((ext_vector_type(VEC), aligned(4)));
    __shared__ __attribute__((aligned(16))) float part[kDeep][kColumns];
    const int tx = threadIdx.x % kWide, ty = threadIdx.x / kWide;
    const long column = (long)blockIdx.x * kColumns + tx * VEC;
    const long first = (long)blockIdx.y * range, last = min(rows, first + range);
    const bool inside = column + VEC <= n;          // (VEC = 4 takes only n that are multiples of four)
    const float* at = s.in[blockIdx.z] + (inside ? column : 0);
    const long stride = s.row_stride[blockIdx.z];
    vec level[kLevels] = {};
    unsigned trees = 0;
    long r = first + ty;
    for (; r + (kFlight - 1) * kDeep < last; r += kFlight * kDeep) {
        vec v[kFlight];
#pragma unroll
        for (int u = 0; u < kFlight; ++u) v[u] = *reinterpret_cast<const vec_any*>(at + (r + u * kDeep) * stride);
        level[0] += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        ++trees;
        unsigned whole = kChain;
#pragma unroll
        for (int l = 0; l + 1 < kLevels; ++l, whole *= kChain)
            if (trees % whole == 0) { level[l + 1] += level[l]; level[l] = 0.0f; }
    }
    vec total = 0.0f;
    for (; r < last; r += kDeep) total += *reinterpret_cast<const vec_any*>(at + r * stride);
#pragma unroll
    for (int l = 0; l < kLevels; ++l) total += level[l];
    *reinterpret_cast<vec*>(&part[ty][tx * VEC]) = total;
    for (int half = kDeep / 2; half >= 1; half /= 2) {
        __syncthreads();
        for (int i = threadIdx.x; i < half * kColumns; i += kThreads) part[i / kColumns][i % kColumns] += part[i / kColumns + half][i % kColumns];
    }
    __syncthreads();
    if (threadIdx.x < kColumns) {
        const long c = (long)blockIdx.x * kColumns + threadIdx.x;
        if (c < n) s.out[blockIdx.z][(long)blockIdx.y * n + c] = part[0][threadIdx.x];
    }
}

// rows per range and number of ranges
struct Cut { long range, ranges; };
Cut cut_rows(long rows, long n)
{
    const long groups = (n + kColumns - 1) / kColumns;
    const long most = std::max(1L, std::min({rows / kLeastRows, kMostGroups / groups, 65535L}));
    const long range = (rows + most - 1) / most;
    return Cut{range, (rows + range - 1) / range};
}

void launch(const Sums& s, int matrices, long rows, long n, const Cut& cut, hipStream_t st)
{
    const dim3 grid((unsigned)((n + kColumns - 1) / kColumns), (unsigned)cut.ranges, (unsigned)matrices);
    if (n % 4 == 0) hipLaunchKernelGGL(column_sums_kernel<4>, grid, dim3(kThreads), 0, st, s, rows, n, cut.range);
    else hipLaunchKernelGGL(column_sums_kernel<1>, grid, dim3(kThreads), 0, st, s, rows, n, cut.range);
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
