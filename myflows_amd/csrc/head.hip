// The network head and loss around the last convolution: the global average pool (forward and
// backward), the mean squared error (loss and gradient) and FP64 column sums (a Linear layer's
// bias gradient). Each repeats the float32 rounding steps of the operator it replaces, with the
// sums formed in FP64 in a fixed order, so every result is reproducible bit for bit:
//   * plane means y[p] = float(FP64 sum of x[p, 0..hw) / hw)              (mean in FP64, rounded once)
//   * their gradient dx[p, i] (+)= dy[p] / float(hw)                     (one float32 division)
//   * loss = float(FP64 sum of float32 (d * d) / count), d = pred - target (float32 difference and
//     square, as the operator's diff * diff)
//   * its gradient g[i] (+)= seed * ((2 * d) / float(count))             (float32, in that order)
//   * column sums out[j] = float(FP64 sum over rows of src[r, j]): in 1, 4 or 16 runs of rows, each in
//     order, then in run order.
#include <algorithm>
#include <cstdint>

#include "common.h"
#include "plane_walk.h"

namespace mfh {
namespace {

constexpr int HEAD_THREADS = 256;
constexpr int LOSS_THREADS = 1024;  // of a workgroup of the loss

// LANES lanes share a plane: lane l adds elements l, l + LANES, ... in FP64 (four loads in flight),
// then a fixed butterfly adds the lanes. One thread per plane read a cache line per lane and element
// and left all but planes / 64 waves idle: 64 x 64 planes of 29 x 39 took 327 us for 18.5 MB in a
// training pass, with 64 lanes 5.1.
template <int LANES>
__global__ __launch_bounds__(HEAD_THREADS) void plane_mean_kernel(const float* __restrict__ x, float* __restrict__ y,
                                                                  long long planes, int hw) {
    const long long p = (static_cast<long long>(blockIdx.x) * HEAD_THREADS + threadIdx.x) / LANES;
    if (p >= planes) return;  // uniform over the LANES lanes of a plane
    const int lane = threadIdx.x % LANES;
    const float* __restrict__ src = x + p * hw;
    double s = 0.0;
    walk_plane<LANES, 4>(
        lane, hw,
        [&](unsigned i) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = src[i + u * LANES];
#pragma unroll
            for (int u = 0; u < 4; ++u) s += static_cast<double>(v[u]);
        },
        [&](unsigned i) { s += static_cast<double>(src[i]); });
#pragma unroll
    for (int offset = LANES / 2; offset > 0; offset >>= 1) s += __shfl_xor(s, offset, LANES);
    if (lane == 0) y[p] = static_cast<float>(s / static_cast<double>(hw));
}

__global__ __launch_bounds__(HEAD_THREADS) void plane_mean_backward_kernel(const float* __restrict__ dy, float* dx,
                                                                           long long count, int hw, int add) {
#pragma clang fp contract(off)
    const long long i = static_cast<long long>(blockIdx.x) * HEAD_THREADS + threadIdx.x;
    if (i >= count) return;
    const float v = dy[i / hw] / static_cast<float>(hw);
    dx[i] = add ? dx[i] + v : v;
}

// Thread t of the grid adds the squares of elements t, t + threads, ... in that order in FP64, with
// LOSS_AHEAD loads of each operand in flight; a workgroup's thread sums are combined by a fixed tree in
// LDS. A single workgroup writes the loss; several write their sums to partials, which mse_finish_kernel
// adds. One workgroup with a load in flight took 70 us for 256 x 1000 elements in a training pass, a
// CU's own latency and bandwidth bounding it; 32 workgroups take 5.1 and the finish 2.7.
constexpr int LOSS_AHEAD = 8;
// A fixed cap, so that the order of the sum does not depend on the device; the finish reads one partial
// a thread.
constexpr int LOSS_GROUPS_MAX = 256;
static_assert(LOSS_GROUPS_MAX <= LOSS_THREADS, "mse_finish_kernel reads one partial per thread");

__device__ __forceinline__ double tree_sum(double* partial, double s) {
    partial[threadIdx.x] = s;
    __syncthreads();
    for (int half = LOSS_THREADS / 2; half > 0; half >>= 1) {
        if (static_cast<int>(threadIdx.x) < half) partial[threadIdx.x] += partial[threadIdx.x + half];
        __syncthreads();
    }
    return partial[0];
}

// The mean of no elements is NaN, as the operator's FP64 mean of an empty array.
__device__ __forceinline__ float mean_of(double sum, long long count) {
    return count > 0 ? static_cast<float>(sum / static_cast<double>(count)) : __builtin_nanf("");
}

__global__ __launch_bounds__(LOSS_THREADS) void mse_loss_kernel(const float* __restrict__ pred,
                                                                const float* __restrict__ target,
                                                                float* __restrict__ loss,
                                                                double* __restrict__ partials, long long count) {
#pragma clang fp contract(off)
    __shared__ double partial[LOSS_THREADS];
    const long long step = static_cast<long long>(gridDim.x) * LOSS_THREADS;
    long long i = static_cast<long long>(blockIdx.x) * LOSS_THREADS + threadIdx.x;
    double s = 0.0;
    for (; i + (LOSS_AHEAD - 1) * step < count; i += LOSS_AHEAD * step) {
        float p[LOSS_AHEAD], t[LOSS_AHEAD];
#pragma unroll
        for (int u = 0; u < LOSS_AHEAD; ++u) {
            p[u] = pred[i + u * step];
            t[u] = target[i + u * step];
        }
#pragma unroll
        for (int u = 0; u < LOSS_AHEAD; ++u) {
            const float d = p[u] - t[u];
            const float square = d * d;
            s += static_cast<double>(square);
        }
    }
    for (; i < count; i += step) {
        const float d = pred[i] - target[i];
        const float square = d * d;
        s += static_cast<double>(square);
    }
    const double sum = tree_sum(partial, s);
    if (threadIdx.x != 0) return;
    if (partials) partials[blockIdx.x] = sum;
    else loss[0] = mean_of(sum, count);
}

// The workgroups' sums (at most LOSS_GROUPS_MAX), added by the same tree.
__global__ __launch_bounds__(LOSS_THREADS) void mse_finish_kernel(const double* __restrict__ partials, int groups,
                                                                  float* __restrict__ loss, long long count) {
    __shared__ double partial[LOSS_THREADS];
    const double sum = tree_sum(partial, static_cast<int>(threadIdx.x) < groups ? partials[threadIdx.x] : 0.0);
    if (threadIdx.x == 0) loss[0] = mean_of(sum, count);
}

__global__ __launch_bounds__(HEAD_THREADS) void mse_grad_kernel(const float* __restrict__ pred,
                                                                const float* __restrict__ target,
                                                                const float* __restrict__ seed, float* grad,
                                                                long long count, float divisor, int add) {
#pragma clang fp contract(off)
    const long long i = static_cast<long long>(blockIdx.x) * HEAD_THREADS + threadIdx.x;
    if (i >= count) return;
    const float d = pred[i] - target[i];
    const float v = seed[0] * ((2.0f * d) / divisor);
    grad[i] = add ? grad[i] + v : v;
}

// A workgroup of SPAN columns by GROUPS row groups: group g adds its run of rows in order in FP64, eight
// loads in flight; the groups' sums are then added in group order through LDS.
template <int GROUPS, int SPAN>
__global__ __launch_bounds__(SPAN* GROUPS) void column_sums_kernel(const float* __restrict__ src,
                                                                   float* __restrict__ out, long long rows,
                                                                   long long cols) {
    __shared__ double group_sum[GROUPS][SPAN];
    const int c = threadIdx.x % SPAN, g = threadIdx.x / SPAN;
    const long long j = static_cast<long long>(blockIdx.x) * SPAN + c;
    const long long per = (rows + GROUPS - 1) / GROUPS;
    const long long last = min(rows, (g + 1) * per);
    double s = 0.0;
    if (j < cols) {
        long long r = g * per;
        for (; r + 8 <= last; r += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = src[(r + u) * cols + j];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += static_cast<double>(v[u]);
        }
        for (; r < last; ++r) s += static_cast<double>(src[r * cols + j]);
    }
    if constexpr (GROUPS > 1) {
        group_sum[g][c] = s;
        __syncthreads();
        if (g != 0) return;
#pragma unroll
        for (int h = 1; h < GROUPS; ++h) s += group_sum[h][c];
    }
    if (j < cols) out[j] = static_cast<float>(s);
}

}  // namespace

int launch_plane_mean(const float* x, float* y, std::int64_t planes, int hw, hipStream_t stream) {
    if (planes == 0) return OK;
    // A wave per plane from two full passes of it on; 16 lanes for the small planes of a network's end
    // (4 x 5, 7 x 7), of which a wave then takes four; one thread where 16 lanes would mostly idle. us for
    // 4096 planes by one thread each / as here: of 16 elements 3.4 / 2.1, of 49 7.5 / 2.4, of 127 17.4 /
    // 2.5, of 128 16.2 / 2.7, of 1131 148 / 4.1; for 32768 of 128, 17.0 / 6.9 (of 127 by 16 lanes 3.8).
    const auto run = [&](auto kernel, int lanes) {
        launch(kernel, blocks_for(planes * lanes, HEAD_THREADS), HEAD_THREADS, 0, stream, x, y, planes, hw);
    };
    if (hw >= 128) run(plane_mean_kernel<64>, 64);
    else if (hw >= 16) run(plane_mean_kernel<16>, 16);
    else run(plane_mean_kernel<1>, 1);
    return MFH_CHECK_LAUNCH("plane_mean", stream);
}

int launch_plane_mean_backward(const float* dy, float* dx, std::int64_t planes, int hw, bool add, hipStream_t stream) {
    const std::int64_t count = planes * hw;
    if (count == 0) return OK;
    launch(plane_mean_backward_kernel, blocks_for(count, HEAD_THREADS), HEAD_THREADS, 0, stream, dy, dx, count, hw,
                                                                                           add ? 1 : 0);
    return MFH_CHECK_LAUNCH("plane_mean_backward", stream);
}

// Workgroups of the loss of count elements: one while its loads are a few rounds (32768 elements 4.3 us,
// 6.0 before its loads were LOSS_AHEAD deep), as the finish is a second launch, else one per LOSS_AHEAD
// rounds up to LOSS_GROUPS_MAX (32769 elements 5.6 us, 65536 5.4 where one workgroup took 9.8).
int mse_loss_groups(std::int64_t count) {
    if (count <= 4LL * LOSS_AHEAD * LOSS_THREADS) return 1;
    return static_cast<int>(std::min<std::int64_t>(LOSS_GROUPS_MAX, blocks_for(count, LOSS_AHEAD * LOSS_THREADS)));
}

int launch_mse_loss(const float* pred, const float* target, float* loss, std::int64_t count, double* partials,
                    hipStream_t stream) {
    const int groups = partials ? mse_loss_groups(count) : 1;
    if (groups == 1) partials = nullptr;
    launch(mse_loss_kernel, groups, LOSS_THREADS, 0, stream, pred, target, loss, partials, count);
    MFH_TRY(MFH_CHECK_LAUNCH("mse_loss", stream));
    if (groups == 1) return OK;
    launch(mse_finish_kernel, 1, LOSS_THREADS, 0, stream, partials, groups, loss, count);
    return MFH_CHECK_LAUNCH("mse_finish", stream);
}

int launch_mse_grad(const float* pred, const float* target, const float* seed, float* grad, std::int64_t count,
                    bool add, hipStream_t stream) {
    if (count == 0) return OK;
    const float divisor = static_cast<float>(count > 0 ? count : 1);
    launch(mse_grad_kernel, blocks_for(count, HEAD_THREADS), HEAD_THREADS, 0, stream, pred, target, seed, grad, count,
                                                                                divisor, add ? 1 : 0);
    return MFH_CHECK_LAUNCH("mse_grad", stream);
}

int launch_column_sums(const float* src, float* out, std::int64_t rows, std::int64_t cols, hipStream_t stream) {
    if (cols == 0) return OK;
    // Few rows: one thread a column, whose loads are in flight in a few rounds (groups would leave most of
    // their block idle: 8 x 1000000 4.0 us, by 4 groups 9.6, by 16 26). More rows: a column's chain of loads
    // bounds it, and groups share it, 16 of them while the columns alone do not fill the GPU (256 x 1000
    // 6.4 us by one thread, 2.9 by 4 groups, 2.5 by 16; 2048 x 4096 44 / 12.5 / 7.1), 4 from 32769 columns
    // on (64 x 100000 4.5 / 3.2 / 7.1, 256 x 65536 14.1 / 11.0 / 10.8).
    const auto run = [&](auto kernel, int groups, int span) {
        launch(kernel, blocks_for(cols, span), groups * span, 0, stream, src, out, rows, cols);
    };
    const bool wide = cols > 32768;
    if (rows < (wide ? 64 : 48)) run(column_sums_kernel<1, 256>, 1, 256);
    else if (wide) run(column_sums_kernel<4, 64>, 4, 64);
    else run(column_sums_kernel<16, 64>, 16, 64);
    return MFH_CHECK_LAUNCH("column_sums", stream);
}

}  // namespace mfh
