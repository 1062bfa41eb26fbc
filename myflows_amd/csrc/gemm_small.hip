// Small FP32 products C(M x N) = op(A) op(B) (+ bias) (activation) on the matrix cores: one
// workgroup of SMALL_WAVES wave64s per 32 x 32 output tile, every wave on its own run of K.
//
// What bounds these products is latency, not the matrix cores: the LDS tiles of gemm.hip walk K in
// 16-deep stages with a barrier each, and a 100 x 130 output over K = 257 is six 64 x 64 tiles of
// nine stages (two groups of waves share them), 13.1 us against 6.6 here. Here a wave reads its operands straight into the MFMA's lanes
// (no LDS, no barrier, two 16-deep steps in flight), K is shared by eight waves of the same
// workgroup, and the eight partial tiles are added through LDS in wave order in FP64 and rounded
// once (the automatic plan split many of these products, and its slices are summed so): one launch,
// no workspace, each output summed in one fixed order.
#include <algorithm>

#include "common.h"
#include "gemm_core.h"

namespace mfh {
namespace {

constexpr int SMALL_TILE = 32, SMALL_WAVES = 8, SMALL_STEP = 16;
constexpr int SMALL_THREADS = SMALL_WAVES * 64;

// One operand's share of a 16-deep step. Lane l holds row (of op(A), or column of op(B)) l % 32 and,
// as MFMA s takes one k from either lane half, the terms k0 + (l / 32) * 8 + s, s = 0 .. 7. RUNS: the
// operand is contiguous along k, so a lane's eight terms are a run, two 16-byte loads wherever it
// starts, but in the step across k_end; otherwise it is contiguous along the rows and each load is
// one row of 32 lanes. Terms from k_end on are zeros and never read; a row past the last reads the
// last one, which only reaches outputs that are not stored.
template <bool RUNS>
struct SmallOperand {
    const float* base;
    int ld, k_half;
    float v[8];

    __device__ __forceinline__ void init(const float* p, int stride, int row, int rows, int lane) {
        ld = stride;
        k_half = (lane / 32) * 8;
        const int r = min(row + lane % 32, rows - 1);
        base = RUNS ? p + static_cast<long long>(r) * stride : p + r;
    }

    __device__ __forceinline__ void load(int k0, int k_end) {
        const int first = k0 + k_half;
        if (RUNS && k0 + SMALL_STEP <= k_end) {  // uniform over the wave
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const UnalignedQuad x = *reinterpret_cast<const UnalignedQuad*>(base + first + 4 * q);
                v[4 * q] = x.x;
                v[4 * q + 1] = x.y;
                v[4 * q + 2] = x.z;
                v[4 * q + 3] = x.w;
            }
            return;
        }
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int k = first + s;
            float x = 0.0f;
            if (k < k_end) x = base[RUNS ? static_cast<long long>(k) : static_cast<long long>(k) * ld];
            v[s] = x;
        }
    }
};

template <bool TA, bool TB>
__global__ __launch_bounds__(SMALL_THREADS) void gemm_small_kernel(GemmParams p) {
    __shared__ float partial[SMALL_WAVES][SMALL_TILE * SMALL_TILE];
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int m0 = blockIdx.y * SMALL_TILE, n0 = blockIdx.x * SMALL_TILE;
    const int k_begin = wave * p.k_chunk, k_end = min(p.K, k_begin + p.k_chunk);

    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    if (k_begin < k_end) {  // uniform over the wave
        SmallOperand<!TA> a[2];
        SmallOperand<TB> b[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            a[t].init(p.A, p.lda, m0, p.M, lane);
            b[t].init(p.B, p.ldb, n0, p.N, lane);
            a[t].load(k_begin + t * SMALL_STEP, k_end);
            b[t].load(k_begin + t * SMALL_STEP, k_end);
        }
        for (int k0 = k_begin; k0 < k_end; k0 += 2 * SMALL_STEP) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int s = 0; s < 8; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t].v[s], b[t].v[s], acc, 0, 0, 0);
                a[t].load(k0 + (t + 2) * SMALL_STEP, k_end);
                b[t].load(k0 + (t + 2) * SMALL_STEP, k_end);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r)
        partial[wave][(8 * (r / 4) + 4 * (lane / 32) + r % 4) * SMALL_TILE + lane % 32] = acc[r];
    __syncthreads();
#pragma unroll
    for (int i = threadIdx.x; i < SMALL_TILE * SMALL_TILE; i += SMALL_THREADS) {
        const int row = m0 + i / SMALL_TILE, col = n0 + i % SMALL_TILE;
        if (row >= p.M || col >= p.N) continue;
        // FP64, rounded once, as the reduction of a split plan adds its slices.
        double sum = static_cast<double>(partial[0][i]);
#pragma unroll
        for (int w = 1; w < SMALL_WAVES; ++w) sum += static_cast<double>(partial[w][i]);
        float v = static_cast<float>(sum);
        if (p.bias_mode == BIAS_COLUMN) v += p.bias[col];
        else if (p.bias_mode == BIAS_ROW) v += p.bias[row];
        write_output(p, p.C, row, col, activate(v, p.act, p.alpha));
    }
}

}  // namespace

// Where one launch of these tiles is the faster one (us on the GPU, gemm.hip's automatic plan / here, the
// slowest of the layouts): 64 x 10 over 16 6.2 / 4.2, 100 x 130 over 257 13.1 / 6.6, over 1000 17.8 /
// 11.3, 256 x 1000 over 512 17.3 / 8.0, 500 x 500 over 1000 19.1 / 12.5, 512 x 1000 over 257 12.4 / 10.2,
// over 512 16.6 / 12.6. A wave's serial run of K, and the operands' traffic (each 32 x 32 tile reads its
// rows and columns again) bound it: 128 x 128 over 2048 14.4 / 18.1 (split K), 1000 x 1000 over 512 17.2 /
// 21.9. The lines leave out sizes that would still gain, by layout: up to 256 tiles K to about 1500 (128 x
// 128 over 1280 16.3 / 13.1, over 1536 15.6 / 15.1), up to 512 tiles K to about 1000 (512 x 1000 over 640
// 19.2 / 16.7 and, B transposed, 20.9 / 15.3; over 1024 22.3 / 21.2 and 23.4 / 19.5).
bool gemm_takes_small(int M, int N, int K) {
    const std::int64_t tiles = static_cast<std::int64_t>(blocks_for(M, SMALL_TILE)) * blocks_for(N, SMALL_TILE);
    return M > 0 && N > 0 && K > 0 && K <= (tiles <= 256 ? 1024 : 512) && tiles <= 512;
}

int launch_gemm_small(GemmParams p, bool trans_a, bool trans_b, hipStream_t stream) {
    p.k_chunk = ((p.K + SMALL_WAVES - 1) / SMALL_WAVES + SMALL_STEP - 1) / SMALL_STEP * SMALL_STEP;  // whole steps
    const auto kernel = trans_a ? (trans_b ? gemm_small_kernel<true, true> : gemm_small_kernel<true, false>)
                                : (trans_b ? gemm_small_kernel<false, true> : gemm_small_kernel<false, false>);
    launch(kernel, dim3(blocks_for(p.N, SMALL_TILE), blocks_for(p.M, SMALL_TILE)), SMALL_THREADS, 0, stream, p);
    return MFH_CHECK_LAUNCH("gemm_small", stream);
}

}  // namespace mfh
