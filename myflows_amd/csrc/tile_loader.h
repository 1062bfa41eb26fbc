// The global-to-LDS tile loads of operands that are read with plain (not buffer) loads. Free of other
// headers, so that a host test can run the very loads against guarded memory.
#pragma once

namespace mfh {

// Four floats at any float's address (the hardware's 16-byte loads need 4-byte alignment only).
typedef float UnalignedQuad __attribute__((ext_vector_type(4), aligned(4)));

// A ROWS x COLS tile whose COLS dimension is contiguous in global memory (row stride ld), staged
// through registers in quads: load() issues the global reads, store() writes them to LDS. VEC: every
// row's start is 16-byte aligned and col_limit a multiple of 4. Otherwise (odd sizes) quads are read
// from wherever they start, and the quad across col_limit needs care:
//  * COLS along k: its terms past col_limit must be zeros, so its floats are read singly. Only the last
//    stage of a run of k has one.
//  * ROWS along k (ROWS_K): columns past col_limit only reach outputs that are not stored, so it may
//    hold the first floats of the next row, and its floats are read singly only in the last stage, whose
//    rows may have no next one.
// The single floats come after the quads, for the lanes that have none. As the other way of a branch
// around the quads they cost every stage of every tile: whichever of the two the compiler places second
// waits for all loads in flight before it fills the same registers.
// us a product on MI355X, single floats everywhere / in such a branch / as here: A^T B 1000 x 1001 over
// 3000 78.7 / 93.1 / 72.8, 2047 x 2047 over 1023 104.8 / 113.3 / 89.6, 3001 x 129 over 513 20.2 / 24.9 /
// 17.9; A B^T 1531 x 1000 over 777 42.7 / 39.0 / 38.9.
template <int ROWS, int COLS, int THREADS, bool VEC, bool ROWS_K>
struct TileLoader {
    static constexpr int ELEMS = ROWS * COLS / 4;
    static constexpr int PER_THREAD = (ELEMS + THREADS - 1) / THREADS;
    static constexpr int VCOLS = COLS / 4;
    static_assert(COLS % 4 == 0 && THREADS % VCOLS == 0, "whole quads per row, one column per thread");
    float4 v[PER_THREAD];

    // Reads the quads; true where this lane's floats are left for load_singles (same arguments).
    __device__ __forceinline__ bool load_quads(const float* __restrict__ base, int ld, int row0, int row_limit,
                                                int col0, int col_limit, int tid) {
        const int col = col0 + (tid % VCOLS) * 4;
        // Whether the tile has no quad to read singly. A quad that spills over ends at most three floats
        // past its row, and a row holds one at least: with four more rows there is always enough.
        // (Differences, not sums: a limit may be 2^31 - 1.)
        const bool whole = VEC || col_limit - col0 >= COLS || (ROWS_K && row_limit - row0 > ROWS + 3);
        const bool quad = VEC || (ROWS_K && whole) ? col < col_limit : col_limit - col > 3;
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
            const int f = tid + i * THREADS, row = row0 + f / VCOLS;
            float4 value = make_float4(0.f, 0.f, 0.f, 0.f);
            if (f < ELEMS && row < row_limit && quad) {
                const float* at = base + static_cast<long long>(row) * ld + col;
                if constexpr (VEC) {
                    value = *reinterpret_cast<const float4*>(at);
                } else {
                    const UnalignedQuad q = *reinterpret_cast<const UnalignedQuad*>(at);
                    value = make_float4(q.x, q.y, q.z, q.w);
                }
            }
            v[i] = value;
        }
        return !whole && !quad && col < col_limit;
    }

    __device__ __forceinline__ void load_singles(const float* __restrict__ base, int ld, int row0, int row_limit,
                                                  int col0, int col_limit, int tid) {
        const int col = col0 + (tid % VCOLS) * 4;
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
            const int f = tid + i * THREADS, row = row0 + f / VCOLS;
            const float* at = base + static_cast<long long>(row) * ld + col;
            float e[3] = {0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < 3; ++u)
                if (f < ELEMS && row < row_limit && u < col_limit - col) e[u] = at[u];
            v[i] = make_float4(e[0], e[1], e[2], 0.f);
        }
    }

    __device__ __forceinline__ void load(const float* __restrict__ base, int ld, int row0, int row_limit, int col0,
                                          int col_limit, int tid) {
        if (load_quads(base, ld, row0, row_limit, col0, col_limit, tid))
            load_singles(base, ld, row0, row_limit, col0, col_limit, tid);
    }

    template <int LD>
    __device__ __forceinline__ void store(float* lds, int tid) const {
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
            const int f = tid + i * THREADS;
            if (f < ELEMS) *reinterpret_cast<float4*>(lds + f / VCOLS * LD + f % VCOLS * 4) = v[i];
        }
    }
};

}  // namespace mfh
