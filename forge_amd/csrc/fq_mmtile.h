// fq_mmtile.h -- row tiles of one or several matrices over the same tokens,
// shared by the prefill kernels (128 tokens x 256 rows per work-group, eight
// waves of 64 x 64).
//
// Several matrices in one launch share the token operands and fill the chip
// together (a 1024-row K or V matrix is four tiles), and the results need no
// pass of their own: a concatenated result is written at its columns, a
// gate/up pair is multiplied in the epilogue.  A work-group's tile never spans
// two matrices of a concatenation; in a pair it holds 128 gate rows and the
// same 128 up rows, so that lane c of a wave's row tiles j = 0 and 1 has gate
// and up of one row.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fq_kernels.h"

namespace fq {

// The row tile of work-group bx: its matrix, that matrix's rows, the tile's
// first row, and the matrix's first column in the result.
struct RowTile {
    const uint8_t* w;   // (MM_PAIR: the gate matrix)
    int rows, n0, col;
};
template <bool PAIR>
__device__ __forceinline__ RowTile row_tile(const MmqArgs& a, int bx, int bn) {
    if constexpr (PAIR) return RowTile{a.w, a.n1, bx * (bn / 2), 0};
    const int t1 = (a.n1 + bn - 1) / bn;
    if (a.mm == MM_ONE || bx < t1) return RowTile{a.w, a.n1, bx * bn, 0};
    const int t2 = (a.n2 + bn - 1) / bn;
    if (bx < t1 + t2) return RowTile{a.w2, a.n2, (bx - t1) * bn, a.n1};
    return RowTile{a.w3, a.n3, (bx - t1 - t2) * bn, a.n1 + a.n2};
}
// Work-groups along the rows
inline int row_tiles(const MmqArgs& a, int bn) {
    if (a.mm == MM_PAIR) return (a.n1 + bn / 2 - 1) / (bn / 2);
    int t = (a.n1 + bn - 1) / bn;
    if (a.mm == MM_CAT) t += (a.n2 + bn - 1) / bn + (a.n3 + bn - 1) / bn;
    return t;
}

__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// The results of a wave's two row tiles (acc[.][0], acc[.][1]) of 32 x 32
// tokens x rows: lane (c, g) holds column c of each, tokens 8 (e / 4) + 4 g +
// e % 4.  n: the lane's row of tile j = 0 within its matrix (PAIR: of both);
// split: the partial slab of split z.  EX: times 2^a.ex[token].
template <bool PAIR, bool EX, class V>
__device__ __forceinline__ void store_tiles(const MmqArgs& a, const RowTile& rt, int m, int n, int g,
                                            const V (&acc)[2], bool split, int z) {
    const int cols = PAIR ? 2 * a.N : a.N;
    float* const slab = split ? a.part + (size_t)z * a.M * cols : a.y;
    int ei[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) ei[e] = !EX ? 0 : a.ex[min(m + 8 * (e >> 2) + 4 * g + (e & 3), a.M - 1)];
    if constexpr (PAIR) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int t = m + 8 * (e >> 2) + 4 * g + (e & 3);
            if (t >= a.M || n >= rt.rows) continue;
            const float u = __builtin_amdgcn_ldexpf(acc[0][e], ei[e]);
            const float v = __builtin_amdgcn_ldexpf(acc[1][e], ei[e]);
            if (split) {
                slab[(size_t)t * cols + n] = u;
                slab[(size_t)t * cols + a.N + n] = v;
            } else {
                slab[(size_t)t * cols / 2 + n] = silu_mul(u, v);
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int nj = n + 32 * j;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int t = m + 8 * (e >> 2) + 4 * g + (e & 3);
                if (t >= a.M || nj >= rt.rows) continue;
                float v = __builtin_amdgcn_ldexpf(acc[j][e], ei[e]);
                if (!split) {
                    if (a.bias_mode == 1) v += nj < a.bias_len ? a.bias[nj] : 0.0f;
                    else if (a.bias_mode == 2) v += a.bias[(size_t)t * a.N + nj];
                }
                slab[(size_t)t * cols + rt.col + nj] = v;
            }
        }
    }
}

}  // namespace fq
