// fq_dequant.hip -- the bit-exact dequant kernel (fq_dequant_rows) and small
// elementwise kernels: a fill kernel used instead of memset nodes (so callers
// may capture it) and the SiLU-multiply of the fused FFN.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "fq_formats.h"
#include "fq_kernels.h"
#include "fq_mmtile.h"

namespace fq {

// Dequantize.  The kernel writes 4 bytes per weight and reads 0.4 to 1.1, so
// the stores bound it: a wave owns a chunk of 256 consecutive elements of one
// row and each lane four consecutive ones, stored as one 16-byte piece, so a
// store instruction covers 1 KiB of contiguous bytes.  14336 x 4096 Q4_K:
// 40 us, 6.7 TB/s, the rate of a plain fill (one thread per 32-weight unit,
// each storing its 32 values 4 bytes at a time: 260 us).  A quad's codes lie in one dword (or byte
// run) of its block; the block's scales are read by every lane of the block
// and come from the cache.
//
// Quad<F>::get: elements 4 j .. 4 j + 3 of a row, bit-identical to the
// reference's row routines (scalar fp16 conversion f16_ref, the reference's
// expression order).
template <int F>
struct Quad;

__device__ __forceinline__ float byte_f(uint32_t w, int b) {
    return (float)((w >> (8 * b)) & 0xFFu);
}

// nibble formats: elements 0..15 of a block are the low nibbles of qs[16],
// 16..31 the high ones
__device__ __forceinline__ uint32_t nib4(const uint8_t* qs, int e) {
    return (ld_u32(qs + (e & 15)) >> (e < 16 ? 0 : 4)) & 0x0F0F0F0Fu;
}

template <>
struct Quad<Q4_0> {  // w = (q - 8) d
    __device__ static void get(const uint8_t* row, int j, float* v) {
        const uint8_t* p = row + 18 * (j >> 3);
        const uint32_t q = nib4(p + 2, 4 * (j & 7));
        const float d = f16_ref(ld_u16(p));
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = (byte_f(q, b) - 8.0f) * d;
    }
};
template <>
struct Quad<Q4_1> {  // w = q d + m (q d is exact: the fused form rounds as the sum does)
    __device__ static void get(const uint8_t* row, int j, float* v) {
        const uint8_t* p = row + 20 * (j >> 3);
        const uint32_t q = nib4(p + 4, 4 * (j & 7)), dm = ld_u32(p);
        const float d = f16_ref(dm & 0xFFFFu), m = f16_ref(dm >> 16);
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = __builtin_fmaf(byte_f(q, b), d, m);
    }
};
template <>
struct Quad<Q8_0> {  // w = q d
    __device__ static void get(const uint8_t* row, int j, float* v) {
        const uint8_t* p = row + 34 * (j >> 3);
        const uint32_t q = ld_u32(p + 2 + 4 * (j & 7)) ^ 0x80808080u;
        const float d = f16_ref(ld_u16(p));
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = (byte_f(q, b) - 128.0f) * d;
    }
};
template <>
struct Quad<Q5_0> {  // w = (q - 16) d
    __device__ static void get(const uint8_t* row, int j, float* v) {
        const uint8_t* p = row + 22 * (j >> 3);
        const int e = 4 * (j & 7);
        const uint32_t q = five_bit(nib4(p + 6, e), ld_u32(p + 2) >> e);
        const float d = f16_ref(ld_u16(p));
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = (byte_f(q, b) - 16.0f) * d;
    }
};
template <>
struct Quad<Q5_1> {  // w = q d + m (exact product, as Q4_1)
    __device__ static void get(const uint8_t* row, int j, float* v) {
        const uint8_t* p = row + 24 * (j >> 3);
        const int e = 4 * (j & 7);
        const uint32_t q = five_bit(nib4(p + 8, e), ld_u32(p + 4) >> e), dm = ld_u32(p);
        const float d = f16_ref(dm & 0xFFFFu), m = f16_ref(dm >> 16);
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = __builtin_fmaf(byte_f(q, b), d, m);
    }
};
template <>
struct Quad<IQ4_NL> {  // w = d T[q]
    __device__ static void get(const uint8_t* row, int j, float* v) {
        const uint8_t* p = row + 18 * (j >> 3);
        const uint32_t t = iq4_lookup(nib4(p + 2, 4 * (j & 7)));
        const float d = f16_ref(ld_u16(p));
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = d * (float)(int8_t)(t >> (8 * b));
    }
};

// Q4_K / Q5_K: w = (d sc) q - dmin m; (d sc) q is exact (11 + 6 + 5 bits), so
// the fused form rounds as the difference does.  Sub-block e / 32 of the
// super-block, its pair e / 64 sharing the 32 qs bytes.
template <int F>
struct QuadK {
    __device__ static void get(const uint8_t* row, int j, float* v) {
        const uint8_t* p = row + Fmt<F>::BB * (j >> 6);
        const int e = 4 * (j & 63), g = e >> 6, h = (e >> 5) & 1, l = e & 31;
        const uint4 hdr = ld_u128(p);
        uint32_t q = (ld_u32(p + (F == Q5_K ? 48 : 16) + 32 * g + l) >> (4 * h)) & 0x0F0F0F0Fu;
        if constexpr (F == Q5_K)
            q |= ((ld_u32(p + 16 + l) >> (2 * g + h)) & 0x01010101u) << 4;
        uint32_t sa, ma, sb, mb;
        Fmt<Q4_K>::scale_min(hdr, g, sa, ma, sb, mb);
        const float A = f16_ref(hdr.x & 0xFFFFu) * (float)(h ? sb : sa);
        const float B = -(f16_ref(hdr.x >> 16) * (float)(h ? mb : ma));
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = __builtin_fmaf(A, byte_f(q, b), B);
    }
};
template <>
struct Quad<Q4_K> : QuadK<Q4_K> {};
template <>
struct Quad<Q5_K> : QuadK<Q5_K> {};

// Q6_K: element 128 n + 32 u + l is nibble u / 2 of ql[64 n + 32 (u % 2) + l]
// with bits 2 u .. of qh[32 n + l]; w = (d sc)(q - 32), d sc exact.
template <>
struct Quad<Q6_K> {
    __device__ static void get(const uint8_t* row, int j, float* v) {
        const uint8_t* p = row + 210 * (j >> 6);
        const int e = 4 * (j & 63), n = e >> 7, u = (e >> 5) & 3, l = e & 31;
        const uint32_t lo = ld_u32(p + 64 * n + 32 * (u & 1) + l) >> (4 * (u >> 1));
        const uint32_t hi = ld_u32(p + 128 + 32 * n + l) >> (2 * u);
        const uint32_t q = (lo & 0x0F0F0F0Fu) | ((hi & 0x03030303u) << 4);
        const float A = f16_ref(ld_u16(p + 208)) * (float)(int8_t)p[192 + (e >> 4)];
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = A * (byte_f(q, b) - 32.0f);
    }
};
// Q3_K: element 128 n + 32 u + l: bits 2 u .. of qs[32 n + l], plus 4 where
// bit 4 n + u of hmask[l] is set; w = (d (sc - 32))(q - 4).
template <>
struct Quad<Q3_K> {
    __device__ static void get(const uint8_t* row, int j, float* v) {
        const uint8_t* p = row + 110 * (j >> 6);
        const int e = 4 * (j & 63), n = e >> 7, u = (e >> 5) & 3, l = e & 31, i = e >> 4;
        const uint32_t q = ((ld_u32(p + 32 + 32 * n + l) >> (2 * u)) & 0x03030303u) |
                           (((ld_u32(p + l) >> (4 * n + u)) & 0x01010101u) << 2);
        const uint32_t lo = (p[96 + (i & 7)] >> (4 * (i >> 3))) & 15u;
        const uint32_t hi = (p[104 + (i & 3)] >> (2 * (i >> 2))) & 3u;
        const float A = f16_ref(ld_u16(p + 108)) * (float)((int)(lo | (hi << 4)) - 32);
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = A * (byte_f(q, b) - 4.0f);
    }
};

// CH chunks of a wave per iteration, so that their loads are in flight
// together.  K need not be a multiple of 4 or of the block: the last quad of
// a row is cut (its codes lie inside the row's last whole block), and rows
// that are not whole 16-byte pieces are stored value by value.
constexpr int CH = 4;
// chunks per row (K up to the largest int)
__host__ __device__ inline int dequant_chunks(int K) { return K / 256 + (K % 256 != 0); }
template <int F>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ w,
                                                      float* __restrict__ out, int N, int K,
                                                      int row_bytes, int vec) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int cpr = dequant_chunks(K);
    const int64_t total = (int64_t)N * cpr, stride = (int64_t)gridDim.x * 4 * CH;
    for (int64_t c0 = ((int64_t)blockIdx.x * 4 + wave) * CH; c0 < total; c0 += stride) {
        int64_t row = c0 / cpr;
        int c = (int)(c0 - row * cpr);
        float v[CH][4];
        int64_t at[CH];
        int k[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            k[i] = row < N ? 256 * c + 4 * lane : K;
            at[i] = row * K + k[i];
            if (k[i] < K) Quad<F>::get(w + row * row_bytes, k[i] >> 2, v[i]);
            if (++c == cpr) {
                c = 0;
                ++row;
            }
        }
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            if (k[i] >= K) continue;
            float* o = out + at[i];
            if (vec) {
                typedef float f32x4 __attribute__((ext_vector_type(4)));
                __builtin_nontemporal_store(f32x4{v[i][0], v[i][1], v[i][2], v[i][3]},
                                            reinterpret_cast<f32x4*>(o));
            } else {
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    if (k[i] + b < K) o[b] = v[i][b];
            }
        }
    }
}

// Clears n words.
__global__ __launch_bounds__(256) void zero_kernel(uint32_t* p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        p[i] = 0u;
}

// y = silu(gate) * up = gate / (1 + exp(-gate)) * up, as the reference's
// silu_multiply (src/operators/cpu/elementwise.cpp:89-150).
__global__ __launch_bounds__(256) void silu_mul_kernel(const float* __restrict__ gate,
                                                       const float* __restrict__ up,
                                                       float* __restrict__ y, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        y[i] = silu_mul(gate[i], up[i]);
    }
}

hipError_t launch_silu_mul(const float* gate, const float* up, float* y, size_t n, int cus,
                           hipStream_t st) {
    const size_t want = (n + 255) / 256, cap = (size_t)cus * 8;
    hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)(want < cap ? want : cap)), dim3(256), 0, st,
                       gate, up, y, n);
    return hipGetLastError();
}

// y[m][off + n] = src[m][n]: places one matrix's outputs into the
// concatenated rows of a fused QKV result.
__global__ __launch_bounds__(256) void copy_cols_kernel(const float* __restrict__ src,
                                                        float* __restrict__ y, int M, int n_src,
                                                        int ld, int off) {
    const size_t total = (size_t)M * n_src;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total;
         i += (size_t)gridDim.x * 256) {
        const int m = (int)(i / n_src), n = (int)(i % n_src);
        y[(size_t)m * ld + off + n] = src[i];
    }
}

hipError_t launch_copy_cols(const float* src, float* y, int M, int n_src, int ld, int off, int cus,
                            hipStream_t st) {
    const size_t want = ((size_t)M * n_src + 255) / 256, cap = (size_t)cus * 8;
    hipLaunchKernelGGL(copy_cols_kernel, dim3((unsigned)(want < cap ? want : cap)), dim3(256), 0,
                       st, src, y, M, n_src, ld, off);
    return hipGetLastError();
}

hipError_t launch_zero(uint32_t* p, size_t n, int grid, hipStream_t st) {
    hipLaunchKernelGGL(zero_kernel, dim3(grid), dim3(256), 0, st, p, n);
    return hipGetLastError();
}

hipError_t launch_dequant(int dtype, const uint8_t* w, float* out, int N, int K, int row_bytes,
                          int cus, hipStream_t st) {
    // whole 16-byte pieces: every row then starts on one
    const int vec = K % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    const int64_t chunks = (int64_t)N * dequant_chunks(K);
    const int grid = (int)std::min<int64_t>((chunks + 4 * CH - 1) / (4 * CH), (int64_t)cus * 32);
    return with_format(dtype, hipErrorInvalidValue, [&](auto f) {
        hipLaunchKernelGGL(dequant_kernel<decltype(f)::value>, dim3(grid), dim3(256), 0, st, w,
                           out, N, K, row_bytes, vec);
        return hipGetLastError();
    });
}

}  // namespace fq
