// fq_mmqk.hip -- prefill (M > 32 tokens) for Q4_K and Q5_K on
// v_mfma_f32_32x32x16_f16, the sub-block scales inside the weight operand.
//
// A weight of these formats is d (sc q) - dmin m with 6-bit integers sc, m per
// 32-element sub-block and fp16 d, dmin per 256-element super-block.  With c
// the middle of the code range (8, Q5_K: 16), sc (q - c) is at most 1008 in
// magnitude, exact in fp16, so the B operand holds sc (q - c) and one chain of
// MFMAs runs over a whole super-block:
//
//   D   = sum over the super-block of (x_hi + x_lo) sc (q - c)   (fp32, 32
//         MFMAs per 32 x 32 tile) + c sum over its sub-blocks of S sc, S the
//         token's sub-block sums as fp16 hi + lo (one MFMA: 16 slots)
//   Dm  = sum over its sub-blocks of S m                       (one MFMA)
//   acc += 2^e (d D - dmin Dm)                       (three per output)
//
// with x 2^-e as x_hi + x_lo, e the token's exponent.  S's low part is kept 2^12
// larger and meets weights 2^12 smaller, exact in fp16: it keeps its bits down to
// 2^-29 of the token's largest, where fp16's least value alone ends at 2^-17.
// Q5_K (FINE), whose tokens had an exponent per 64 elements in the fp16 MFMA
// kernel, has one per super-block, and x_lo kept in the same way (xprepk_kernel;
// its fold, acc += 2^e (..), costs 2 to 3 %: Q4_K 3584 -> 18944 pair, M = 1999,
// 1125 -> 1157 us).
//
// (codes about zero keep the chain's partial sums small: with q as it stands
// the result's error against 64 bits was 40 % larger, 3.2e-7 at K = 4096)
//
// against one FMA per output and 32-element block and an fp32 MFMA per 64
// elements for the minimum.  A loop of nothing but v_mfma_f32_32x32x16_f16 runs
// at 2.49 PFLOP/s on zeros with one wave per SIMD, 1.64 on random operands, and
// with two waves, as here, at 1.66 and 1.21: the rate falls with what the
// operands and the waves cost in power, and 128 FMAs and 16 LDS reads beside each
// 32 MFMAs took a fifth of it.  This kernel reaches 0.93 with its matrix cores
// busy 55 % of the cycles, so every vector instruction taken out of a step
// counts, also where it would have overlapped a matrix instruction.
// The multiply by sc replaces the subtract that removes the 1024 of the
// byte-to-half trick: with the code in the top bits of its byte the half reads
// 1024 + 16 q (Q5_K 1024 + 8 q), and (1024 + 16 q) (sc / 16) - 72 sc =
// sc (q - 8) is one packed FMA whose operands and result are exact (72 sc =
// 9 * 63 * 8 at most: 10 bits).
//
// Measured (whole calls): Q4_K 3584 -> 18944, M = 1999 698 -> 595 us; 4096 ->
// 14336, M = 512 170 -> 134; Q5_K, which had no such kernel, 4096 -> 14336 at
// M = 77 101 -> 44, M = 512 149; Q4_K error against 64 bits 2.0e-7 (3.2e-7).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fq_dma.h"
#include "fq_formats.h"
#include "fq_kernels.h"
#include "fq_mfma16.h"
#include "fq_mmtile.h"

namespace fq {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int BMT = 128, BNT = 256;  // tokens, rows per work-group
constexpr int KS = 64;               // K elements per step: one sub-block pair
constexpr int XT = 1024;             // halves per (32-token tile, 16-k quarter): hi then lo
constexpr int NBUF = 3;              // buffers of a step's operands: steps s, s + 1, s + 2
constexpr int NW = 8;                // waves per work-group
constexpr int SEXP = 1024;           // bytes of a tile's sub-block sums: [hi, lo][token][sub-block]
constexpr int STILE_FINE = SEXP + 128;  // and 2^e of its tokens
constexpr float LO = 0x1p12f;        // what the kept low parts are larger by

// ------------------------------------------------------------- token prep
// FINE: the A operand as xprep4_kernel lays it out, an exponent per token and
// super-block.  A work-group is a tile and super-block, a wave four of
// its tokens: lane t + 4 j has pieces (2 kq + g = j and j + 16) of token t, so that
// four lanes write one 64-byte run and the exponent and the sums need no barrier.
__global__ __launch_bounds__(512) void xprepk_kernel(const float* __restrict__ x, int M, int K,
                                                     _Float16* __restrict__ xop,
                                                     uint8_t* __restrict__ xs) {
    const int lane = threadIdx.x & 63, t = lane & 3, j = lane >> 2;
    const int sb = blockIdx.x, T = blockIdx.y, lm = 4 * (threadIdx.x >> 6) + t, m = 32 * T + lm;
    float v[2][8] = {};
    float mx = 0.0f;
    if (m < M) {
        const float* const xr = x + (size_t)m * K + 256 * sb;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int gq = j + 16 * i;
            const float* s = xr + 32 * (gq >> 2) + 16 * (gq & 1) + 8 * ((gq >> 1) & 1);
            const float4 a = *reinterpret_cast<const float4*>(s), b = *reinterpret_cast<const float4*>(s + 4);
            const float u[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                v[i][k] = u[k];
                mx = fmaxf(mx, fabsf(u[k]));
            }
        }
    }
#pragma unroll
    for (int o = 4; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    // (2^e a normal number)
    const int e = (mx > 0.0f && mx <= 3.0e38f) ? max(ilogbf(mx) - 14, -126) : 0;
    uint8_t* const sbk = xs + ((size_t)T * (K / 256) + sb) * STILE_FINE;
    if (j == 0) *reinterpret_cast<float*>(sbk + SEXP + 4 * lm) = __builtin_amdgcn_ldexpf(1.0f, e);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int gq = j + 16 * i;
        float w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = __builtin_amdgcn_ldexpf(v[i][k], -e);
        h8 hi, lo;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float u = w[slot_elem(k)];
            hi[k] = (_Float16)u;
            lo[k] = (_Float16)((u - (float)hi[k]) * LO);
        }
        _Float16* const dst = xop + ((size_t)T * (K / 16) + 16 * sb + (gq >> 1)) * XT + (lm + 32 * (gq & 1)) * 8;
        *reinterpret_cast<h8*>(dst) = hi;
        *reinterpret_cast<h8*>(dst + 512) = lo;
        // the sum over sub-block gq / 4: four pieces, times 2^-5 (below 2^15)
        float s = ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
        s += __shfl_xor(s, 4, 64);
        s += __shfl_xor(s, 8, 64);
        if ((gq & 3) == 0) {
            s *= 0x1p-5f;
            const _Float16 h = (_Float16)s;
            _Float16* const d = reinterpret_cast<_Float16*>(sbk) + lm * 8 + (gq >> 2);
            d[0] = h;
            d[256] = (_Float16)((s - (float)h) * LO);
        }
    }
}

// Super-block layout: header (d dmin scales[12]) @0, Q5_K: qh[32] @16, then
// qs[128].  The header and qh are copied once per super-block as HP planes of
// one 16-byte chunk per row, a step's 32 code bytes as two.
template <int F>
struct KQ {
    static constexpr int BB = F == Q5_K ? 176 : 144;
    static constexpr int HP = F == Q5_K ? 3 : 1;
    static constexpr int QOFF = 16 * HP;
    static constexpr float UNIT = F == Q5_K ? 8.0f : 16.0f;  // value of a code step in the half
    static constexpr float MID = F == Q5_K ? 16.0f : 8.0f;   // c
    static constexpr bool FINE = F == Q5_K;
    static constexpr int STILE = FINE ? STILE_FINE : SEXP;
    // LDS: token operands, code planes (NBUF each), super-block planes, sums (2 each)
    static constexpr int XBUF = 16 * XT * 2;
    static constexpr int QBUF = 2 * BNT * 16;
    static constexpr int HBUF = HP * BNT * 16;
    static constexpr int SBUF = 4 * STILE;
    static constexpr int LDS = NBUF * (XBUF + QBUF) + 2 * (HBUF + SBUF);
    // copy instructions per wave: every step, and more with a super-block's first
    static constexpr int CS = 4 + 1;
    static constexpr int CB = (HP + 1) / 2 + 1;
    static_assert(LDS <= 160 * 1024, "LDS");
};

// Byte J of the scale bytes (dwords y, z, w of the header): 6-bit scale and
// minimum of sub-block b (get_scale_min_k4, matmul.cpp:232-240).
__device__ __forceinline__ uint32_t sub_scale(const fq_u32x4& h, int b) {
    if (b < 4) return (h.y >> (8 * b)) & 63u;
    return ((h.w >> (8 * (b - 4))) & 15u) | (((h.y >> (8 * (b - 4) + 6)) & 3u) << 4);
}
__device__ __forceinline__ uint32_t sub_min(const fq_u32x4& h, int b) {
    if (b < 4) return (h.z >> (8 * b)) & 63u;
    return ((h.w >> (8 * (b - 4) + 4)) & 15u) | (((h.z >> (8 * (b - 4) + 6)) & 3u) << 4);
}

// The four codes of w (top bits of its bytes) as slots 0..3: sc (q - c), with
// sc / 16 (Q5_K: / 8) in s and -72 sc (-144 sc) in off
__device__ __forceinline__ void scaled_pairs(uint32_t w, h2 s, h2 off, h2& p0, h2& p1) {
    p0 = __builtin_elementwise_fma(
        __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w, 0x04020400u)), s, off);
    p1 = __builtin_elementwise_fma(
        __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w, 0x04030401u)), s, off);
}
__device__ __forceinline__ h8 scaled8(uint32_t w0, uint32_t w1, h2 s, h2 off) {
    h2 a, b, c, d;
    scaled_pairs(w0, s, off, a, b);
    scaled_pairs(w1, s, off, c, d);
    return h8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

__device__ __forceinline__ fq_u32x4 lds16(const uint8_t* p) {
    typedef const __attribute__((address_space(3))) fq_u32x4* lds_v4;
    return *reinterpret_cast<lds_v4>(reinterpret_cast<uintptr_t>(p));
}

// A work-group owns 128 tokens x 256 rows and a K range of whole super-blocks
// (split-K when that shortens the busiest CU's work).  Eight waves, each 64
// tokens x 64 rows (2 x 2 tiles of 32 x 32), tokens as the A operand
// (xprep4_kernel, xprepk_kernel), weights as B, so that a
// lane's 16 results of a tile belong to one row and d, dmin are one value per
// lane.  All operands reach LDS by direct copies, three buffers deep for a
// step's, two for a super-block's; one barrier per step publishes step s and
// frees the buffers that step s + 2 refills.
template <int F, bool PAIR>
__global__ __launch_bounds__(512) void mmqk_kernel(MmqArgs a, int steps_per_split) {
    using Q = KQ<F>;
    constexpr int STILE = Q::STILE;
    constexpr int RJ = PAIR ? BNT / 2 : 32;  // tile rows between a wave's two row tiles
    __shared__ __attribute__((aligned(16))) uint8_t lds[Q::LDS];
    uint8_t* const xs0 = lds;
    uint8_t* const qs0 = xs0 + NBUF * Q::XBUF;
    uint8_t* const hs0 = qs0 + NBUF * Q::QBUF;
    uint8_t* const ss0 = hs0 + 2 * Q::HBUF;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;  // 64-token / 64-row quadrant
    const RowTile rt = row_tile<PAIR>(a, blockIdx.x, BNT);
    const int m0 = blockIdx.y * BMT;
    const int nsteps = a.K / KS;
    const int s0 = blockIdx.z * steps_per_split, s1 = min(nsteps, s0 + steps_per_split);
    const int Tn = (a.M + 31) / 32;
    const int KQ16 = a.K / 16, NSB = a.K / 256;

    // copy sources: token run (tile wave / 2, half wave & 1 of its 8 KiB per
    // step), 64 rows of code plane wave / 4, half the sums of tile wave / 2
    const int T = min(m0 / 32 + (wave >> 1), Tn - 1);
    const uint8_t* const xbase =
        reinterpret_cast<const uint8_t*>(a.xop) + ((size_t)T * KQ16 * XT) * 2 + (wave & 1) * 4096;
    const uint8_t* const sbase =
        reinterpret_cast<const uint8_t*>(a.xsum) + (size_t)T * NSB * STILE + (wave & 1) * (STILE / 2);
    // tile row r is row r % 128 of the gate (r < 128) or up matrix of a pair
    auto row_off = [&](int r) {
        return (uint32_t)min(rt.n0 + (PAIR ? r & (BNT / 2 - 1) : r), rt.rows - 1) *
               (uint32_t)a.row_bytes;
    };
    auto row_base = [&](int r) { return PAIR && r >= BNT / 2 ? a.w2 : rt.w; };  // wave-uniform r
    const uint32_t qoff = row_off(64 * (wave & 3) + lane) + Q::QOFF + 16 * (wave >> 2);
    const uint8_t* const qbase = row_base(64 * (wave & 3));
    // super-block planes: 64 rows of planes 2 q and 2 q + 1 each (all eight
    // waves), 32 rows of an odd last plane
    constexpr int HR = (Q::HP + 1) / 2;
    uint32_t hoff[HR];
    const uint8_t* hbase[HR];
#pragma unroll
    for (int q = 0; q < HR; ++q) {
        const bool half = 2 * q + 1 == Q::HP;
        const int r0 = half ? 32 * wave : 64 * (wave & 3), pl = half ? 2 * q : 2 * q + (wave >> 2);
        hoff[q] = row_off(min(r0 + lane, BNT - 1)) + 16 * pl;
        hbase[q] = row_base(r0);
    }
    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds);
    auto issue = [&](int s, bool first) __attribute__((always_inline)) {  // first: s is its super-block's first step
        const int buf = s % NBUF, sb = s >> 2;
        const uint32_t xl = lds_base + buf * Q::XBUF + wave * 4096;
        const uint8_t* xg = xbase + (size_t)s * 4 * XT * 2;
#pragma unroll
        for (int i = 0; i < 4; ++i) dma16s(16 * lane + 1024 * i, xg, xl + 1024 * i);
        const size_t wsb = (size_t)sb * Q::BB;
        dma16s(qoff, qbase + wsb + 32 * (s & 3), lds_base + NBUF * Q::XBUF + buf * Q::QBUF + wave * 1024);
        if (first) {
            const uint32_t hl = lds_base + NBUF * (Q::XBUF + Q::QBUF) + (sb & 1) * Q::HBUF;
#pragma unroll
            for (int q = 0; q < HR; ++q) {
                if (2 * q + 1 < Q::HP) dma16s(hoff[q], hbase[q] + wsb, hl + 8192 * q + 1024 * wave);
                else if (lane < 32) dma16s(hoff[q], hbase[q] + wsb, hl + 8192 * q + 512 * wave);
            }
            if (lane < STILE / 32)
                dma16s(16 * lane, sbase + (size_t)sb * STILE,
                       lds_base + NBUF * (Q::XBUF + Q::QBUF) + 2 * Q::HBUF + (sb & 1) * Q::SBUF +
                           wave * (STILE / 2));
        }
    };

    f32x16 acc[2][2], D[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    const int g = lane >> 5, c = lane & 31;
    auto read_a = [&](const _Float16* xs, int b, int i, h8 (&r)[4]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const _Float16* xp = xs + ((2 * wm + i) * 4 + 2 * b + h) * XT + lane * 8;
            r[2 * h] = *reinterpret_cast<const h8*>(xp);
            r[2 * h + 1] = *reinterpret_cast<const h8*>(xp + 512);
        }
    };
    // one step, sub-block pair U of its super-block; NI: the wave's token tiles
    // that hold tokens
    auto step = [&](auto u, auto ni, const _Float16* xs, const uint8_t* qs, const uint8_t* hs,
                    const uint8_t* ss) {
        constexpr int U = decltype(u)::value, NI = decltype(ni)::value;
        if constexpr (NI == 0) return;
        h8 A[2][4];
        read_a(xs, 0, 0, A[0]);
        const int rl = PAIR ? 32 * wn + c : 64 * wn + c;
        fq_u32x4 hdr[2], qh[2], qv[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            hdr[j] = lds16(hs + (rl + RJ * j) * 16);
            qv[j] = lds16(qs + (g * BNT + rl + RJ * j) * 16);
            if constexpr (F == Q5_K) qh[j] = lds16(hs + ((1 + g) * BNT + rl + RJ * j) * 16);
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            h8 B[2][2], Bl[2][2];  // Bl: for x_lo
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float sf = (float)sub_scale(hdr[j], 2 * U + b);
                const _Float16 s1 = (_Float16)(sf * (1.0f / Q::UNIT));
                const h2 sc = {s1, s1}, off = sc * h2{(_Float16)-1152.0f, (_Float16)-1152.0f};
                uint32_t w[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if constexpr (F == Q5_K) {
                        // fifth bit 2 U + b of the qh byte on top of the nibble
                        w[k] = (b ? qv[j][k] >> 1 : qv[j][k] << 3) & 0x78787878u;
                        w[k] |= (qh[j][k] << (7 - 2 * U - b)) & 0x80808080u;
                    } else {
                        w[k] = (b ? qv[j][k] : qv[j][k] << 4) & 0xF0F0F0F0u;
                    }
                }
                B[j][0] = scaled8(w[0], w[1], sc, off);
                B[j][1] = scaled8(w[2], w[3], sc, off);
#pragma unroll
                for (int h = 0; h < 2; ++h) Bl[j][h] = Q::FINE ? B[j][h] * (_Float16)(1.0f / LO) : B[j][h];
            }
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int st = NI * b + i;
                h8(&cur)[4] = A[st & 1];
                if (st + 1 < 2 * NI) read_a(xs, (st + 1) / NI, (st + 1) % NI, A[(st + 1) & 1]);
                const f32x16 z = {};
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    D[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                        cur[0], B[j][0], U == 0 && b == 0 ? z : D[i][j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    D[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur[1], Bl[j][0], D[i][j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    D[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur[2], B[j][1], D[i][j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    D[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur[3], Bl[j][1], D[i][j], 0, 0, 0);
            }
        }
        if constexpr (U == 3) {
            // the super-block's fold: acc += d D - dmin Dm (FINE: times 2^e).
            // Sums operand: lane (c, g) the hi (g = 0) or lo parts of token c,
            // times 2^-5 (lo: times LO)
            const float gs = g ? 1.0f / LO : 1.0f;
            h8 Mb[2], Sb[2];
            float d[2], dn[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                h8 m, sc;
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    m[b] = (_Float16)((float)sub_min(hdr[j], b) * gs);
                    sc[b] = (_Float16)((float)sub_scale(hdr[j], b) * (gs * 32.0f * Q::MID));
                }
                Mb[j] = m;
                Sb[j] = sc;
                d[j] = f16_hw(hdr[j].x & 0xFFFFu);
                dn[j] = -32.0f * f16_hw(hdr[j].x >> 16);
            }
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const h8 S = *reinterpret_cast<const h8*>(ss + (2 * wm + i) * STILE + 16 * lane);
                const f32x16 z = {};
                f32x16 dm[2];
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    D[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(S, Sb[j], D[i][j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    dm[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(S, Mb[j], z, 0, 0, 0);
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {  // the lane's tokens 8 e4 + 4 g ..
                    float4 f4 = {};
                    if constexpr (Q::FINE)
                        f4 = *reinterpret_cast<const float4*>(ss + (2 * wm + i) * STILE + SEXP + 32 * e4 + 16 * g);
                    const float f[4] = {f4.x, f4.y, f4.z, f4.w};
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const int e = 4 * e4 + k;
                            if constexpr (Q::FINE) {
                                const float v = __builtin_fmaf(d[j], D[i][j][e], dn[j] * dm[j][e]);
                                acc[i][j][e] = __builtin_fmaf(v, f[k], acc[i][j][e]);
                            } else {
                                acc[i][j][e] = __builtin_fmaf(d[j], D[i][j][e], acc[i][j][e]);
                                acc[i][j][e] = __builtin_fmaf(dn[j], dm[j][e], acc[i][j][e]);
                            }
                        }
                }
            }
        }
    };
    // s0 and s1 are multiples of four steps
    if (s0 < s1) {
        issue(s0, true);
        issue(s0 + 1, false);
    }
    auto run = [&](auto u, auto ni, int s) __attribute__((always_inline)) {
        constexpr int U = decltype(u)::value;
        // this wave's copies of step s are complete; those of step s + 1 may
        // be in flight
        if (s + 1 >= s1) wait_vm<0>();
        else wait_vm<Q::CS + (U == 3 ? Q::CB : 0)>();
        __syncthreads();
        if (s + 2 < s1) issue(s + 2, U == 2);
        const int buf = s % NBUF, sb = (s >> 2) & 1;
        step(u, ni, reinterpret_cast<const _Float16*>(xs0 + buf * Q::XBUF), qs0 + buf * Q::QBUF,
             hs0 + sb * Q::HBUF, ss0 + sb * Q::SBUF);
    };
    // Token tiles past M are copied and waited for, not computed: the matrix
    // cores' pace is the kernel's, so a tile of zeros costs as much as any
    // (Q4_K 4096 -> 14336 at M = 77, preparation included, 49 -> 43 us).  Deeper
    // buffers in the LDS that fewer tiles would leave measured no faster.
    auto loop = [&](auto ni) __attribute__((always_inline)) {
        for (int s = s0; s < s1; s += 4) {
            run(std::integral_constant<int, 0>{}, ni, s);
            run(std::integral_constant<int, 1>{}, ni, s + 1);
            run(std::integral_constant<int, 2>{}, ni, s + 2);
            run(std::integral_constant<int, 3>{}, ni, s + 3);
        }
    };
    const int live = Tn - (m0 / 32 + 2 * wm);  // wave-uniform
    if (live >= 2) loop(std::integral_constant<int, 2>{});
    else if (live == 1) loop(std::integral_constant<int, 1>{});
    else loop(std::integral_constant<int, 0>{});
#pragma unroll
    for (int i = 0; i < 2; ++i)
        store_tiles<PAIR, !Q::FINE>(a, rt, m0 + 64 * wm + 32 * i, rt.n0 + (PAIR ? 32 : 64) * wn + c, g, acc[i],
                          gridDim.z > 1, blockIdx.z);
}

}  // namespace

bool mmqk_supported(int dtype) { return dtype == Q4_K || dtype == Q5_K; }

bool mmqk_fine(int dtype) { return dtype == Q5_K; }

// Bytes of the sub-block sums of one 32-token tile
size_t mmqk_sum_bytes(int dtype, int K) {
    return (size_t)(K / 256) * (mmqk_fine(dtype) ? KQ<Q5_K>::STILE : KQ<Q4_K>::STILE);
}

hipError_t launch_xprepk(const float* x, int M, int K, _Float16* xop, uint8_t* xs, hipStream_t st) {
    if (K % 256 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(xprepk_kernel, dim3(K / 256, (M + 31) / 32), dim3(512), 0, st, x, M, K, xop, xs);
    return hipGetLastError();
}

hipError_t launch_mmqk(int dtype, const MmqArgs& a, int splits, hipStream_t st) {
    const int nsteps = a.K / KS;
    const int sps = ((nsteps + splits - 1) / splits + 3) & ~3;  // whole super-blocks
    if (a.K % 256 != 0 || (long)sps * (splits - 1) >= nsteps) return hipErrorInvalidValue;
    const dim3 grid(row_tiles(a, BNT), (a.M + BMT - 1) / BMT, splits), wg(64 * NW);
    const bool pair = a.mm == MM_PAIR;
    if (dtype == Q4_K && pair)
        hipLaunchKernelGGL((mmqk_kernel<Q4_K, true>), grid, wg, 0, st, a, sps);
    else if (dtype == Q4_K)
        hipLaunchKernelGGL((mmqk_kernel<Q4_K, false>), grid, wg, 0, st, a, sps);
    else if (dtype == Q5_K && pair)
        hipLaunchKernelGGL((mmqk_kernel<Q5_K, true>), grid, wg, 0, st, a, sps);
    else if (dtype == Q5_K)
        hipLaunchKernelGGL((mmqk_kernel<Q5_K, false>), grid, wg, 0, st, a, sps);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace fq
