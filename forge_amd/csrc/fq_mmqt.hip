// fq_mmqt.hip -- small batches (M <= 32 tokens) of every format but Q3_K on the
// fp16 matrix cores, the token operands shared by the rows of a work-group.
//
// A work-group owns a range of steps: super-blocks (256 elements of K) of tiles
// of 64, 128 or 256 rows.  Per super-block it copies into LDS, two or three
// buffers deep and with no registers in between,
//
//   the rows' super-blocks (or eight 32-element blocks) as they lie in memory
//   (16-byte pieces along each row: contiguous runs of 144 to 272 bytes), each
//   wave its own 16 rows,
//   the tokens' operands (16 KiB per 16 tokens), an equal share per wave,
//   the tokens' sub-block sums and scales,
//
// and one barrier per super-block publishes them.  In the band kernel of
// fq_mmqs.hip every wave reads the token operands of its own super-blocks from
// L2, for 32 or 64 rows: 3.5 times the weight bytes for a Q6_K head at 16
// tokens (1.1 GB).  Here the operands of a super-block serve all rows of the
// work-group.  152064 x 3584 Q6_K, M = 16: 216 -> 131 us; Q4_K, M = 8 131 ->
// 94; 14336 x 4096 Q4_K, M = 8 18.7 -> 16.3, M = 32 (fp16 MFMA kernel) 40.2 ->
// 24.0, gate and up of that size in one launch 37.7 -> 23.8 and 82.5 -> 35.8.
// What bounds it: vector and matrix issue, then the LDS reads of the token
// operands (Q6_K head, M = 16: vector issue 69 % of the cycles, the matrix
// cores 28 %, LDS 32 %; an earlier form with a work-group per tile half and
// without the x_lo W_lo product, 139 us in all, took 117 without the copies, 105
// without the arithmetic), so the waves per SIMD count: that form with 256 rows
// on eight waves of two tiles each ran the head in 152 us, on sixteen waves 139.
//
// Tokens are the A operand of v_mfma_f32_16x16x32_f16 (lane 16 q + c: token c,
// eight elements of k group q) and weights the B operand (lane 16 q + c: row
// c), so that a lane's results belong to one row.  Lane group q takes the
// q-th quarter of the super-block: Q4_K / Q5_K sub-block pair q (its 32 qs
// bytes, two scales), Q6_K unit q (16 l positions of a half, four scales), and
// decodes no scale but its own.  The scale goes into the weight operand:
//
//   Q4_K, Q5_K: sc (q - c) as in fq_mmqk.hip, exact in fp16 (at most 1008);
//   Q6_K: sc (q - 32) has up to 13 bits: W = W_hi + W_lo, W_hi its fp16
//   rounding and W_lo the exact rest; all four products are formed (without
//   x_lo W_lo, up to 2^-22 of a product, the codes would not be exact; the
//   head at M = 16 takes 131 us with it, 125 without).
//
//   the 32-element blocks: the integer code, d on the results (TQB below).
//
// Short MFMA chains, added up per super-block, then acc += 2^e (d D + Dm), e the
// token's exponent (x 2^-e below 2^15, split into fp16 hi + lo: 22 significant
// bits) and Dm the minimum and centring terms, an fp32 product of the token's
// sub-block sums.  The 32-element blocks have an exponent per 64 elements.  The
// K-quants have one per super-block, whose 64-element quarters one MFMA spans;
// their x_lo is kept 2^12 larger, in a chain of its own, so that an element
// keeps its bits down to 2^-29 of the super-block's largest (fp16's least
// value alone: 2^-17) and is 2^-51 of that largest off at most.
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

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int XSB = 16384;  // operand bytes of a (16-token tile, super-block): [ks][hi, lo][lane][8]
// sums and scales of a (tile, super-block), floats: lane 16 q + c's sums of token
// c's sub-blocks 2 q and 2 q + 1, then 2^e of tokens 0 .. 15, of each 64-element
// group (K-quants: the first alone, of the super-block)
constexpr int SEXP = 64 * 8, SSB = SEXP + 4 * 64;
constexpr float LO = 0x1p12f;  // what the K-quants' x_lo is larger by

// ------------------------------------------------------------- token prep
// One work-group per super-block and 16-token tile; thread 16 c + p holds
// elements 16 p .. 16 p + 15 of token c.  Eight elements 8 e8 .. + 7 are slots
// (slot_elem order) of lane group q in MFMA ks: Q4_K / Q5_K (MAP 0) q = e8 /
// 8, ks = e8 % 8; Q6_K (MAP 1) element 128 n + 32 u + 16 h + 8 i: q = 2 n + h,
// ks = 2 u + i; 32-element blocks (MAP 2) ks the block, q = e8 % 4.
template <int MAP>
__global__ __launch_bounds__(256) void xprept_kernel(const float* __restrict__ x, int M, int K,
                                                     uint8_t* __restrict__ xop,
                                                     uint8_t* __restrict__ xs) {
    const int tid = threadIdx.x, c = tid >> 4, p = tid & 15;
    const int sb = blockIdx.x, T = blockIdx.y, m = 16 * T + c, nsb = K / 256;
    float v[16] = {};
    if (m < M) {
        const float4* s = reinterpret_cast<const float4*>(x + (size_t)m * K + 256 * sb + 16 * p);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 t = s[i];
            v[4 * i] = t.x;
            v[4 * i + 1] = t.y;
            v[4 * i + 2] = t.z;
            v[4 * i + 3] = t.w;
        }
    }
    float mx = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, fabsf(v[i]));
#pragma unroll
    for (int o = 1; o < (MAP == 2 ? 4 : 16); o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    // (2^e a normal number: -e up to 126 brings every x but the subnormal ones
    // to 2^0 and more, and those into fp16 exactly)
    const int e = (mx > 0.0f && mx <= 3.0e38f) ? max(ilogbf(mx) - 14, -126) : 0;
    float sum = 0.0f;
    uint8_t* const ob = xop + ((size_t)T * nsb + sb) * XSB;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int e8 = 2 * p + i;
        const int q = MAP == 2 ? e8 & 3 : MAP == 1 ? 2 * (e8 >> 4) + ((e8 >> 1) & 1) : e8 >> 3;
        const int ks = MAP == 2 ? e8 >> 2 : MAP == 1 ? 2 * ((e8 >> 2) & 3) + (e8 & 1) : e8 & 7;
        float w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] = __builtin_amdgcn_ldexpf(v[8 * i + j], -e);
        h8 hi, lo;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float u = w[slot_elem(j)];
            hi[j] = (_Float16)u;
            lo[j] = (_Float16)((u - (float)hi[j]) * (MAP == 2 ? 1.0f : LO));
        }
        h8* o = reinterpret_cast<h8*>(ob + ks * 2048 + (16 * q + c) * 16);
        o[0] = hi;
        o[64] = lo;
        sum += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
    }
    float* const sbk = reinterpret_cast<float*>(xs + ((size_t)T * nsb + sb) * SSB);
    if (p % (MAP == 2 ? 4 : 16) == 0) sbk[SEXP / 4 + 4 * p + c] = __builtin_amdgcn_ldexpf(1.0f, e);
    if constexpr (MAP != 1) {
        sum += __shfl_xor(sum, 1, 64);
        const int b = p >> 1;
        // (K-quants: times 2^-e; the others, of several e, as they are, times
        // 2^-5: no larger than the largest x)
        if ((p & 1) == 0)
            sbk[2 * (16 * (b >> 1) + c) + (b & 1)] = MAP == 2 ? __builtin_amdgcn_ldexpf(sum, e - 5) : sum;
    }
}

// ------------------------------------------------------------- weights
// BLOCKS: a scale per 32-element block, outside the operand (below).  PPR: 16-byte pieces of a row's super-block in LDS; SHIFT: rows start at even
// addresses only, each super-block copied from its aligned-down start and read
// at its shift (Q6_K: 14 pieces always hold some of its 210 bytes; a 15th,
// a repeat, keeps 16 rows' 16-byte units on distinct banks).
template <int F>
struct TQ;

__device__ __forceinline__ fq_u32x4 lds16(const uint8_t* p) {
    typedef const __attribute__((address_space(3))) fq_u32x4* lds_v4;
    return *reinterpret_cast<lds_v4>(reinterpret_cast<uintptr_t>(p));
}
__device__ __forceinline__ uint32_t lds4(const uint8_t* p) {
    typedef const __attribute__((address_space(3))) uint32_t* lds_v1;
    return *reinterpret_cast<lds_v1>(reinterpret_cast<uintptr_t>(p));
}

template <int F>
struct TQK {
    static constexpr int SBB = F == Q5_K ? 176 : 144, PPR = SBB / 16, LAST = PPR - 1;
    static constexpr bool SHIFT = false, MIN = true, SPLITW = false, BLOCKS = false;
    static constexpr float UNIT = F == Q5_K ? 8.0f : 16.0f, MID = F == Q5_K ? 16.0f : 8.0f;
    uint32_t w[8], h[8];
    h2 s[2], off[2];
    float d, wm[2];
    // row's super-block at p (LDS), lane group q
    __device__ void load(const uint8_t* p, int, int q) {
        const fq_u32x4 hd = lds16(p);
        const uint8_t* qs = p + (F == Q5_K ? 48 : 16) + 32 * q;
        const fq_u32x4 a = lds16(qs), b = lds16(qs + 16);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            w[k] = a[k];
            w[4 + k] = b[k];
        }
        if constexpr (F == Q5_K) {  // bits 2 q, 2 q + 1 of each qh byte to bits 6, 7
            const fq_u32x4 ha = lds16(p + 16), hb = lds16(p + 32);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                h[k] = ha[k] << (6 - 2 * q);
                h[4 + k] = hb[k] << (6 - 2 * q);
            }
        }
        uint32_t sa, ma, sb, mi;
        Fmt<Q4_K>::scale_min(uint4{hd.x, hd.y, hd.z, hd.w}, q, sa, ma, sb, mi);
        const float f0 = (float)sa, f1 = (float)sb;
        const _Float16 u0 = (_Float16)(f0 * (1.0f / UNIT)), u1 = (_Float16)(f1 * (1.0f / UNIT));
        s[0] = h2{u0, u0};
        s[1] = h2{u1, u1};
        off[0] = s[0] * h2{(_Float16)-1152.0f, (_Float16)-1152.0f};
        off[1] = s[1] * h2{(_Float16)-1152.0f, (_Float16)-1152.0f};
        d = f16_hw(hd.x & 0xFFFFu);
        const float dm = f16_hw(hd.x >> 16);
        wm[0] = __builtin_fmaf(d * MID, f0, -(dm * (float)ma));
        wm[1] = __builtin_fmaf(d * MID, f1, -(dm * (float)mi));
    }
    template <int KSI>
    __device__ uint32_t code(int k) const {
        if constexpr (F == Q5_K) {
            const uint32_t n = (KSI < 4 ? w[k] << 3 : w[k] >> 1) & 0x78787878u;
            return n | ((KSI < 4 ? h[k] << 1 : h[k]) & 0x80808080u);
        } else {
            return (KSI < 4 ? w[k] << 4 : w[k]) & 0xF0F0F0F0u;
        }
    }
    // the weight operand of MFMA KSI
    template <int KSI>
    __device__ void ops(h8& whi, h8&) const {
        constexpr int k = 2 * (KSI & 3), t = KSI >> 2;
        const uint32_t c0 = code<KSI>(k), c1 = code<KSI>(k + 1);
        auto pr = [&](uint32_t c, uint32_t sel) {
            return __builtin_elementwise_fma(
                __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, c, sel)), s[t], off[t]);
        };
        const h2 a = pr(c0, 0x04020400u), b = pr(c0, 0x04030401u), e = pr(c1, 0x04020400u),
                 f = pr(c1, 0x04030401u);
        whi = h8{a[0], a[1], b[0], b[1], e[0], e[1], f[0], f[1]};
    }
};
template <>
struct TQ<Q4_K> : TQK<Q4_K> {};
template <>
struct TQ<Q5_K> : TQK<Q5_K> {};

// Q6_K (210 B: ql[128] qh[64] sc[16] d), unit q = 2 n + h: 16 bytes each of
// ql[64 n + 16 h], ql[64 n + 32 + 16 h] and qh[32 n + 16 h]; u = 0..3: nibble
// u / 2 of the first (u even) or second run, bits 2 u of the third, scale
// sc[8 n + 2 u + h]; MFMA ks = 2 u + i takes its bytes 8 i .. 8 i + 7.
template <>
struct TQ<Q6_K> {
    static constexpr int SBB = 210, PPR = 15, LAST = 13;
    static constexpr bool SHIFT = true, MIN = false, SPLITW = true, BLOCKS = false;
    uint32_t lo[4], hi[4], qh[4];
    h2 s[4];
    float d;
    __device__ static void run16(const uint8_t* p, uint32_t sh, uint32_t (&o)[4]) {
        uint32_t t[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) t[k] = lds4(p + 4 * k);
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = __builtin_amdgcn_alignbyte(t[k + 1], t[k], sh);
    }
    // the row's pieces at p, its super-block sh bytes in
    __device__ void load(const uint8_t* p, int sh, int q) {
        const uint32_t r = sh & 3;  // 0 or 2
        const uint8_t* a = p + (sh & ~3);
        const int n = q >> 1, h = q & 1;
        run16(a + 64 * n + 16 * h, r, lo);
        run16(a + 64 * n + 32 + 16 * h, r, hi);
        run16(a + 128 + 32 * n + 16 * h, r, qh);
        const uint32_t s0 = lds4(a + 192 + 8 * n), s1 = lds4(a + 196 + 8 * n), s2 = lds4(a + 200 + 8 * n);
        const uint32_t sa = __builtin_amdgcn_alignbyte(s1, s0, r) >> (8 * h);
        const uint32_t sb = __builtin_amdgcn_alignbyte(s2, s1, r) >> (8 * h);
        const uint32_t sv[4] = {sa, sa >> 16, sb, sb >> 16};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const _Float16 f = (_Float16)(float)(int8_t)(sv[u] & 0xFFu);
            s[u] = h2{f, f};
        }
        d = f16_hw((lds4(a + 208) >> (8 * r)) & 0xFFFFu);
    }
    template <int KSI>
    __device__ void ops(h8& whi, h8& wlo) const {
        constexpr int u = KSI >> 1, k = 2 * (KSI & 1);
        h2 vh[4], vl[4];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const uint32_t l = u & 1 ? hi[k + t] : lo[k + t];
            const uint32_t hb = u < 2 ? qh[k + t] << (4 - 2 * u) : qh[k + t] >> (2 * u - 4);
            const uint32_t c = ((u < 2 ? l : l >> 4) & 0x0F0F0F0Fu) | (hb & 0x30303030u);
            h2 p0, p1;
            byte_pairs(c, (_Float16)1056.0f, p0, p1);  // q - 32
            vh[2 * t] = p0 * s[u];
            vh[2 * t + 1] = p1 * s[u];
            vl[2 * t] = __builtin_elementwise_fma(p0, s[u], -vh[2 * t]);
            vl[2 * t + 1] = __builtin_elementwise_fma(p1, s[u], -vh[2 * t + 1]);
        }
        whi = h8{vh[0][0], vh[0][1], vh[1][0], vh[1][1], vh[2][0], vh[2][1], vh[3][0], vh[3][1]};
        wlo = h8{vl[0][0], vl[0][1], vl[1][0], vl[1][1], vl[2][0], vl[2][1], vl[3][0], vl[3][1]};
    }
};

// The 32-element block formats (eight blocks are 144 / 160 / 272 / 176 / 192 /
// 144 bytes of a row: Q4_0, Q4_1, Q8_0, Q5_0, Q5_1, IQ4_NL).  MFMA ks is block
// ks of the super-block, lane group q its elements 8 q .. 8 q + 7: q < 2 the low
// nibbles of qs bytes 8 q .., else the high ones of 8 (q - 2) ..; bits 8 q .. of
// qh.  The operand holds the integer code (IQ4_NL: the table value), the
// block's scale d multiplies the MFMA pair's results (d codes have up to 19
// bits).  Q4_1 and Q5_1, w = d q + m, enter as d (q - c) + (m + c d), c 8 or 16,
// the second term on the sub-block sums.  Rows of 160 and 192
// bytes take a repeated piece, so that 16 rows start on eight banks, not four
// or two.
template <int F>
struct TQB {
    static constexpr int BB = Fmt<F>::BB, SBB = 8 * BB;
    static constexpr int LAST = SBB / 16 - 1, PPR = SBB / 16 + (F == Q4_1 || F == Q5_1 ? 1 : 0);
    static constexpr bool SHIFT = false, MIN = F == Q4_1 || F == Q5_1, SPLITW = false, BLOCKS = true;
    static constexpr int QS = F == Q4_0 || F == IQ4_NL || F == Q8_0 ? 2 : F == Q4_1 ? 4 : F == Q5_0 ? 6 : 8;
    static constexpr int QH = F == Q5_0 ? 2 : 4;
    static constexpr float MID = F == Q5_0 || F == Q5_1 ? 16.0f : 8.0f;  // subtracted from a code
    uint32_t w[16], h[8];
    float db[8], wm[2];
    int sh;
    // the dword at p + o, o even and known at compile time
    template <int O>
    __device__ static uint32_t dw(const uint8_t* p) {
        if constexpr (O % 4 == 0) return lds4(p + O);
        else return __builtin_amdgcn_alignbyte(lds4(p + O + 2), lds4(p + O - 2), 2);
    }
    template <int B>
    __device__ void block(const uint8_t* p, const uint8_t* pq, int q) {
        constexpr int O = BB * B;
        if constexpr ((O + QS) % 4 == 0) {
            w[2 * B] = lds4(pq + O + QS);
            w[2 * B + 1] = lds4(pq + O + QS + 4);
        } else {
            const uint32_t a = lds4(pq + O + QS - 2), b = lds4(pq + O + QS + 2), c = lds4(pq + O + QS + 6);
            w[2 * B] = __builtin_amdgcn_alignbyte(b, a, 2);
            w[2 * B + 1] = __builtin_amdgcn_alignbyte(c, b, 2);
        }
        if constexpr (F == Q5_0 || F == Q5_1) h[B] = dw<O + QH>(p) >> (8 * q);
        db[B] = f16_hw(*reinterpret_cast<const uint16_t*>(p + O));
    }
    __device__ void load(const uint8_t* p, int, int q) {
        const uint8_t* pq = p + (F == Q8_0 ? 8 * q : 8 * (q & 1));
        sh = 4 * (q >> 1);
        block<0>(p, pq, q);
        block<1>(p, pq, q);
        block<2>(p, pq, q);
        block<3>(p, pq, q);
        block<4>(p, pq, q);
        block<5>(p, pq, q);
        block<6>(p, pq, q);
        block<7>(p, pq, q);
        if constexpr (MIN) {  // m + c d of this lane group's sub-blocks 2 q, 2 q + 1
            const uint32_t d0 = lds4(p + 2 * BB * q), d1 = lds4(p + 2 * BB * q + BB);
            wm[0] = __builtin_fmaf(MID, f16_hw(d0 & 0xFFFFu), f16_hw(d0 >> 16));
            wm[1] = __builtin_fmaf(MID, f16_hw(d1 & 0xFFFFu), f16_hw(d1 >> 16));
        }
    }
    template <int KSI>
    __device__ h8 op() const {
        if constexpr (F == Q8_0) {
            return byte8(w[2 * KSI] ^ 0x80808080u, w[2 * KSI + 1] ^ 0x80808080u, (_Float16)1152.0f);
        } else {
            uint32_t a = (w[2 * KSI] >> sh) & 0x0F0F0F0Fu, b = (w[2 * KSI + 1] >> sh) & 0x0F0F0F0Fu;
            if constexpr (F == IQ4_NL)
                return byte8(iq4_lookup(a) ^ 0x80808080u, iq4_lookup(b) ^ 0x80808080u, (_Float16)1152.0f);
            if constexpr (F == Q5_0 || F == Q5_1) {
                a = five_bit(a, h[KSI]);
                b = five_bit(b, h[KSI] >> 4);
            }
            return byte8(a, b, (_Float16)(1024.0f + MID));
        }
    }
};
template <>
struct TQ<Q4_0> : TQB<Q4_0> {};
template <>
struct TQ<Q4_1> : TQB<Q4_1> {};
template <>
struct TQ<Q8_0> : TQB<Q8_0> {};
template <>
struct TQ<Q5_0> : TQB<Q5_0> {};
template <>
struct TQ<Q5_1> : TQB<Q5_1> {};
template <>
struct TQ<IQ4_NL> : TQB<IQ4_NL> {};

// TT 16-token tiles; RW waves along the rows, 16 each (PAIR: the first half
// gate, the second half up rows), in KG groups: step j of a row tile is group
// k's super-block KG j + k.
template <int F, int TT, int RW, int KG>
struct Thin {
    using Q = TQ<F>;
    static constexpr int NW = RW * KG, BN = 16 * RW;      // waves; rows of a work-group
    static constexpr int PI = (16 * Q::PPR + 63) / 64;    // copies per 16-row tile
    static constexpr int PANEL = BN * Q::PPR * 16;
    static constexpr int GBUF = PANEL + TT * (XSB + SSB), BUF = KG * GBUF;
    static constexpr int NB = 3 * BUF <= 160 * 1024 ? 3 : 2;
    static constexpr int LDS = NB * BUF;
    static constexpr int XC = 16 / RW;                    // 1 KiB token copies per wave and tile
    static constexpr int SW = RW < 8 ? RW : 8;            // waves that copy a tile's sums
    static_assert(LDS <= 160 * 1024, "LDS");
    static_assert(NW * TT * 1024 <= BUF, "the sums exchanged at a tile's end");
};

__device__ __forceinline__ float biased(const MmqArgs& a, float v, int m, int n) {
    if (a.bias_mode == 1) return v + (n < a.bias_len ? a.bias[n] : 0.0f);
    return a.bias_mode == 2 ? v + a.bias[(size_t)m * a.N + n] : v;
}

// The parts of row tile t, of nst steps, when each work-group takes per steps of
// all tiles' in a row: the work-groups first .. first + n - 1.
struct Parts {
    int first, n;
};
__device__ __forceinline__ Parts tile_parts(int t, int nst, int per) {
    const int f = t * nst / per;
    return Parts{f, (t * nst + nst - 1) / per - f + 1};
}

// Work-group j takes steps per j .. of the row tiles' steps laid end to end, and
// its copies run ahead over the tiles' ends: one work-group fills a CU's LDS, so
// that work-groups in turn each fill and drain the pipeline alone (a step and
// 1.5 us more), and a last round of them leaves CUs idle.  A tile within one
// work-group goes to y, the parts of one cut by a range's end to slabs that
// reducet_kernel adds.  Against a work-group per tile or K-split of one: Q6_K
// 152064 x 3584 M = 16 140 -> 129 us, Q4_K M = 24 138 -> 126, gate and up of
// 18944 x 3584 Q4_0 at M = 4 34 -> 29.
// ONE: per divides the steps of a tile, so that a work-group has one tile or a
// part of it; the code for several cost such a call 3 to 5 % (14336 x 4096 Q4_K
// M = 8 16.9 -> 17.7).
template <int F, bool PAIR, int TT, int RW, int KG, bool ONE>
__global__ __launch_bounds__(64 * RW * KG) void mmqt_kernel(MmqArgs a, int per, int total) {
    using Q = TQ<F>;
    using TH = Thin<F, TT, RW, KG>;
    __shared__ __attribute__((aligned(16))) uint8_t lds[TH::LDS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rw = wave % RW, kg = wave / RW;
    const int c = lane & 15, q = lane >> 4;
    const int nsb = a.K / 256, nst = (nsb + KG - 1) / KG;  // mmqt_steps
    const int s0 = blockIdx.x * per, s1 = min(total, s0 + per);
    // this wave's 16 rows of a tile
    const bool up = PAIR && rw >= RW / 2;
    const int wrow = 16 * (PAIR ? rw % (RW / 2) : rw);

    // copy sources in tile it, step ij.  SHIFT: offsets from the matrix's
    // aligned-down base, not yet aligned themselves (the super-block's start is
    // added first)
    int it = s0 / nst, ij = s0 - it * nst;
    const uint8_t* wb;
    uint32_t woff[TH::PI], wp[TH::PI];
    auto source = [&](int t) __attribute__((always_inline)) {
        const RowTile rt = row_tile<PAIR>(a, t, TH::BN);
        const uint8_t* const base = up ? a.w2 : rt.w;
        const uint32_t mis = Q::SHIFT ? (uint32_t)(reinterpret_cast<uintptr_t>(base) & 15) : 0u;
        wb = base - mis;
#pragma unroll
        for (int i = 0; i < TH::PI; ++i) {
            const int L = min(64 * i + lane, 16 * Q::PPR - 1), r = L / Q::PPR;
            wp[i] = 16u * (uint32_t)min(L - r * Q::PPR, Q::LAST);
            woff[i] = (uint32_t)min(rt.n0 + wrow + r, rt.rows - 1) * (uint32_t)a.row_bytes + mis +
                      (Q::SHIFT ? 0u : wp[i]);
        }
    };
    source(it);
    constexpr int XB = XSB / RW, SB = SSB / TH::SW;  // this wave's share of a tile's operands
    const uint8_t* const xb = reinterpret_cast<const uint8_t*>(a.xop) + XB * rw;
    const uint8_t* const sbase = reinterpret_cast<const uint8_t*>(a.xsum) + SB * rw;
    const uint32_t l0 = __builtin_amdgcn_readfirstlane(lds_addr(lds)) + kg * TH::GBUF;
    const bool sums = rw < TH::SW;  // wave-uniform
    auto copy = [&](int sb, int n) __attribute__((always_inline)) {
        const uint32_t lb = l0 + (uint32_t)(n % TH::NB) * TH::BUF;
        const uint32_t lp = lb + (uint32_t)(16 * rw) * (Q::PPR * 16), so = (uint32_t)sb * Q::SBB;
#pragma unroll
        for (int i = 0; i < TH::PI; ++i) {
            if (64 * (i + 1) > 16 * Q::PPR && lane >= 16 * Q::PPR - 64 * i) continue;
            if constexpr (Q::SHIFT) dma16s(((woff[i] + so) & ~15u) + wp[i], wb, lp + 1024 * i);
            else dma16s(woff[i], wb + so, lp + 1024 * i);
        }
#pragma unroll
        for (int T = 0; T < TT; ++T) {
            const size_t blk = (size_t)T * nsb + sb;
            const uint32_t lx = lb + TH::PANEL + T * XSB + XB * rw;
#pragma unroll
            for (int i = 0; i < TH::XC; ++i)
                dma16s(16 * lane + 1024 * i, xb + blk * XSB, lx + 1024 * i);
            if (sums && lane < SB / 16)
                dma16s(16 * lane, sbase + blk * SSB, lb + TH::PANEL + TT * XSB + T * SSB + SB * rw);
        }
    };
    // the copies of this wave for the next step, the n-th of the work-group
    auto issue = [&](int n) __attribute__((always_inline)) {
        const int sb = KG * ij + kg;
        if (KG == 1 || sb < nsb) copy(sb, n);
        if (++ij == nst && !ONE) {
            ij = 0;
            if (s0 + n + 1 < s1) source(++it);
        }
    };
    // wait until this wave's copies of a step are complete; later: those of the
    // next are under way and nothing else is
    auto wait = [&](bool later) {
        constexpr int C = TH::PI + TH::XC * TT;
        if (TH::NB == 2 || !later) wait_vm<0>();
        else if (sums) wait_vm<C + TT>();
        else wait_vm<C>();
    };

    // a tile's steps enter two sums in turn (Q6_K 152064 x 3584: error against 64
    // bits 1.17e-7 with one, 1.11e-7 with two)
    f32x4 acc[TT], acc2[TT];
#pragma unroll
    for (int T = 0; T < TT; ++T) acc[T] = acc2[T] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // the tile and step computed
    int ct = it, cj = ij;
    RowTile rt = row_tile<PAIR>(a, ct, TH::BN);
    // byte shift of lane row c's super-block in its pieces, before sb's
    auto row_shift = [&]() __attribute__((always_inline)) {
        return (uint32_t)(reinterpret_cast<uintptr_t>(up ? a.w2 : rt.w) & 15) +
               (uint32_t)min(rt.n0 + wrow + c, rt.rows - 1) * (uint32_t)a.row_bytes;
    };
    uint32_t rsh = row_shift();

    auto compute = [&](int sb, int n) __attribute__((always_inline)) {
        const uint8_t* buf = lds + kg * TH::GBUF + (n % TH::NB) * TH::BUF;
        const uint8_t* xs = buf + TH::PANEL;
        const uint8_t* ss = xs + TT * XSB;
        Q w;
        w.load(buf + (16 * rw + c) * (Q::PPR * 16),
               Q::SHIFT ? (int)((rsh + (uint32_t)sb * Q::SBB) & 15u) : 0, q);
        // The matrix cores' additions round toward zero, so a chain's error
        // grows with its length times its magnitude: four chains of two for
        // the large products (x_hi W_hi), one each for those of x_lo and W_lo.
        // 32-element blocks: D[0] the sum of d D over a 64-element group, Dl those
        // groups' sum (added to the tile's sums one by one: 1.10e-7 against
        // 1.02e-7, Q4_0 at K = 3584)
        f32x4 D[4][TT], Dl[TT], Dw[TT];
        auto exps = [&](int T, int g) {
            return *reinterpret_cast<const f32x4*>(ss + T * SSB + SEXP + 64 * g + 16 * q);
        };
        // a value joins a tile's sums, the two in turn
        auto add = [&](int T, int i, float v, float f) {
            v = __builtin_fmaf(v, f, acc[T][i]);
            acc[T][i] = acc2[T][i];
            acc2[T][i] = v;
        };
        const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
        auto ks = [&](auto ki) {
            constexpr int KSI = decltype(ki)::value;
            h8 whi, wlo;
            if constexpr (Q::BLOCKS) whi = w.template op<KSI>();
            else w.template ops<KSI>(whi, wlo);
#pragma unroll
            for (int T = 0; T < TT; ++T) {
                const uint8_t* xp = xs + T * XSB + KSI * 2048 + 16 * lane;
                const h8 xh = *reinterpret_cast<const h8*>(xp);
                const h8 xl = *reinterpret_cast<const h8*>(xp + 1024);
                if constexpr (Q::BLOCKS) {
                    // (x_lo first: 1.8e-7 against 1.2e-7 at K = 18944)
                    f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, whi, z, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, whi, d, 0, 0, 0);
                    f32x4& dd = D[0][T];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        dd[i] = KSI & 1 ? __builtin_fmaf(w.db[KSI], d[i], dd[i]) : w.db[KSI] * d[i];
                    if constexpr (KSI & 1) {
                        const f32x4 f = exps(T, KSI >> 1);
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            Dl[T][i] = KSI > 1 ? __builtin_fmaf(dd[i], f[i], Dl[T][i]) : dd[i] * f[i];
                    }
                    continue;
                }
                f32x4& d = D[KSI >> 1][T];
                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, whi, KSI & 1 ? d : z, 0, 0, 0);
                Dl[T] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, whi, KSI ? Dl[T] : z, 0, 0, 0);
                if constexpr (Q::SPLITW) {
                    Dl[T] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, wlo, Dl[T], 0, 0, 0);
                    Dw[T] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, wlo, KSI ? Dw[T] : z, 0, 0, 0);
                }
            }
        };
        ks(std::integral_constant<int, 0>{});
        ks(std::integral_constant<int, 1>{});
        ks(std::integral_constant<int, 2>{});
        ks(std::integral_constant<int, 3>{});
        ks(std::integral_constant<int, 4>{});
        ks(std::integral_constant<int, 5>{});
        ks(std::integral_constant<int, 6>{});
        ks(std::integral_constant<int, 7>{});
#pragma unroll
        for (int T = 0; T < TT; ++T) {
            f32x4 Dm = z;
            if constexpr (Q::MIN) {
                const float2 S = *reinterpret_cast<const float2*>(ss + T * SSB + 8 * lane);
                Dm = __builtin_amdgcn_mfma_f32_16x16x4f32(S.x, w.wm[0], z, 0, 0, 0);
                Dm = __builtin_amdgcn_mfma_f32_16x16x4f32(S.y, w.wm[1], Dm, 0, 0, 0);
            }
            if constexpr (!Q::BLOCKS) {
                const f32x4 f = exps(T, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float v = (D[0][T][i] + D[1][T][i]) + (D[2][T][i] + D[3][T][i]);
                    if constexpr (Q::SPLITW) v += __builtin_fmaf(Dl[T][i], 1.0f / LO, Dw[T][i]);
                    else v = __builtin_fmaf(Dl[T][i], 1.0f / LO, v);
                    add(T, i, __builtin_fmaf(w.d, v, Dm[i]), f[i]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    add(T, i, Q::MIN ? __builtin_fmaf(Dm[i], 32.0f, Dl[T][i]) : Dl[T][i], 1.0f);
            }
        }
    };

    // the sums of tile ct, step n of the work-group its last one here
    auto flush = [&](int n) __attribute__((always_inline)) {
        const Parts ps = ONE && per == nst ? Parts{0, 1} : tile_parts(ct, nst, per);
        const bool split = ps.n > 1;
#pragma unroll
        for (int T = 0; T < TT; ++T) acc[T] += acc2[T];
        // exchanged in the buffer just read: the next copies into it come after
        // the next step's barrier
        f32x4* const gs = reinterpret_cast<f32x4*>(lds + (n % TH::NB) * TH::BUF);
        if constexpr (KG > 1) {  // the groups' sums, added in group order
            __syncthreads();
#pragma unroll
            for (int T = 0; T < TT; ++T)
                if (kg > 0) gs[(wave * TT + T) * 64 + lane] = acc[T];
            __syncthreads();
            if (kg == 0) {
#pragma unroll
                for (int k = 1; k < KG; ++k)
#pragma unroll
                    for (int T = 0; T < TT; ++T) acc[T] += gs[((k * RW + rw) * TT + T) * 64 + lane];
            }
        }
        if constexpr (PAIR) {  // the up waves hand their sums to the gate waves
            __syncthreads();
#pragma unroll
            for (int T = 0; T < TT; ++T)
                if (kg == 0 && up && !split) gs[(wave * TT + T) * 64 + lane] = acc[T];
            __syncthreads();
        }
        // lane (c, q): row c of the wave's tile, tokens 16 T + 4 q + i (m0, opaque: the
        // compiler would keep every address in registers through the steps)
        int m0 = 4 * q;
        asm volatile("" : "+v"(m0));
        const int cols = PAIR ? 2 * a.N : a.N, nr = rt.n0 + wrow + c;
        if (kg > 0 || (PAIR && up && !split) || nr >= rt.rows) return;
        if (split) {
            float* const out = a.part + (size_t)(blockIdx.x - ps.first) * a.M * cols + rt.col + nr;
#pragma unroll
            for (int T = 0; T < TT; ++T)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int m = 16 * T + m0 + i;
                    if (m < a.M) out[(size_t)m * cols + (up ? a.N : 0)] = acc[T][i];
                }
            return;
        }
#pragma unroll
        for (int T = 0; T < TT; ++T) {
            f32x4 v = acc[T];
            if constexpr (PAIR) {
                const f32x4 u = gs[((rw + RW / 2) * TT + T) * 64 + lane];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = silu_mul(v[i], u[i]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = 16 * T + m0 + i;
                if (m < a.M) a.y[(size_t)m * a.N + rt.col + nr] = PAIR ? v[i] : biased(a, v[i], m, nr);
            }
        }
    };

#pragma unroll
    for (int i = 0; i < TH::NB - 1; ++i)
        if (s0 + i < s1) issue(i);
    bool stored = false;  // the step before ended a tile: its stores are under way too
    for (int s = s0; s < s1; ++s) {
        const int n = s - s0, nj = cj + 1 == nst ? 0 : cj + 1;
        wait((ONE || !stored) && s + 1 < s1 && (KG == 1 || KG * nj + kg < nsb));
        __syncthreads();
        if (s + TH::NB - 1 < s1) issue(n + TH::NB - 1);
        const int sb = KG * cj + kg;
        if (KG == 1 || sb < nsb) compute(sb, n);
        cj = nj;
        if constexpr (ONE) continue;
        stored = nj == 0;
        if (!stored || s + 1 == s1) continue;
        flush(n);
        rt = row_tile<PAIR>(a, ++ct, TH::BN);
        rsh = row_shift();
#pragma unroll
        for (int T = 0; T < TT; ++T) acc[T] = acc2[T] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    flush(s1 - 1 - s0);
}

// y of the tiles in parts, added in order: a work-group per tile and 256 R of
// its results.  R = 4 where a tile has few parts (a head's thousands of
// work-groups of one result per thread, most with nothing to add, took 10 us),
// else 1: a thread's loads are a serial chain of few at a time.
template <bool PAIR, int R>
__global__ __launch_bounds__(256) void reducet_kernel(MmqArgs a, int bn, int nst, int per) {
    const Parts ps = tile_parts(blockIdx.x, nst, per);
    if (ps.n == 1) return;
    const RowTile rt = row_tile<PAIR>(a, blockIdx.x, bn);
    const int nc = PAIR ? bn / 2 : bn, cols = PAIR ? 2 * a.N : a.N;
    const size_t slab = (size_t)a.M * cols;
    const float* p[R];
    float v[R], u[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {  // past the end: the last one's values, not stored
        const int i = blockIdx.y * (256 * R) + 256 * k + threadIdx.x;
        p[k] = a.part + (size_t)min(i / nc, a.M - 1) * cols + rt.col + min(rt.n0 + i % nc, rt.rows - 1);
        v[k] = p[k][0];
        u[k] = PAIR ? p[k][a.N] : 0.0f;
    }
#pragma unroll(R == 1 ? 8 : 1)
    for (int z = 1; z < ps.n; ++z)
#pragma unroll
        for (int k = 0; k < R; ++k) {
            v[k] += p[k][z * slab];
            if constexpr (PAIR) u[k] += p[k][z * slab + a.N];
        }
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int i = blockIdx.y * (256 * R) + 256 * k + threadIdx.x, m = i / nc, n = rt.n0 + i % nc;
        if (m >= a.M || n >= rt.rows) continue;
        if constexpr (PAIR) a.y[(size_t)m * a.N + n] = silu_mul(v[k], u[k]);
        else a.y[(size_t)m * cols + rt.col + n] = biased(a, v[k], m, n);
    }
}
template <bool PAIR>
void reducet(const MmqArgs& a, int bn, int nst, int per, hipStream_t st) {
    const int tiles = row_tiles(a, bn), n = a.M * (PAIR ? bn / 2 : bn);
    if (mmqt_parts(nst, per) <= 3)
        hipLaunchKernelGGL((reducet_kernel<PAIR, 4>), dim3(tiles, (n + 1023) / 1024), dim3(256), 0, st, a,
                           bn, nst, per);
    else
        hipLaunchKernelGGL((reducet_kernel<PAIR, 1>), dim3(tiles, (n + 255) / 256), dim3(256), 0, st, a,
                           bn, nst, per);
}

template <int F, int TT, int RW, int KG>
hipError_t go(const MmqArgs& a, int per, hipStream_t st) {
    const int tiles = row_tiles(a, 16 * RW), nst = mmqt_steps(a.K, KG), total = tiles * nst;
    const bool parts = mmqt_parts(nst, per) > 1;
    const dim3 grid((total + per - 1) / per), wg(64 * RW * KG);
    auto run = [&](auto pair) {
        constexpr bool P = decltype(pair)::value;
        if (nst % per == 0)
            hipLaunchKernelGGL((mmqt_kernel<F, P, TT, RW, KG, true>), grid, wg, 0, st, a, per, total);
        else
            hipLaunchKernelGGL((mmqt_kernel<F, P, TT, RW, KG, false>), grid, wg, 0, st, a, per, total);
        if (parts) reducet<P>(a, 16 * RW, nst, per, st);
    };
    if (a.mm == MM_PAIR) run(std::true_type{});
    else run(std::false_type{});
    return hipGetLastError();
}
// Work-groups of 256, 128 or 64 rows, each in wave groups of as many waves as
// fit: has<F, TT>(rows) is the group count, 0 where two buffers do not fit LDS.
template <int F, int TT, int RW, int KG>
constexpr bool fits() {
    return 2 * KG * (16 * RW * TQ<F>::PPR * 16 + TT * (XSB + SSB)) <= 160 * 1024;
}
template <int F, int TT>
constexpr int groups(int rows) {
    return rows == 256   ? (fits<F, TT, 16, 1>() ? 1 : 0)
           : rows == 128 ? (fits<F, TT, 8, 2>() ? 2 : fits<F, TT, 8, 1>() ? 1 : 0)
           : rows == 64  ? (fits<F, TT, 4, 2>() ? 2 : 0)
                         : 0;
}
template <int F, int TT>
hipError_t go_f(const MmqArgs& a, int rows, int per, hipStream_t st) {
    if constexpr (groups<F, TT>(256) != 0) {
        if (rows == 256) return go<F, TT, 16, 1>(a, per, st);
    }
    if constexpr (groups<F, TT>(128) != 0) {
        if (rows == 128) return go<F, TT, 8, groups<F, TT>(128)>(a, per, st);
    }
    if constexpr (groups<F, TT>(64) != 0) {
        if (rows == 64) return go<F, TT, 4, 2>(a, per, st);
    }
    return hipErrorInvalidValue;
}
template <class R, class Fn>
R with_thin(int dtype, R dflt, Fn&& fn) {
    if (dtype == Q3_K) return dflt;
    return with_format(dtype, dflt, [&](auto f) -> R {
        if constexpr (decltype(f)::value == Q3_K) return dflt;
        else return fn(f);
    });
}

}  // namespace

bool mmqt_supported(int dtype) { return with_thin(dtype, false, [](auto) { return true; }); }
int mmqt_groups(int dtype, int M, int rows) {
    return with_thin(dtype, 0, [&](auto f) {
        constexpr int F = decltype(f)::value;
        return M <= 16 ? groups<F, 1>(rows) : groups<F, 2>(rows);
    });
}
int mmqt_row_tiles(const MmqArgs& a, int rows) { return row_tiles(a, rows); }
size_t mmqt_xop_bytes(int M, int K) { return (size_t)((M + 15) / 16) * (K / 256) * XSB; }
size_t mmqt_sum_bytes(int M, int K) { return (size_t)((M + 15) / 16) * (K / 256) * SSB; }

hipError_t launch_xprept(int dtype, const float* x, int M, int K, uint8_t* xop, uint8_t* xs,
                         hipStream_t st) {
    const dim3 grid(K / 256, (M + 15) / 16);
    if (dtype == Q6_K)
        hipLaunchKernelGGL(xprept_kernel<1>, grid, dim3(256), 0, st, x, M, K, xop, xs);
    else if (dtype == Q4_K || dtype == Q5_K)
        hipLaunchKernelGGL(xprept_kernel<0>, grid, dim3(256), 0, st, x, M, K, xop, xs);
    else
        hipLaunchKernelGGL(xprept_kernel<2>, grid, dim3(256), 0, st, x, M, K, xop, xs);
    return hipGetLastError();
}

hipError_t launch_mmqt(int dtype, const MmqArgs& a, int rows, int per, hipStream_t st) {
    if (a.M > 32 || a.K % 256 != 0 || per < 1) return hipErrorInvalidValue;
    return with_thin(dtype, hipErrorInvalidValue, [&](auto f) {
        constexpr int F = decltype(f)::value;
        return a.M <= 16 ? go_f<F, 1>(a, rows, per, st) : go_f<F, 2>(a, rows, per, st);
    });
}

}  // namespace fq
