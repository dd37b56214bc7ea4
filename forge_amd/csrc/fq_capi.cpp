// fq_capi.cpp -- the extern "C" entry points declared in include/forge_q.h:
// argument validation, launch planning and the per-stream scratch memory.
//
// Dispatch by token count (run_matmul): M = 1 runs the batch-1 GEMV kernels
// (fq_gemvp.hip over GGUF bytes or the aligned layout, fq_gemvt.hip for Q8_0
// matrices of 64k rows and more on the aligned layout, the row-step kernels
// of fq_gemv1.hip under about 4 MB of weights); M = 2..4
// the same batch-1 kernels with each weight unit dotted with every token;
// M = 2..16 (by format and shape) the band kernel of fq_mmqs.hip
// (Q6_K M = 4 on wide matrices of 24 to 32 MiB: three tokens, then the fourth);
// M = 4..16 on matrices of 24 to 48 MiB and more and M = 17..32 the kernel of
// fq_mmqt.hip; M > 32 the prefill kernels
// of fq_mmqk.hip and fq_mmqp.hip (rows in 16-byte chunks, K a multiple of 256); the rest --
// the reference's batched GEMV (1 < M <= 32) and dequant + GEMM prefill
// (M > 32), matmul.cpp:1150-1286 -- the int8 and fp16 MFMA kernels of
// fq_mmqi.hip and fq_mmq.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <cstdio>
#include <cstdint>
#include <map>
#include <memory>
#include <vector>
#include <tuple>
#include <mutex>
#include <utility>

#include "../../include/forge_q.h"
#include "fq_kernels.h"
#include "fq_pack.h"

namespace {

thread_local int g_last_hip = 0;

int hip_fail(hipError_t e) {
    g_last_hip = (int)e;
    return FQ_ERR_HIP;
}

struct Geometry {
    int be, bb, ng;
};

bool geometry(uint32_t dtype, Geometry& g) {
    switch (dtype) {
        case FQ_DTYPE_Q4_0: g = {32, 18, 1}; return true;
        case FQ_DTYPE_Q4_1: g = {32, 20, 1}; return true;
        case FQ_DTYPE_Q8_0: g = {32, 34, 1}; return true;
        case FQ_DTYPE_Q4_K: g = {256, 144, 2}; return true;
        case FQ_DTYPE_Q6_K: g = {256, 210, 4}; return true;
        case FQ_DTYPE_Q5_0: g = {32, 22, 1}; return true;
        case FQ_DTYPE_Q5_1: g = {32, 24, 1}; return true;
        case FQ_DTYPE_Q3_K: g = {256, 110, 4}; return true;
        case FQ_DTYPE_Q5_K: g = {256, 176, 2}; return true;
        case FQ_DTYPE_IQ4_NL: g = {32, 18, 1}; return true;
        default: return false;
    }
}

// Whether a row's bytes fit the kernels' int.
bool row_fits(const Geometry& g, int K) { return (int64_t)(K / g.be) * g.bb <= INT32_MAX; }

// Formats with the aligned packed layout (fq_pack.h).
bool packable(uint32_t dtype) { return fq::packed_row_bytes((int)dtype, 256) > 0; }

struct DevInfo {
    int cus = 0;
    size_t lds = 0;
};

DevInfo device_info(int dev) {
    static std::mutex mu;
    static std::map<int, DevInfo> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(dev);
    if (it != cache.end()) return it->second;
    DevInfo d;
    if (hipDeviceGetAttribute(&d.cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) d.cus = 0;
    int lds = 0;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) lds = 0;
    d.lds = (size_t)lds;
    if (d.cus <= 0) d.cus = 256;
    if (d.lds == 0) d.lds = 64 * 1024;
    cache[dev] = d;
    return d;
}

// Device scratch per (device, stream, slot) for the MFMA path (slot 0: token
// operands, group sums, exponents and split-K partial slabs) and the GGUF
// fused FFN / QKV (slot 1: the gate/up or per-matrix rows).
//
// A call holds its slot's lock (StreamScratch::Lease) from taking the pointer
// until its launches are enqueued, so two host threads sharing a stream never
// see a buffer change under them.  The buffer only grows, at least doubling;
// a superseded buffer is not freed inside a compute call (queued work may
// still read it, and waiting for it would block the host mid-stream): it is
// kept until fq_release_workspace(), so the workspace of a stream holds less
// than twice its largest request.  fq_reserve_workspace() sizes it up front;
// during HIP-graph capture a call that would have to grow it fails with
// FQ_ERR_WORKSPACE instead of allocating.
struct StreamScratch {
    std::mutex mu;
    uint8_t* p = nullptr;
    size_t n = 0;
    std::vector<uint8_t*> retired;

    class Lease {
      public:
        explicit Lease(StreamScratch& s) : lk_(s.mu), s_(s) {}
        // the slot's buffer, at least `bytes` long
        int get(size_t bytes, hipStream_t st, uint8_t** out) {
            if (s_.n < bytes) {
                hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
                if (st && hipStreamIsCapturing(st, &cs) == hipSuccess &&
                    cs != hipStreamCaptureStatusNone)
                    return FQ_ERR_WORKSPACE;
                const size_t want = std::max(bytes, 2 * s_.n);
                uint8_t* np = nullptr;
                const hipError_t e = hipMalloc(reinterpret_cast<void**>(&np), want);
                if (e != hipSuccess) return hip_fail(e);
                if (s_.p) s_.retired.push_back(s_.p);
                s_.p = np;
                s_.n = want;
            }
            *out = s_.p;
            return FQ_OK;
        }
        size_t held() const { return s_.n; }

      private:
        std::unique_lock<std::mutex> lk_;
        StreamScratch& s_;
    };
};

std::mutex g_scratch_mu;
std::map<std::tuple<int, hipStream_t, int>, std::unique_ptr<StreamScratch>> g_scratch;

StreamScratch& stream_scratch(int dev, hipStream_t st, int slot) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    auto& p = g_scratch[{dev, st, slot}];
    if (!p) p.reset(new StreamScratch);
    return *p;
}

// Workspace bytes of the MFMA path for one call (the same plan run_mmq makes).
struct MmqPlan {
    int Tp, NC, shape, gx, gy, splits;
    size_t xop_b, xsum_b, ex_b, part_b, total;
};

MmqPlan plan_mmq(int M, int K, int N, int cus) {
    MmqPlan p{};
    p.Tp = (M + 15) / 16;
    p.NC = (K + 63) / 64;
    p.shape = p.Tp == 1 ? fq::MMQ_SMALL1 : p.Tp == 2 ? fq::MMQ_SMALL2
              : p.Tp <= 4 ? fq::MMQ_MID : fq::MMQ_BIG;
    int bn = 0, bm = 0;
    fq::mmq_shape(p.shape, &bn, &bm);
    p.gx = (N + bn - 1) / bn;
    p.gy = (p.Tp + bm / 16 - 1) / (bm / 16);
    const long tiles = (long)p.gx * p.gy;
    // K-splits only when the tiles alone leave CUs idle, to about two
    // work-groups per CU for the 128x128 prefill tiles and three for the
    // small-batch tiles (measured: cfg4 448 tiles fastest unsplit, 128 tiles
    // with 4 splits; 18944-row Q5_K at M = 8 41 -> 37 us with 6 splits)
    const long per_cu = p.shape == fq::MMQ_BIG ? 2 : 3;
    int splits = tiles >= cus ? 1
                              : (int)std::max(1L, std::min<long>((per_cu * cus + tiles - 1) / tiles, 8));
    p.splits = std::max(1, std::min(splits, p.NC / 4));
    p.xop_b = (size_t)p.Tp * p.NC * 2048 * 2;
    p.xsum_b = (size_t)p.Tp * p.NC * 64 * 4;
    p.ex_b = (size_t)p.Tp * p.NC * 16 * 4;
    p.part_b = p.splits > 1 ? (size_t)p.splits * M * N * 4 : 0;
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    p.total = 256 + al(p.xop_b) + al(p.xsum_b) + al(p.ex_b) + al(p.part_b);
    return p;
}

// Rows per band and K-splits of the small-batch band kernel.  Short rows:
// bands of up to four 16-row tiles, as few rows per band as fill every CU,
// unsplit.  Long rows (32 super-blocks and more) with few rows: each band
// re-reads the token operands of all of K, 4 KiB per 64 elements, for as
// few as 16 rows, so the bands take four tiles and K is split to fill the
// CUs (each wave keeping at least one super-block per split; the slabs are
// summed in split order).  Measured at 3584 x 18944 (M = 4 / 16): 30.3 /
// 30.8 us unsplit on 16-row bands, 27.1 / 28.0 us on 64-row bands in four
// splits; at K = 4096 every split measured slower.
int mmqs_plan(int N, int K, int cus, int* rows_per_wg, int mt) {
    const int nsb = K / 256;
    const long bands4 = (N + 16 * mt - 1) / (16 * mt);
    if (nsb >= 32 && 2 * bands4 <= cus) {
        *rows_per_wg = 16 * mt;
        const int s = (int)std::max(1L, std::min<long>(cus / bands4, nsb / 8));
        const int sps = (nsb + s - 1) / s;
        return (nsb + sps - 1) / sps;
    }
    *rows_per_wg = 16 * std::min(mt, std::max(1, (N + 16 * cus - 1) / (16 * cus)));
    return 1;
}

// Workspace bytes of a band-kernel call: the token operands of plan_mmq's
// single token tile and, when K is split, the slabs.
size_t mmqs_need(int M, int K, int N, int cus, int mt) {
    const MmqPlan pl = plan_mmq(M, K, N, cus);
    int rpw = 0;
    const int splits = mmqs_plan(N, K, cus, &rpw, mt);
    const size_t part_b = splits > 1 ? (size_t)splits * M * N * 4 : 0;
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    return 256 + al(pl.xop_b) + al(pl.xsum_b) + al(pl.ex_b) + al(part_b);
}

// Bytes of the fixed workspace of fq_matmul_transB_noalloc.
constexpr size_t kNoAllocBytes = (size_t)64 << 20;

// Workspace bytes and K-splits of the prefill kernels (M > 32, K a multiple
// of 256): one work-group per CU and tile, each split a multiple of four
// 64-element steps.
struct MmqpPlan {
    int splits;
    size_t xop_b, ex_b, sum_b, part_b, q6c_b, total;
};

// Of `splits` slabs; cols: columns of a partial slab, q6_rows: Q6_K rows to
// rewrite (0: another format).
MmqpPlan mmqp_sizes(uint32_t dtype, int M, int K, int cols, int q6_rows, int splits) {
    MmqpPlan p{};
    const int Tn = (M + 31) / 32;
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    p.splits = splits;
    p.xop_b = (size_t)Tn * K * 64 * 2;
    p.ex_b = (size_t)M * 4;
    // sub-block sums (formats with a min term): floats, or mmqk's hi + lo
    p.sum_b = (size_t)Tn * (fq::mmqk_supported((int)dtype) ? fq::mmqk_sum_bytes((int)dtype, K) : (size_t)K * 4);
    p.q6c_b = (size_t)fq::mmqp_q6c_bytes(q6_rows, K);  // Q6_K rows as 36-byte blocks
    p.part_b = splits > 1 ? (size_t)splits * M * cols * 4 : 0;
    p.total = 256 + al(p.xop_b) + al(p.ex_b) + al(p.sum_b) + al(p.q6c_b) + al(p.part_b);
    return p;
}

// The fewest tokens the prefill kernels can run at a time with the bits of the
// whole call: with a minimum per block (fq_mmqp.hip), a token's additions come in
// an order that depends on which 32 of a wave's 64 tokens it is in, and whether
// both hold tokens.
int prefill_granule(uint32_t dtype) { return dtype == FQ_DTYPE_Q4_1 || dtype == FQ_DTYPE_Q5_1 ? 64 : 1; }

// Slabs of one prefill call at most (they only even out the rounds of
// work-groups: of 2 million sizes up to 4096 x 160000 x 20480 under 1 % would
// take more, 9 % faster at best by the estimate below), and rewritten Q6_K rows
// of several matrices in one launch (gate and up of 18944 x 3584: 146 MiB): what
// fq_reserve_workspace has to set aside.
constexpr size_t kMaxSlabs = (size_t)256 << 20, kMaxRewrite = (size_t)160 << 20;

// Estimated time of a prefill launch over K in sp splits (0: some would be
// empty): rounds of work-groups x (steps per split at 2.1 us, 3 us to fill the
// pipeline and store), and for a split the launch of the slab sum.  Beside it each
// slab element is written and read once at 4 TB/s, kSlabUs per element and slab.
// (Counting steps alone took 16 splits for a 14336-row gate/up pair at K = 4096,
// M = 77: 117 + 23 us against 80 + 7 with 2, and 8 for a 6144-row QKV at M = 512:
// 82 + 19 us against 72 + 8.)
constexpr double kSlabUs = 4.0 / 4e6;
double mmqp_us(long tiles, int nsteps, int sp, int cus) {
    const int sps = ((nsteps + sp - 1) / sp + 3) & ~3;
    if ((nsteps + sps - 1) / sps != sp) return 0.0;
    return (double)((tiles * sp + cus - 1) / cus) * (2.1 * sps + 3.0) + (sp > 1 ? 4.0 : 0.0);
}

// tiles_n: work-groups along the rows.  one: a single matrix, whose plan
// fq_matmul_transB_noalloc runs in a fixed array, fewer tokens at a time if
// need be (run_prefill): so the slabs of the fewest have to fit there where the
// operands of all do.
MmqpPlan plan_mmqp(uint32_t dtype, int M, int K, long tiles_n, int cols, int q6_rows, bool one, int cus) {
    const int nsteps = K / 64;
    const int tm = fq::mmqp_tile_tokens();
    const long tiles = tiles_n * ((M + tm - 1) / tm);
    MmqpPlan p = mmqp_sizes(dtype, M, K, cols, q6_rows, 1);
    const bool fits = p.total <= kNoAllocBytes || dtype == FQ_DTYPE_Q5_K;
    double best = 0.0;  // the split count of the smallest estimated time
    for (int sp = 1; sp <= std::max(1, std::min(16, nsteps / 4)); ++sp) {
        double t = mmqp_us(tiles, nsteps, sp, cus);
        if (t == 0.0) continue;
        if (sp > 1) {
            if ((size_t)sp * M * cols * 4 > kMaxSlabs) break;
            if (one && fits &&
                mmqp_sizes(dtype, std::min(M, prefill_granule(dtype)), K, cols, q6_rows, sp).total > kNoAllocBytes)
                break;
            t += (sp + 1.0) * M * cols * kSlabUs;
        }
        if (sp == 1 || t < best) {
            best = t;
            p.splits = sp;
        }
    }
    return mmqp_sizes(dtype, M, K, cols, q6_rows, p.splits);
}

// No plan_mmqp of up to M tokens, K elements (whole super-blocks) and cols
// columns has more bytes of slabs: for every K and tile count, a split count is
// the best only while there are few enough elements that its slabs cost less than
// the time they save over each smaller count.
size_t mmqp_max_slabs(int M, int K, int64_t cols, int cus) {
    const int tm = fq::mmqp_tile_tokens(), tn = fq::mmqp_tile_rows();
    const long tiles_max = (long)((M + tm - 1) / tm) * (long)((cols + tn - 1) / tn + 2);
    double most = 0.0;
    for (int nsteps = K / 64; nsteps >= 8; nsteps -= 4)
        for (long tiles = 1; tiles <= tiles_max; ++tiles) {
            const double n = std::min((double)M * (double)cols, (double)tiles * tm * tn);
            double us[17];
            for (int sp = 1; sp <= std::min(16, nsteps / 4); ++sp) {
                us[sp] = mmqp_us(tiles, nsteps, sp, cus);
                if (us[sp] == 0.0 || sp * n <= most) continue;
                double ns = n;
                for (int q = 1; q < sp; ++q)
                    if (us[q] != 0.0)
                        ns = std::min(ns, (us[q] - us[sp]) / ((q == 1 ? sp + 1 : sp - q) * kSlabUs) + 1.0);
                if (sp > 1) most = std::max(most, sp * ns);
            }
            if (most * 4.0 >= (double)kMaxSlabs) return kMaxSlabs;
        }
    return (size_t)(most * 4.0) + 64;
}

// M > 1 on the matrix cores: token operand preparation, then one tile per
// work-group (K-split when the tiles alone do not fill the chip).  The
// workspace is `fixed` (fixed_cap bytes) when given, else the stream's.
int run_mmq(uint32_t dtype, const Geometry& g, const float* x, const void* w, const float* bias,
            int bias_mode, int64_t bias_len, float* y, int M, int K, int N, int dev,
            const DevInfo& di, hipStream_t st, uint8_t* fixed, size_t fixed_cap) {
    const MmqPlan pl = plan_mmq(M, K, N, di.cus);
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    std::unique_ptr<StreamScratch::Lease> lease;
    uint8_t* buf = fixed;
    if (fixed) {
        if (pl.total > fixed_cap) return FQ_ERR_WORKSPACE;
    } else {
        lease.reset(new StreamScratch::Lease(stream_scratch(dev, st, 0)));
        const int rc = lease->get(pl.total, st, &buf);
        if (rc != FQ_OK) return rc;
    }
    fq::MmqArgs a{};
    a.w = static_cast<const uint8_t*>(w);
    a.xop = buf;
    a.xsum = reinterpret_cast<const float*>(buf + al(pl.xop_b));
    a.ex = reinterpret_cast<const int*>(buf + al(pl.xop_b) + al(pl.xsum_b));
    a.part = pl.splits > 1
                 ? reinterpret_cast<float*>(buf + al(pl.xop_b) + al(pl.xsum_b) + al(pl.ex_b))
                 : nullptr;
    a.y = y;
    a.bias = bias;
    a.bias_len = bias_mode ? bias_len : 0;
    a.bias_mode = bias_mode;
    a.M = M;
    a.N = N;
    a.K = K;
    a.NC = pl.NC;
    a.row_bytes = (K / g.be) * g.bb;
    hipError_t e = hipSuccess;
    if (pl.NC > 0) {  // K == 0 only writes the bias (or zeros)
        e = fq::launch_xprep((int)dtype, x, M, K, pl.NC, reinterpret_cast<_Float16*>(buf),
                             const_cast<float*>(a.xsum), const_cast<int*>(a.ex), st);
        if (e != hipSuccess) return hip_fail(e);
    }
    e = fq::launch_mmq((int)dtype, a, pl.shape, pl.gx, pl.gy, pl.splits, st);
    return e == hipSuccess ? FQ_OK : hip_fail(e);
}

// The matrices of one prefill call: fq::MM_ONE w[0]; fq::MM_PAIR the gate and
// up matrices w[0], w[1] of n[0] rows each; fq::MM_CAT up to three whose
// results are concatenated (empty ones last).
struct Mats {
    int mm;
    const void* w[3];
    int n[3];
};

// Prefill on v_mfma_f32_32x32x16_f16 (fq_mmqk.hip for Q4_K and Q5_K,
// fq_mmqp.hip for the other formats): rows that are whole 16-byte chunks (K a
// multiple of 256, 16-byte aligned weights, under 4 GiB of them: the copies
// take 32-bit offsets): per-token operands, then one work-group per CU and
// tile (K-split while the tiles leave CUs idle).  Q6_K rows are first
// rewritten into 36-byte blocks in the workspace.  kNotTaken: another kernel
// runs the call (several matrices: one call each, also where the workspace
// cannot grow to this call's size under graph capture).
constexpr int kNotTaken = -1;
int run_prefill(uint32_t dtype, const Geometry& g, const float* x, const Mats& ms,
                const float* bias, int bias_mode, int64_t bias_len, float* y, int M, int K, int N,
                int dev, const DevInfo& di, hipStream_t st, uint8_t* fixed, size_t fixed_cap) {
    const bool q6k = dtype == FQ_DTYPE_Q6_K, mmqk = fq::mmqk_supported((int)dtype);
    if (!(mmqk || fq::mmqp_supported((int)dtype)) || M <= 32 || K <= 0 || K % 256 != 0)
        return kNotTaken;
    const int64_t rb = q6k ? fq::mmqp_q6c_bytes(1, K) : (int64_t)(K / g.be) * g.bb;
    int rows = 0;  // of all matrices
    for (int i = 0; i < 3; ++i) {
        const int n = ms.mm == fq::MM_PAIR && i < 2 ? ms.n[0] : ms.n[i];
        if (n == 0) continue;
        if ((!q6k && (reinterpret_cast<uintptr_t>(ms.w[i]) & 15) != 0) || n * rb >= ((int64_t)1 << 32))
            return kNotTaken;
        rows += n;
    }
    if (q6k && ms.mm != fq::MM_ONE && (size_t)fq::mmqp_q6c_bytes(rows, K) > kMaxRewrite) return kNotTaken;
    fq::MmqArgs a{};
    a.mm = ms.mm;
    a.w = static_cast<const uint8_t*>(ms.w[0]);
    a.w2 = static_cast<const uint8_t*>(ms.w[1]);
    a.w3 = static_cast<const uint8_t*>(ms.w[2]);
    a.n1 = ms.n[0];
    a.n2 = ms.n[1];
    a.n3 = ms.n[2];
    a.row_bytes = (K / g.be) * g.bb;
    a.N = N;
    a.K = K;
    const int cols = fq::mm_cols(a), q6_rows = q6k ? rows : 0;
    MmqpPlan pl = plan_mmqp(dtype, M, K, fq::mmqp_row_tiles(a), cols, q6_rows, ms.mm == fq::MM_ONE, di.cus);
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    std::unique_ptr<StreamScratch::Lease> lease;
    uint8_t* buf = fixed;
    int mc = M;  // tokens at a time
    if (fixed) {
        // The operands of all tokens have to fit (Q5_K: those of the fp16 MFMA
        // kernel may, which differ by a few per cent for rows of 46 thousand
        // elements); where the slabs beside them do not, the same launches run
        // for as many tokens as do: a token's sums do not depend on the others,
        // so the bits are those of the call on a stream's workspace (642 x 18944
        // x 14336: four splits, 194 MB of slabs).
        if (mmqp_sizes(dtype, M, K, cols, q6_rows, 1).total > fixed_cap &&
            !(dtype == FQ_DTYPE_Q5_K && plan_mmq(M, K, N, di.cus).total <= fixed_cap))
            return FQ_ERR_WORKSPACE;
        while (pl.total > fixed_cap && mc > prefill_granule(dtype)) {
            mc = mc > 64 ? (mc - 1) / 64 * 64 : mc / 2;
            pl = mmqp_sizes(dtype, mc, K, cols, q6_rows, pl.splits);
        }
        if (pl.total > fixed_cap) return FQ_ERR_WORKSPACE;
    } else {
        lease.reset(new StreamScratch::Lease(stream_scratch(dev, st, 0)));
        int rc = lease->get(pl.total, st, &buf);
        if (rc == FQ_ERR_WORKSPACE) {
            // capture on a workspace that another call sized: fewer tokens can
            // take more splits, one split takes the operands alone
            pl = mmqp_sizes(dtype, M, K, cols, q6_rows, 1);
            if (pl.total > lease->held()) return ms.mm != fq::MM_ONE ? kNotTaken : rc;
            rc = lease->get(pl.total, st, &buf);
        }
        if (rc != FQ_OK) return rc;
    }
    const int splits = pl.splits;
    hipError_t e = hipSuccess;
    if (q6k) {
        uint8_t* conv = buf + al(pl.xop_b) + al(pl.ex_b) + al(pl.sum_b) + al(pl.part_b);
        const uint8_t** w[3] = {&a.w, &a.w2, &a.w3};
        for (int i = 0; i < 3; ++i) {
            const int n = ms.mm == fq::MM_PAIR && i < 2 ? ms.n[0] : ms.n[i];
            if (n == 0) continue;
            e = fq::launch_q6c(*w[i], n, K, a.row_bytes, conv, st);
            if (e != hipSuccess) return hip_fail(e);
            *w[i] = conv;
            conv += n * rb;
        }
        a.row_bytes = (int)rb;
    }
    _Float16* const xop = reinterpret_cast<_Float16*>(buf);
    int* const ex = reinterpret_cast<int*>(buf + al(pl.xop_b));
    uint8_t* const sums = mmqk || dtype == FQ_DTYPE_Q4_1 || dtype == FQ_DTYPE_Q5_1
                              ? buf + al(pl.xop_b) + al(pl.ex_b)
                              : nullptr;
    a.xop = buf;
    a.ex = ex;
    a.xsum = reinterpret_cast<const float*>(sums);
    a.part = splits > 1 ? reinterpret_cast<float*>(buf + al(pl.xop_b) + al(pl.ex_b) + al(pl.sum_b))
                        : nullptr;
    a.bias_len = bias_mode ? bias_len : 0;
    a.bias_mode = bias_mode;
    for (int t0 = 0; t0 < M; t0 += mc) {
        const float* const xt = x + (size_t)t0 * K;
        a.M = std::min(mc, M - t0);
        a.y = y + (size_t)t0 * N;
        a.bias = bias_mode == 2 ? bias + (size_t)t0 * N : bias;
        if (fq::mmqk_fine((int)dtype))
            e = fq::launch_xprepk(xt, a.M, K, xop, sums, st);
        else
            e = fq::launch_xprep32(xt, a.M, K, xop, ex, mmqk ? nullptr : reinterpret_cast<float*>(sums),
                                   mmqk ? reinterpret_cast<_Float16*>(sums) : nullptr, q6k, st);
        if (e != hipSuccess) return hip_fail(e);
        e = mmqk ? fq::launch_mmqk((int)dtype, a, splits, st) : fq::launch_mmqp((int)dtype, a, splits, st);
        if (e == hipSuccess && splits > 1) e = fq::launch_reduce(a, splits, st);
        if (e != hipSuccess) return hip_fail(e);
    }
    return FQ_OK;
}

// Small batches with the token operands shared by the rows of a work-group
// (fq_mmqt.hip: every format but Q3_K).
struct MmqtPlan {
    int rows, per, parts;
    size_t xop_b, sum_b, part_b, total;
};

// Rows per tile and steps per work-group of the smallest estimated time:
// whole tiles, or the steps of all tiles shared out over the CUs (or over
// half, a quarter .. of them, with fewer parts of a tile), at most one
// work-group per CU: 1.5 us to fill the pipeline, the steps, 1 us per tile
// ended, and for tiles in parts their sum (3.5 us and each slab written and
// read at 4 TB/s).  A step's time is what 14336 x 4096 measured on 224
// work-groups (Q6_K without the product of its low parts, 4 % of it), or its
// weight bytes on all busy CUs at 5 TB/s (Q8_0 152064 x 3584 at M = 16: 134 us on
// 128 rows, 156 on 64).  Of Q8_0's tiles 128 rows run in one wave group and 64 in two:
// a step of either reads the same bytes, and where tiles outnumber the CUs 64 rows take
// as long per step, up to 16 tokens (at 1.3 us a step a pair of 17408 x 8192 took 98
// us on 64 rows at M = 3, 72 on 128, 18944 x 4096 48.8 and 39.2; fewer tiles, parts to
// sum: 3072 x 2816 12.6 on 64, 15.5 on 128).
//
// No plan takes more than the fixed array of fq_matmul_transB_noalloc, so that
// the plan is the same there (cap: what a workspace under capture holds).
MmqtPlan plan_mmqt(const fq::MmqArgs& a, uint32_t dtype, int cus, size_t cap = kNoAllocBytes) {
    const bool q6 = dtype == FQ_DTYPE_Q6_K, q8 = dtype == FQ_DTYPE_Q8_0, wide = a.M > 16;
    MmqtPlan p{};
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    p.xop_b = fq::mmqt_xop_bytes(a.M, a.K);
    p.sum_b = fq::mmqt_sum_bytes(a.M, a.K);
    const size_t ops_b = 256 + al(p.xop_b) + al(p.sum_b);
    const double sb_bytes = (double)a.row_bytes / (a.K / 256);
    double best = 0.0;
    for (int rows : {256, 128, 64}) {
        const int kg = fq::mmqt_groups((int)dtype, a.M, rows);
        if (kg == 0) continue;
        const int tiles = fq::mmqt_row_tiles(a, rows), nst = fq::mmqt_steps(a.K, kg);
        const double it = rows == 256 ? (q6 ? 2.7 : wide ? 2.6 : 2.0)
                          : rows == 128 ? (q6 ? (wide ? 2.2 : 1.7) : wide ? 1.6 : 1.7)
                                        : (q6 ? 1.8 : q8 && !wide && tiles > cus ? 1.8 : 1.3);
        const int whole = nst * ((tiles + cus - 1) / cus);
        const int64_t total = (int64_t)tiles * nst;
        if (total >= (int64_t)1 << 31) continue;
        for (int per = (int)((total + cus - 1) / cus);; per *= 2) {
            per = std::min(per, whole);
            const int parts = fq::mmqt_parts(nst, per);
            const size_t part_b = parts > 1 ? (size_t)parts * a.M * fq::mm_cols(a) * 4 : 0;
            if (parts <= 16 && ops_b + al(part_b) <= cap) {
                const double busy = (double)((total + per - 1) / per);
                const double step = std::max(it, busy * kg * rows * sb_bytes / 5e6);
                const double t = 1.5 + step * per + (double)((per + nst - 1) / nst) +
                                 (parts > 1 ? 3.5 + (parts + 1.0) * a.M * fq::mm_cols(a) * 4.0 / 4e6 : 0.0);
                if (p.rows == 0 || t < best) {
                    best = t;
                    p.rows = rows;
                    p.per = per;
                    p.parts = parts;
                    p.part_b = part_b;
                }
            }
            if (per == whole) break;
        }
    }
    p.total = ops_b + al(p.part_b);
    return p;
}

// Estimates of whole calls up to 16 tokens, us, for the choice between this kernel and
// the band kernel, fitted to 5632 .. 18944 rows x 1024 .. 8192 (this kernel: 5750 calls,
// 3.1 % rms, band: 840, 3.2 %).  thin: a super-block of 128 rows here (256 rows take
// 1.7 times as long, 64 0.66 where 128 run in two wave groups, 0.61 in one); band: a
// super-block of a 16-row tile there.
struct SmallUs {
    double thin, band;
};
SmallUs small_us(uint32_t dtype) {
    switch (dtype) {
        case FQ_DTYPE_Q4_0: return {1.00, 0.145};
        case FQ_DTYPE_Q4_1: return {1.04, 0.169};
        case FQ_DTYPE_Q8_0: return {1.30, 0.168};
        case FQ_DTYPE_Q5_0: return {1.24, 0.185};
        case FQ_DTYPE_Q5_1: return {1.41, 0.185};
        case FQ_DTYPE_IQ4_NL: return {1.27, 0.199};
        case FQ_DTYPE_Q4_K: return {0.91, 0.161};
        case FQ_DTYPE_Q5_K: return {1.02, 0.173};
        default: return {1.53, 0.246};  // Q6_K
    }
}
double thin_us(const MmqtPlan& p, const fq::MmqArgs& a, uint32_t dtype) {
    const double r = p.rows == 256                                ? 1.7
                     : p.rows == 128                              ? 1.0
                     : fq::mmqt_groups((int)dtype, a.M, 128) == 2 ? 0.66
                                                                  : 0.61;
    return 6.0 + r * small_us(dtype).thin * p.per * fq::mmqt_groups((int)dtype, a.M, p.rows) +
           (p.parts > 1 ? 4.6 + 0.37e-6 * (double)p.part_b : 0.0) +
           0.033e-6 * a.row_bytes * fq::mm_cols(a);
}

// Whether 4..32 tokens on one matrix of this size go there, up to 16 unless the
// band kernel is estimated faster by 4 %.  17..32 tokens
// always (the fp16 MFMA path: Q4_K 4096 x 4096 at M = 32 20.8 -> 14.1 us, 14336 x
// 4096 40.2 -> 24.0, Q8_0 40.5 -> 28.6, Q6_K 4096 x 14336 56.4 -> 30.3).  Up to
// 16 from 24 MiB of Q4_K and Q5_K, 48 of Q8_0, 32 of the others: below, the band
// kernel's bands fill the chip without a K split and its slab sum (M = 8: Q4_K
// 8192 x 4096, 19 MB, 12.6 us there, 13.5 here, 14336 x 4096, 33 MB, 18.7 and
// 16.3; Q6_K 28 MB 16.5 and 16.8, 48 MB 27.6 and 21.7; Q8_0 36 MB 14.1 and
// 15.3, 62 MB 23.5 and 20.0; Q4_0 33 MB 17.8 and 16.7, 38 MB 24.0 and 20.6;
// 152064 x 3584: Q4_0 132 and 96, Q8_0 171 and 131, Q6_K 211 and 127).
bool thin_takes(uint32_t dtype, int M, int64_t bytes) {
    if (!fq::mmqt_supported((int)dtype) || M < 4 || M > 32) return false;
    const int64_t mib = dtype == FQ_DTYPE_Q4_K || dtype == FQ_DTYPE_Q5_K ? 24
                        : dtype == FQ_DTYPE_Q8_0                        ? 48
                                                                        : 32;
    return M > 16 || bytes >= mib << 20;
}

// Whether a gate/up pair of such matrices goes there: as one matrix of both's rows,
// or two to four tokens, which otherwise take two launches and a SiLU pass (M = 4: Q4_0
// 5632 x 2048 18.4 -> 10.9 us, 18944 x 3584 52.4 -> 31.2; M = 2: 13.9 -> 10.8), but
// not two on large matrices of the formats whose batch-1 kernel then reads at
// nearly the rate of one token (M = 2: Q4_0 18944 x 3584 30.2 against 35.8, Q6_K
// 37.6 against 44.3, Q8_0 14336 x 4096 33.8 against 34.5).  Two tokens of other formats
// stay, also where two launches are faster (Q5_0 17408 x 2048 21.9 against 24.3): the
// batch-1 kernel's limbs err by 1.4..1.9e-6 there, this one by 1.6e-7.
bool thin_takes_pair(uint32_t dtype, int M, int64_t bytes) {
    if (!fq::mmqt_supported((int)dtype) || M < 2) return false;
    if (M == 2 && (dtype == FQ_DTYPE_Q4_0 || dtype == FQ_DTYPE_Q6_K || dtype == FQ_DTYPE_Q8_0))
        return bytes < 24 << 20;
    return M <= 4 || thin_takes(dtype, M, 2 * bytes);
}

// kNotTaken: another kernel runs the call (also where the workspace cannot grow
// to this one's operands under capture).  kSlower: estimated above limit_us.
constexpr int kSlower = -2;
int run_thin(uint32_t dtype, const Geometry& g, const float* x, const Mats& ms, const float* bias,
             int bias_mode, int64_t bias_len, float* y, int M, int K, int N, int dev,
             const DevInfo& di, hipStream_t st, uint8_t* fixed, size_t fixed_cap, double limit_us) {
    if (!fq::mmqt_supported((int)dtype) || M < 2 || M > 32 || K <= 0 || K % 256 != 0) return kNotTaken;
    const bool q6k = dtype == FQ_DTYPE_Q6_K;
    const int64_t rb = (int64_t)(K / g.be) * g.bb;
    for (int i = 0; i < 3; ++i) {
        const int n = ms.mm == fq::MM_PAIR && i < 2 ? ms.n[0] : ms.n[i];
        if (n == 0) continue;
        if ((reinterpret_cast<uintptr_t>(ms.w[i]) & (q6k ? 1 : 15)) != 0 ||
            n * rb + 16 >= ((int64_t)1 << 32))
            return kNotTaken;
    }
    fq::MmqArgs a{};
    a.mm = ms.mm;
    a.w = static_cast<const uint8_t*>(ms.w[0]);
    a.w2 = static_cast<const uint8_t*>(ms.w[1]);
    a.w3 = static_cast<const uint8_t*>(ms.w[2]);
    a.n1 = ms.n[0];
    a.n2 = ms.n[1];
    a.n3 = ms.n[2];
    a.row_bytes = (int)rb;
    a.M = M;
    a.N = N;
    a.K = K;
    MmqtPlan pl = plan_mmqt(a, dtype, di.cus);
    if (pl.rows == 0) return kNotTaken;
    if (thin_us(pl, a, dtype) > limit_us) return kSlower;
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    std::unique_ptr<StreamScratch::Lease> lease;
    uint8_t* buf = fixed;
    if (fixed) {
        if (pl.total > fixed_cap) return FQ_ERR_WORKSPACE;
    } else {
        lease.reset(new StreamScratch::Lease(stream_scratch(dev, st, 0)));
        int rc = lease->get(pl.total, st, &buf);
        if (rc == FQ_ERR_WORKSPACE) {
            // capture on a workspace that another call sized: fewer tokens can
            // take more parts (14336 x 4096 Q4_K pair, 17 tokens 8.3 MB, 32 0.5)
            pl = plan_mmqt(a, dtype, di.cus, std::min(kNoAllocBytes, lease->held()));
            if (pl.rows == 0) return kNotTaken;
            rc = lease->get(pl.total, st, &buf);
        }
        if (rc != FQ_OK) return rc;
    }
    a.xop = buf;
    uint8_t* const sums = buf + al(pl.xop_b);
    a.xsum = reinterpret_cast<const float*>(sums);
    a.part = pl.parts > 1 ? reinterpret_cast<float*>(sums + al(pl.sum_b)) : nullptr;
    a.y = y;
    a.bias = bias;
    a.bias_len = bias_mode ? bias_len : 0;
    a.bias_mode = bias_mode;
    hipError_t e = fq::launch_xprept((int)dtype, x, M, K, buf, sums, st);
    if (e != hipSuccess) return hip_fail(e);
    e = fq::launch_mmqt((int)dtype, a, pl.rows, pl.per, st);
    return e == hipSuccess ? FQ_OK : hip_fail(e);
}

// Whether the band kernel (fq_mmqs.hip) takes a call of 2..16 tokens; block:
// a 32-element-block format there, ahead of the batch-1 kernel with several
// tokens.
struct BandRule {
    bool block, takes;
};
BandRule band_rule(uint32_t dtype, const Geometry& g, int M, int K, int N, const void* w, int cus) {
    // Q4_0 and Q8_0: rows that start 16-byte aligned
    // (K a multiple of 256), 5..16 tokens, or 4 from 16 MB (below, other
    // kernels take M = 4 0.4-0.7 us faster for Q4_0; Q8_0 only
    // while the bands number at most one per CU: lm_head 157 us on the
    // batch-1 kernel against 173), or, Q4_0 only, 3 from 16 MB with K of
    // 14336 and more (3584 x 18944: 26.4 us on the batch-1 kernel).  At 3
    // and 4 tokens Q4_0 needs at most one band per CU or at least eight
    // (152064 rows at M = 4 129 against 151 us); from 5 tokens any count
    // (18944 rows in three-tile bands, below: 24.5 against 27.5 us at M =
    // 8).  Q8_0 takes any count (the fp16 MFMA path is slower at every one
    // measured: 14336 x 4096 at M = 8 24.1 against 37.6 us)
    const int bmt = fq::mmqs_max_tiles((int)dtype);
    const long bands = ((long)N + 16 * bmt - 1) / (16 * bmt);
    // (Q4_1 as Q4_0)
    const bool q4x = dtype == FQ_DTYPE_Q4_0 || dtype == FQ_DTYPE_Q4_1;
    const bool blk_band = (q4x || dtype == FQ_DTYPE_Q8_0) && K % 256 == 0 &&
                          (reinterpret_cast<uintptr_t>(w) & 15) == 0 &&
                          (M >= 5 ||
                           ((M == 4 ? q4x || bands <= cus : M == 3 && q4x && K >= 14336) &&
                            (int64_t)N * (K / g.be) * g.bb >= (16 << 20))) &&
                          (dtype == FQ_DTYPE_Q8_0 || M >= 5 || bands <= cus ||
                           bands >= 8L * cus);
    // Q5_K (rows 16-byte aligned): 5..16 tokens; 4 while the bands number at
    // most one per CU or at least eight per CU (18944 x 3584: 33.4 against
    // 31.7 us on the fp16 MFMA path); 3 at K >= 14336 or eight bands per CU
    // and more (3584 x 18944 54.1 -> 27.0 us at M = 4, lm_head at M = 3 166
    // against about 150; 18944 x 3584 at M = 3 26.0 against 33); 2 at K >=
    // 14336 (3584 x 18944: 53.9 on the fp16 MFMA path; lm_head at M = 2
    // 111.5 against about 150 stays there)
    const bool al16 = K % 256 == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0;
    // Q5_0 and IQ4_NL: K >= 14336 from 2 tokens (3584 x 18944 at M = 2..8:
    // 55.3 -> 27.9 and 47.4 -> 28.3 us), or 4..16 tokens in one round of
    // bands (14336 x 4096 at M = 8: 33.2 -> 21.3, 29.2 -> 21.6); 18944 rows
    // at M = 8 measured slower (35.5 against 32.7, 36.1 against 28.4).
    // Q5_1 (160 KB of LDS per work-group): K >= 14336 only (43.8 -> 37.5;
    // lm_head at M = 8 216 against 159)
    const bool q5x_band =
        al16 && M >= 2 &&
        (((dtype == FQ_DTYPE_Q5_0 || dtype == FQ_DTYPE_IQ4_NL) &&
          (K >= 14336 || (M >= 4 && bands <= cus))) ||
         (dtype == FQ_DTYPE_Q5_1 && K >= 14336));
    // Q3_K (rows at even addresses): K >= 14336 from two tokens (3584 x 18944
    // 61 -> 28.7 us), 4..16 tokens for any row count (152064 x 3584 at M = 8
    // 262 -> 184, 14336 x 4096 41.9 -> 32.0; equal at M = 4)
    const bool q3k_band = dtype == FQ_DTYPE_Q3_K && K % 256 == 0 &&
                          (reinterpret_cast<uintptr_t>(w) & 1) == 0 && M >= 2 &&
                          (K >= 14336 || M >= 4);
    const bool q5k_band =
        q3k_band || (dtype == FQ_DTYPE_Q5_K && al16 &&
         (M >= 5 || (M == 4 && (bands <= cus || bands >= 8L * cus)) ||
          (M == 3 && (K >= 14336 || bands >= 8L * cus)) || (M == 2 && K >= 14336))) ||
        q5x_band;
    // Q4_K beyond one band per CU only above 8 tokens, which the int8 kernel
    // does not take (18944 x 3584 at M = 16 31.2 against 34.4 us on the fp16
    // MFMA path, 152064 x 3584 143.5 against 170.4; at M = 4..8 the int8
    // kernel is faster, 21.1-27.5 against 30.2-30.4 and 108-130 against
    // 137-139); Q4_K at M = 2, 3 is faster on the batch-1 and int8 kernels
    const bool takes =
        fq::mmqs_supported((int)dtype) && M >= (q5k_band ? 2 : blk_band ? 3 : 4) && M <= 16 && K > 0 &&
        (dtype == FQ_DTYPE_Q4_K   ? N <= 16 * bmt * cus || M > 8
         : dtype == FQ_DTYPE_Q6_K ? (reinterpret_cast<uintptr_t>(w) & 1) == 0
         : (q4x || dtype == FQ_DTYPE_Q8_0) ? blk_band
                                           : q5k_band);
    return {blk_band, takes};
}

// Tiles of the band kernel's bands over N rows.
int band_tiles(uint32_t dtype, int K, int N, int cus) {
    const int bmt = fq::mmqs_max_tiles((int)dtype);
    // Q8_0: two- or three-tile bands, whichever the estimate (rounds of
    // work-groups x tiles x super-blocks per split) puts lower, three
    // within 5 % (14336 x 4096 at M = 8: 24.2 us on two, 30.1 on three;
    // 152064 x 3584: 175.4 / 170.0; 18944 x 3584: 31.3 / 29.6)
    int tiles = bmt;
    if (bmt == 4 && K / 256 < 32) {
        // four-tile bands whose last round of work-groups is mostly idle
        // (18944 rows: 296 bands on 256 CUs) take three tiles when those
        // fill their rounds better (395 bands: Q4_0 at M = 8 27.5 ->
        // 24.5 us, Q4_K at M = 16 31.3 -> 26.4, Q5_K 33.2 -> 27.7; at
        // 14336 and 152064 rows four tiles measured faster)
        auto fill = [&](int t) {
            const long b = ((long)N + 16 * t - 1) / (16 * t);
            return (double)b / (double)(((b + cus - 1) / cus) * cus);
        };
        if (N > 64L * cus && fill(4) < 0.6 && fill(3) > fill(4)) tiles = 3;
    } else if (dtype == FQ_DTYPE_Q8_0) {
        auto est = [&](int mt) {
            int r = 0;
            const long sp = mmqs_plan(N, K, cus, &r, mt);
            const long wgs = ((long)N + r - 1) / r * sp;
            return (double)((wgs + cus - 1) / cus) * (r / 16) *
                   (double)((K / 256 + sp - 1) / sp);
        };
        tiles = est(3) <= 1.05 * est(2) ? 3 : 2;
    }
    return tiles;
}

// Rows per band (a pair: gate rows, as many up rows) and K-splits of a band call.
struct BandPlan {
    int tiles, rpw, splits;
};
BandPlan band_plan(uint32_t dtype, int K, int N, bool pair, int cus) {
    BandPlan p{band_tiles(dtype, K, N, cus), 0, 1};
    if (pair) p.tiles = p.tiles >= 4 ? 4 : 2;
    p.splits = mmqs_plan(pair ? 2 * N : N, K, cus, &p.rpw, p.tiles);
    if (pair) p.rpw = 16 * ((p.rpw / 16 + 1) / 2);
    return p;
}
// Its estimated time: rounds of work-groups, each its super-blocks of its tiles, a
// K split's slab sum and the weight bytes (SmallUs).
double band_us(uint32_t dtype, const Geometry& g, int K, int N, bool pair, int cus) {
    const BandPlan p = band_plan(dtype, K, N, pair, cus);
    const int nsb = K / 256, sb = (nsb + p.splits - 1) / p.splits;
    const long wgs = ((long)N + p.rpw - 1) / p.rpw * p.splits, rounds = (wgs + cus - 1) / cus;
    const double mats = pair ? 2.0 : 1.0, tiles = mats * (p.rpw / 16);
    return 5.9 + 1.74 * (rounds - 1.0) + (double)rounds * sb * (small_us(dtype).band * tiles + 0.037) +
           (p.splits > 1 ? 1.75 : 0.0) + 0.071e-6 * mats * N * ((double)(K / g.be) * g.bb);
}

// 2..16 tokens (by format and shape): token operands, then one pass over the
// weights on the fp16 matrix cores, one band of rows per work-group (Q4_K at
// 14336 x 4096: 19.2-19.7 us for every M in 4..16, against 21-30 us on the
// int8 matrix-core and fp16 MFMA paths).  Several matrices (unsplit K only):
// one token preparation and one launch, the same bits as one call per matrix.
int run_band(uint32_t dtype, const Geometry& g, const float* x, const Mats& ms, const float* bias,
             int bias_mode, int64_t bias_len, float* y, int M, int K, int N, int dev,
             const DevInfo& di, hipStream_t st, uint8_t* fixed, size_t fixed_cap, bool x_ready) {
    const int NC = K / 64;
    const MmqPlan pl = plan_mmq(M, K, N, di.cus);
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    hipError_t e = hipSuccess;
    const bool pair = ms.mm == fq::MM_PAIR;
    const BandPlan bp = band_plan(dtype, K, N, pair, di.cus);
    const int rpw = bp.rpw, splits = bp.splits;
    const size_t need = mmqs_need(M, K, N, di.cus, bp.tiles);
    std::unique_ptr<StreamScratch::Lease> lease;
    uint8_t* buf = fixed;
    if (fixed) {
        if (need > fixed_cap) return FQ_ERR_WORKSPACE;
    } else {
        lease.reset(new StreamScratch::Lease(stream_scratch(dev, st, 0)));
        const int rc = lease->get(need, st, &buf);
        if (rc != FQ_OK) return rc;
    }
    fq::MmqArgs a{};
    a.mm = ms.mm;
    a.w = static_cast<const uint8_t*>(ms.w[0]);
    a.w2 = static_cast<const uint8_t*>(ms.w[1]);
    a.w3 = static_cast<const uint8_t*>(ms.w[2]);
    a.n1 = ms.n[0];
    a.n2 = ms.n[1];
    a.n3 = ms.n[2];
    a.xop = buf;
    a.xsum = reinterpret_cast<const float*>(buf + al(pl.xop_b));
    a.ex = reinterpret_cast<const int*>(buf + al(pl.xop_b) + al(pl.xsum_b));
    a.part = splits > 1 ? reinterpret_cast<float*>(buf + al(pl.xop_b) + al(pl.xsum_b) +
                                                   al(pl.ex_b))
                        : nullptr;
    a.y = y;
    a.bias = bias;
    a.bias_len = bias_mode ? bias_len : 0;
    a.bias_mode = bias_mode;
    a.M = M;
    a.N = N;
    a.K = K;
    a.NC = NC;
    a.row_bytes = (K / g.be) * g.bb;
    if (!x_ready) {
        e = fq::launch_xprep((int)dtype, x, M, K, NC, reinterpret_cast<_Float16*>(buf),
                             const_cast<float*>(a.xsum), const_cast<int*>(a.ex), st);
        if (e != hipSuccess) return hip_fail(e);
    }
    e = fq::launch_mmqs((int)dtype, a, rpw, 512, splits, st);
    if (e != hipSuccess) return hip_fail(e);
    return FQ_OK;
}

// band_x (optional): in, true when the stream's slot-0 workspace already
// holds the band kernel's token operands of this x, M, K and format (a call
// just before with the same x, M, K, N and format took the band kernel:
// same plan, same workspace size, so the buffer was not replaced); out,
// whether this call took the band kernel.
int run_matmul(uint32_t dtype, const float* x, const void* w, const float* bias, int bias_mode,
               int64_t bias_len, float* y, int M, int K, int N, hipStream_t st,
               uint8_t* fixed = nullptr, size_t fixed_cap = 0, bool* band_x = nullptr);

// Fixed workspace of fq_matmul_transB_noalloc, for callers that cannot
// allocate (HIP-graph capture, serving loops that forbid hipMalloc).  Every
// GPU the library runs on holds its own copy until the process ends.  It is
// shared by every call of that entry point on the device: calls that overlap
// on one GPU race on it.  Nothing in it has to start at zero (the token
// preparation writes every operand, each K-split writes its whole slab).
__device__ __align__(256) uint8_t scratch[kNoAllocBytes];

// The device address of `scratch` on the current device, looked up once per
// device (the host-side name is only a stand-in for the symbol).
int noalloc_workspace(int dev, uint8_t** out) {
    static std::mutex mu;
    static std::map<int, uint8_t*> ptrs;
    std::lock_guard<std::mutex> lk(mu);
    auto it = ptrs.find(dev);
    if (it == ptrs.end()) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e);
        it = ptrs.emplace(dev, static_cast<uint8_t*>(p)).first;
    }
    *out = it->second;
    return FQ_OK;
}

int packed_gemv(uint32_t dtype, const float* x, const void* w_packed, const void* w2_packed,
                const void* w3_packed, int n1, int n2, int mode, const float* bias,
                int64_t bias_len, float* y, int K, int N, hipStream_t st, bool gguf, int M = 1,
                bool bias_full = false, uint8_t* fixed = nullptr, size_t fixed_cap = 0);

int run_matmul(uint32_t dtype, const float* x, const void* w, const float* bias, int bias_mode,
               int64_t bias_len, float* y, int M, int K, int N, hipStream_t st, uint8_t* fixed,
               size_t fixed_cap, bool* band_x) {
    const bool x_ready = band_x && *band_x;
    if (band_x) *band_x = false;
    Geometry g;
    if (!geometry(dtype, g)) return FQ_ERR_DTYPE;
    if (M < 0 || N < 0 || K < 0) return FQ_ERR_SHAPE;
    if (K % g.be != 0) return FQ_ERR_SHAPE;
    if (M == 0 || N == 0) return FQ_OK;
    if (!x || !w || !y) return FQ_ERR_NULL;
    if (bias_mode != 0 && !bias) return FQ_ERR_NULL;
    if (bias_mode == 2 && bias_len < (int64_t)M * N) return FQ_ERR_SHAPE;
    if (!row_fits(g, K)) return FQ_ERR_SHAPE;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    const DevInfo di = device_info(dev);
    if (K == 0 && bias_mode == 0) {
        // a zero-length contraction: y = 0 (with a bias the kernel writes y = bias)
        e = fq::launch_zero(reinterpret_cast<uint32_t*>(y), (size_t)M * N, di.cus, st);
        return e == hipSuccess ? FQ_OK : hip_fail(e);
    }

    if (M == 1 && K > 0 && packable(dtype) &&
        (dtype == FQ_DTYPE_Q6_K || (int64_t)N * (K / g.be) * g.bb >= (4 << 20))) {
        // batch 1 on the five benchmark formats: the aligned-layout kernel,
        // reading the GGUF rows through per-wave LDS buffers (with one token a
        // full [1][N] bias is a row vector of N).  Below ~4 MB of weights the
        // row-step kernels start faster (2048 x 2048 Q4_0, 2.4 MB: 3.6 us
        // against 4.2); from 4.5 MB this one is (2048 x 2048 Q8_0 4.4 against
        // 4.7 us, TinyLlama Q4_0 5632 x 2048 4.8 against 5.15); Q6_K always
        // runs here.
        const int rc = packed_gemv(dtype, x, w, nullptr, nullptr, 0, 0, 0,
                                   bias_mode ? bias : nullptr, bias_mode == 2 ? N : bias_len, y,
                                   K, N, st, true);
        if (rc != FQ_ERR_SHAPE) return rc;
    }

    const BandRule rule = band_rule(dtype, g, M, K, N, w, di.cus);
    if (thin_takes(dtype, M, (int64_t)N * (K / g.be) * g.bb)) {
        // (where bands fill their rounds the band kernel is faster: at M = 8 Q5_0 12288
        // x 4096 16.7 us there, 20.6 here, 14336 x 4096 20.5 and 20.9; Q4_0 12288 x 5632
        // 19.6 and 23.1, 13824 x 5632 23.3 and 23.6, 17408 x 5632, two rounds, 33.4 and 25.7)
        const double limit = M <= 16 && K < 32 * 256 && rule.takes
                                 ? 1.04 * band_us(dtype, g, K, N, false, di.cus)
                                 : HUGE_VAL;
        const Mats ms{fq::MM_ONE, {w}, {N}};
        int rc = run_thin(dtype, g, x, ms, bias, bias_mode, bias_len, y, M, K, N, dev, di, st, fixed,
                          fixed_cap, limit);
        if (rc == kSlower) {
            rc = run_band(dtype, g, x, ms, bias, bias_mode, bias_len, y, M, K, N, dev, di, st, fixed,
                          fixed_cap, x_ready);
            if (rc == FQ_OK && band_x) *band_x = true;
            if (rc == FQ_ERR_WORKSPACE)  // capture on a workspace that another call sized
                rc = run_thin(dtype, g, x, ms, bias, bias_mode, bias_len, y, M, K, N, dev, di, st,
                              fixed, fixed_cap, HUGE_VAL);
        }
        if (rc != kNotTaken) return rc;
    }

    if (dtype == FQ_DTYPE_Q6_K && M == 4 && K > 0 && N > 16384 &&
        (int64_t)N * (K / g.be) * g.bb >= (24 << 20)) {
        // four Q6_K tokens on 24 MB and more of more than 16384 rows that the
        // shared-operand kernel above does not take (under 32 MiB; 152064 x 3584
        // 126 us there, 203 this way, 18944 x 3584 26.2 and 36.2, 20000 x 2048,
        // 32.0 MiB, 19.2 and 31.6): three on the batch-1 kernel, whose four-token
        // form spills, then the fourth (18944 x 3584 34.7 against 37.3 on the
        // band kernel); fewer rows take the band kernel below (14336 x 4096 27.8
        // against 30.8)
        for (int t0 = 0; t0 < M; t0 += 3) {
            const int m = std::min(3, M - t0);
            const int rc = run_matmul(dtype, x + (size_t)t0 * K, w,
                                      bias_mode == 2 ? bias + (size_t)t0 * N : bias, bias_mode,
                                      bias_mode == 2 ? (int64_t)m * N : bias_len,
                                      y + (size_t)t0 * N, m, K, N, st, fixed, fixed_cap);
            if (rc != FQ_OK) return rc;
        }
        return FQ_OK;
    }

    if (M >= 2 && M <= 4 && !rule.block && K > 0 && packable(dtype) &&
        (dtype == FQ_DTYPE_Q6_K || (int64_t)N * (K / g.be) * g.bb >= (8 << 20))) {
        // two to four tokens: the same kernel dots each weight unit it reads
        // with every token's limbs, K split into slabs where the tokens'
        // records of a whole row do not fit LDS (FQ_ERR_SHAPE: no split fits,
        // or the slabs need workspace the call cannot have)
        const int rc = packed_gemv(dtype, x, w, nullptr, nullptr, 0, 0, 0,
                                   bias_mode ? bias : nullptr, bias_mode == 2 ? N : bias_len, y,
                                   K, N, st, true, M, bias_mode == 2, fixed, fixed_cap);
        if (rc != FQ_ERR_SHAPE) return rc;
    }

    if (rule.takes) {
        const int rc = run_band(dtype, g, x, Mats{fq::MM_ONE, {w}, {N}}, bias, bias_mode, bias_len, y, M,
                                K, N, dev, di, st, fixed, fixed_cap, x_ready);
        if (rc == FQ_OK && band_x) *band_x = true;
        return rc;
    }

    if ((M == 1 || M == 2) && K > 0) {
        // batch 1 (and two tokens on rows of at most 128 units, where the
        // row-step kernel keeps both tokens' limbs in registers): persistent
        // work-groups, as many as fit on every CU
        const int U1 = K / 32;
        int wg = 1024;
        size_t lds = M == 1 ? fq::gemv1_lds_bytes((int)dtype, U1, wg) : 0;
        const void* fn = M == 1 ? fq::gemv1_kernel_fn((int)dtype, bias_mode != 0, wg) : nullptr;
        int npr = 0;
        size_t lds_r = 0;
        int wg_r = 0;
        const void* fr = fq::gemv1r_kernel_fn((int)dtype, U1, (K / g.be) * g.bb, bias_mode != 0,
                                              &npr, &lds_r, &wg_r, M);
        if (fr && lds_r <= std::min<size_t>(di.lds, 160 * 1024)) {
            fn = fr;
            lds = lds_r;
            wg = wg_r;
        }
        if (fn && lds <= std::min<size_t>(di.lds, 160 * 1024)) {
            int per_cu = 0;
            e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, wg, lds);
            if (e != hipSuccess) return hip_fail(e);
            if (per_cu >= 1) {
                fq::GemvArgs a{};
                a.x = x;
                a.w = static_cast<const uint8_t*>(w);
                a.y = y;
                a.bias = bias;
                a.bias_len = bias_mode == 0 ? 0 : bias_len;
                a.bias_mode = bias_mode;
                a.M = M;
                a.K = K;
                a.N = N;
                a.U = U1;
                a.Uc = U1;
                a.row_bytes = (K / g.be) * g.bb;
                const int wpb = wg / 64;
                const long waves = (long)di.cus * per_cu * wpb;
                const long need = std::min<long>(waves, N);
                const int grid = (int)std::max(1L, (need + wpb - 1) / wpb);
                e = fq::launch_raw(fn, a, grid, wg, lds, st);
                return e == hipSuccess ? FQ_OK : hip_fail(e);
            }
        }
    }

    if (fq::mmqi_supported((int)dtype) && M >= 3 && M <= 8 && K > 0) {
        // Q4_K, 3..8 tokens that the kernels above do not take: three tokens
        // on weights under 8 MB (from 8 MB the batch-1 kernel takes them, with
        // K split where the records overflow its LDS), and 4..8 tokens on more
        // rows than one mmqs band per CU covers.  The int8 matrix-core kernel
        // runs them in one pass (M = 9..16 takes the band kernel above)
        const long T = (N + 15) / 16;
        const long G = std::max(1L, std::min<long>(di.cus, T));
        const int tpw = (int)((T + G - 1) / G);
        bool ok = true;
        for (int m0 = 0; m0 < M && ok; m0 += 8) {
            const int mt = std::min(8, M - m0);
            size_t lds = 0;
            int wg = 0;
            // chunk: >= 3 steps, about 4 per wave
            int chunk = 3;
            const void* fn = nullptr;
            for (int pass = 0; pass < 2; ++pass) {
                const int waves = (pass == 0 && mt <= 4) ? 16 : 8;
                chunk = (int)std::max(3L, std::min(16L, (long)tpw * (K / 256) / (4L * waves)));
                fn = fq::mmqi_kernel_fn(mt, bias_mode != 0, K, tpw, chunk,
                                        std::min<size_t>(di.lds, 160 * 1024), &lds, &wg);
                if (fn && wg / 64 == waves) break;
            }
            if (!fn) {
                ok = false;
                break;
            }
            fq::GemvArgs a{};
            a.x = x + (size_t)m0 * K;
            a.w = static_cast<const uint8_t*>(w);
            a.y = y + (size_t)m0 * N;
            a.bias = bias_mode == 2 ? bias + (size_t)m0 * N : bias;
            a.bias_len = bias_mode == 0 ? 0 : bias_len;
            a.bias_mode = bias_mode;
            a.M = mt;
            a.K = K;
            a.N = N;
            a.U = (int)T;
            a.Uc = chunk;
            a.row_bytes = (K / g.be) * g.bb;
            e = fq::launch_raw(fn, a, (int)G, wg, lds, st);
            if (e != hipSuccess) return hip_fail(e);
        }
        if (ok) return FQ_OK;
    }

    if (M >= 2 && M <= 4 && K > 0) {
        // a few tokens: the batch-1 chunk kernel reads and unpacks each weight
        // unit once and dots it with every token's activation limbs
        const int U1 = K / 32;
        size_t lds = 0;
        const void* fn = fq::gemv1_multi_fn((int)dtype, bias_mode != 0, M, &lds, U1);
        if (fn && lds <= std::min<size_t>(di.lds, 160 * 1024)) {
            int per_cu = 0;
            e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 1024, lds);
            if (e != hipSuccess) return hip_fail(e);
            if (per_cu >= 1) {
                fq::GemvArgs a{};
                a.x = x;
                a.w = static_cast<const uint8_t*>(w);
                a.y = y;
                a.bias = bias;
                a.bias_len = bias_mode == 0 ? 0 : bias_len;
                a.bias_mode = bias_mode;
                a.M = M;
                a.K = K;
                a.N = N;
                a.U = U1;
                a.Uc = U1;
                a.row_bytes = (K / g.be) * g.bb;
                const long waves = (long)di.cus * per_cu * 16;
                const long need = std::min<long>(waves, N);
                const int grid = (int)std::max(1L, (need + 15) / 16);
                e = fq::launch_raw(fn, a, grid, 1024, lds, st);
                return e == hipSuccess ? FQ_OK : hip_fail(e);
            }
        }
    }

    if (M > 32) {
        const int rc = run_prefill(dtype, g, x, Mats{fq::MM_ONE, {w}, {N}}, bias, bias_mode,
                                   bias_len, y, M, K, N, dev, di, st, fixed, fixed_cap);
        if (rc != kNotTaken) return rc;
    }

    // M > 4, and rows too long for the batch-1 kernels' LDS
    return run_mmq(dtype, g, x, w, bias, bias_mode, bias_len, y, M, K, N, dev, di, st, fixed,
                   fixed_cap);
}

// Batch-1 GEMV over the tiled aligned layout, one row per lane
// (fq_gemvt.hip; every matrix involved satisfies packed_tiled()).  N output
// rows (mode 1: rows of each of the two matrices).  W waves per work-group
// (one K range each), 16 / W work-groups per CU, the tiles dealt out in turn
// so every work-group gets the same number within one; W shrinks until a
// work-group's tiles fit its LDS (gemvt_max_tiles()).
int run_gemvt(uint32_t dtype, const float* x, const void* w, const void* w2, const void* w3,
              int n1, int n2, int mode, const float* bias, int64_t bias_len, float* y, int K,
              int N, hipStream_t st, const DevInfo& di) {
    const int U = fq::gemvt_units((int)dtype, K);
    if (U % 4 != 0) return FQ_ERR_SHAPE;
    const int GR = U / 4;
    const int TRW = fq::gemvt_tile_rows();
    const long tiles = mode == 2 ? (long)(n1 + TRW - 1) / TRW + (n2 + TRW - 1) / TRW +
                                       (N - n1 - n2 + TRW - 1) / TRW
                                 : (long)(N + TRW - 1) / TRW;
    if (tiles > INT32_MAX / TRW) return FQ_ERR_SHAPE;
    // the kernel addresses each matrix through a 32-bit buffer offset
    const int64_t RB = fq::packed_row_bytes((int)dtype, K);
    if ((int64_t)(mode == 2 ? std::max(n1, std::max(n2, N - n1 - n2)) : N) * RB >= ((int64_t)1 << 32))
        return FQ_ERR_SHAPE;
    const int WM = fq::gemvt_max_waves(), ntmax = fq::gemvt_max_tiles();
    const int maxrec = fq::gemvt_max_records(), RBY = fq::gemvt_record_bytes();
    const int NV = mode == 1 ? 2 : 1;
    const size_t cu_lds = std::min<size_t>(di.lds, 160 * 1024);
    auto recs_of = [&](int w) { return ((GR + w - 1) / w) * 4; };
    auto lds_of = [&](int w, long nt) {
        return (size_t)w * recs_of(w) * RBY + (size_t)nt * NV * w * 64 * 4;
    };
    // the fewest waves per work-group (more work-groups per CU, the same 16
    // waves) whose records fit and whose tiles stay within gemvt_max_tiles()
    // and the CU's LDS
    int W = 0;
    long GT = 0;
    for (int w = std::min(WM, GR); w >= 1; w = w > 1 ? std::max(1, w / 2) : 0) {
        if (recs_of(w) > maxrec) break;
        const int wpc = std::max(1, WM / w);
        const long gt = std::min<long>(tiles, (long)di.cus * wpc);
        const long nt = (tiles + gt - 1) / gt;
        if (nt <= ntmax && lds_of(w, nt) * wpc <= cu_lds) {
            W = w;
            GT = gt;
            if (nt * 2 > ntmax) break;  // fewer waves would not fit the next halving
        } else if (W) {
            break;
        }
    }
    if (!W) {  // very long rows or very many tiles: the smallest fitting W, more work-groups
        W = std::min(WM, GR);
        while (W < WM && recs_of(W) > maxrec) W = std::min(WM, 2 * W);
        if (recs_of(W) > maxrec) return FQ_ERR_SHAPE;
        const size_t fixed = lds_of(W, 0);
        if (fixed >= cu_lds) return FQ_ERR_SHAPE;
        const long ntcap = std::max<long>(1, std::min<long>(ntmax, (long)((cu_lds - fixed) / ((size_t)NV * W * 64 * 4))));
        GT = (tiles + ntcap - 1) / ntcap;
    }
    const int recs = recs_of(W);
    const int nt_max = (int)((tiles + GT - 1) / GT);
    const size_t lds = lds_of(W, nt_max);
    if (lds > cu_lds) return FQ_ERR_SHAPE;
    const void* fn = fq::gemvt_kernel_fn((int)dtype, mode);
    if (!fn) return FQ_ERR_DTYPE;
    fq::TArgs a{};
    a.x = x;
    a.w = static_cast<const uint8_t*>(w);
    a.w2 = static_cast<const uint8_t*>(w2);
    a.w3 = static_cast<const uint8_t*>(w3);
    a.n1 = n1;
    a.n2 = n2;
    a.y = y;
    a.bias = bias;
    a.bias_len = bias ? bias_len : 0;
    a.mode = mode;
    a.N = N;
    a.K = K;
    a.U = U;
    a.GR = GR;
    a.recs = recs;
    a.T = (int)tiles;
    a.row_bytes = RB;
    const hipError_t e = fq::launch_gemvt(fn, a, (int)GT, W, lds, st);
    return e == hipSuccess ? FQ_OK : hip_fail(e);
}

// Batch-1 GEMV over packed rows.  mode 0: y = x . w (+ bias).  mode 1 (fused
// gate/up): y[n] = silu(x . w[n]) * (x . w2[n]), run as one GEMV over 2 N
// interleaved rows.  mode 2 (fused QKV): y = [x . w | x . w2 | x . w3] with
// n1 and n2 rows in w and w2 and N rows in all.
// gguf: the same kernel over the unmodified GGUF rows (the caller has
// validated the arguments as run_matmul does).
int packed_gemv(uint32_t dtype, const float* x, const void* w_packed, const void* w2_packed,
                const void* w3_packed, int n1, int n2, int mode, const float* bias,
                int64_t bias_len, float* y, int K, int N, hipStream_t st, bool gguf, int M,
                bool bias_full, uint8_t* fixed, size_t fixed_cap) {
    Geometry g;
    if (!geometry(dtype, g) || !packable(dtype)) return FQ_ERR_DTYPE;
    if (N < 0 || K < 0 || K % (gguf ? g.be : 256) != 0) return FQ_ERR_SHAPE;
    if (N == 0) return FQ_OK;
    if (!x || !w_packed || !y) return FQ_ERR_NULL;
    if (M != 1 && !(gguf && mode == 0 && M >= 2 && M <= 4)) return FQ_ERR_SHAPE;
    const uintptr_t amask = gguf ? 1 : 15;
    if ((reinterpret_cast<uintptr_t>(w_packed) & amask) != 0) return FQ_ERR_ALIGN;
    for (const void* p : {w2_packed, w3_packed})
        if (p && (reinterpret_cast<uintptr_t>(p) & amask) != 0) return FQ_ERR_ALIGN;
    const bool dual = mode == 1;
    const int NV = dual ? 2 * N : N;  // rows the kernel walks
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    const DevInfo di = device_info(dev);
    if (K == 0) {  // y = 0 (silu(0) * 0 = 0 for the fused form)
        if (bias) return FQ_ERR_SHAPE;
        e = fq::launch_zero(reinterpret_cast<uint32_t*>(y), (size_t)N, di.cus, st);
        return e == hipSuccess ? FQ_OK : hip_fail(e);
    }
    if (!gguf) {
        // the arrangement of each packed matrix follows from its rows
        const int nr[3] = {mode == 2 ? n1 : N, mode == 2 ? n2 : N, mode == 2 ? N - n1 - n2 : N};
        const int nm = mode == 0 ? 1 : mode == 1 ? 2 : 3;
        int tiled = 0;
        for (int i = 0; i < nm; ++i) tiled += fq::packed_tiled((int)dtype, nr[i]) ? 1 : 0;
        if (tiled == nm)
            return run_gemvt(dtype, x, w_packed, w2_packed, w3_packed, n1, n2, mode, bias,
                             bias_len, y, K, N, st, di);
        if (tiled > 0) {  // fused QKV over both arrangements: one GEMV per matrix
            const void* ws[3] = {w_packed, w2_packed, w3_packed};
            int off = 0;
            for (int i = 0; i < 3; ++i) {
                if (nr[i] > 0) {
                    const int rc = packed_gemv(dtype, x, ws[i], nullptr, nullptr, 0, 0, 0, nullptr,
                                               0, y + off, K, nr[i], st, false);
                    if (rc != FQ_OK) return rc;
                }
                off += nr[i];
            }
            return FQ_OK;
        }
    }
    int units = 0, records = 0;
    fq::gemvp_geometry((int)dtype, K, &units, &records);
    size_t lds = 0;
    int wg = 0;
    const size_t lds_cap = std::min<size_t>(di.lds, 160 * 1024);
    // partial sums a work-group can buffer: a static 4096-entry array for the
    // packed kernel, the LDS left after the records and wave buffers for GGUF
    long pcap = 4096;
    int nl = 1;
    const void* fn =
        gguf ? fq::gemvg_kernel_fn((int)dtype, units, records, bias != nullptr, &lds, &wg, &nl, NV,
                                   M, mode)
             : fq::gemvp_kernel_fn((int)dtype, units, records, bias != nullptr, &lds, &wg, &nl,
                                   mode);
    // K split over blockIdx.y for several tokens whose records of a whole row
    // do not fit LDS (K = 18944: 2 x 85 KB): each work-group stages only the
    // records of its own K-slices and writes partial sums, [splits][M][N],
    // which the slab sum adds with the bias (the fewest splits that fit)
    int splits = 1, spl = 0;
    if (gguf && fn && M >= 2 && lds + 64 * 4 * M + 256 > lds_cap) {
        fn = fq::gemvg_kernel_fn((int)dtype, units, records, false, &lds, &wg, &nl, NV, M, mode);
        if (!fn) return FQ_ERR_SHAPE;
        const size_t rb = (size_t)fq::gemvp_record_bytes();
        const size_t wbufs = lds - (size_t)M * records * rb;
        const int nrec = records / units, ns_all = (units + 64 * nl - 1) / (64 * nl);
        for (int s = 2; s <= 8 && !spl; ++s) {
            const int sp = (ns_all + s - 1) / s;
            const size_t l = (size_t)M * std::min(units, sp * 64 * nl) * nrec * rb + wbufs;
            if (l + 64 * 4 * M * (size_t)sp + 256 <= lds_cap) {
                spl = sp;
                splits = (ns_all + sp - 1) / sp;
                lds = l;
            }
        }
        if (!spl) return FQ_ERR_SHAPE;
    }
    std::unique_ptr<StreamScratch::Lease> lease;
    uint8_t* slab = fixed;
    if (splits > 1) {
        const size_t need = (size_t)splits * M * NV * sizeof(float);
        if (fixed) {
            if (need > fixed_cap) return FQ_ERR_SHAPE;
        } else {
            lease.reset(new StreamScratch::Lease(stream_scratch(dev, st, 0)));
            const int rc = lease->get(need, st, &slab);
            // under graph capture without a reserved workspace: another kernel
            if (rc == FQ_ERR_WORKSPACE) return FQ_ERR_SHAPE;
            if (rc != FQ_OK) return rc;
        }
    }
    if (gguf) {
        // M tokens' partial sums per row and K-slice
        // (256 bytes left for the kernel's static LDS: its step counter)
        if (lds + 64 * 4 * M + 256 > lds_cap) return FQ_ERR_SHAPE;
        pcap = std::min<long>(4096, (long)(lds_cap - lds - 256) / (4 * M));
    }
    if (!fn || lds > lds_cap) return FQ_ERR_SHAPE;
    int per_cu = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, wg,
                                                     gguf ? lds + 4 * (size_t)M * pcap : lds);
    if (e != hipSuccess) return hip_fail(e);
    if (per_cu < 1) return FQ_ERR_SHAPE;
    const int wpb = wg / 64;
    // one work-group per resident slot, each owning a contiguous row range
    // with at least one row per wave, and whose row x K-slice partial sums fit
    // its LDS buffer (slices of 64 lane units)
    const long ns = spl ? spl : (units + 64 * nl - 1) / (64 * nl);
    long G = ((long)di.cus * per_cu + splits - 1) / splits;
    G = std::max(1L, std::min<long>(G, ((long)NV + wpb - 1) / wpb));
    auto max_rows = [&](long g) { return dual ? 2 * ((N + g - 1) / g) : (NV + g - 1) / g; };
    G = std::max<long>(G, ((long)NV * ns + pcap - 1) / pcap);
    while (max_rows(G) * ns > pcap) ++G;
    if (gguf) lds += 4 * (size_t)M * (max_rows(G) * ns);
    fq::GemvArgs a{};
    a.x = x;
    a.w = static_cast<const uint8_t*>(w_packed);
    a.w2 = static_cast<const uint8_t*>(w2_packed);
    a.w3 = static_cast<const uint8_t*>(w3_packed);
    a.n1 = n1;
    a.n2 = n2;
    a.y = y;
    a.bias = bias;
    a.bias_len = bias ? bias_len : 0;
    a.bias_mode = bias ? (bias_full ? 2 : 1) : 0;
    a.M = M;
    a.K = K;
    a.N = NV;
    a.U = units;
    a.Uc = records;
    a.row_bytes = gguf ? (K / g.be) * g.bb : (int)fq::packed_row_bytes((int)dtype, K);
    if (splits > 1) {
        a.part = reinterpret_cast<float*>(slab);
        a.spl = spl;
        a.bias = nullptr;
        a.bias_len = 0;
        a.bias_mode = 0;
    }
    e = fq::launch_raw(fn, a, (int)G, wg, lds, st, splits);
    if (e != hipSuccess || splits == 1) return e == hipSuccess ? FQ_OK : hip_fail(e);
    fq::MmqArgs r{};
    r.part = a.part;
    r.y = y;
    r.bias = bias;
    r.bias_len = bias ? bias_len : 0;
    r.bias_mode = bias ? (bias_full ? 2 : 1) : 0;
    r.M = M;
    r.N = NV;
    e = fq::launch_reduce(r, splits, st);
    return e == hipSuccess ? FQ_OK : hip_fail(e);
}

}  // namespace

extern "C" {

int fq_block_info(uint32_t dtype, int* block_elems, int* block_bytes) {
    Geometry g;
    if (!geometry(dtype, g)) return FQ_ERR_DTYPE;
    if (block_elems) *block_elems = g.be;
    if (block_bytes) *block_bytes = g.bb;
    return FQ_OK;
}

const char* fq_status_str(int status) {
    switch (status) {
        case FQ_OK: return "ok";
        case FQ_ERR_DTYPE: return "unsupported quantized type";
        case FQ_ERR_SHAPE: return "invalid shape";
        case FQ_ERR_NULL: return "null pointer";
        case FQ_ERR_HIP: return "HIP runtime error";
        case FQ_ERR_NO_DEVICE: return "no HIP device";
        case FQ_ERR_ALIGN: return "packed buffer not 16-byte aligned";
        case FQ_ERR_WORKSPACE:
            return "workspace too small (reserve it with fq_reserve_workspace before graph "
                   "capture; fq_matmul_transB_noalloc: the call needs more than its fixed "
                   "64 MiB)";
        default: return "unknown status";
    }
}

int fq_last_hip_error(void) { return g_last_hip; }

int fq_gemv(uint32_t dtype, const float* x, const void* w, float* y, int K, int N, void* stream) {
    return run_matmul(dtype, x, w, nullptr, 0, 0, y, 1, K, N,
                      static_cast<hipStream_t>(stream));
}

int fq_gemv_batch(uint32_t dtype, const float* x, const void* w, float* y, int M, int K, int N,
                  void* stream) {
    if (M < 1 || M > 32) return FQ_ERR_SHAPE;
    return run_matmul(dtype, x, w, nullptr, 0, 0, y, M, K, N,
                      static_cast<hipStream_t>(stream));
}

int fq_matmul_prefill(uint32_t dtype, const float* x, const void* w, float* y, int M, int K,
                      int N, void* stream) {
    if (M < 1) return FQ_ERR_SHAPE;
    return run_matmul(dtype, x, w, nullptr, 0, 0, y, M, K, N,
                      static_cast<hipStream_t>(stream));
}

int fq_matmul_transB(uint32_t dtype, const float* x, const void* w, const float* bias,
                     int bias_ndim, int64_t bias_len, float* y, int M, int K, int N,
                     void* stream) {
    int mode = 0;
    if (bias && bias_ndim == 1) mode = 1;
    else if (bias && bias_ndim == 2) mode = 2;
    else if (bias && bias_ndim != 0) return FQ_ERR_SHAPE;
    return run_matmul(dtype, x, w, bias, mode, bias_len, y, M, K, N,
                      static_cast<hipStream_t>(stream));
}

int fq_matmul_transB_noalloc(uint32_t dtype, const float* x, const void* w, const float* bias,
                             int bias_ndim, int64_t bias_len, float* y, int M, int K, int N,
                             void* stream) {
    int mode = 0;
    if (bias && bias_ndim == 1) mode = 1;
    else if (bias && bias_ndim == 2) mode = 2;
    else if (bias && bias_ndim != 0) return FQ_ERR_SHAPE;
    int dev = 0;
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    uint8_t* ws = nullptr;
    const int rc = noalloc_workspace(dev, &ws);
    if (rc != FQ_OK) return rc;
    return run_matmul(dtype, x, w, bias, mode, bias_len, y, M, K, N,
                      static_cast<hipStream_t>(stream), ws, kNoAllocBytes);
}

int fq_dequant_rows(uint32_t dtype, const void* w, float* out, int N, int K, void* stream) {
    Geometry g;
    if (!geometry(dtype, g)) return FQ_ERR_DTYPE;
    if (N < 0 || K < 0) return FQ_ERR_SHAPE;
    if (N == 0 || K == 0) return FQ_OK;
    if (!w || !out) return FQ_ERR_NULL;
    const int64_t row_b = ((int64_t)K / g.be + (K % g.be != 0)) * g.bb;
    if (row_b > INT32_MAX) return FQ_ERR_SHAPE;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    const DevInfo di = device_info(dev);
    e = fq::launch_dequant((int)dtype, static_cast<const uint8_t*>(w), out, N, K, (int)row_b,
                           di.cus, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? FQ_OK : hip_fail(e);
}

int64_t fq_packed_row_bytes(uint32_t dtype, int K) {
    Geometry g;
    if (!geometry(dtype, g) || !packable(dtype) || K <= 0 || K % 256 != 0) return 0;
    return fq::packed_row_bytes((int)dtype, K);
}

static int pack_common(uint32_t dtype, const void* src, void* dst, int N, int K, bool pack,
                       void* stream) {
    Geometry g;
    if (!geometry(dtype, g) || !packable(dtype)) return FQ_ERR_DTYPE;
    if (N < 0 || K < 0 || K % 256 != 0) return FQ_ERR_SHAPE;
    if (N == 0 || K == 0) return FQ_OK;
    if (!src || !dst) return FQ_ERR_NULL;
    const void* packed = pack ? dst : src;
    const void* gguf = pack ? src : dst;
    if ((reinterpret_cast<uintptr_t>(packed) & 15) != 0) return FQ_ERR_ALIGN;
    if ((reinterpret_cast<uintptr_t>(gguf) & 1) != 0) return FQ_ERR_ALIGN;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    const DevInfo di = device_info(dev);
    e = fq::launch_pack((int)dtype, static_cast<const uint8_t*>(src), static_cast<uint8_t*>(dst),
                        N, K, pack, di.cus * 8, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? FQ_OK : hip_fail(e);
}

int fq_pack_weights(uint32_t dtype, const void* w_gguf, void* w_packed, int N, int K,
                    void* stream) {
    return pack_common(dtype, w_gguf, w_packed, N, K, true, stream);
}

int fq_unpack_weights(uint32_t dtype, const void* w_packed, void* w_gguf, int N, int K,
                      void* stream) {
    return pack_common(dtype, w_packed, w_gguf, N, K, false, stream);
}


int fq_gemv_packed(uint32_t dtype, const float* x, const void* w_packed, const float* bias,
                   int64_t bias_len, float* y, int K, int N, void* stream) {
    return packed_gemv(dtype, x, w_packed, nullptr, nullptr, 0, 0, 0, bias, bias_len, y, K, N,
                       static_cast<hipStream_t>(stream), false);
}

int fq_ffn_up_fused_packed(uint32_t dtype, const float* x, const void* w_gate_packed,
                           const void* w_up_packed, float* y, int K, int N, void* stream) {
    if (!w_up_packed) return FQ_ERR_NULL;
    return packed_gemv(dtype, x, w_gate_packed, w_up_packed, nullptr, 0, 0, 1, nullptr, 0, y, K,
                       N, static_cast<hipStream_t>(stream), false);
}

int fq_fused_qkv_packed(uint32_t dtype, const float* x, const void* wq, const void* wk,
                        const void* wv, float* y, int K, int Nq, int Nk, int Nv, void* stream) {
    if (Nq < 0 || Nk < 0 || Nv < 0 || (int64_t)Nq + Nk + Nv > INT32_MAX) return FQ_ERR_SHAPE;
    if ((Nk && !wk) || (Nv && !wv)) return FQ_ERR_NULL;
    return packed_gemv(dtype, x, wq, wk, wv, Nq, Nk, 2, nullptr, 0, y, K, Nq + Nk + Nv,
                       static_cast<hipStream_t>(stream), false);
}

int fq_fused_qkv(uint32_t dtype, const float* x, const void* wq, const void* wk, const void* wv,
                 float* y, int M, int K, int Nq, int Nk, int Nv, void* stream) {
    Geometry g;
    if (!geometry(dtype, g)) return FQ_ERR_DTYPE;
    if (M < 0 || K < 0 || Nq < 0 || Nk < 0 || Nv < 0 || K % g.be != 0) return FQ_ERR_SHAPE;
    if ((int64_t)Nq + Nk + Nv > INT32_MAX) return FQ_ERR_SHAPE;
    const int Nt = Nq + Nk + Nv;
    if (M == 0 || Nt == 0) return FQ_OK;
    if (!x || !y || (Nq && !wq) || (Nk && !wk) || (Nv && !wv)) return FQ_ERR_NULL;
    if (!row_fits(g, K)) return FQ_ERR_SHAPE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const void* ws[3] = {wq, wk, wv};
    const int ns[3] = {Nq, Nk, Nv};
    if (M == 1) {  // the three outputs are contiguous slices of y
        // one launch over the three matrices' GGUF rows (the five formats
        // the batch-1 kernel reads; at every size: against three launches,
        // TinyLlama QKV 9.4 -> 4.5 us for Q4_0, 12.3 -> 4.5 us for Q8_0)
        if (packable(dtype)) {
            // a matrix of no rows is never read: any valid pointer stands in
            const void* any = Nq ? wq : Nk ? wk : wv;
            const int rc = packed_gemv(dtype, x, Nq ? wq : any, Nk ? wk : any, Nv ? wv : any, Nq,
                                       Nk, 2, nullptr, 0, y, K, Nt, st, true);
            if (rc != FQ_ERR_SHAPE) return rc;
        }
        int off = 0;
        for (int i = 0; i < 3; ++i) {
            if (ns[i] > 0) {
                const int rc = run_matmul(dtype, x, ws[i], nullptr, 0, 0, y + off, 1, K, ns[i], st);
                if (rc != FQ_OK) return rc;
            }
            off += ns[i];
        }
        return FQ_OK;
    }
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    const DevInfo di = device_info(dev);
    Mats ms{fq::MM_CAT, {}, {}};
    for (int i = 0, n = 0; i < 3; ++i)
        if (ns[i] > 0) {
            ms.w[n] = ws[i];
            ms.n[n++] = ns[i];
        }
    if (M > 16) {  // one launch over the three matrices
        int rc = kNotTaken;
        if (M > 32)
            rc = run_prefill(dtype, g, x, ms, nullptr, 0, 0, y, M, K, Nt, dev, di, st, nullptr, 0);
        else if (thin_takes(dtype, M, 0))
            rc = run_thin(dtype, g, x, ms, nullptr, 0, 0, y, M, K, Nt, dev, di, st, nullptr, 0, HUGE_VAL);
        if (rc != kNotTaken) return rc;
    }
    if (M >= 5 && M <= 16 && K < 32 * 256) {
        // where each matrix would run on the band kernel (K unsplit): one
        // launch over the three (Q4_K 4096 -> 4096 + 1024 + 1024 at M = 8: 33
        // -> 12 us against a preparation, three bands and three copies)
        bool band = true;
        for (int i = 0; i < 3; ++i)
            band = band && (ns[i] == 0 ||
                            (band_rule(dtype, g, M, K, ns[i], ws[i], di.cus).takes &&
                             !thin_takes(dtype, M, (int64_t)ns[i] * (K / g.be) * g.bb)));
        if (band) {
            const int rc = run_band(dtype, g, x, ms, nullptr, 0, 0, y, M, K, Nt, dev, di, st, nullptr,
                                    0, false);
            if (rc != FQ_ERR_WORKSPACE) return rc;
        }
    }
    uint8_t* buf = nullptr;
    const int nmax = std::max(Nq, std::max(Nk, Nv));
    StreamScratch::Lease lease(stream_scratch(dev, st, 1));
    const int rs = lease.get((size_t)M * nmax * sizeof(float), st, &buf);
    if (rs != FQ_OK) return rs;
    float* tmp = reinterpret_cast<float*>(buf);
    // The band kernel's token operands serve every matmul here that takes
    // it, one after another: the stream's slot-0 workspace is first grown to
    // the largest of their band-kernel needs, so none of these calls replaces
    // it (a call on another path clears the flag, and the next band call
    // prepares again).  Where that growth is refused (graph capture with a
    // smaller reserve) each call prepares its own.
    bool share = false;
    if (M <= 16 && K % 256 == 0) {
        size_t need = 0;
        for (int i = 0; i < 3; ++i)
            if (ns[i] > 0)
                for (int mt : {4, 3, 2}) need = std::max(need, mmqs_need(M, K, ns[i], di.cus, mt));
        StreamScratch::Lease l0(stream_scratch(dev, st, 0));
        uint8_t* p0 = nullptr;
        share = l0.get(need, st, &p0) == FQ_OK;
    }
    bool band_x = false;
    int off = 0;
    for (int i = 0; i < 3; ++i) {
        if (ns[i] > 0) {
            const int rc = run_matmul(dtype, x, ws[i], nullptr, 0, 0, tmp, M, K, ns[i], st,
                                      nullptr, 0, share ? &band_x : nullptr);
            if (rc != FQ_OK) return rc;
            e = fq::launch_copy_cols(tmp, y, M, ns[i], Nt, off, di.cus, st);
            if (e != hipSuccess) return hip_fail(e);
        }
        off += ns[i];
    }
    return FQ_OK;
}

int fq_ffn_down_residual(uint32_t dtype, const float* x, const void* w, const float* residual,
                         float* y, int M, int K, int N, void* stream) {
    if (!residual) return FQ_ERR_NULL;
    return run_matmul(dtype, x, w, residual, 2, (int64_t)M * N, y, M, K, N,
                      static_cast<hipStream_t>(stream));
}

int fq_ffn_down_residual_packed(uint32_t dtype, const float* x, const void* w_packed,
                                const float* residual, float* y, int K, int N, void* stream) {
    if (!residual) return FQ_ERR_NULL;
    return packed_gemv(dtype, x, w_packed, nullptr, nullptr, 0, 0, 0, residual, N, y, K, N,
                       static_cast<hipStream_t>(stream), false);
}

int fq_ffn_up_fused(uint32_t dtype, const float* x, const void* w_gate, const void* w_up, float* y,
                    int M, int K, int N, void* stream) {
    Geometry g;
    if (!geometry(dtype, g)) return FQ_ERR_DTYPE;
    if (M < 0 || N < 0 || K < 0 || K % g.be != 0) return FQ_ERR_SHAPE;
    if (M == 0 || N == 0) return FQ_OK;
    if (!x || !w_gate || !w_up || !y) return FQ_ERR_NULL;
    if (!row_fits(g, K)) return FQ_ERR_SHAPE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (M == 1 && packable(dtype)) {
        // one launch at every size: gate and up rows interleaved,
        // silu(gate) * up in the epilogue, straight from the GGUF bytes
        // (against two matmuls and the SiLU-multiply launch)
        const int rc = packed_gemv(dtype, x, w_gate, w_up, nullptr, 0, 0, 1, nullptr, 0, y, K, N,
                                   st, true);
        if (rc != FQ_ERR_SHAPE) return rc;
    }
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    const DevInfo di = device_info(dev);
    if (M > 32) {  // one prefill launch, gate and up rows in each tile
        const int rc = run_prefill(dtype, g, x, Mats{fq::MM_PAIR, {w_gate, w_up}, {N}}, nullptr, 0, 0,
                                   y, M, K, N, dev, di, st, nullptr, 0);
        if (rc != kNotTaken) return rc;
    }
    if (M > 1 && M <= 32) {  // gate and up rows in one launch
        const Mats ms{fq::MM_PAIR, {w_gate, w_up}, {N}};
        const int64_t bytes = (int64_t)N * (K / g.be) * g.bb;
        const bool band = M >= 5 && M <= 16 && K < 32 * 256 &&  // K unsplit
                          band_rule(dtype, g, M, K, N, w_gate, di.cus).takes &&
                          band_rule(dtype, g, M, K, N, w_up, di.cus).takes;
        // 5..16 tokens: the band kernel where it is estimated faster, for matrices that
        // it takes one by one unless 10 % slower (M = 8: Q4_1 9472 x 5632 42.9 us there,
        // 28.0 here, Q5_0 9472 x 4096 35.7 and 28.2); what it does not take here too
        const bool thin = thin_takes_pair(dtype, M, bytes);
        const double limit =
            band ? (thin_takes(dtype, M, bytes) ? 1.04 : 0.9) * band_us(dtype, g, K, N, true, di.cus)
                 : HUGE_VAL;
        auto run = [&](double us) {
            return run_thin(dtype, g, x, ms, nullptr, 0, 0, y, M, K, N, dev, di, st, nullptr, 0, us);
        };
        int rc = thin || (M >= 5 && !band) ? run(limit) : kNotTaken;
        if (band && (rc == kSlower || rc == kNotTaken)) {
            rc = run_band(dtype, g, x, ms, nullptr, 0, 0, y, M, K, N, dev, di, st, nullptr, 0, false);
            if (rc == FQ_ERR_WORKSPACE) rc = run(HUGE_VAL);  // capture on what another call sized
        }
        if (rc != kNotTaken) return rc;
    }
    uint8_t* buf = nullptr;
    StreamScratch::Lease lease(stream_scratch(dev, st, 1));
    const int rs = lease.get(2 * (size_t)M * N * sizeof(float), st, &buf);
    if (rs != FQ_OK) return rs;
    float* gate = reinterpret_cast<float*>(buf);
    float* up = gate + (size_t)M * N;
    // gate and up share x, M, K, N and the format: when the gate call takes
    // the band kernel, the up call does too and reuses its token operands
    // (one token-prep launch fewer: about 5 us)
    bool band_x = false;
    int rc = run_matmul(dtype, x, w_gate, nullptr, 0, 0, gate, M, K, N, st, nullptr, 0, &band_x);
    if (rc != FQ_OK) return rc;
    rc = run_matmul(dtype, x, w_up, nullptr, 0, 0, up, M, K, N, st, nullptr, 0, &band_x);
    if (rc != FQ_OK) return rc;
    e = fq::launch_silu_mul(gate, up, y, (size_t)M * N, di.cus, st);
    return e == hipSuccess ? FQ_OK : hip_fail(e);
}

int fq_reserve_workspace(int M_max, int K_max, int N_max, void* stream) {
    if (M_max < 0 || K_max < 0 || N_max < 0) return FQ_ERR_SHAPE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    const DevInfo di = device_info(dev);
    // slot 0: the largest plan of up to M_max tokens, K_max columns and N_max rows
    // per matrix, up to three of them in one launch
    size_t need0 = 0;
    const int Kp = K_max - K_max % 256;
    const int64_t cols = 3 * (int64_t)N_max;
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    // the fp16 MFMA kernel (the split-K slabs grow with splits x N, and fewer rows
    // can mean more splits: every row count that changes the tile count is
    // tried), and the batch-1 kernel's K-split slabs for 2..4 tokens (at most 8)
    for (int n = N_max; n > 0; n = n > 128 ? ((n - 1) / 128) * 128 : 0)
        for (int m = 2; m <= M_max; ++m) {
            need0 = std::max(need0, plan_mmq(m, K_max, n, di.cus).total);
            if (m <= 4) need0 = std::max(need0, (size_t)8 * m * n * sizeof(float));
        }
    if (M_max >= 2 && N_max > 0 && Kp > 0) {  // the band kernel (at most nsb / 8 splits of cus bands)
        const int m = std::min(M_max, 16);
        const MmqPlan pl = plan_mmq(m, Kp, N_max, di.cus);
        const int64_t slabs = std::min<int64_t>(64LL * di.cus, (int64_t)(Kp / 2048) * N_max);
        need0 = std::max(need0, 256 + al(pl.xop_b) + al(pl.xsum_b) + al(pl.ex_b) + al((size_t)slabs * m * 4));
        // the shared-operand kernel: parts - 2 of a tile's columns are at most a
        // step of every CU, so (parts - 2) cols <= 256 cus; 64 MiB in all
        const int mt = std::min(M_max, 32);
        const size_t ops = 256 + al(fq::mmqt_xop_bytes(mt, Kp)) + al(fq::mmqt_sum_bytes(mt, Kp));
        const int64_t parts = std::min<int64_t>(16 * cols, 2 * cols + 256LL * di.cus);
        need0 = std::max(need0, std::min(kNoAllocBytes, ops + al((size_t)parts * mt * 4)));
    }
    if (M_max > 32 && N_max > 0 && Kp > 0) {  // the prefill kernels
        // (the larger sums of Q5_K, the rewritten rows of Q6_K)
        const MmqpPlan pl = mmqp_sizes(FQ_DTYPE_Q5_K, M_max, Kp, 0, 0, 1);
        const size_t row_b = (size_t)fq::mmqp_q6c_bytes(1, Kp);
        const size_t q6c_b = std::max(row_b * N_max, std::min(row_b * (size_t)cols, kMaxRewrite));
        need0 = std::max(need0, pl.total + al(q6c_b) + al(mmqp_max_slabs(M_max, Kp, cols, di.cus)));
    }
    const size_t need1 = 2 * (size_t)M_max * N_max * sizeof(float);
    uint8_t* p = nullptr;
    if (need0) {
        StreamScratch::Lease l(stream_scratch(dev, st, 0));
        const int rc = l.get(need0, st, &p);
        if (rc != FQ_OK) return rc;
    }
    if (need1) {
        StreamScratch::Lease l(stream_scratch(dev, st, 1));
        const int rc = l.get(need1, st, &p);
        if (rc != FQ_OK) return rc;
    }
    return FQ_OK;
}

int fq_release_workspace(void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    e = hipStreamSynchronize(st);  // queued work may still read the buffers
    if (e != hipSuccess) return hip_fail(e);
    for (int slot = 0; slot < 2; ++slot) {
        StreamScratch& s = stream_scratch(dev, st, slot);
        std::lock_guard<std::mutex> lk(s.mu);
        for (uint8_t* r : s.retired) hipFree(r);
        s.retired.clear();
        if (s.p) hipFree(s.p);
        s.p = nullptr;
        s.n = 0;
    }
    return FQ_OK;
}

}  // extern "C"
