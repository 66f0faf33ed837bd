// MFMA GEMMs (NT / NN / TN) with fused epilogues for the linears of the GPT layer at tensor-parallel size 1: which kernel
// runs a product (the plan), the sums of k splits, and the C entry points.  The kernels are in the gemm_*.hip beside.
#include "gemm_epilogue.h"
#include "vec_grads.h"

#include <mutex>

namespace tp {

// The tiles of gemm_dma.hip (configurations 0, 3, 5, 8, 11, 12, 13; fp32: 0) and of gemm_tall.hip (2, 17 to 20; a grouped
// launch, TN, of 2, 19 or 20): launch `cfg` on `grid` = (column tiles, row tiles, k splits); false when there is no such
// kernel.
bool launch_gemm_dma(int cfg, int op, int dtype, dim3 grid, const GemmArgs& a, hipStream_t s);
bool launch_gemm_tall(int cfg, int op, int dtype, dim3 grid, const GemmArgs& a, hipStream_t s);
bool launch_gemm_tall_group(int cfg, int dtype, int tiles, const GemmGroupArgs& ga, const VecGradArgs* vec, hipStream_t s);

// Sums the split-K partials and applies the epilogue.  A block of 256 threads covers 256 columns
// (32 threads x 8 columns) by 8 rows, one vector of 8 columns a thread; column sums are combined across the
// rows in LDS so that they cost one atomic per column per block.  Bound by the latency of its loads (4 partial
// sums of 256 x 2048 are 8 MB, 1.6 us of bandwidth): four rows a thread, one split at a time, took 14.0 us.
// One row a thread with four splits' loads in flight takes 7.2.
template <typename T>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(GemmArgs a) {
    __shared__ float cs[8][256];
    const int cl = threadIdx.x & 31, rl = threadIdx.x >> 5;
    const int col0 = (blockIdx.x * 32 + cl) * 8;
    const int row = blockIdx.y * 8 + rl;
    float csum[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) csum[e] = 0.f;
    if (col0 < a.N && row < a.M) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = 0.f;
        const long plane = (long)a.M * a.N;
        const float* src = a.partial + (long)row * a.N + col0;
        // four splits' loads under way at a time (the partial sums are added in the order of the splits)
        for (int z = 0; z < a.nsplit; z += 4) {
            float4 p[4][2];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (z + u < a.nsplit) {
                    p[u][0] = *reinterpret_cast<const float4*>(src + (z + u) * plane);
                    p[u][1] = *reinterpret_cast<const float4*>(src + (z + u) * plane + 4);
                }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (z + u < a.nsplit) {
                    v[0] += p[u][0].x; v[1] += p[u][0].y; v[2] += p[u][0].z; v[3] += p[u][0].w;
                    v[4] += p[u][1].x; v[5] += p[u][1].y; v[6] += p[u][1].z; v[7] += p[u][1].w;
                }
        }
        epilogue_vec8<T>(a, row, col0, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) csum[e] = v[e];
    }
    if (a.colsum) {
#pragma unroll
        for (int e = 0; e < 8; ++e) cs[rl][cl * 8 + e] = csum[e];
        __syncthreads();
        const int c = threadIdx.x;
        const int col = blockIdx.x * 256 + c;
        if (col < a.N) {
            float t = 0.f;
#pragma unroll
            for (int r = 0; r < 8; ++r) t += cs[r][c];
            atomicAdd(a.colsum + col, t);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
static constexpr int kNumCU = 256;  // MI355X

// Tile configurations of the 16-bit kernels by number (the numbers are what the measured plan table, the
// `reserved` field of tp_gemm_desc and the tuning script refer to; numbers not listed do not exist).
struct TileCfg { int bm, bn, bk, stages; };
static bool tile_cfg(int id, TileCfg& c) {
    switch (id) {
    case 0: c = {64, 64, 64, 2}; return true;      // gemm_kernel, register-staged (fp32 runs it with 64 x 64 x 16 tiles)
    // gemm_dma_kernel: four waves 2 x 2 (configuration 3: eight waves of 64 x 64)
    case 3: c = {128, 256, 64, 3}; return true;
    case 5: c = {128, 128, 64, 2}; return true;
    case 8: c = {64, 64, 64, 4}; return true;
    case 11: c = {64, 256, 64, 3}; return true;
    case 12: c = {64, 64, 128, 4}; return true;    // NT and NN on weights up to 4096 x 4096: the deep rings of gemm_deep.hip
    case 13: c = {128, 128, 64, 3}; return true;
    // gemm_tall_kernel: 256-row tiles
    case 2: c = {256, 256, 32, 4}; return true;    // gemm_tall_kernel, 20 on 16 x 16 x 32 MFMA blocks
    // gemm_pipe_kernel: four waves, 16 x 16 x 32 MFMA blocks, software-pipelined k-loop
    case 6: c = {192, 160, 64, 3}; return true;    // 2 x 2 waves of 96 x 80 (NT only, like 7)
    case 7: c = {160, 160, 64, 3}; return true;    // 2 x 2 waves of 80 x 80
    case 14: c = {192, 128, 64, 3}; return true;   // 2 x 2 waves of 96 x 64
    case 15: c = {256, 128, 64, 3}; return true;   // 4 x 1 waves of 64 x 128
    case 16: c = {128, 128, 64, 3}; return true;   // 2 x 2 waves of 64 x 64
    case 17: c = {256, 160, 64, 3}; return true;   // 4 waves stacked in M, 64 x 160 each (NT only)
    case 18: c = {256, 128, 64, 3}; return true;   // 64 x 128 each
    case 19: c = {256, 256, 64, 2}; return true;   // 8 waves (4 x 2) of 64 x 128
    case 20: c = {256, 256, 32, 4}; return true;   // the same with half the k-tile and twice the stages
    // gemm_stream_kernel (gemm_stream.hip; NT and NN): whole-slice row tiles of 64 * RB rows, separate activation /
    // weight rings (stages = the weight ring's); 4 waves unless noted
    case 21: c = {192, 128, 64, 5}; return true;
    case 22: c = {256, 128, 64, 4}; return true;
    case 23: c = {256, 128, 64, 6}; return true;   // two activation stages
    case 24: c = {192, 80, 64, 8}; return true;    // NT only
    case 25: c = {256, 80, 64, 6}; return true;    // NT only
    case 26: c = {128, 128, 64, 7}; return true;
    case 27: c = {256, 64, 64, 8}; return true;
    case 28: c = {192, 64, 64, 10}; return true;
    case 29: c = {256, 128, 64, 4}; return true;   // 8 waves
    case 30: c = {192, 128, 64, 5}; return true;   // 8 waves
    case 31: c = {192, 128, 64, 5}; return true;   // 16 waves
    case 32: c = {256, 128, 64, 4}; return true;   // 16 waves
    case 33: c = {192, 256, 64, 3}; return true;   // 16 waves
    case 34: c = {256, 256, 64, 3}; return true;   // 16 waves
    case 35: c = {128, 256, 64, 3}; return true;   // 16 waves
    case 36: c = {64, 256, 64, 4}; return true;    // 16 waves
    case 37: c = {128, 128, 64, 7}; return true;   // 16 waves
    case 38: c = {64, 128, 64, 8}; return true;    // 16 waves
    case 39: c = {128, 256, 64, 3}; return true;   // 8 waves
    case 40: c = {64, 256, 64, 4}; return true;    // 8 waves
    // gemm_pipe_kernel again: row tiles that fit slices of 224 and of 160 / 320 rows (whole 16-row blocks, so
    // nothing of a tile lies beyond the slice)
    case 41: c = {224, 128, 64, 3}; return true;   // 2 x 2 waves of 112 x 64
    case 42: c = {160, 128, 64, 3}; return true;   // 2 x 2 waves of 80 x 64
    case 43: c = {224, 160, 64, 3}; return true;   // 2 x 2 waves of 112 x 80 (NT only, like 6 and 7)
    // gemm_wide_kernel: eight waves (2 x 4) of 128 x 64, software-pipelined
    case 44: c = {256, 256, 64, 2}; return true;   // NT and NN
    default: return false;
    }
}
static constexpr int kFirstStreamCfg = 21, kLastStreamCfg = 40;
static constexpr int kWideCfg = 44;
static constexpr int kSkinnyRows = 32;

// Measured plans: for NT / NN the weight extents (N, K) match exactly and M (tokens of the slice) picks the
// nearest measured M at or above it (at least half of it, so that a much shorter slice falls through to the
// heuristics); on weights of up to 4096 x 4096, which have an estimate of their own, rows that end in the same 16 as M (128 rows on
// 8192 x 2048 with the entry of 256, 128 x 128 tiles, 22.8 us; 64 x 64 as the estimate has it 13.9).  TN (parameter gradients) matches all three extents.
struct TunedPlan { int op, M, N, K, cfg, nsplit; };
static const TunedPlan kTuned[] = {
#include "gemm_tuned.inc"
    {-1, 0, 0, 0, 0, 0},
};
// Those of its entries that are not the best beside other streams' launches (reserved bit 24).  A sliced step on one stream, three,
// with the entries for products alone / these for all: 44B, 32-token slices 134 and 112 ms / 167 and 102; 175B, 128 tokens 63.4 and
// 60.9 / 70.8 and 58.3; 13B 27.1 and 24.8 / 28.4 and 24.6.
static const TunedPlan kTunedBeside[] = {
#include "gemm_tuned_beside.inc"
    {-1, 0, 0, 0, 0, 0},
};
constexpr int kBeside = 1 << 24, kForced = 0xffffff;        // of tp_gemm_desc.reserved (and kNoBackward, gemm_epilogue.h)

static bool small_weight(const tp_gemm_desc* d) { return (long)d->N * d->K <= (16L << 20); }
static const TunedPlan* find_tuned(const tp_gemm_desc* d) {
    const TunedPlan* best = nullptr;
    for (const TunedPlan* t = kTuned; t->op >= 0; ++t) {
        if (t->op != d->op || t->N != d->N || t->K != d->K) continue;
        if (d->op == TP_GEMM_TN) {
            if (t->M == d->M) return t;
            continue;
        }
        if (t->M >= d->M && (small_weight(d) ? (t->M + 15) / 16 == (d->M + 15) / 16 : t->M <= 2 * d->M) && (!best || t->M < best->M)) best = t;
    }
    if (best && (d->reserved & kBeside))
        for (const TunedPlan* t = kTunedBeside; t->op >= 0; ++t)
            if (t->op == best->op && t->M == best->M && t->N == best->N && t->K == best->K) return t;
    return best;
}

struct GemmPlan {
    int cfg;
    int nsplit;
    int kper, bk;   // k per split, and the k-tile it is a multiple of
    int gx, gy;
    int deep;       // columns of the deep-ring tile (gemm_deep.hip) that runs configuration 12, 0: none
    int wide;       // columns of the eight-wave tile (gemm_wide.hip) that runs configuration 44: 256 or 192
};

static void finish_plan(const tp_gemm_desc* d, GemmPlan& p, int bk, int nsplit) {
    long kt = (d->K + bk - 1) / bk;
    if (nsplit > kt) nsplit = (int)kt;
    if (nsplit < 1) nsplit = 1;
    long per = (kt + nsplit - 1) / nsplit;
    p.bk = bk;
    p.kper = (int)(per * bk);
    p.nsplit = (int)((d->K + p.kper - 1) / p.kper);
}

// The time (us) of `tiles` workgroups of a tile configuration over k: rounds of one workgroup per CU, each a fixed part
// (prologue, epilogue) and a part per k; a partly filled round runs somewhat faster per k (less traffic, higher clocks).
// Where the operands outgrow the memory-side cache (`spill`) a tile that reads them more often falls behind.  NT and NN: fitted to
// 1300 products (520 to 8192 rows, hidden 512 to 12288, alone on the chip, weights from memory), rms 5 to 9 %, then moved to
// where the choice is best: 1.006 times the fastest of 64 x 64 to 256 x 256 tiles and their splits in the mean.  TN: fitted to 66
// (hidden 1024 to 6144; k of 1024, 2048 and 4096).
struct TileCost { int cfg, bm, bn; float fixed, per_k, per_k_spill, partial; };
static const TileCost kTileCost[] = {
    {16, 128, 128, 3.86f, 0.00845f, 0.00950f, 0.927f},
    {14, 192, 128, 5.74f, 0.01031f, 0.01179f, 0.982f},
    {15, 256, 128, 6.60f, 0.01257f, 0.01245f, 0.920f},
    {kWideCfg, 256, 256, 6.70f, 0.02276f, 0.02220f, 0.832f},
    {kWideCfg, 256, 192, 5.62f, 0.01992f, 0.02102f, 0.970f},
};
static const TileCost kTileCostTN[] = {
    {16, 128, 128, 4.8f, 0.0068f, 0.0084f, 0.72f},
    {15, 256, 128, 12.0f, 0.0115f, 0.0125f, 0.72f},
    {2, 256, 256, 11.5f, 0.0248f, 0.0248f, 0.72f},
};
static float tile_time(const TileCost& c, long tiles, float k, bool spill) {
    const float per_k = spill ? c.per_k_spill : c.per_k;
    const long full = tiles / kNumCU, rest = tiles % kNumCU;
    return full * (c.fixed + per_k * k) + (rest ? c.fixed + per_k * k * (c.partial + (1.f - c.partial) * rest / kNumCU) : 0.f);
}
static bool tile_serves(const TileCost& c, int K) { return c.cfg != kWideCfg || K >= 64; }

// Products on weights of up to 4096 x 4096, NT and NN.  The time (us) of `tiles` workgroups, one round per 256: a fixed part
// and a part per k, which grows from `lo` for a few workgroups to `hi` for a full round (they share the caches' and the
// memory's bandwidth).  64 x 64 tiles fit a CU twice: theirs is a round per 512, `lo` to `mid` while each has a CU to itself, `two`
// to `hi` when a second one comes beside.  Fitted to 1300 products (hidden 512 to 2816, 33 to 512 rows, up to 4 splits, no weight used
// twice within 400 MB): rms error 6 to 11 %, then moved to where the choice is best: 1.004 times the fastest of these tiles in the
// mean, 1.11 at most.  (With a round per 256 of the 64 x 64 tiles the estimate gave up to 512 of them to the 128 x 128 tile: 640 x 2304 x
// 768 8.2 us, 11.0 with it; 1500 x 1024 x 1024 9.7 and 11.8.)
struct SliceCost { float fixed, round, lo, hi; };
struct PairCost { float fixed, round, lo, mid, two, hi; };
static const PairCost kSlice64[2] = {{3.14f, 1.12f, 0.00402f, 0.00448f, 0.00630f, 0.00811f},     // cfg 8: NT, NN
                                     {3.12f, 0.66f, 0.00438f, 0.00450f, 0.00682f, 0.00936f}};
static const SliceCost kSlice128[2] = {{3.83f, 2.19f, 0.00909f, 0.00922f}, {3.96f, 2.10f, 0.00742f, 0.00802f}};   // cfg 16
static const SliceCost kDeep32[2] = {{4.18f, 2.47f, 0.00237f, 0.00264f}, {4.06f, 1.87f, 0.00359f, 0.00399f}};
static const SliceCost kDeep64[2] = {{4.29f, 2.40f, 0.00341f, 0.00383f}, {4.05f, 1.93f, 0.00422f, 0.00422f}};
static const SliceCost kDeep128[2] = {{4.76f, 2.31f, 0.00608f, 0.00611f}, {4.50f, 1.88f, 0.00690f, 0.00690f}};
static float slice_time(const SliceCost& c, long tiles, float k) {
    const long full = (tiles - 1) / kNumCU;
    const float part = (float)(tiles - full * kNumCU) / kNumCU;
    return c.fixed + full * (c.round + k * c.hi) + k * (c.lo + (c.hi - c.lo) * part);
}
static float slice_time(const PairCost& c, long tiles, float k) {
    const long full = (tiles - 1) / (2 * kNumCU);
    const float part = (float)(tiles - full * 2 * kNumCU) / kNumCU;
    return c.fixed + full * (c.round + k * c.hi) + k * (part <= 1.f ? c.lo + (c.mid - c.lo) * part : c.two + (c.hi - c.two) * (part - 1.f));
}
// (the deep rings have no column sums, and no tiles for weights that stream from HBM beside other launches)
static bool deep_serves(const tp_gemm_desc* d) { return d->op != TP_GEMM_TN && d->dtype != TP_F32 && small_weight(d) && !d->colsum_acc; }
// The deep ring's time at `ns` splits and its tile's columns.
static float deep_time(const tp_gemm_desc* d, int ns, int* columns) {
    const int op = d->op == TP_GEMM_NN;
    const long rows = (d->M + 63) / 64;
    float best = 0.f;
    *columns = 0;
    auto take = [&](int c, const SliceCost& cost) {
        const float t = slice_time(cost, rows * ((d->N + c - 1) / c) * ns, (float)d->K / ns);
        if (!*columns || t < best) { best = t; *columns = c; }
    };
    take(32, kDeep32[op]);
    take(64, kDeep64[op]);
    take(128, kDeep128[op]);
    return best;
}
// Products whose sums of k splits the layer calls and the runner leave to the LayerNorm behind them: the two with a residual,
// and the data gradients of the widening linears (the LM head's, which has no LayerNorm behind it, comes as `ragged`).
static bool feeds_layernorm(const tp_gemm_desc* d) {
    return d->epilogue == TP_EPI_BIAS_RESIDUAL || (d->op == TP_GEMM_NN && d->epilogue == TP_EPI_STORE && !d->ragged && d->K >= 3L * d->N);
}
// A split's partial sums and the launch that adds them, or the LayerNorm's reads of them (264 products with the LayerNorm behind,
// 96 to 3072 rows, hidden 768 to 2560: the choice takes 1.011 times the fastest in the mean; priced like the launch the splits went
// unused, 768 x 1024 x 4096 NN with the LayerNorm 22.2 us in four splits, 27.6 in one piece).
static float reduce_time(const tp_gemm_desc* d, int ns) {
    if (ns == 1) return 0.f;
    const float sums = 4.f * ns * d->M * d->N;
    return feeds_layernorm(d) ? 1.5f + 0.15e-6f * sums : 3.19f + 0.21e-6f * sums;
}
static void plan_slice(const tp_gemm_desc* d, int& cfg, int& ns) {
    const int op = d->op == TP_GEMM_NN;
    const long t64 = (long)((d->M + 63) / 64) * ((d->N + 63) / 64), t128 = (long)((d->M + 127) / 128) * ((d->N + 127) / 128);
    float best = 0.f;
    for (int n = 1; n <= 8; ++n) {
        if (n > 1 && (d->N % 8 || d->K / n < 1536 || t128 * n > kNumCU)) break;
        const float k = (float)d->K / n, r = reduce_time(d, n);
        int columns;
        auto take = [&](int c, float t) { if (best == 0.f || t < best) { best = t; cfg = c; ns = n; } };
        if (n == 1 || t64 * n <= 2 * kNumCU) {
            if (deep_serves(d)) take(12, r + deep_time(d, n, &columns));
            take(8, r + slice_time(kSlice64[op], t64 * n, k));
        }
        if (d->M > 64) take(16, r + slice_time(kSlice128[op], t128 * n, k));
    }
}

// The columns of the eight-wave tile at `ns` splits.
static int wide_columns(const tp_gemm_desc* d, int ns) {
    const bool spill = 2.0 * ((double)d->M + d->N) * d->K > 225e6;
    int columns = 0;
    float best = 0.f;
    for (const TileCost& c : kTileCost) {
        if (c.cfg != kWideCfg) continue;
        const long tiles = (long)((d->M + c.bm - 1) / c.bm) * ((d->N + c.bn - 1) / c.bn);
        const float t = tile_time(c, tiles * ns, (float)d->K / ns, spill);
        if (!columns || t < best) { best = t; columns = c.bn; }
    }
    return columns;
}

// Products of more than 512 rows and parameter gradients: the tile and the k split with the smallest estimate.  A split
// costs its fp32 partial sums (written and read once at 5.5 TB/s) and the launch that adds them, and has to be 4 % ahead (NT, NN:
// part of the same fit); less where a LayerNorm takes them.  The rules this replaces
// named 256 x 256 tiles from 192 of them on and split or shrank them otherwise, without regard for the last round: the
// estimate's choice takes 0.61 to 1.0 of their time (1024 x 5120 x 20480: 284 -> 188 us; 4096 x 1600 x 6400: 117 -> 80).
static void plan_large(const tp_gemm_desc* d, int& cfg, int& ns) {
    const float K = (float)d->K;
    // 48 to 63 tiles of 256 x 256 on a long k are split to one round: the estimate has too little for the 128 x 128 tiles it
    // names there.  2048 x 1792 x 16384: 121 us against 141, 2048 x 1600 x 12800: 97 against 113; at k = 8192 the
    // estimate is right (1536 x 2048: 65 against 55, 1700 x 2048: 67 against 54), from 24576 on it names the same.
    const long t256 = (long)((d->M + 255) / 256) * ((d->N + 255) / 256);
    if (d->op != TP_GEMM_TN && d->K >= 12288 && t256 >= 48 && t256 < 64) {
        cfg = kWideCfg;
        ns = (int)(kNumCU / t256);
        return;
    }
    const bool spill = 2.0 * ((double)d->M + d->N) * d->K > 225e6;
    // 64 x 64 tiles (TN: two per CU): where the larger ones leave most of the chip idle
    const long t64 = (long)((d->M + 63) / 64) * ((d->N + 63) / 64);
    float best = d->op != TP_GEMM_TN ? slice_time(kSlice64[d->op == TP_GEMM_NN], t64, K)
                 : t64 <= kNumCU ? 4.6f + 0.0038f * K : (float)((t64 + 511) / 512) * (3.5f + 0.0066f * K);
    cfg = 8;
    ns = 1;
    int columns;
    if (deep_serves(d) && t64 <= 2 * kNumCU) {      // (1024 x 768 x 3072: 16.3 -> 13.4 us, 1024 x 512 x 2048 11.9 -> 8.8)
        const float t = deep_time(d, 1, &columns);
        if (t < best) { best = t; cfg = 12; }
    }
    const bool layernorm = feeds_layernorm(d);
    auto consider = [&](const TileCost& c) {
        if (!tile_serves(c, d->K)) return;
        const long tiles = (long)((d->M + c.bm - 1) / c.bm) * ((d->N + c.bn - 1) / c.bn);
        for (int n = 1; n <= 8; ++n) {
            if (n > 1 && (d->N % 8 || d->K / n < 512 || tiles * n > 2 * kNumCU)) break;
            float t = tile_time(c, tiles * n, K / n, spill);
            if (n > 1 && layernorm) t += 2.5f + 1.2e-6f * n * d->M * d->N;
            else if (n > 1) t = (t + 4.f + (float)((double)n * d->M * d->N * 8 / 5.5e6)) * (d->op == TP_GEMM_TN ? 1.f : 1.044f);
            if (t < best * (n > 1 && layernorm ? 0.98f : 1.f)) { best = t; cfg = c.cfg; ns = n; }       // (a tie goes to fewer splits)
        }
    };
    if (d->op == TP_GEMM_TN) for (const TileCost& c : kTileCostTN) consider(c);
    else for (const TileCost& c : kTileCost) consider(c);
}

// Forward products of up to kSkinnyRows rows on a weight of up to 4096 x 4096 run without LDS tiles: the plan's k splits,
// whatever its tile.  (Beyond, both are bound by the weight stream and the tile kernels read the activation less often:
// 16 rows on 20480 x 5120 49 us against 58.  A forced tile, and column sums, take the tile kernels.)
// Only where no backward follows (another order of the sums turns ReLU units near zero on or off, and the weight gradients behind them
// move by 2e-2 in fp16), up to 8 rows: without k splits, unless the rows of a weight are longer than 8192 and its tiles of 16 of
// them do not come to whole rounds of the CUs (5120 x 20480, 1.25 of them: 48 us against 40 on tiles with three splits).
static inline bool skinny_unsplit(const tp_gemm_desc* d) {
    return (d->reserved & kNoBackward) && d->M <= 8 && (d->K <= 8192 || d->N % 4096 == 0);
}
// Those also on larger weights, where tiles of 64 columns, the alternative, would leave half of their last round of CUs or more
// without one, or split k.  us, 4 and 8 rows, tiles / these: 5120 x 5120 20.4 / 17.9 and 20.1 / 18.5, 7680 x 2560 14.6 / 10.1 and 14.4 / 10.4,
// 20480 x 5120 48.4 / 41.0 and 47.5 / 43.3, 24576 x 4096 44.6 / 40.1 and 42.2 / 42.5, 4096 x 16384 37.1 / 31.4 and 37.1 / 33.0.  Where
// they fill it (12288 x 4096 23.8 / 24.9 and 24.0 / 25.3, 15360 x 5120 30.5 / 31.6 and 30.7 / 32.7, 28672 x 4096 48.0 / 51.0) these are taken
// for the LayerNorm's launch that they save, 3.7 us, and from k = 8192 on (15360 x 8192 57.9 / 53.2 and 57.2 / 52.3).  Weights with few and
// long rows keep the tiles' k splits: 4608 x 6144 17.8 / 19.4, 5120 x 8192 22.7 / 24.4.
static inline bool skinny_large(const tp_gemm_desc* d) {
    const bool filled = ((d->N + 63) / 64 - 1) % kNumCU >= kNumCU / 2;
    return skinny_unsplit(d) && (long)d->N * d->K <= 256L << 20 && (d->N % 4096 == 0 || 4L * d->K <= 5L * d->N) &&
           (!filled || d->K >= 8192 || skinny_takes_ln(d->M, d->K));
}
static inline bool runs_skinny(const tp_gemm_desc* d) {
    return d->op == TP_GEMM_NT && d->dtype != TP_F32 && d->M <= kSkinnyRows && (d->reserved & 0xff) == 0 && !d->colsum_acc &&
           ((long)d->N * d->K <= 16L << 20 || skinny_large(d));
}

// fp32 products that run on tiles of 32 x 32 whose waves share k, in one launch (gemm_f32.hip): where the tiles come to at
// most two workgroups per CU and eight waves take all of k at once.  Against 64 x 64 tiles with splits: k = 256 1.9 (up to 128
// tiles) to 1.4 (512) times as fast, k = 64 1.25 to 1.05 up to 256 tiles, less beyond.  The rule ends with the first turn: k = 512, in
// two, was measured on products alone only (1.45 to 1.15), k = 1024 at 1.1 to 0.8.  (A forced tile or split, and column sums, take
// the tile kernel.)
void launch_gemm_f32_small(int op, const GemmArgs& a, hipStream_t s);
static bool runs_f32_small(const tp_gemm_desc* d) {
    if (d->dtype != TP_F32 || d->colsum_acc || (d->reserved & kForced)) return false;
    const long tiles = (long)((d->M + 31) / 32) * ((d->N + 31) / 32);
    return d->K <= 256 && tiles <= (d->K < 128 ? kNumCU : 2 * kNumCU);
}

static GemmPlan plan_gemm(const tp_gemm_desc* d) {
    GemmPlan p;
    p.deep = p.wide = 0;
    if (d->dtype == TP_F32) {
        p.cfg = 0;
        p.gx = (d->N + 63) / 64; p.gy = (d->M + 63) / 64;
        if (runs_f32_small(d)) {
            finish_plan(d, p, 16, 1);
            return p;
        }
        long tiles = (long)p.gx * p.gy;
        int nsplit = 1;
        if (tiles < 2 * kNumCU) {
            long want = (2 * kNumCU + tiles - 1) / tiles;
            long kt = (d->K + 15) / 16;
            long maxs = kt / 8 > 0 ? kt / 8 : 1;
            nsplit = (int)(want < maxs ? want : maxs);
            if (nsplit > 32) nsplit = 32;       // (16 at most: 8 rows on 1024 x 4096 18.0 -> 16.6 us alone, 20.9 -> 16.6 with the LayerNorm)
        }
        if (d->N % 8) nsplit = 1;       // (partial sums are rows of N)
        finish_plan(d, p, 16, nsplit);
        return p;
    }
    // reserved: bits 0-7 force a tile configuration (1-based index + 1 so that 0 means automatic),
    // bits 8-15 force the number of k splits.  For tuning and tests.
    int forced_cfg = (d->reserved & 0xff) - 1;
    int forced_split = (d->reserved >> 8) & 0xff;
    const long t128 = (long)((d->M + 127) / 128) * ((d->N + 127) / 128);
    const long t64 = (long)((d->M + 63) / 64) * ((d->N + 63) / 64);
    int cfg, ns = 1;
    const long t256n = (d->N + 255) / 256;
    const long t256 = (long)((d->M + 255) / 256) * t256n;
    // k splits that bring `tiles` workgroups as near to one per CU as they get without exceeding it (a second, partly
    // filled round costs more than the idle CUs) while every split keeps at least min_k of k
    auto splits_for = [&](long tiles, int min_k) {
        int v = (int)(kNumCU / tiles);
        const int maxs = d->K / min_k;
        if (v > maxs) v = maxs;
        if (v > 8) v = 8;
        return v < 1 ? 1 : v;
    };
    if (d->op != TP_GEMM_TN && d->M <= 512) {
        // A slice's linears, forward (NT) and data gradient (NN): up to 512 rows against a weight.  The rules are the
        // common ground of sweeps over every tile configuration and split on layer geometries that have no entry in
        // the measured table (hidden 3072 to 10240, 64 to 512 rows): about one workgroup per CU is the target -- fewer
        // leave CUs without a share of the weight stream, every extra split adds a round of fp32 partial sums and
        // does not pay below 1536-2048 of k per split -- and the tile grows with the slice so that the activation,
        // which every column tile re-reads, stays the smaller part of what a CU has to fill.
        const long t3 = (long)((d->M + 127) / 128) * t256n;          // 128 x 256 tiles
        if (runs_skinny(d)) {
            cfg = 8;                // (its k splits are what counts)
            ns = skinny_unsplit(d) ? 1 : splits_for(t64, 2048);
        } else if (small_weight(d)) {
            plan_slice(d, cfg, ns);
        } else if (d->M <= 64) {
            // one row of tiles: 64 x 64 until they come to more than two per CU, then 64 x 256
            if (t64 >= 2 * kNumCU) { cfg = 11; ns = splits_for(t256n, 2048); }
            else { cfg = 8; ns = splits_for(t64, 2048); }
        } else if (d->M <= 128) {
            const int ns13 = splits_for(t128, 1536);
            if (t128 > kNumCU) { cfg = 3; ns = splits_for(t3, 2048); }                      // many column tiles: 128 x 256
            else if (t128 * ns13 < 192 && t64 >= 192 && t64 <= 2 * kNumCU) { cfg = 8; }     // too few 128 x 128 tiles for the chip
            else { cfg = 13; ns = ns13; }
        } else if (d->M > 448 && d->K % 64 == 0 && t256 >= 160) {
            cfg = 19;               // two full rows of 256 x 256 tiles for most of the CUs
        } else if (d->M > 256 && d->M <= 384 && d->K % 64 == 0 && t3 > kNumCU) {
            cfg = 33;               // two row tiles of 192 x 256 (the weight-streaming kernel) where 128 x 256 tiles are too many
            ns = splits_for(2 * t256n, 2048);
        } else {
            // 128 x 256 tiles when a split still keeps 4096 of k, to amortise the larger tile's prologue; else 128 x 128
            const int ns3 = splits_for(t3, 2048);
            if (d->K / ns3 >= 4096 || t128 > kNumCU) { cfg = 3; ns = ns3; }
            else { cfg = 13; ns = splits_for(t128, 2048); }
        }
    } else {
        plan_large(d, cfg, ns);
    }
    // The pipelined 16 x 16 x 32 tiles in place of the 32 x 32 ones the rules above name, where a sweep over other
    // geometries (hidden 3072, 4096, 8192; 128 to 512 rows; 144 slice products) has them ahead: 128 x 128 for
    // 128 x 128 (0.94 to 0.99 of the time), 192 x 128 for 128 x 256 at 129 to 192 rows and at 257 to 384 (0.83 to 0.91),
    // 256 x 128 above 384 rows (0.92), and the 160- and 224-row tiles where they end with the slice (0.95 to 1.0 of
    // the padded tile's time on the 13B shapes); a k-split stays within one round of workgroups of the new tile.
    if (d->op != TP_GEMM_TN && d->M <= 512 && (cfg == 13 || cfg == 3)) {
        int bm = 128, bn = 128, to = 16;
        if (cfg == 3) {
            // row tiles that end with the slice where whole 16-row blocks allow it: 160 (one or two tiles), 192 (one
            // or two), 224 (one or two), else 256
            if ((d->M > 128 && d->M <= 160) || (d->M > 256 && d->M <= 320)) { to = 42; bm = 160; }
            else if ((d->M > 160 && d->M <= 192) || (d->M > 320 && d->M <= 384)) { to = 14; bm = 192; }
            else if ((d->M > 192 && d->M <= 224) || (d->M > 384 && d->M <= 448)) { to = 41; bm = 224; }
            else if (d->M > 448) { to = 15; bm = 256; }
            else to = 3;
        }
        if (to != 3) {
            cfg = to;
            const long tiles = (long)((d->M + bm - 1) / bm) * ((d->N + bn - 1) / bn);
            const int cap = (int)(kNumCU / tiles);
            if (ns > 1 && ns > cap) ns = cap < 1 ? 1 : cap;
        }
    }
    if (const TunedPlan* t = find_tuned(d)) {
        cfg = t->cfg;
        ns = t->nsplit;
        // An entry that fewer rows take with fewer row tiles keeps its number of workgroups (NN 80 to 128 x 5120 x 5120 with the 160-row
        // entry's three splits 25.1 to 27.2 us, with six 20.0 to 22.6), unless other streams' launches are to have the rest of the chip.
        TileCfg tt;
        if (ns > 1 && !(d->reserved & kBeside) && tile_cfg(cfg, tt)) {
            const int more = ns * ((t->M + tt.bm - 1) / tt.bm) / ((d->M + tt.bm - 1) / tt.bm);
            if (d->K / more >= 768) ns = more;
        }
    }
    if (ns < 1) ns = 1;
    if (ns > 16) ns = 16;
    TileCfg tc;
    if (forced_cfg >= 0 && tile_cfg(forced_cfg, tc)) cfg = forced_cfg;
    if (forced_split) ns = forced_split;
    // The tiles that exist for some operand orders only (a token-major tile 160 or 192 wide has no XOR swizzle: the chunk
    // index would leave the row; the streaming and the wide kernel have no TN form).  A ragged k: the weight-streaming
    // and the 32 x 32-block tall tiles load whole k-tiles only; the pipelined tiles copy the ragged part first, but a tile
    // FORCED through the descriptor keeps to whole k-tiles (it falls back to the 128 x 128 tile).
    const bool ragged = d->K % 64 != 0, forced = forced_cfg >= 0;
    if ((cfg == 6 || cfg == 7 || cfg == 43) && ((ragged && forced) || d->op != TP_GEMM_NT)) cfg = 5;
    if ((cfg == 41 || cfg == 42 || cfg == 14) && ((ragged && forced) || d->op == TP_GEMM_TN)) cfg = 5;
    if ((cfg == 15 || cfg == 16 || cfg == 2) && ragged && forced) cfg = 5;
    if (cfg == kWideCfg && ((ragged && forced) || d->op == TP_GEMM_TN || d->K < 64)) cfg = 5;
    if (cfg >= 17 && cfg <= 20 && (ragged || (cfg == 17 && d->op != TP_GEMM_NT))) cfg = 5;
    if (cfg >= kFirstStreamCfg && cfg <= kLastStreamCfg &&
        (d->op == TP_GEMM_TN || ragged || ((cfg == 24 || cfg == 25) && d->op != TP_GEMM_NT))) cfg = 5;
    if (d->N % 8) ns = 1;               // (partial sums are rows of N)
    p.cfg = cfg;
    tile_cfg(cfg, tc);
    p.gx = (d->N + tc.bn - 1) / tc.bn;
    p.gy = (d->M + tc.bm - 1) / tc.bm;
    finish_plan(d, p, tc.bk, ns);
    if (cfg == 12 && deep_serves(d)) {
        deep_time(d, p.nsplit, &p.deep);
        if ((d->reserved >> 16) & 0xff) p.deep = (d->reserved >> 16) & 0xff;    // forced (tuning, tests)
        p.gx = (d->N + p.deep - 1) / p.deep;
    }
    if (cfg == kWideCfg) {
        const int columns = (d->reserved >> 16) & 0xff;     // forced (tuning, tests): 192, else 256
        p.wide = columns ? (columns == 192 ? 192 : 256) : wide_columns(d, p.nsplit);
        p.gx = (d->N + p.wide - 1) / p.wide;
    }
    return p;
}

static size_t plan_bytes(const tp_gemm_desc* d, const GemmPlan& p) {
    return p.nsplit > 1 ? (size_t)p.nsplit * d->M * d->N * sizeof(float) : 0;
}

// The plan of tp_gemm_static_ws: splits of the library's own that need more than the built-in workspace are cut to what fits,
// on the same tile, so that what fits it does not hang on how the plan weighs splits.
static GemmPlan plan_static_ws(const tp_gemm_desc* d) {
    GemmPlan p = plan_gemm(d);
    if (plan_bytes(d, p) > (size_t)TP_GEMM_STATIC_WS_BYTES && !((d->reserved >> 8) & 0xff))
        finish_plan(d, p, p.bk, (int)((size_t)TP_GEMM_STATIC_WS_BYTES / ((size_t)d->M * d->N * sizeof(float))));
    return p;
}

// the tile configurations of gemm_pipe.hip
static inline bool is_pipe_cfg(int cfg) { return cfg == 6 || cfg == 7 || (cfg >= 14 && cfg <= 16) || (cfg >= 41 && cfg <= 43); }

// false: the plan names a (tile configuration, op, dtype) that no kernel is built for -- nothing was launched
template <typename T>
static bool launch_gemm(const tp_gemm_desc* d, const GemmPlan& p, const GemmArgs& a, hipStream_t s, const SkinnyLn* ln) {
    if (runs_skinny(d)) {
        launch_gemm_skinny(d->dtype, a, d->reserved & kNoBackward, ln, s);
    } else if (runs_f32_small(d)) {
        launch_gemm_f32_small(d->op, a, s);
    } else if (p.deep) {
        if (!launch_gemm_deep(p.deep, d->op, d->dtype, dim3(p.gx, p.gy, p.nsplit), a, s)) return false;
    } else if (p.cfg >= kFirstStreamCfg && p.cfg <= kLastStreamCfg) {
        if (!launch_gemm_stream(p.cfg, d->op, d->dtype, dim3(p.gx, p.gy, p.nsplit), a, s)) return false;
    } else if (is_pipe_cfg(p.cfg) && d->dtype != TP_F32) {
        if (!launch_gemm_pipe(p.cfg, d->op, d->dtype, dim3(p.gx, p.gy, p.nsplit), a, s)) return false;
    } else if (p.cfg == kWideCfg && d->dtype != TP_F32) {
        if (!launch_gemm_wide(p.wide, d->op, d->dtype, dim3(p.gx, p.gy, p.nsplit), a, s)) return false;
    } else if (p.cfg == 2 || (p.cfg >= 17 && p.cfg <= 20)) {
        if (!launch_gemm_tall(p.cfg, d->op, d->dtype, dim3(p.gx, p.gy, p.nsplit), a, s)) return false;
    } else if (!launch_gemm_dma(p.cfg, d->op, d->dtype, dim3(p.gx, p.gy, p.nsplit), a, s)) {
        return false;
    }
    if (p.nsplit > 1 && !d->defer_reduce) {
        dim3 grid((d->N + 255) / 256, (d->M + 7) / 8);
        gemm_splitk_reduce_kernel<T><<<grid, 256, 0, s>>>(a);
    }
    return true;
}

static int validate_gemm(const tp_gemm_desc* d) {
    if (!d) { set_error("tp_gemm: null descriptor"); return TP_ERR_ARG; }
    if (d->dtype < TP_F32 || d->dtype > TP_BF16) { set_error("tp_gemm: bad dtype %d", d->dtype); return TP_ERR_ARG; }
    if (d->op < TP_GEMM_NT || d->op > TP_GEMM_TN) { set_error("tp_gemm: bad op %d", d->op); return TP_ERR_ARG; }
    if (d->epilogue < TP_EPI_STORE || d->epilogue > TP_EPI_GELU_GRAD) { set_error("tp_gemm: bad epilogue %d", d->epilogue); return TP_ERR_ARG; }
    if (d->M <= 0 || d->N <= 0 || d->K <= 0) { set_error("tp_gemm: non-positive shape M=%d N=%d K=%d", d->M, d->N, d->K); return TP_ERR_ARG; }
    if (!d->A || !d->B) { set_error("tp_gemm: null operand"); return TP_ERR_ARG; }
    const int ch = d->dtype == TP_F32 ? 4 : 8;
    // contiguous extents of the operands as stored
    int a_cols = d->op == TP_GEMM_TN ? d->M : d->K;
    int b_cols = d->op == TP_GEMM_NT ? d->K : d->N;
    // With `ragged`, A's contiguous extent may end inside a chunk that its row holds in full where what it multiplies is
    // bounded by rows: k of NN (the weight's rows past k count as zeros; A's columns there have to be finite), M of TN
    const bool a_ragged = d->ragged && d->op != TP_GEMM_NT && d->lda >= (a_cols + ch - 1) / ch * ch;
    if ((a_cols % ch && !a_ragged) || b_cols % ch || d->lda % ch || d->ldb % ch) {
        set_error("tp_gemm: contiguous extents / leading dimensions must be multiples of %d elements "
                  "(A cols %d lda %ld, B cols %d ldb %ld)", ch, a_cols, (long)d->lda, b_cols, (long)d->ldb);
        return TP_ERR_UNSUPPORTED;
    }
    if (d->lda < a_cols || d->ldb < b_cols) { set_error("tp_gemm: leading dimension smaller than row"); return TP_ERR_ARG; }
    if (((uintptr_t)d->A | (uintptr_t)d->B) & 15) { set_error("tp_gemm: operands must be 16-byte aligned"); return TP_ERR_ARG; }
    // with `ragged`, so may N of a plain NT product in C's rows (the columns past N get the last one's values)
    if (d->N % 8 && (!d->ragged || d->op != TP_GEMM_NT || d->epilogue != TP_EPI_STORE || d->defer_reduce || d->colsum_acc || d->ldc < (d->N + 7) / 8 * 8)) {
        set_error("tp_gemm: N=%d must be a multiple of 8", d->N);
        return TP_ERR_UNSUPPORTED;
    }
    if (d->defer_reduce && ((d->epilogue != TP_EPI_STORE && d->epilogue != TP_EPI_BIAS_RESIDUAL) || d->colsum_acc)) {
        set_error("tp_gemm: defer_reduce needs the STORE or BIAS_RESIDUAL epilogue and no colsum_acc");
        return TP_ERR_ARG;
    }
    if (d->epilogue != TP_EPI_QKV_SCATTER) {
        if (!d->C || d->ldc < d->N || d->ldc % ch || ((uintptr_t)d->C & 15)) { set_error("tp_gemm: bad C / ldc / alignment"); return TP_ERR_ARG; }
    }
    if (((uintptr_t)d->bias | (uintptr_t)d->residual | (uintptr_t)d->aux | (uintptr_t)d->aux_out |
         (uintptr_t)d->q | (uintptr_t)d->k_cache | (uintptr_t)d->v_cache) & 15) {
        set_error("tp_gemm: epilogue tensors must be 16-byte aligned"); return TP_ERR_ARG;
    }
    if ((d->residual && d->ldr % ch) || (d->aux && d->ldaux % ch) || (d->aux_out && d->ldauxo % ch)) {
        set_error("tp_gemm: epilogue leading dimensions must be multiples of %d", ch); return TP_ERR_ARG;
    }
    switch (d->epilogue) {
    case TP_EPI_BIAS: case TP_EPI_BIAS_RELU: case TP_EPI_BIAS_GELU:
        if (!d->bias) { set_error("tp_gemm: epilogue needs bias"); return TP_ERR_ARG; }
        break;
    case TP_EPI_BIAS_RESIDUAL:
        if (!d->bias || !d->residual || d->ldr < d->N) { set_error("tp_gemm: epilogue needs bias and residual"); return TP_ERR_ARG; }
        break;
    case TP_EPI_RELU_GRAD: case TP_EPI_GELU_GRAD:
        if (!d->aux || d->ldaux < d->N) { set_error("tp_gemm: epilogue needs aux"); return TP_ERR_ARG; }
        break;
    case TP_EPI_QKV_SCATTER:
        if (!d->bias || !d->q || !d->k_cache || !d->v_cache) { set_error("tp_gemm: qkv scatter needs bias, q, k_cache, v_cache"); return TP_ERR_ARG; }
        if (d->batch <= 0 || d->heads <= 0 || d->head_dim <= 0 || d->head_dim % 8 || d->cache_len < 0) { set_error("tp_gemm: bad qkv geometry"); return TP_ERR_ARG; }
        if (d->N != 3 * d->heads * d->head_dim) { set_error("tp_gemm: qkv scatter needs N == 3*heads*head_dim (N=%d)", d->N); return TP_ERR_ARG; }
        if (d->M % d->batch) { set_error("tp_gemm: qkv scatter needs M %% batch == 0"); return TP_ERR_ARG; }
        if ((long)d->cache_len + d->M / d->batch > d->cache_rows) {
            set_error("tp_gemm: slice [%d, %d) does not fit a cache of %ld rows", d->cache_len,
                      d->cache_len + d->M / d->batch, (long)d->cache_rows);
            return TP_ERR_ARG;
        }
        break;
    default: break;
    }
    return TP_OK;
}

}  // namespace tp

extern "C" int tp_gemm_splits(const tp_gemm_desc* d) {
    if (tp::validate_gemm(d) != TP_OK) return 0;
    return tp::plan_gemm(d).nsplit;
}

extern "C" int tp_gemm_plan(const tp_gemm_desc* d, int* tile_cfg, int* nsplit) {
    int rc = tp::validate_gemm(d);
    if (rc != TP_OK) return rc;
    tp::GemmPlan p = tp::plan_gemm(d);
    if (tile_cfg) *tile_cfg = p.cfg;
    if (nsplit) *nsplit = p.nsplit;
    return TP_OK;
}

extern "C" int tp_gemm_tile(const tp_gemm_desc* d, int static_ws, int* rows, int* columns, int* nsplit) {
    int rc = tp::validate_gemm(d);
    if (rc != TP_OK) return rc;
    const tp::GemmPlan p = static_ws ? tp::plan_static_ws(d) : tp::plan_gemm(d);
    tp::TileCfg tc = {};
    if (tp::runs_f32_small(d)) tc = {32, 32, 0, 0};
    else if (!tp::runs_skinny(d)) tp::tile_cfg(p.cfg, tc);
    if (rows) *rows = tc.bm;
    if (columns) *columns = p.deep ? p.deep : p.wide ? p.wide : tc.bn;
    if (nsplit) *nsplit = p.nsplit;
    return TP_OK;
}

extern "C" size_t tp_gemm_workspace_bytes(const tp_gemm_desc* d) {
    if (tp::validate_gemm(d) != TP_OK) return 0;
    return tp::plan_bytes(d, tp::plan_gemm(d));
}

namespace tp {
static GemmArgs fill_args(const tp_gemm_desc* d, const GemmPlan& p, void* workspace) {
    GemmArgs a;
    a.A = d->A; a.B = d->B; a.C = d->C;
    a.lda = d->lda; a.ldb = d->ldb; a.ldc = d->ldc;
    a.M = d->M; a.N = d->N; a.K = d->K;
    a.epi = d->epilogue;
    a.bias = d->bias; a.resid = d->residual; a.ldr = d->ldr;
    a.aux = d->aux; a.ldaux = d->ldaux; a.aux_out = d->aux_out; a.ldauxo = d->ldauxo;
    a.colsum = d->colsum_acc;
    a.q = d->q; a.kc = d->k_cache; a.vc = d->v_cache;
    a.batch = d->batch; a.heads = d->heads; a.hd = d->head_dim;
    a.T = d->epilogue == TP_EPI_QKV_SCATTER ? d->M / d->batch : 0;
    a.q_rows = d->q_bh_rows > 0 ? d->q_bh_rows : a.T;
    a.P = d->cache_len; a.cache_rows = d->cache_rows; a.qscale = d->q_scale;
    a.kper = p.kper; a.nsplit = p.nsplit; a.partial = reinterpret_cast<float*>(workspace);
    return a;
}

static int run_gemm(const tp_gemm_desc* d, const GemmPlan& p, void* workspace, void* stream, const SkinnyLn* ln = nullptr, const void* ln_x = nullptr) {
    GemmArgs a = fill_args(d, p, workspace);
    if (ln) { a.A = ln_x; a.lda = d->K; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    bool launched;
    switch (d->dtype) {
    case TP_F32: launched = launch_gemm<float>(d, p, a, s, ln); break;
    case TP_F16: launched = launch_gemm<f16>(d, p, a, s, ln); break;
    default: launched = launch_gemm<bf16>(d, p, a, s, ln); break;
    }
    if (!launched) {
        set_error("tp_gemm: no kernel for tile configuration %d with op %d, dtype %d", p.cfg, d->op, d->dtype);
        return TP_ERR_UNSUPPORTED;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { set_error("tp_gemm: launch failed: %s", hipGetErrorString(e)); return TP_ERR_LAUNCH; }
    return TP_OK;
}

bool gemm_takes_layernorm(const tp_gemm_desc& d, const LayerNormOf& l) {
    return (d.reserved & kNoBackward) && runs_skinny(&d) && skinny_takes_ln(d.M, d.K) && d.lda == d.K && l.x && l.gamma && l.beta &&
           !(((uintptr_t)l.x | (uintptr_t)l.gamma | (uintptr_t)l.beta) & 15) && plan_gemm(&d).nsplit <= 1;
}
int gemm_of_layernorm(const tp_gemm_desc& d, const LayerNormOf& l, float eps, void* stream) {
    const int rc = validate_gemm(&d);
    if (rc != TP_OK) return rc;
    const SkinnyLn ln = {l.gamma, l.beta, eps};
    return run_gemm(&d, plan_gemm(&d), nullptr, stream, &ln, l.x);
}

// One launch for the whole group when every member is a 16-bit TN product (parameter gradients) of the same dtype and
// k (whole 64-wide k-tiles), on the tile with the smallest estimate for all members' tiles together (or the largest
// member's measured or forced one; the 256 x 256 tile unless another is a tenth ahead): the configuration of that
// launch, or 0 when the group runs member by member.
static int group_cfg(const tp_gemm_desc* descs, int n) {
    if (n < 2 || n > kGroupMax) return 0;
    int big = 0;
    for (int i = 0; i < n; ++i) {
        const tp_gemm_desc& d = descs[i];
        if (d.op != TP_GEMM_TN || d.dtype != descs[0].dtype || d.dtype == TP_F32 || d.K != descs[0].K || d.K % 64 != 0 ||
            d.reserved != descs[0].reserved ||      // a forced plan (tuning, tests) must be the same for all members
            d.defer_reduce != 0 || d.epilogue == TP_EPI_QKV_SCATTER)
            return 0;
        if ((double)d.M * d.N > (double)descs[big].M * descs[big].N) big = i;
    }
    if ((descs[0].reserved & kForced) || find_tuned(&descs[big])) {
        const GemmPlan pb = plan_gemm(&descs[big]);
        return ((pb.cfg == 2 || pb.cfg == 15 || pb.cfg == 16 || pb.cfg == 19 || pb.cfg == 20) && pb.nsplit == 1) ? pb.cfg : 0;
    }
    const bool spill = 2.0 * ((double)descs[big].M + descs[big].N) * descs[0].K > 225e6;
    int cfg = 0;
    float best = 0.f;
    for (const TileCost& c : kTileCostTN) {
        long tiles = 0;
        for (int i = 0; i < n; ++i) tiles += (long)((descs[i].M + c.bm - 1) / c.bm) * ((descs[i].N + c.bn - 1) / c.bn);
        const float t = tile_time(c, tiles, (float)descs[0].K, spill) * (c.cfg == 2 ? 0.9f : 1.f);
        if (!cfg || t < best) { best = t; cfg = c.cfg; }
    }
    return cfg;
}

// Groups of a short k on tiles of 128 x 128, two workgroups per CU (gemm_short.hip; the same k order, and bits, as the 256 x 256
// tile, whose configuration they report): plain or added results, where the estimate has them a twentieth ahead.  Both were
// fitted to a layer's four products (hidden 768 to 5120, k 64 to 1024): a launch, the tiles' part of C's traffic, the rounds'
// part of k, the last one's partly by how full it is.  Calls taken gain 1.04 to 1.32: 1600 wide, added over 256 rows 51.3 -> 40.9 us,
// over 768 86 -> 75; 5120 wide over 256 381 -> 346; those left 0.83 to 1.07, at k = 1024 the two were level at best (768: 1.27).
struct GroupCost { float fixed, tile, per_k, partial; };
static float group_time(const GroupCost& c, long tiles, int round, int K) {
    const long full = tiles / round, rest = tiles % round;
    const float rounds = full + (rest ? c.partial + (1.f - c.partial) * rest / round : 0.f);
    return c.fixed + c.tile * tiles / round + c.per_k * K * rounds;
}
bool launch_gemm_short_group(bool add, int dtype, int tiles, const GemmGroupArgs& ga, hipStream_t s);
static bool runs_short(const tp_gemm_desc* descs, int n) {
    static const GroupCost kWide[2] = {{4.6f, 8.1f, 0.0246f, 0.75f}, {3.7f, 15.1f, 0.0227f, 0.92f}};      // plain, added
    static const GroupCost kShort[2] = {{6.2f, 2.9f, 0.0167f, 0.04f}, {6.5f, 5.5f, 0.0164f, 0.06f}};
    long t256 = 0, t128 = 0;
    for (int i = 0; i < n; ++i) {
        const tp_gemm_desc& d = descs[i];
        if (d.K > 768 || d.N % 8 || d.colsum_acc || (d.reserved & kForced) || d.epilogue != descs[0].epilogue ||
            (d.epilogue != TP_EPI_STORE && d.epilogue != TP_EPI_ACCUMULATE)) return false;
        t256 += (long)((d.M + 255) / 256) * ((d.N + 255) / 256);
        t128 += (long)((d.M + 127) / 128) * ((d.N + 127) / 128);
    }
    const int add = descs[0].epilogue == TP_EPI_ACCUMULATE, K = descs[0].K;
    return group_time(kShort[add], t128, 2 * kNumCU, K) < 0.95f * group_time(kWide[add], t256, kNumCU, K);
}

// vec: blocks behind the tiles (takes_vec_grads)
static bool launch_group(const tp_gemm_desc* descs, int n, int cfg, const VecGradArgs* vec, hipStream_t s) {
    GemmGroupArgs ga;
    int tiles = 0;
    for (int i = 0; i < n; ++i) {
        GemmPlan p = {};            // every member on the group's tiles, its whole k in one piece
        p.cfg = cfg;
        TileCfg tc;
        tile_cfg(cfg, tc);
        p.gx = (descs[i].N + tc.bn - 1) / tc.bn;
        p.gy = (descs[i].M + tc.bm - 1) / tc.bm;
        p.kper = descs[i].K; p.nsplit = 1;
        ga.g[i] = fill_args(&descs[i], p, nullptr);
        ga.first_tile[i] = tiles;
        ga.tiles_x[i] = p.gx;
        ga.tiles_y[i] = p.gy;
        tiles += p.gx * p.gy;
    }
    for (int i = n; i < kGroupMax; ++i) { ga.g[i] = ga.g[0]; ga.first_tile[i] = tiles; ga.tiles_x[i] = 1; ga.tiles_y[i] = 1; }
    ga.n = n;
    if (cfg == 2 && runs_short(descs, n)) {
        tiles = 0;
        for (int i = 0; i < n; ++i) {
            ga.first_tile[i] = tiles;
            ga.tiles_x[i] = (descs[i].N + 127) / 128;
            ga.tiles_y[i] = (descs[i].M + 127) / 128;
            tiles += ga.tiles_x[i] * ga.tiles_y[i];
        }
        return launch_gemm_short_group(descs[0].epilogue == TP_EPI_ACCUMULATE, descs[0].dtype, tiles, ga, s);
    }
    if (cfg == 15 || cfg == 16) return launch_gemm_pipe_group(cfg, descs[0].dtype, tiles, ga, s);
    return launch_gemm_tall_group(cfg, descs[0].dtype, tiles, ga, vec, s);
}
// Whether a layer's vector-parameter gradients run as blocks behind the group's tiles, where those are of 256 x 256: on the CUs that the
// tiles' last round leaves, then, when it ends, on all of them.  A layer's four weight gradients alone / its vector gradients alone /
// the two launches / this one, us: 1024 wide, 4096 rows (64 CUs left) 100 / 24 / 125 / 102; 2048 wide, 2048 rows (three full rounds,
// none left) 177 / 25 / 197 / 191; 2560 wide, 2048 rows 294 / 26 / 314 / 295; 6144 wide, 4096 rows 2974 / 116 / 3077 / 3073.
static bool takes_vec_grads(const tp_gemm_desc* descs, int n, int cfg) {
    return (cfg == 2 && !runs_short(descs, n)) || cfg == 19 || cfg == 20;
}
}  // namespace tp

// ---------------------------------------------------------------------------------------------
// Workspace for callers that cannot allocate (tp_gemm_static_ws): the k-split partial sums go to a
// file-scope device array instead of a caller's buffer.  In host code the array's name is only a
// stand-in; its device address is asked for once per device and kept.
// ---------------------------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[TP_GEMM_STATIC_WS_BYTES];

namespace tp {
static constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[kMaxDevices] = {};

// device address of `scratch` on the CURRENT device (nullptr + error text on failure)
static void* scratch_on_current_device() {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        set_error("tp_gemm_static_ws: hipGetDevice failed or device index %d out of range: %s", dev, hipGetErrorString(e));
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error("tp_gemm_static_ws: hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(e));
            return nullptr;
        }
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}
}  // namespace tp

// Also looks up the array's address on the current device (a module and symbol lookup that must not happen while a
// stream capture is open): callers that capture tp_gemm_static_ws call this once per device beforehand.
extern "C" size_t tp_gemm_static_ws_capacity(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) == hipSuccess && n > 0) (void)tp::scratch_on_current_device();
    return (size_t)TP_GEMM_STATIC_WS_BYTES;
}

extern "C" int tp_gemm_static_ws(const tp_gemm_desc* d, void* stream) {
    int rc = tp::validate_gemm(d);
    if (rc != TP_OK) return rc;
    if (d->defer_reduce) {
        tp::set_error("tp_gemm_static_ws: defer_reduce hands the workspace to a later call; use tp_gemm");
        return TP_ERR_ARG;
    }
    const tp::GemmPlan p = tp::plan_static_ws(d);
    const size_t need = tp::plan_bytes(d, p);
    if (need > (size_t)TP_GEMM_STATIC_WS_BYTES) {
        tp::set_error("tp_gemm_static_ws: this product needs %zu bytes of k-split workspace, the built-in one holds %zu "
                      "(M=%d N=%d K=%d, %d splits); use tp_gemm with a caller workspace",
                      need, (size_t)TP_GEMM_STATIC_WS_BYTES, d->M, d->N, d->K, p.nsplit);
        return TP_ERR_WORKSPACE;
    }
    void* ws = nullptr;
    if (need > 0) {
        ws = tp::scratch_on_current_device();
        if (!ws) return TP_ERR_LAUNCH;
    }
    return tp::run_gemm(d, p, ws, stream);
}

extern "C" int tp_gemm(const tp_gemm_desc* d, void* workspace, size_t workspace_bytes, void* stream) {
    int rc = tp::validate_gemm(d);
    if (rc != TP_OK) return rc;
    const tp::GemmPlan p = tp::plan_gemm(d);
    const size_t need = tp::plan_bytes(d, p);
    if (need > 0 && (!workspace || workspace_bytes < need)) {
        tp::set_error("tp_gemm: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
        return TP_ERR_WORKSPACE;
    }
    return tp::run_gemm(d, p, workspace, stream);
}

extern "C" int tp_gemm_group_cfg(const tp_gemm_desc* descs, int n) {
    if (!descs || n < 1) return 0;
    for (int i = 0; i < n; ++i)
        if (tp::validate_gemm(&descs[i]) != TP_OK) return 0;
    return tp::group_cfg(descs, n);
}

extern "C" int tp_gemm_group_tile(const tp_gemm_desc* descs, int n, int* rows, int* columns) {
    const int cfg = tp_gemm_group_cfg(descs, n);
    tp::TileCfg tc = {};
    if (cfg) tp::tile_cfg(cfg, tc);
    if (cfg == 2 && tp::runs_short(descs, n)) tc.bm = tc.bn = 128;
    if (rows) *rows = tc.bm;
    if (columns) *columns = tc.bn;
    return TP_OK;
}

extern "C" int tp_gemm_grouped(const tp_gemm_desc* descs, int n, void* workspace, size_t workspace_bytes, void* stream) {
    return tp_gemm_grouped_vec(descs, n, nullptr, 0, workspace, workspace_bytes, stream);
}

extern "C" int tp_gemm_grouped_vec(const tp_gemm_desc* descs, int n, const tp_vecgrad_desc* vecs, int n_vecs, void* workspace,
                                   size_t workspace_bytes, void* stream) {
    if (!descs || n < 1) { tp::set_error("tp_gemm_grouped: bad argument"); return TP_ERR_ARG; }
    for (int i = 0; i < n; ++i) {
        int rc = tp::validate_gemm(&descs[i]);
        if (rc != TP_OK) return rc;
    }
    tp::VecGradArgs vec;
    int blocks = 0;
    if (n_vecs) {
        const int rc = tp::fill_vec_grads(vecs, n_vecs, descs[0].dtype, vec, blocks);
        if (rc != TP_OK) return rc;
    }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int cfg = tp::group_cfg(descs, n);
    const bool together = n_vecs && tp::takes_vec_grads(descs, n, cfg);
    if (n_vecs && !together) {
        const int rc = tp_vec_param_grads(vecs, n_vecs, descs[0].dtype, stream);
        if (rc != TP_OK) return rc;
    }
    if (cfg) {
        if (!tp::launch_group(descs, n, cfg, together ? &vec : nullptr, s)) {
            tp::set_error("tp_gemm_grouped: no kernel for tile configuration %d, dtype %d", cfg, descs[0].dtype);
            return TP_ERR_UNSUPPORTED;
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) { tp::set_error("tp_gemm_grouped: launch failed: %s", hipGetErrorString(e)); return TP_ERR_LAUNCH; }
        return TP_OK;
    }
    // any other group: its members one after the other (they share the workspace: same stream, in order)
    for (int i = 0; i < n; ++i) {
        int rc = tp_gemm(&descs[i], workspace, workspace_bytes, stream);
        if (rc != TP_OK) return rc;
    }
    return TP_OK;
}
