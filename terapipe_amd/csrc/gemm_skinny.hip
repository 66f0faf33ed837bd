// Y = X W^T for a handful of rows (decoding: one token of each sequence), 16-bit.
#include "gemm_epilogue.h"

namespace tp {

// ---------------------------------------------------------------------------------------------
// At most 16 * MB rows.  The product reads the whole weight and computes next to nothing: for weights of a few MB it is
// bound by latency and by the bytes kept in flight, which a tile kernel that stages 64 rows through LDS with a barrier
// per k-tile keeps low.  Here a workgroup owns 16 * NT weight rows and its eight waves share their k: a wave reads 16
// rows x 128 k (NT x 16 rows; of NT = 4 half the k) per turn, straight into the
// registers the MFMA takes (lane l: row l & 15, k 8 * (l >> 4) .. + 7 of each 32), the activation rows the same way
// (they stay in the caches; NT weight tiles share one read of them), the next turn's loads under way meanwhile.  No LDS and no
// barrier until the eight partial tiles are added at the end.
// Measured (4 rows, weights from memory, launches of one graph back to back, us): 8192 x 2048 9.6 (3.5 TB/s; without the second turn's
// loads under way 10.3), 6144 x 2048 8.7 (9.0), 4096 x 4096 12.3 (13.0; without k splits 10.2), 20480 x 5120 41.0 (5.1 TB/s); tiles of 8
// rows: 2048 x 2048 4.9 (of 16: 5.7), 2048 x 8192 10.3 (of 16 with four k splits and the launch that adds them 12.6), 768 x 3072 5.2 (6.6).  In a
// decoding step's chain with the LayerNorm: 8192 x 2048 12.2 (10.5 + 3.6), 6144 x 2048 11.0 (9.4 + 3.6).
// ---------------------------------------------------------------------------------------------
// HALF (up to 8 rows, where tiles of 16 weight rows would leave half of the CUs without one): a tile is 8 weight rows, the 16 rows
// of the MFMA are those at two k ranges, and so are its columns; the two diagonal quarters are the tile's sums.  With it a weight of
// 2048 rows needs no k split.
// LN (up to 8 rows): the activation rows are the LayerNorm of a.A, taken by each workgroup for itself while its first
// weight rows come (two-pass fp32 statistics, rounded to T in LDS); neither they nor their statistics are kept.  A launch less in a
// chain where a LayerNorm of four rows takes 3.7 us.
template <typename T, int MB, int NT, bool HALF, bool LN>
__global__ __launch_bounds__(512, MB == 1 && !HALF ? 4 : 2) void gemm_skinny_kernel(GemmArgs a, SkinnyLn ln) {
    constexpr int WAVES = 8, U = HALF ? 8 : NT == 4 ? 2 : 4, UK = HALF ? 64 : 32, STEP = UK * U, TN = HALF ? 8 : 16, PITCH = NT * TN + 4;
    constexpr int LNC = 5;          // 16-byte chunks of a row per lane
    __shared__ float part[WAVES][MB * 16][PITCH];
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn[];
    T* xs = reinterpret_cast<T*>(dyn);          // LN: [M][K + 8]
    // Some of the epilogue's arguments, one of each line of the scalar cache, come with the first ones: asked for behind the last barrier,
    // where the compiler would have them, they cost a small product 0.2 us (4 rows, us: 256 x 256 3.3 -> 3.1, 768 x 768 4.0 -> 3.8; all of
    // the arguments asked for here 0 to 0.1 more); with the wave's number in a scalar register 3.0 and 3.8.
    asm volatile("" :: "s"(a.epi), "s"(a.bias), "s"(a.C), "s"(a.q), "s"(a.partial), "s"(a.nsplit));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);     // (its turns branch on scalars)
    const int n0 = blockIdx.x * TN * NT;
    const int kbeg = blockIdx.z * a.kper, kend = min(a.K, kbeg + a.kper);
    const int r = lane & (HALF ? 7 : 15), kq = 8 * (lane >> 4) + (HALF ? 32 * ((lane >> 3) & 1) : 0);
    const T *w[NT], *x[MB];
#pragma unroll
    for (int n = 0; n < NT; ++n) w[n] = reinterpret_cast<const T*>(a.B) + (long)min(n0 + TN * n + r, a.N - 1) * a.ldb + kq;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const int row = min(16 * m + r, a.M - 1);
        x[m] = LN ? xs + row * (a.K + 8) + kq : reinterpret_cast<const T*>(a.A) + (long)row * a.lda + kq;
    }
    float4v acc[NT][MB];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MB; ++m) acc[n][m] = float4v{0.f, 0.f, 0.f, 0.f};
    struct Turn { uint4 w[NT][U], x[MB][U]; };
    auto load_if = [](bool in, const T* p) __attribute__((always_inline)) {
        uint4 v = make_uint4(0, 0, 0, 0);
        if (in) v = *reinterpret_cast<const uint4*>(p);
        return v;
    };
    auto load_x = [&](Turn& t, int k) __attribute__((always_inline)) {
        if (__builtin_expect(k + STEP <= kend, 1)) {         // wave-uniform
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int u = 0; u < U; ++u) t.x[m][u] = *reinterpret_cast<const uint4*>(x[m] + k + UK * u);
        } else {
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int u = 0; u < U; ++u) t.x[m][u] = load_if(k + UK * u + kq < kend, x[m] + k + UK * u);      // (k is a multiple of 8)
        }
    };
    auto load = [&](Turn& t, int k) __attribute__((always_inline)) {
        if (__builtin_expect(k + STEP <= kend, 1)) {
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int u = 0; u < U; ++u) t.w[n][u] = *reinterpret_cast<const uint4*>(w[n] + k + UK * u);
        } else {
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int u = 0; u < U; ++u) t.w[n][u] = load_if(k + UK * u + kq < kend, w[n] + k + UK * u);
        }
        if constexpr (!LN) load_x(t, k);
    };
    auto use = [&](Turn& t, int k) __attribute__((always_inline)) {
        if constexpr (LN) load_x(t, k);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int m = 0; m < MB; ++m) acc[n][m] = Mfma16x16x32<T>::run(t.w[n][u], t.x[m][u], acc[n][m]);
    };
    Turn t, t1;
    // a wave's turns: two beside each other with one tile of 16 rows, else a turn of all waves apart
    constexpr int FROM = NT == 1 && !HALF ? 2 * STEP : STEP, APART = NT == 1 && !HALF ? STEP : WAVES * STEP;
    int k = kbeg + wave * FROM;
    if constexpr (LN) {
        // 8, 4, 2 or 1 waves to a row; everything is asked for at once, the wave's first weights too
        const int share = a.M > 4 ? 1 : a.M > 2 ? 2 : a.M > 1 ? 4 : 8, row = min(wave / share, a.M - 1), part_of = wave % share;
        const int nch = a.K / 8, c0 = part_of * 64 + lane, step = 64 * share;
        float* red = &part[0][0][0];
        uint4 raw[LNC], gm[LNC], bt[LNC];
#pragma unroll
        for (int i = 0; i < LNC; ++i) {
            const int c = min(c0 + i * step, nch - 1) * 8;
            raw[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(a.A) + (long)row * a.lda + c);
            gm[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(ln.gamma) + c);
            bt[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(ln.beta) + c);
        }
        load(t, k);             // (behind the rows': loads come back in order)
        auto row_sum = [&](float v, float* buf) __attribute__((always_inline)) {
            v = wave_sum(v);
            if (lane == 0) buf[wave] = v;
            __syncthreads();
            v = 0.f;
            for (int i = 0; i < share; ++i) v += buf[wave - part_of + i];
            return v;
        };
        float sum = 0.f, sq = 0.f;
#pragma unroll
        for (int i = 0; i < LNC; ++i)
            if (c0 + i * step < nch) {
                const float8v v = unpack8<T>(Raw8<T>{{raw[i]}});
#pragma unroll
                for (int e = 0; e < 8; ++e) sum += v[e];
            }
        const float mu = row_sum(sum, red) / (float)a.K;
#pragma unroll
        for (int i = 0; i < LNC; ++i)
            if (c0 + i * step < nch) {
                const float8v v = unpack8<T>(Raw8<T>{{raw[i]}});
#pragma unroll
                for (int e = 0; e < 8; ++e) { const float d = v[e] - mu; sq += d * d; }
            }
        const float rs = 1.0f / sqrtf(row_sum(sq, red + WAVES) / (float)a.K + ln.eps);
        const bool mine = wave / share < a.M;
#pragma unroll
        for (int i = 0; i < LNC; ++i)
            if (mine && c0 + i * step < nch) {
                const int c = (c0 + i * step) * 8;
                const float8v v = unpack8<T>(Raw8<T>{{raw[i]}}), g = unpack8<T>(Raw8<T>{{gm[i]}}), b = unpack8<T>(Raw8<T>{{bt[i]}});
                float8v y;
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] = (v[e] - mu) * rs * g[e] + b[e];
                store8<T>(xs, row * (a.K + 8) + c, y);
            }
        __syncthreads();
    }
    // the next turn's loads are under way while this one's MFMAs wait for theirs
    if (!LN && k < kend) load(t, k);
    for (; k < kend; k += 2 * WAVES * STEP) {
        const int k1 = k + APART;
        if (k1 < kend) load(t1, k1);
        use(t, k);
        if (k1 < kend) {
            if (k + 2 * WAVES * STEP < kend) load(t, k + 2 * WAVES * STEP);
            use(t1, k1);
        }
    }
    // register j of the lane: weight row 4 * (lane >> 4) + j, activation row lane & 15
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            if constexpr (HALF) {
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[n][m][j] += __shfl_xor(acc[n][m][j], 40, 64);
                if (lane < 32 && (lane & 8) == 0) *reinterpret_cast<float4v*>(&part[wave][r][TN * n + 4 * (lane >> 4)]) = acc[n][m];
            } else {
                *reinterpret_cast<float4v*>(&part[wave][16 * m + r][TN * n + 4 * (lane >> 4)]) = acc[n][m];
            }
        }
    __syncthreads();
    // 8 consecutive columns of one row per thread
    constexpr int VEC = NT * TN / 8;
    const int row = threadIdx.x / VEC, c = (threadIdx.x % VEC) * 8;
    if (row >= MB * 16 || row >= a.M || n0 + c >= a.N) return;
    float8v v = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < WAVES; ++s) {
        const float4v lo = *reinterpret_cast<const float4v*>(&part[s][row][c]), hi = *reinterpret_cast<const float4v*>(&part[s][row][c + 4]);
        v += __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
    if (a.nsplit > 1) {
        store8<float>(a.partial, ((long)blockIdx.z * a.M + row) * a.N + n0 + c, v);
    } else {
        with_epilogue(a.epi, [&](auto epic) __attribute__((always_inline)) {
            constexpr int EPI = decltype(epic)::value;
            Raw8<T> bias = {}, side = {};
            if constexpr (kEpiBias<EPI>) bias = load_raw8<T>(a.bias, n0 + c);
            if constexpr (kEpiSide<EPI>) side = load_raw8<T>(epi_side<EPI>(a), (long)row * epi_side_ld<EPI>(a) + n0 + c);
            epilogue_apply8<T, EPI>(a, row, n0 + c, v, bias, side);
        });
    }
}

// Weight tiles per workgroup: two workgroups fit a CU, so the estimate counts half rounds of 256 workgroups (the first)
// and rounds of 512, each as long as the tiles a workgroup has; the activation rows' reads, M / (16 NT) of the weight's,
// cost half as much as those (they hit the caches).  (Of 17 to 32 rows one fits: two turns of loads take 130 to 174 registers.  Its
// estimate is the same, since the tiles decide a forward's order of sums.  Two workgroups of one turn are slower: 24 rows, us, 6144 x 2048 10.3 /
// 10.8, 8192 x 2048 11.9 / 12.4, 2048 x 8192 14.3 / 15.0; one turn of twice the loads, as before: 10.9, 12.1, 14.4.)
static int skinny_tiles(const GemmArgs& a) {
    const int tiles = (a.N + 15) / 16;
    int best = 1;
    float best_cost = 0.f;
    for (int nt = 1; nt <= 4; nt *= 2) {
        const int blocks = (tiles + nt - 1) / nt * a.nsplit;
        const float rounds = blocks <= 256 ? 0.5f : (float)((blocks + 511) / 512);
        const float cost = rounds * nt * (1.f + 0.5f * a.M / (16 * nt));
        if (nt == 1 || cost <= best_cost) { best = nt; best_cost = cost; }
    }
    return best;
}

template <typename T, int MB, int NT, bool HALF> static void launch_tile(const GemmArgs& a, const SkinnyLn* ln, hipStream_t s) {
    constexpr int COLS = NT * (HALF ? 8 : 16);
    const dim3 grid((a.N + COLS - 1) / COLS, 1, a.nsplit);
    if constexpr (MB == 1)
        if (ln) {
            gemm_skinny_kernel<T, MB, NT, HALF, true><<<grid, 512, (size_t)a.M * (a.K + 8) * sizeof(T), s>>>(a, *ln);
            return;
        }
    gemm_skinny_kernel<T, MB, NT, HALF, false><<<grid, 512, 0, s>>>(a, SkinnyLn{});
}
template <typename T, int MB> static void launch_skinny(const GemmArgs& a, bool half, const SkinnyLn* ln, hipStream_t s) {
    const int nt = skinny_tiles(a);
    if (MB == 1 && half && skinny_half(a.M, a.N)) launch_tile<T, 1, 1, true>(a, ln, s);
    else if (nt == 4) launch_tile<T, MB, 4, false>(a, ln, s);
    else if (nt == 2) launch_tile<T, MB, 2, false>(a, ln, s);
    else launch_tile<T, MB, 1, false>(a, ln, s);
}

// (five chunks of 8 per lane, 64 * (8 / rows) lanes to a row)
bool skinny_takes_ln(int M, int K) { return M <= 8 && K <= (M > 4 ? 2560 : M > 2 ? 5120 : M > 1 ? 10240 : 20480); }

void launch_gemm_skinny(int dtype, const GemmArgs& a, bool half, const SkinnyLn* ln, hipStream_t s) {
    if (dtype == TP_F16) { if (a.M <= 16) launch_skinny<f16, 1>(a, half, ln, s); else launch_skinny<f16, 2>(a, half, ln, s); }
    else { if (a.M <= 16) launch_skinny<bf16, 1>(a, half, ln, s); else launch_skinny<bf16, 2>(a, half, ln, s); }
}

}  // namespace tp
