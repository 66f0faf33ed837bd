// Y = X W^T for a handful of rows (decoding: one token of each sequence), 16-bit.
#include "gemm_epilogue.h"

namespace tp {

// ---------------------------------------------------------------------------------------------
// At most 16 * MB rows.  The product reads the whole weight and computes next to nothing: for weights of a few MB it is
// bound by latency and by the bytes kept in flight, which a tile kernel that stages 64 rows through LDS with a barrier
// per k-tile keeps low.  Here a workgroup owns 16 * NT weight rows and its eight waves share their k: a wave reads 16
// rows x 256 k (NT x 16 rows of less k) per turn, eight 16-byte weight loads per lane outstanding, straight into the
// registers the MFMA takes (lane l: row l & 15, k 8 * (l >> 4) .. + 7 of each 32), the activation rows the same way
// (they stay in the caches; NT weight tiles share one read of them).  No LDS and no barrier until the eight partial
// tiles are added at the end.
// Measured (4 rows, weights from HBM, the same launch back to back): 6144 x 2048 10.3 -> 8.4 us, 2048 x 2048 8.5 -> 5.3,
// 2048 x 8192 (four k splits) 14.6 -> 8.2 (4.1 TB/s), 2304 x 768 6.1 -> 3.7.  In a decoding step's chain of dependent
// launches: 9.9 (2.6 TB/s), 6.0 (1.4), 9.8 (3.4), 8192 x 2048 11.6 (2.9).
// ---------------------------------------------------------------------------------------------
template <typename T, int MB, int NT>
__global__ __launch_bounds__(512) void gemm_skinny_kernel(GemmArgs a) {
    constexpr int WAVES = 8, U = 8 / NT, STEP = 32 * U, PITCH = NT * 16 + 4;
    __shared__ float part[WAVES][MB * 16][PITCH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = blockIdx.x * 16 * NT;
    const int kbeg = blockIdx.z * a.kper, kend = min(a.K, kbeg + a.kper);
    const int r = lane & 15, kq = 8 * (lane >> 4);
    const T *w[NT], *x[MB];
#pragma unroll
    for (int n = 0; n < NT; ++n) w[n] = reinterpret_cast<const T*>(a.B) + (long)min(n0 + 16 * n + r, a.N - 1) * a.ldb + kq;
#pragma unroll
    for (int m = 0; m < MB; ++m) x[m] = reinterpret_cast<const T*>(a.A) + (long)min(16 * m + r, a.M - 1) * a.lda + kq;
    float4v acc[NT][MB];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MB; ++m) acc[n][m] = float4v{0.f, 0.f, 0.f, 0.f};
    const uint4 zero = make_uint4(0, 0, 0, 0);
    for (int k = kbeg + wave * STEP; k < kend; k += WAVES * STEP) {
        uint4 fw[NT][U], fx[MB][U];
        if (k + STEP <= kend) {         // wave-uniform
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int u = 0; u < U; ++u) fw[n][u] = *reinterpret_cast<const uint4*>(w[n] + k + 32 * u);
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int u = 0; u < U; ++u) fx[m][u] = *reinterpret_cast<const uint4*>(x[m] + k + 32 * u);
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool in = k + 32 * u + kq < kend;         // k is a multiple of 8
#pragma unroll
                for (int n = 0; n < NT; ++n) fw[n][u] = in ? *reinterpret_cast<const uint4*>(w[n] + k + 32 * u) : zero;
#pragma unroll
                for (int m = 0; m < MB; ++m) fx[m][u] = in ? *reinterpret_cast<const uint4*>(x[m] + k + 32 * u) : zero;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int m = 0; m < MB; ++m) acc[n][m] = Mfma16x16x32<T>::run(fw[n][u], fx[m][u], acc[n][m]);
    }
    // register j of the lane: weight row 4 * (lane >> 4) + j, activation row lane & 15
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MB; ++m) *reinterpret_cast<float4v*>(&part[wave][16 * m + r][16 * n + 4 * (lane >> 4)]) = acc[n][m];
    __syncthreads();
    // 8 consecutive columns of one row per thread
    const int row = threadIdx.x / (2 * NT), c = (threadIdx.x % (2 * NT)) * 8;
    if (threadIdx.x >= 32 * MB * NT || row >= a.M || n0 + c >= a.N) return;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
#pragma unroll
    for (int s = 0; s < WAVES; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += part[s][row][c + e];
    if (a.nsplit > 1) {
        float* dst = a.partial + ((long)blockIdx.z * a.M + row) * a.N + n0 + c;
#pragma unroll
        for (int e = 0; e < 8; ++e) dst[e] = v[e];
    } else {
        epilogue_vec8<T>(a, row, n0 + c, v);
    }
}

// Weight tiles per workgroup: two workgroups fit a CU, so the estimate counts half rounds of 256 workgroups (the first)
// and rounds of 512, each as long as the tiles a workgroup has; the activation rows' reads, M / (16 NT) of the weight's,
// cost half as much as those (they hit the caches).
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

template <typename T, int MB> static void launch_skinny(const GemmArgs& a, hipStream_t s) {
    const int nt = skinny_tiles(a);
    const dim3 grid(((a.N + 15) / 16 + nt - 1) / nt, 1, a.nsplit);
    if (nt == 4) gemm_skinny_kernel<T, MB, 4><<<grid, 512, 0, s>>>(a);
    else if (nt == 2) gemm_skinny_kernel<T, MB, 2><<<grid, 512, 0, s>>>(a);
    else gemm_skinny_kernel<T, MB, 1><<<grid, 512, 0, s>>>(a);
}

void launch_gemm_skinny(int dtype, const GemmArgs& a, hipStream_t s) {
    if (dtype == TP_F16) { if (a.M <= 16) launch_skinny<f16, 1>(a, s); else launch_skinny<f16, 2>(a, s); }
    else { if (a.M <= 16) launch_skinny<bf16, 1>(a, s); else launch_skinny<bf16, 2>(a, s); }
}

}  // namespace tp
