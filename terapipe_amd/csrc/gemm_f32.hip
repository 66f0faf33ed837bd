// fp32 products with few tiles: k shared by a workgroup's waves, operands straight from memory into registers.
#include "gemm_epilogue.h"

namespace tp {

// ---------------------------------------------------------------------------------------------
// 32 x 32 tile, eight waves that share its k (v_mfma_f32_32x32x2_f32).  A product of a few hundred rows and columns has
// about a hundred such tiles and is over in the time of its launches: gemm_kernel brings it to 512 workgroups of 64 x 64
// with k splits, each a chain of 16-wide k-tiles that wait for memory, and a second launch adds the splits.  Here a wave asks
// for all of its share of k at once (32 positions of both operands; products of up to 256 of k come here), no LDS and no barrier
// stand between, and the eight partial tiles are added through LDS, in pairs.
// A lane (row or column lane & 31 of its operand, g = lane >> 5) takes k-positions 4 g .. 4 g + 3 of every 8 from a
// k-contiguous operand as one 16-byte load, position by position from the other kind: MFMA j of 4 sees k = 4 g + j from both.
// ---------------------------------------------------------------------------------------------
template <bool AKM, bool BKM>
__global__ __launch_bounds__(512) void gemm_f32_small_kernel(GemmArgs a) {
    constexpr int WAVES = 8, STEP = 32, NV = STEP / 8, PITCH = 36;
    __shared__ float part[WAVES][32][PITCH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 31, g = lane >> 5;
    const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
    const float* A = reinterpret_cast<const float*>(a.A);
    const float* B = reinterpret_cast<const float*>(a.B);
    const int m = min(m0 + li, a.M - 1), n = min(n0 + li, a.N - 1);     // (rows and columns past the edge are not stored)
    const long sa = AKM ? 1 : a.lda, sb = BKM ? 1 : a.ldb;              // from one k to the next
    const float* pa = AKM ? A + (long)m * a.lda : A + m;
    const float* pb = BKM ? B + (long)n * a.ldb : B + n;
    float16v acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    // 4 consecutive k from k0 on; positions past K are zero (K is a multiple of 4 where one of them is contiguous)
    auto load = [&](const float* p, long stride, bool contiguous, int k0) __attribute__((always_inline)) -> float4v {
        float4v v = {0.f, 0.f, 0.f, 0.f};
        if (contiguous) {
            if (k0 < a.K) v = *reinterpret_cast<const float4v*>(p + k0);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (k0 + j < a.K) v[j] = p[(long)(k0 + j) * stride];
        }
        return v;
    };
    for (int k = wave * STEP; k < a.K; k += WAVES * STEP) {
        float4v fa[NV], fb[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            fa[i] = load(pa, sa, AKM, k + 8 * i + 4 * g);
            fb[i] = load(pb, sb, BKM, k + 8 * i + 4 * g);
        }
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][j], fb[i][j], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][acc_row(r, g)][li] = acc[r];
    __syncthreads();
    if (threadIdx.x >= 128) return;
    const int row = threadIdx.x >> 2, c = (threadIdx.x & 3) * 8;
    if (m0 + row >= a.M || n0 + c >= a.N) return;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {           // pairwise
        float p[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) p[w] = part[w][row][c + e];
        v[e] = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    }
    epilogue_vec8<float>(a, m0 + row, n0 + c, v);
}

void launch_gemm_f32_small(int op, const GemmArgs& a, hipStream_t s) {
    const dim3 grid((a.N + 31) / 32, (a.M + 31) / 32);
    if (op == TP_GEMM_NT) gemm_f32_small_kernel<true, true><<<grid, 512, 0, s>>>(a);
    else if (op == TP_GEMM_NN) gemm_f32_small_kernel<true, false><<<grid, 512, 0, s>>>(a);
    else gemm_f32_small_kernel<false, false><<<grid, 512, 0, s>>>(a);
}

}  // namespace tp
