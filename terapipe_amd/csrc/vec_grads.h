// The vector-parameter gradients of a layer as blocks of 512 threads: of a launch of their own (layernorm.hip), or behind the tiles of
// the launch that takes the weight gradients of the same rows (gemm_tall.hip).
#pragma once
#include "common.h"

namespace tp {

// (fp32 chunks change type by value: taken apart through a pointer some are put into scratch memory)
template <typename T> __device__ __forceinline__ void load_chunk(const T* p, float* out) {
    constexpr int CH = 16 / sizeof(T);
    uint4 raw = *reinterpret_cast<const uint4*>(p);
    if constexpr (sizeof(T) == 2) {
        const T* h = reinterpret_cast<const T*>(&raw);
#pragma unroll
        for (int e = 0; e < CH; ++e) out[e] = Elem<T>::to_float(h[e]);
    } else {
        const float4v f = __builtin_bit_cast(float4v, raw);
#pragma unroll
        for (int e = 0; e < CH; ++e) out[e] = f[e];
    }
}

// The vector-parameter gradients of a layer in ONE launch: up to kVecGradMax reductions over the rows of a step,
// each either column sums of dy (a bias gradient) or the LayerNorm pair (dgamma += sum dy * xhat, dbeta += sum dy).
// A block of 512 threads = 32 column chunks (8 columns, 16-byte loads for 16-bit types) x 16 row lanes covers
// 256 columns x kVecGradRows rows of one problem; the row lanes are combined in LDS and every column then costs one
// atomic per block.  Blocks are numbered problem by problem (first_block[]).
constexpr int kVecGradMax = 8;
constexpr int kVecGradLanes = 16, kVecGradRows = 256;
struct VecGradProblem {
    const void* dy; const void* x; const float* mean; const float* rstd;
    float* acc0; float* acc1;
    long ld; int M, N;
};
// In a kernel: VEC_GRAD_PICK(args, block, pr, first) declares the problem of a block and its first one.  (Constant indices only, and no reference
// to the argument: either would have it copied to scratch memory.)
#define VEC_GRAD_PICK(args, block, pr, first)                                       \
    VecGradProblem pr = (args).p[0];                                                \
    int first = (args).first_block[0];                                              \
    _Pragma("unroll") for (int i = 1; i < kVecGradMax; ++i)                         \
        if (i < (args).n && (block) >= (args).first_block[i]) { pr = (args).p[i]; first = (args).first_block[i]; }
struct VecGradArgs {
    VecGradProblem p[kVecGradMax];
    int first_block[kVecGradMax + 1];
    int n;
};

// lds: kVecGradLds bytes; U: rows of a thread under way (1 where four blocks share a CU, more for one alone on it)
constexpr int kVecGradLds = 2 * kVecGradLanes * 256 * 4;
template <typename T> using Chunk = T __attribute__((ext_vector_type(8)));
template <typename T, int U> __device__ __forceinline__ void vec_param_grads_block(VecGradProblem pr, int local, void* lds) {
    typedef float Row[256];
    Row *sg = reinterpret_cast<Row*>(lds), *sb = sg + kVecGradLanes;
    const int ncb = (pr.N + 255) / 256;
    const int cb = local % ncb, rb = local / ncb;
    const int cl = threadIdx.x & 31, rl = threadIdx.x >> 5;
    const int col0 = (cb * 32 + cl) * 8;
    const int r0 = rb * kVecGradRows, r1 = min(pr.M, r0 + kVecGradRows);
    const T* dy = reinterpret_cast<const T*>(pr.dy);
    const T* x = reinterpret_cast<const T*>(pr.x);
    float ag[8], ab[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) { ag[e] = 0.f; ab[e] = 0.f; }
    if (col0 < pr.N) {
        int row = r0 + rl;
        if constexpr (U > 1) {
            static_assert(sizeof(T) == 2, "16-byte chunks");
            for (; row + (U - 1) * kVecGradLanes < r1; row += U * kVecGradLanes) {
                Chunk<T> rd[U], rx[U];
#pragma unroll
                for (int u = 0; u < U; ++u) rd[u] = *reinterpret_cast<const Chunk<T>*>(dy + (long)(row + u * kVecGradLanes) * pr.ld + col0);
                if (x) {
#pragma unroll
                    for (int u = 0; u < U; ++u) rx[u] = *reinterpret_cast<const Chunk<T>*>(x + (long)(row + u * kVecGradLanes) * pr.ld + col0);
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const float mu = pr.mean[row + u * kVecGradLanes], rs = pr.rstd[row + u * kVecGradLanes];
#pragma unroll
                        for (int e = 0; e < 8; ++e) ag[e] += (float)rd[u][e] * ((float)rx[u][e] - mu) * rs;
                    }
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int e = 0; e < 8; ++e) ab[e] += (float)rd[u][e];
            }
        }
        for (; row < r1; row += kVecGradLanes) {
            float d[8];
            load_chunk<T>(dy + (long)row * pr.ld + col0, d);
            if constexpr (sizeof(T) == 4) load_chunk<T>(dy + (long)row * pr.ld + col0 + 4, d + 4);
            if (x) {
                const float mu = pr.mean[row], rs = pr.rstd[row];
                float xv[8];
                load_chunk<T>(x + (long)row * pr.ld + col0, xv);
                if constexpr (sizeof(T) == 4) load_chunk<T>(x + (long)row * pr.ld + col0 + 4, xv + 4);
#pragma unroll
                for (int e = 0; e < 8; ++e) ag[e] += d[e] * (xv[e] - mu) * rs;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) ab[e] += d[e];
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) { sg[rl][cl * 8 + e] = ag[e]; sb[rl][cl * 8 + e] = ab[e]; }
    __syncthreads();
    const int c = threadIdx.x, col = cb * 256 + c;
    if (c < 256 && col < pr.N) {
        float tg = 0.f, tb = 0.f;
#pragma unroll
        for (int r = 0; r < kVecGradLanes; ++r) { tg += sg[r][c]; tb += sb[r][c]; }
        if (x) {
            atomicAdd(pr.acc0 + col, tg);
            atomicAdd(pr.acc1 + col, tb);
        } else {
            atomicAdd(pr.acc0 + col, tb);
        }
    }
}

// Host side: checks the problems and numbers their blocks; TP_OK or an error with its text set (layernorm.hip).
int fill_vec_grads(const tp_vecgrad_desc* descs, int n, int dtype, VecGradArgs& args, int& blocks);

}  // namespace tp
