// Token embedding lookup and vocabulary cross-entropy (the two ends of the layer stack at tensor-parallel
// size 1: reference mpu/layers.py:126-141 and mpu/cross_entropy.py:25-104).
#include "common.h"

namespace tp {

// out[m, :] = W[ids[m], :]; one workgroup per token, 16-byte chunks
template <typename T>
__global__ __launch_bounds__(256) void embedding_fwd_kernel(const int64_t* __restrict__ ids, const T* __restrict__ W,
                                                            T* __restrict__ out, int E, int V) {
    constexpr int CH = 16 / sizeof(T);
    const long m = blockIdx.x;
    const int64_t id = ids[m];
    const bool ok = id >= 0 && id < V;          // out-of-range ids give a zero row (masked rows of the reference)
    const uint4* src = reinterpret_cast<const uint4*>(W + (ok ? id : 0) * (long)E);
    uint4* dst = reinterpret_cast<uint4*>(out + m * (long)E);
    for (int c = threadIdx.x; c < E / CH; c += 256) dst[c] = ok ? src[c] : make_uint4(0, 0, 0, 0);
}

// dW_acc[ids[m], :] += dout[m, :] (fp32 accumulators, atomics: a token id may repeat)
template <typename T>
__global__ __launch_bounds__(256) void embedding_bwd_kernel(const int64_t* __restrict__ ids, const T* __restrict__ dout,
                                                            float* dW, int E, int V) {
    const long m = blockIdx.x;
    const int64_t id = ids[m];
    if (id < 0 || id >= V) return;
    for (int e = threadIdx.x; e < E; e += 256) atomicAdd(dW + id * (long)E + e, Elem<T>::to_float(dout[m * (long)E + e]));
}

// dW[ids[m], :] += sum over the tokens with that id of dout, one rounding per row.  The workgroup of a token's FIRST
// occurrence adds them all up: it looks for the id before its own position (and ends if it finds it), collects the later
// positions in order, and two groups of 256 threads take the collected rows in turn, eight loads under way per thread (a
// text's most frequent token is a sixteenth of it).  Only the rows that occur are touched, and no fp32 copy of the
// whole gradient is zeroed, read and cast: 2048 tokens of 2048 columns into 50257 rows 245 us -> 10, plus the fill of
// the gradient where none exists yet.  The search reads M ids per token, which bounds M (kEmbeddingRowsMax).
constexpr int kEmbeddingRowsMax = 8192;
template <typename T>
__global__ __launch_bounds__(512) void embedding_bwd_rows_kernel(const int64_t* __restrict__ ids, const T* __restrict__ dout,
                                                                 T* dW, int M, int E, int V) {
    constexpr int CH = 16 / sizeof(T);
    __shared__ int list[kEmbeddingRowsMax];
    __shared__ int wave_count[8];
    __shared__ float half[256 * CH];
    const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t id = ids[m];
    if (id < 0 || id >= V) return;
    for (int j0 = 0; j0 < m; j0 += 512) {
        const int j = j0 + tid;
        if (__syncthreads_or(j < m && ids[j] == id)) return;
    }
    int n = 0;
    for (int j0 = m; j0 < M; j0 += 512) {
        const int j = j0 + tid;
        const bool hit = j < M && ids[j] == id;
        const unsigned long long mask = __ballot(hit);
        if (lane == 0) wave_count[wave] = __popcll(mask);
        __syncthreads();
        int at = n, total = 0;
        for (int w = 0; w < 8; ++w) {
            if (w < wave) at += wave_count[w];
            total += wave_count[w];
        }
        if (hit) list[at + __popcll(mask & ((1ull << lane) - 1))] = j;
        n += total;
        __syncthreads();
    }
    const int group = tid >> 8, c = tid & 255;
    for (int c0 = 0; c0 < E / CH; c0 += 256) {
        const bool in = c0 + c < E / CH;
        float sum[CH];
#pragma unroll
        for (int e = 0; e < CH; ++e) sum[e] = 0.f;
        if (in)
            for (int k = group; k < n; k += 16) {
                uint4 raw[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    raw[u] = k + 2 * u < n ? reinterpret_cast<const uint4*>(dout + (long)list[k + 2 * u] * E)[c0 + c] : make_uint4(0, 0, 0, 0);
#pragma unroll
                for (int u = 0; u < 8; ++u)
#pragma unroll
                    for (int e = 0; e < CH; ++e) sum[e] += Elem<T>::to_float(reinterpret_cast<const T*>(&raw[u])[e]);
            }
        if (group == 1)
#pragma unroll
            for (int e = 0; e < CH; ++e) half[c * CH + e] = sum[e];
        __syncthreads();
        if (group == 0 && in) {
            uint4* dst = reinterpret_cast<uint4*>(dW + id * (long)E) + c0 + c;
            uint4 raw = *dst;
            T* w = reinterpret_cast<T*>(&raw);
#pragma unroll
            for (int e = 0; e < CH; ++e) w[e] = Elem<T>::from_float(Elem<T>::to_float(w[e]) + (sum[e] + half[c * CH + e]));
            *dst = raw;
        }
        __syncthreads();
    }
}

__device__ __forceinline__ float block_reduce(float v, float* scratch, bool is_max) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float u = __shfl_xor(v, o, 64);
        v = is_max ? fmaxf(v, u) : v + u;
    }
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float r = scratch[0];
    for (int w = 1; w < nw; ++w) r = is_max ? fmaxf(r, scratch[w]) : r + scratch[w];
    return r;
}

// One workgroup per row of logits [M, ld] (columns >= V are padding and ignored):
//   loss[m] = log(sum_v exp(z_v - max)) + max - z[target[m]]
//   logits[m, v] <- (softmax_v - [v == target[m]]) * grad_scale   (in place, as the reference overwrites its
//   input with the softmax and returns it as the gradient); padding columns <- 0.
template <typename T>
__global__ __launch_bounds__(1024) void cross_entropy_kernel(T* __restrict__ logits, long ld, const int64_t* __restrict__ target,
                                                             float* __restrict__ loss, int V, int Vpad, float grad_scale) {
    __shared__ float scratch[16];
    const long m = blockIdx.x;
    T* z = logits + m * ld;
    float mx = -INFINITY;
    for (int v = threadIdx.x; v < V; v += blockDim.x) mx = fmaxf(mx, Elem<T>::to_float(z[v]));
    mx = block_reduce(mx, scratch, true);
    float s = 0.f;
    for (int v = threadIdx.x; v < V; v += blockDim.x) s += expf(Elem<T>::to_float(z[v]) - mx);
    s = block_reduce(s, scratch, false);
    const int64_t t = target[m];
    const bool tok = t >= 0 && t < V;
    if (threadIdx.x == 0) loss[m] = logf(s) + mx - (tok ? Elem<T>::to_float(z[t]) : 0.f);
    __syncthreads();        // z[t] is read above before any thread overwrites it
    const float inv = 1.0f / s;
    for (int v = threadIdx.x; v < Vpad; v += blockDim.x) {
        float g = 0.f;
        if (v < V) g = (expf(Elem<T>::to_float(z[v]) - mx) * inv - ((tok && v == t) ? 1.f : 0.f)) * grad_scale;
        z[v] = Elem<T>::from_float(g);
    }
}

// The same with 16-byte accesses (rows 16-byte aligned, Vpad a whole number of chunks): the row is read from
// HBM once for the maximum, the two later passes find it in the caches, and the gradient goes out in
// 16-byte stores.
template <typename T>
__global__ __launch_bounds__(1024) void cross_entropy_vec_kernel(T* __restrict__ logits, long ld, const int64_t* __restrict__ target,
                                                                 float* __restrict__ loss, int V, int Vpad, float grad_scale) {
    constexpr int CH = 16 / sizeof(T);
    __shared__ float scratch[16];
    const long m = blockIdx.x;
    T* z = logits + m * ld;
    const uint4* zv = reinterpret_cast<const uint4*>(z);
    const int nch = Vpad / CH;
    float mx = -INFINITY;
    for (int c = threadIdx.x; c < nch; c += blockDim.x) {
        const uint4 raw = zv[c];
        const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (c * CH + i < V) mx = fmaxf(mx, Elem<T>::to_float(e[i]));
    }
    mx = block_reduce(mx, scratch, true);
    float s = 0.f;
    for (int c = threadIdx.x; c < nch; c += blockDim.x) {
        const uint4 raw = zv[c];
        const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (c * CH + i < V) s += expf(Elem<T>::to_float(e[i]) - mx);
    }
    s = block_reduce(s, scratch, false);
    const int64_t t = target[m];
    const bool tok = t >= 0 && t < V;
    if (threadIdx.x == 0) loss[m] = logf(s) + mx - (tok ? Elem<T>::to_float(z[t]) : 0.f);
    __syncthreads();        // z[t] is read above before any thread overwrites it
    const float inv = 1.0f / s;
    for (int c = threadIdx.x; c < nch; c += blockDim.x) {
        const uint4 raw = zv[c];
        const T* e = reinterpret_cast<const T*>(&raw);
        uint4 outv;
        T* o = reinterpret_cast<T*>(&outv);
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int v = c * CH + i;
            float g = 0.f;
            if (v < V) g = (expf(Elem<T>::to_float(e[i]) - mx) * inv - ((tok && v == t) ? 1.f : 0.f)) * grad_scale;
            o[i] = Elem<T>::from_float(g);
        }
        reinterpret_cast<uint4*>(z)[c] = outv;
    }
}

// Rows of up to 1024 * NCH chunks (65536 columns): the row is read once into registers (NCH 16-byte chunks per
// lane), maximum, sum and gradient are taken from there -- one read and one write of the logits in all.
template <typename T, int NCH>
__global__ __launch_bounds__(1024) void cross_entropy_reg_kernel(T* __restrict__ logits, long ld, const int64_t* __restrict__ target,
                                                                 float* __restrict__ loss, int V, int Vpad, float grad_scale) {
    constexpr int CH = 16 / sizeof(T);
    __shared__ float scratch[16];
    const long m = blockIdx.x;
    T* z = logits + m * ld;
    const uint4* zv = reinterpret_cast<const uint4*>(z);
    const int nch = Vpad / CH;
    const int64_t t = target[m];
    const bool tok = t >= 0 && t < V;
    const float zt = tok ? Elem<T>::to_float(z[t]) : 0.f;      // read before anything is overwritten
    // (the row stays in its 16-bit / fp32 form: 8 chunks are 32 registers, which keeps two workgroups on a CU;
    // holding exp(z - max) as floats instead costs 64 registers, one workgroup per CU and 1.5x the time)
    uint4 row[NCH];
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int c = k * 1024 + threadIdx.x;
        row[k] = c < nch ? zv[c] : make_uint4(0, 0, 0, 0);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const T* e = reinterpret_cast<const T*>(&row[k]);
        const int v0 = (k * 1024 + threadIdx.x) * CH;
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (v0 + i < V) mx = fmaxf(mx, Elem<T>::to_float(e[i]));
    }
    mx = block_reduce(mx, scratch, true);
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const T* e = reinterpret_cast<const T*>(&row[k]);
        const int v0 = (k * 1024 + threadIdx.x) * CH;
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (v0 + i < V) s += expf(Elem<T>::to_float(e[i]) - mx);
    }
    s = block_reduce(s, scratch, false);
    if (threadIdx.x == 0) loss[m] = logf(s) + mx - zt;
    const float inv = 1.0f / s;
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int c = k * 1024 + threadIdx.x;
        if (c >= nch) continue;
        const T* e = reinterpret_cast<const T*>(&row[k]);
        uint4 outv;
        T* o = reinterpret_cast<T*>(&outv);
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int v = c * CH + i;
            float g = 0.f;
            if (v < V) g = (expf(Elem<T>::to_float(e[i]) - mx) * inv - ((tok && v == t) ? 1.f : 0.f)) * grad_scale;
            o[i] = Elem<T>::from_float(g);
        }
        reinterpret_cast<uint4*>(z)[c] = outv;
    }
}

// Per-token loss without touching the logits: one read.  max_sum[m] = (row maximum, sum of exp(z - maximum)) for the
// gradient kernel.  A workgroup per row; each thread keeps its own running maximum and sum (a maximum that moves
// rescales the sum), and the workgroup combines them once.  VEC: 16-byte accesses.
template <typename T, bool VEC>
__global__ __launch_bounds__(1024) void cross_entropy_loss_kernel(const T* __restrict__ logits, long ld, const int64_t* __restrict__ target,
                                                                  float* __restrict__ loss, float2* __restrict__ max_sum, int V) {
    constexpr int CH = VEC ? 16 / sizeof(T) : 1;
    __shared__ float scratch[16];
    const long m = blockIdx.x;
    const T* z = logits + m * ld;
    float mx = -INFINITY, s = 0.f;
    const int nch = (V + CH - 1) / CH;
    constexpr int U = VEC ? 4 : 1;          // chunks under way per thread
    for (int c0 = 0; c0 < nch; c0 += U * 1024) {
        float v[U * CH];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = c0 + u * 1024 + threadIdx.x;
            T e[CH];
            if constexpr (VEC) *reinterpret_cast<uint4*>(e) = c < nch ? reinterpret_cast<const uint4*>(z)[c] : make_uint4(0, 0, 0, 0);
            else e[0] = c < nch ? z[c] : T(0);
#pragma unroll
            for (int i = 0; i < CH; ++i) v[u * CH + i] = c * CH + i < V ? Elem<T>::to_float(e[i]) : -INFINITY;
        }
        float top = v[0];
#pragma unroll
        for (int i = 1; i < U * CH; ++i) top = fmaxf(top, v[i]);
        if (top > mx) {
            s *= expf(mx - top);
            mx = top;
        }
        const float base = mx == -INFINITY ? 0.f : mx;
#pragma unroll
        for (int i = 0; i < U * CH; ++i) s += expf(v[i] - base);
    }
    const float all = block_reduce(mx, scratch, true);
    // (a thread without values, or with none above -infinity, has s = 0; one whose values are all NaN has no maximum but s = NaN)
    s = block_reduce(s == 0.f ? 0.f : s * expf(mx - all), scratch, false);
    if (threadIdx.x == 0) {
        const int64_t t = target[m];
        // (the difference first: the logarithm must not be lost in a maximum of -65504, or of 1e38)
        loss[m] = logf(s) + (all - (t >= 0 && t < V ? Elem<T>::to_float(z[t]) : 0.f));
        max_sum[m] = make_float2(all, s);
    }
}

// logits[m, v] <- (softmax_v - [v == target[m]]) * scale[m], padding columns <- 0: one read and one write
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void cross_entropy_grad_kernel(T* __restrict__ logits, long ld, const int64_t* __restrict__ target,
                                                                 const float2* __restrict__ max_sum, const float* __restrict__ scale,
                                                                 int V, int Vpad) {
    constexpr int CH = VEC ? 16 / sizeof(T) : 1;
    const int blocks = (Vpad + 256 * CH - 1) / (256 * CH);       // per row
    const long m = blockIdx.x / blocks;
    const int c = (int)(blockIdx.x % blocks) * 256 + threadIdx.x;
    if (c * CH >= Vpad) return;
    T* z = logits + m * ld + (long)c * CH;
    const float2 ms = max_sum[m];
    const float sc = scale[m], inv = sc / ms.y;
    const int64_t t = target[m];
    T e[CH];
    if constexpr (VEC) *reinterpret_cast<uint4*>(e) = *reinterpret_cast<const uint4*>(z);
    else e[0] = z[0];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int v = c * CH + i;
        float g = 0.f;
        if (v < V) g = expf(Elem<T>::to_float(e[i]) - ms.x) * inv - (v == t ? sc : 0.f);
        e[i] = Elem<T>::from_float(g);
    }
    if constexpr (VEC) *reinterpret_cast<uint4*>(z) = *reinterpret_cast<const uint4*>(e);
    else z[0] = e[0];
}

// x[m, :n] *= scale[m] in place (grad_input.mul_(grad_output.unsqueeze(-1)), mpu/cross_entropy.py:97)
template <typename T>
__global__ __launch_bounds__(256) void scale_rows_kernel(T* __restrict__ x, long ld, const float* __restrict__ scale, int n) {
    const long m = blockIdx.y;
    const float sc = scale[m];
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v < n) x[m * ld + v] = Elem<T>::from_float(Elem<T>::to_float(x[m * ld + v]) * sc);
}

// the same with 16-byte accesses (rows 16-byte aligned, n a whole number of chunks)
template <typename T>
__global__ __launch_bounds__(256) void scale_rows_vec_kernel(T* __restrict__ x, long ld, const float* __restrict__ scale, int nch) {
    constexpr int CH = 16 / sizeof(T);
    const long m = blockIdx.y;
    const float sc = scale[m];
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= nch) return;
    uint4* p = reinterpret_cast<uint4*>(x + m * ld) + c;
    uint4 raw = *p;
    T* e = reinterpret_cast<T*>(&raw);
#pragma unroll
    for (int i = 0; i < CH; ++i) e[i] = Elem<T>::from_float(Elem<T>::to_float(e[i]) * sc);
    *p = raw;
}

static int vocab_status(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { set_error("%s: launch failed: %s", what, hipGetErrorString(e)); return TP_ERR_LAUNCH; }
    return TP_OK;
}

}  // namespace tp

extern "C" int tp_embedding_fwd(const int64_t* ids, const void* weight, void* out, int M, int E, int V, int dtype,
                                void* stream) {
    using namespace tp;
    if (!ids || !weight || !out || M <= 0 || V <= 0) { set_error("tp_embedding_fwd: bad argument"); return TP_ERR_ARG; }
    if (dtype < TP_F32 || dtype > TP_BF16) { set_error("tp_embedding_fwd: bad dtype %d", dtype); return TP_ERR_ARG; }
    const int ch = dtype == TP_F32 ? 4 : 8;
    if (E <= 0 || E % ch || (((uintptr_t)weight | (uintptr_t)out) & 15)) { set_error("tp_embedding_fwd: E=%d must be a multiple of %d and the tensors 16-byte aligned", E, ch); return TP_ERR_UNSUPPORTED; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    switch (dtype) {
    case TP_F32: embedding_fwd_kernel<float><<<M, 256, 0, s>>>(ids, (const float*)weight, (float*)out, E, V); break;
    case TP_F16: embedding_fwd_kernel<f16><<<M, 256, 0, s>>>(ids, (const f16*)weight, (f16*)out, E, V); break;
    default: embedding_fwd_kernel<bf16><<<M, 256, 0, s>>>(ids, (const bf16*)weight, (bf16*)out, E, V); break;
    }
    return vocab_status("tp_embedding_fwd");
}

extern "C" int tp_embedding_bwd(const int64_t* ids, const void* dout, float* dweight_acc, int M, int E, int V, int dtype,
                                void* stream) {
    using namespace tp;
    if (!ids || !dout || !dweight_acc || M <= 0 || E <= 0 || V <= 0) { set_error("tp_embedding_bwd: bad argument"); return TP_ERR_ARG; }
    if (dtype < TP_F32 || dtype > TP_BF16) { set_error("tp_embedding_bwd: bad dtype %d", dtype); return TP_ERR_ARG; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    switch (dtype) {
    case TP_F32: embedding_bwd_kernel<float><<<M, 256, 0, s>>>(ids, (const float*)dout, dweight_acc, E, V); break;
    case TP_F16: embedding_bwd_kernel<f16><<<M, 256, 0, s>>>(ids, (const f16*)dout, dweight_acc, E, V); break;
    default: embedding_bwd_kernel<bf16><<<M, 256, 0, s>>>(ids, (const bf16*)dout, dweight_acc, E, V); break;
    }
    return vocab_status("tp_embedding_bwd");
}

extern "C" int tp_cross_entropy(void* logits, int64_t ld, const int64_t* target, float* loss, int M, int V, int Vpad,
                                float grad_scale, int dtype, void* stream) {
    using namespace tp;
    if (!logits || !target || !loss || M <= 0 || V <= 0 || Vpad < V || ld < Vpad) { set_error("tp_cross_entropy: bad argument (M=%d V=%d Vpad=%d ld=%ld)", M, V, Vpad, (long)ld); return TP_ERR_ARG; }
    if (dtype < TP_F32 || dtype > TP_BF16) { set_error("tp_cross_entropy: bad dtype %d", dtype); return TP_ERR_ARG; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int ch = dtype == TP_F32 ? 4 : 8;
    if (Vpad % ch == 0 && ld % ch == 0 && ((uintptr_t)logits & 15) == 0) {
        if (Vpad / ch <= 1024 * 8) {
            switch (dtype) {
            case TP_F32: cross_entropy_reg_kernel<float, 8><<<M, 1024, 0, s>>>((float*)logits, ld, target, loss, V, Vpad, grad_scale); break;
            case TP_F16: cross_entropy_reg_kernel<f16, 8><<<M, 1024, 0, s>>>((f16*)logits, ld, target, loss, V, Vpad, grad_scale); break;
            default: cross_entropy_reg_kernel<bf16, 8><<<M, 1024, 0, s>>>((bf16*)logits, ld, target, loss, V, Vpad, grad_scale); break;
            }
            return vocab_status("tp_cross_entropy");
        }
        if (dtype == TP_F32 && Vpad / ch <= 1024 * 16) {
            cross_entropy_reg_kernel<float, 16><<<M, 1024, 0, s>>>((float*)logits, ld, target, loss, V, Vpad, grad_scale);
            return vocab_status("tp_cross_entropy");
        }
        switch (dtype) {
        case TP_F32: cross_entropy_vec_kernel<float><<<M, 1024, 0, s>>>((float*)logits, ld, target, loss, V, Vpad, grad_scale); break;
        case TP_F16: cross_entropy_vec_kernel<f16><<<M, 1024, 0, s>>>((f16*)logits, ld, target, loss, V, Vpad, grad_scale); break;
        default: cross_entropy_vec_kernel<bf16><<<M, 1024, 0, s>>>((bf16*)logits, ld, target, loss, V, Vpad, grad_scale); break;
        }
        return vocab_status("tp_cross_entropy");
    }
    switch (dtype) {
    case TP_F32: cross_entropy_kernel<float><<<M, 1024, 0, s>>>((float*)logits, ld, target, loss, V, Vpad, grad_scale); break;
    case TP_F16: cross_entropy_kernel<f16><<<M, 1024, 0, s>>>((f16*)logits, ld, target, loss, V, Vpad, grad_scale); break;
    default: cross_entropy_kernel<bf16><<<M, 1024, 0, s>>>((bf16*)logits, ld, target, loss, V, Vpad, grad_scale); break;
    }
    return vocab_status("tp_cross_entropy");
}

extern "C" int tp_scale_rows(void* x, int64_t ld, const float* scale, int M, int N, int dtype, void* stream) {
    using namespace tp;
    if (!x || !scale || M <= 0 || N <= 0 || ld < N) { set_error("tp_scale_rows: bad argument"); return TP_ERR_ARG; }
    if (dtype < TP_F32 || dtype > TP_BF16) { set_error("tp_scale_rows: bad dtype %d", dtype); return TP_ERR_ARG; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int ch = dtype == TP_F32 ? 4 : 8;
    if (N % ch == 0 && ld % ch == 0 && ((uintptr_t)x & 15) == 0) {
        const int nch = N / ch;
        dim3 vgrid((nch + 255) / 256, M);
        switch (dtype) {
        case TP_F32: scale_rows_vec_kernel<float><<<vgrid, 256, 0, s>>>((float*)x, ld, scale, nch); break;
        case TP_F16: scale_rows_vec_kernel<f16><<<vgrid, 256, 0, s>>>((f16*)x, ld, scale, nch); break;
        default: scale_rows_vec_kernel<bf16><<<vgrid, 256, 0, s>>>((bf16*)x, ld, scale, nch); break;
        }
        return vocab_status("tp_scale_rows");
    }
    dim3 grid((N + 255) / 256, M);
    switch (dtype) {
    case TP_F32: scale_rows_kernel<float><<<grid, 256, 0, s>>>((float*)x, ld, scale, N); break;
    case TP_F16: scale_rows_kernel<f16><<<grid, 256, 0, s>>>((f16*)x, ld, scale, N); break;
    default: scale_rows_kernel<bf16><<<grid, 256, 0, s>>>((bf16*)x, ld, scale, N); break;
    }
    return vocab_status("tp_scale_rows");
}

extern "C" int tp_embedding_bwd_rows(const int64_t* ids, const void* dout, void* dweight, int M, int E, int V, int dtype,
                                     void* stream) {
    using namespace tp;
    if (!ids || !dout || !dweight || M <= 0 || E <= 0 || V <= 0) { set_error("tp_embedding_bwd_rows: bad argument"); return TP_ERR_ARG; }
    if (dtype < TP_F32 || dtype > TP_BF16) { set_error("tp_embedding_bwd_rows: bad dtype %d", dtype); return TP_ERR_ARG; }
    if (M > kEmbeddingRowsMax || E % (dtype == TP_F32 ? 4 : 8) || (((uintptr_t)dout | (uintptr_t)dweight) & 15)) {
        set_error("tp_embedding_bwd_rows: at most %d tokens (M=%d), rows of whole 16-byte chunks (E=%d), 16-byte aligned", kEmbeddingRowsMax, M, E);
        return TP_ERR_UNSUPPORTED;
    }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    switch (dtype) {
    case TP_F32: embedding_bwd_rows_kernel<float><<<M, 512, 0, s>>>(ids, (const float*)dout, (float*)dweight, M, E, V); break;
    case TP_F16: embedding_bwd_rows_kernel<f16><<<M, 512, 0, s>>>(ids, (const f16*)dout, (f16*)dweight, M, E, V); break;
    default: embedding_bwd_rows_kernel<bf16><<<M, 512, 0, s>>>(ids, (const bf16*)dout, (bf16*)dweight, M, E, V); break;
    }
    return vocab_status("tp_embedding_bwd_rows");
}

namespace tp {
template <typename T> static void launch_ce_loss(const void* logits, long ld, const int64_t* target, float* loss, float* max_sum, int M, int V, hipStream_t s) {
    float2* ms = reinterpret_cast<float2*>(max_sum);
    constexpr int CH = 16 / sizeof(T);
    // (whole chunks: the last one may reach past V into the row's padding, which ld covers)
    if (ld % CH == 0 && ((uintptr_t)logits & 15) == 0) cross_entropy_loss_kernel<T, true><<<M, 1024, 0, s>>>((const T*)logits, ld, target, loss, ms, V);
    else cross_entropy_loss_kernel<T, false><<<M, 1024, 0, s>>>((const T*)logits, ld, target, loss, ms, V);
}
template <typename T> static void launch_ce_grad(void* logits, long ld, const int64_t* target, const float* max_sum, const float* scale, int M, int V,
                                                 int Vpad, hipStream_t s) {
    const float2* ms = reinterpret_cast<const float2*>(max_sum);
    constexpr int CH = 16 / sizeof(T);
    if (ld % CH == 0 && Vpad % CH == 0 && ((uintptr_t)logits & 15) == 0)
        cross_entropy_grad_kernel<T, true><<<(unsigned)M * ((Vpad + 256 * CH - 1) / (256 * CH)), 256, 0, s>>>((T*)logits, ld, target, ms, scale, V, Vpad);
    else
        cross_entropy_grad_kernel<T, false><<<(unsigned)M * ((Vpad + 255) / 256), 256, 0, s>>>((T*)logits, ld, target, ms, scale, V, Vpad);
}
}  // namespace tp

extern "C" int tp_cross_entropy_loss(const void* logits, int64_t ld, const int64_t* target, float* loss, float* max_sum, int M, int V,
                                     int dtype, void* stream) {
    using namespace tp;
    if (!logits || !target || !loss || !max_sum || M <= 0 || V <= 0 || ld < V) { set_error("tp_cross_entropy_loss: bad argument (M=%d V=%d ld=%ld)", M, V, (long)ld); return TP_ERR_ARG; }
    if (dtype < TP_F32 || dtype > TP_BF16) { set_error("tp_cross_entropy_loss: bad dtype %d", dtype); return TP_ERR_ARG; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    switch (dtype) {
    case TP_F32: launch_ce_loss<float>(logits, ld, target, loss, max_sum, M, V, s); break;
    case TP_F16: launch_ce_loss<f16>(logits, ld, target, loss, max_sum, M, V, s); break;
    default: launch_ce_loss<bf16>(logits, ld, target, loss, max_sum, M, V, s); break;
    }
    return vocab_status("tp_cross_entropy_loss");
}

extern "C" int tp_cross_entropy_grad(void* logits, int64_t ld, const int64_t* target, const float* max_sum, const float* scale, int M,
                                     int V, int Vpad, int dtype, void* stream) {
    using namespace tp;
    if (!logits || !target || !max_sum || !scale || M <= 0 || V <= 0 || Vpad < V || ld < Vpad) {
        set_error("tp_cross_entropy_grad: bad argument (M=%d V=%d Vpad=%d ld=%ld)", M, V, Vpad, (long)ld);
        return TP_ERR_ARG;
    }
    if (dtype < TP_F32 || dtype > TP_BF16) { set_error("tp_cross_entropy_grad: bad dtype %d", dtype); return TP_ERR_ARG; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    switch (dtype) {
    case TP_F32: launch_ce_grad<float>(logits, ld, target, max_sum, scale, M, V, Vpad, s); break;
    case TP_F16: launch_ce_grad<f16>(logits, ld, target, max_sum, scale, M, V, Vpad, s); break;
    default: launch_ce_grad<bf16>(logits, ld, target, max_sum, scale, M, V, Vpad, s); break;
    }
    return vocab_status("tp_cross_entropy_grad");
}
