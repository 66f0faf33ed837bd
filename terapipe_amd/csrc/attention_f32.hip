// Attention in fp32: a workgroup's waves share the other axis of its 32 rows.
#include "attention_args.h"

namespace tp {

// ------------------------------------------------------------------------------------------------
// A workgroup of four waves owns 32 queries (forward, dQ) or 32 keys (dK / dV) of one (batch, head).  Its waves take the tiles
// of 32 keys (queries) in turn, each through two LDS tiles of its own -- no barrier in the loop -- and add up at the end.
// fp32 MFMAs (32 x 32 x 2) are a sixteenth of the 16-bit ones' rate, so a block of 32 x 32 scores at head dimension 64 is 4
// to 8 thousand cycles of matrix work: what a call takes is how many of them stand one behind the other, and a sequence
// of 128 positions has 32 such rows of blocks for eight (batch, head) pairs on 1024 SIMDs.
// Measured (8 pairs of 64, 128 positions; a wave per 32 rows before): forward 17.3 -> 11.0 us; dQ, delta and dK / dV 55 -> 34 in
// two launches instead of three.  LDS: 70 KB at head dimension 64, 136 at 128 (one workgroup per CU).
// ------------------------------------------------------------------------------------------------
template <int DH> struct F32Tiles {
    static constexpr int DP = (DH + 31) / 32 * 32, LD = DP + 4, TILE = 32 * LD;     // floats
    static constexpr int NDB = DP / 32, NKS = DH / 2, NW = 4;
    typedef TileCopy<float, 32, DP, 64> Copy;
};
// Between a wave's LDS stores and its lanes' reads of each other's: its LDS operations complete in order.
__device__ __forceinline__ void wave_lds_fence() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}
template <int NDB> __device__ __forceinline__ void zero_acc(float16v (&acc)[NDB]) {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
}
// acc[db] += (tile's columns db * 32 .., k over its 32 rows) x p, the 32 x 32 accumulator p as the k x n operand
template <int DH> __device__ __forceinline__ void mul_tile_t(float16v (&acc)[F32Tiles<DH>::NDB], const float* tile, const float16v& p, int lane) {
    const int g = lane >> 5, li = lane & 31;
#pragma unroll
    for (int j = 0; j < 16; ++j)
#pragma unroll
        for (int db = 0; db < F32Tiles<DH>::NDB; ++db)
            acc[db] = Elem<float>::mfma(tile[acc_row(j, g) * F32Tiles<DH>::LD + db * 32 + li], p[j], acc[db]);
}

template <int DH>
__global__ __launch_bounds__(256) void attn_f32_fwd_kernel(AttnArgs a) {
    typedef F32Tiles<DH> F;
    typedef typename F::Copy Copy;
    constexpr int NW = F::NW, NDB = F::NDB, NKS = F::NKS, LD = F::LD, TILE = F::TILE;
    __shared__ __attribute__((aligned(16))) float smem[NW * 2 * TILE];
    __shared__ float sM[NW][32], sL[NW][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5, li = lane & 31;
    const int bh = blockIdx.y, b = bh / a.H, h = bh - b * a.H;
    const int T_ = a.T, P = a.P, S = a.P + a.T;
    const int q0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * 32, tq = q0 + li;       // the longest key ranges start first
    const int ntiles = (P + min(T_, q0 + 32) + 31) / 32;
    float* sK = smem + wave * 2 * TILE;
    float* sV = sK + TILE;
    float qreg[NKS];
    load_row_operands<float, DH>(qreg, reinterpret_cast<const float*>(a.q) + (long)bh * a.q_bhs + (long)min(tq, T_ - 1) * DH, tq < T_, g);
    const float* Kb = reinterpret_cast<const float*>(a.kc) + (long)bh * a.cache_rows * DH;
    const float* Vb = reinterpret_cast<const float*>(a.vc) + (long)bh * a.cache_rows * DH;
    float16v oacc[NDB];
    zero_acc(oacc);
    float m = -INFINITY, lsum = 0.f;
    Copy ck, cv;
    if (wave < ntiles) {
        ck.load(Kb, DH, wave * 32, 0, S, DH, lane);
        cv.load(Vb, DH, wave * 32, 0, S, DH, lane);
    }
    for (int t = wave; t < ntiles; t += NW) {
        wave_lds_fence();
        ck.store(sK, lane);
        cv.store(sV, lane);
        if (t + NW < ntiles) {
            ck.load(Kb, DH, (t + NW) * 32, 0, S, DH, lane);
            cv.load(Vb, DH, (t + NW) * 32, 0, S, DH, lane);
        }
        wave_lds_fence();
        const int key0 = t * 32;
        float16v s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) s = Elem<float>::mfma(sK[li * LD + 2 * ks + g], qreg[ks], s);
        float mt = -INFINITY;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            if (key0 + acc_row(j, g) > P + tq) s[j] = -INFINITY;
            mt = fmaxf(mt, s[j]);
        }
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        const float m_new = fmaxf(m, mt), m_safe = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = exp2f((m - m_safe) * kLog2e);
        float psum = 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            s[j] = exp2f((s[j] - m_safe) * kLog2e);
            psum += s[j];
        }
        lsum = lsum * alpha + psum;
        m = m_new;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
        mul_tile_t<DH>(oacc, sV, s, lane);
    }
    const float lw = lsum + __shfl_xor(lsum, 32, 64);
    if (g == 0) { sM[wave][li] = m; sL[wave][li] = lw; }
    __syncthreads();
    float m_tot = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) m_tot = fmaxf(m_tot, sM[w][li]);
    const float m_ts = m_tot == -INFINITY ? 0.f : m_tot;
    float l_tot = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) l_tot += sL[w][li] * exp2f((sM[w][li] - m_ts) * kLog2e);
    const float f = l_tot > 0.f ? exp2f((m - m_ts) * kLog2e) / l_tot : 0.f;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] *= f;
    if (wave == 0 && g == 0 && tq < T_) a.lse[(long)bh * a.st_bhs + tq] = l_tot > 0.f ? m_tot + logf(l_tot) : -INFINITY;
    acc_to_lds_rows<DH>(oacc, sK, lane);
    __syncthreads();
    const long EE = (long)a.H * DH;
    for (int p = tid; p < 32 * DH / 4; p += 256) {
        const int row = p / (DH / 4), col = (p % (DH / 4)) * 4;
        if (q0 + row >= T_) break;
        float4v v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; ++w) v += *reinterpret_cast<const float4v*>(smem + w * 2 * TILE + row * LD + col);
        *reinterpret_cast<float4v*>(reinterpret_cast<float*>(a.o) + ((long)(q0 + row) * a.B + b) * EE + (long)h * DH + col) = v;
    }
}

// dQ of 32 queries, and their delta = rowsum(dO * O) for the dK / dV kernel that follows on the stream.
template <int DH>
__global__ __launch_bounds__(256) void attn_f32_dq_kernel(AttnArgs a) {
    typedef F32Tiles<DH> F;
    typedef typename F::Copy Copy;
    constexpr int NW = F::NW, NDB = F::NDB, NKS = F::NKS, LD = F::LD, TILE = F::TILE;
    __shared__ __attribute__((aligned(16))) float smem[NW * 2 * TILE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5, li = lane & 31;
    const int bh = blockIdx.y, b = bh / a.H, h = bh - b * a.H;
    const int T_ = a.T, P = a.P, S = a.P + a.T;
    const long EE = (long)a.H * DH;
    const int q0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * 32, tq = q0 + li, tr = min(tq, T_ - 1);
    const bool qok = tq < T_;
    const int ntiles = (P + min(T_, q0 + 32) + 31) / 32;
    float* sK = smem + wave * 2 * TILE;
    float* sV = sK + TILE;
    const float* Kb = reinterpret_cast<const float*>(a.kc) + (long)bh * a.cache_rows * DH;
    const float* Vb = reinterpret_cast<const float*>(a.vc) + (long)bh * a.cache_rows * DH;
    Copy ck, cv;
    if (wave < ntiles) {
        ck.load(Kb, DH, wave * 32, 0, S, DH, lane);
        cv.load(Vb, DH, wave * 32, 0, S, DH, lane);
    }
    float qreg[NKS], doreg[NKS];
    const long orow = ((long)tr * a.B + b) * EE + (long)h * DH;
    load_row_operands<float, DH>(qreg, reinterpret_cast<const float*>(a.q) + (long)bh * a.q_bhs + (long)tr * DH, qok, g);
    load_row_operands<float, DH>(doreg, reinterpret_cast<const float*>(a.d_o) + orow, qok, g);
    float delta_q = 0.f;
    {
        float oreg[NKS];
        load_row_operands<float, DH>(oreg, reinterpret_cast<const float*>(a.o) + orow, qok, g);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) delta_q += oreg[ks] * doreg[ks];
        delta_q += __shfl_xor(delta_q, 32, 64);
        if (wave == 0 && g == 0 && qok) a.delta[(long)bh * a.st_bhs + tq] = delta_q;
    }
    const float lse_q = qok ? a.lse[(long)bh * a.st_bhs + tq] : 0.f;
    float16v dq[NDB];
    zero_acc(dq);
    for (int t = wave; t < ntiles; t += NW) {
        wave_lds_fence();
        ck.store(sK, lane);
        cv.store(sV, lane);
        if (t + NW < ntiles) {
            ck.load(Kb, DH, (t + NW) * 32, 0, S, DH, lane);
            cv.load(Vb, DH, (t + NW) * 32, 0, S, DH, lane);
        }
        wave_lds_fence();
        const int key0 = t * 32;
        float16v s, d;
#pragma unroll
        for (int r = 0; r < 16; ++r) { s[r] = 0.f; d[r] = 0.f; }
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            s = Elem<float>::mfma(sK[li * LD + 2 * ks + g], qreg[ks], s);
            d = Elem<float>::mfma(sV[li * LD + 2 * ks + g], doreg[ks], d);
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const bool vis = qok && key0 + acc_row(j, g) <= P + tq;
            const float p = vis ? exp2f((s[j] - lse_q) * kLog2e) : 0.f;
            d[j] = p * (d[j] - delta_q);
        }
        mul_tile_t<DH>(dq, sK, d, lane);
    }
    wave_lds_fence();
    acc_to_lds_rows<DH>(dq, sK, lane);
    __syncthreads();
    for (int p = tid; p < 32 * DH / 4; p += 256) {
        const int row = p / (DH / 4), col = (p % (DH / 4)) * 4;
        if (q0 + row >= T_) break;
        float4v v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; ++w) v += *reinterpret_cast<const float4v*>(smem + w * 2 * TILE + row * LD + col);
        *reinterpret_cast<float4v*>(reinterpret_cast<float*>(a.dqkv) + ((long)(q0 + row) * a.B + b) * (3 * EE) + (long)h * 3 * DH + col) = v * a.qscale;
    }
}

// dK / dV of 32 keys against the queries of the call; gradient caches as in attn_bwd_dkdv_kernel.
template <int DH>
__global__ __launch_bounds__(256) void attn_f32_dkdv_kernel(AttnArgs a) {
    typedef F32Tiles<DH> F;
    typedef typename F::Copy Copy;
    constexpr int NW = F::NW, NDB = F::NDB, NKS = F::NKS, LD = F::LD, TILE = F::TILE;
    __shared__ __attribute__((aligned(16))) float smem[NW * 2 * TILE];
    __shared__ __attribute__((aligned(16))) float sStat[NW][2][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5, li = lane & 31;
    const int bh = blockIdx.y, b = bh / a.H, h = bh - b * a.H;
    const int T_ = a.T, P = a.P, S = a.P + a.T;
    const long EE = (long)a.H * DH;
    const int key0 = blockIdx.x * 32, key = key0 + li;                  // (the first keys have the most queries)
    if (a.grad_rows > S && !grad_rows_beyond<float, DH, 32, 256>(a, bh, key0, S, tid)) return;
    float* sQ = smem + wave * 2 * TILE;
    float* sdO = sQ + TILE;
    const float* Qb = reinterpret_cast<const float*>(a.q) + (long)bh * a.q_bhs;
    const float* dOb = reinterpret_cast<const float*>(a.d_o) + (long)b * EE + (long)h * DH;      // row t at stride B * E
    const int nqb = (T_ + 31) / 32, qb0 = (key0 > P ? (key0 - P) / 32 : 0) + wave;
    Copy cq, cdo;
    float stat = 0.f;                   // lanes 0 to 31: lse, 32 to 63: delta of the block's rows
    auto load = [&](int qb) {
        cq.load(Qb, DH, qb * 32, 0, T_, DH, lane);
        cdo.load(dOb, (long)a.B * EE, qb * 32, 0, T_, DH, lane);
        const int t = qb * 32 + li;
        stat = t < T_ ? (g ? a.delta : a.lse)[(long)bh * a.st_bhs + t] : 0.f;
    };
    if (qb0 < nqb) load(qb0);
    float kreg[NKS], vreg[NKS];
    const long krow = ((long)bh * a.cache_rows + min(key, S - 1)) * DH;
    load_row_operands<float, DH>(kreg, reinterpret_cast<const float*>(a.kc) + krow, key < S, g);
    load_row_operands<float, DH>(vreg, reinterpret_cast<const float*>(a.vc) + krow, key < S, g);
    float16v dk[NDB], dv[NDB];
    zero_acc(dk);
    zero_acc(dv);
    for (int qb = qb0; qb < nqb; qb += NW) {
        wave_lds_fence();
        cq.store(sQ, lane);
        cdo.store(sdO, lane);
        sStat[wave][g][li] = stat;
        if (qb + NW < nqb) load(qb + NW);
        wave_lds_fence();
        float16v s, d;
#pragma unroll
        for (int r = 0; r < 16; ++r) { s[r] = 0.f; d[r] = 0.f; }
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            s = Elem<float>::mfma(sQ[li * LD + 2 * ks + g], kreg[ks], s);
            d = Elem<float>::mfma(sdO[li * LD + 2 * ks + g], vreg[ks], d);
        }
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
            const float4v l4 = *reinterpret_cast<const float4v*>(&sStat[wave][0][8 * jq + 4 * g]);
            const float4v d4 = *reinterpret_cast<const float4v*>(&sStat[wave][1][8 * jq + 4 * g]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = 4 * jq + e, t = qb * 32 + 8 * jq + 4 * g + e;
                const bool vis = t < T_ && key <= P + t && key < S;
                const float p = vis ? exp2f((s[j] - l4[e]) * kLog2e) : 0.f;
                d[j] = p * (d[j] - d4[e]);
                s[j] = p;
            }
        }
        mul_tile_t<DH>(dv, sdO, s, lane);
        mul_tile_t<DH>(dk, sQ, d, lane);
    }
    wave_lds_fence();
    acc_to_lds_rows<DH>(dk, sQ, lane);
    acc_to_lds_rows<DH>(dv, sdO, lane);
    __syncthreads();
    for (int p = tid; p < 32 * DH / 4; p += 256) {
        const int row = p / (DH / 4), col = (p % (DH / 4)) * 4, k = key0 + row;
        if (k >= S) break;
        float4v vk = {0.f, 0.f, 0.f, 0.f}, vv = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            vk += *reinterpret_cast<const float4v*>(smem + w * 2 * TILE + row * LD + col);
            vv += *reinterpret_cast<const float4v*>(smem + (w * 2 + 1) * TILE + row * LD + col);
        }
        const long goff = ((long)bh * a.cache_rows + k) * DH + col;
        float4v* gK = reinterpret_cast<float4v*>(reinterpret_cast<float*>(a.gk) + goff);
        float4v* gV = reinterpret_cast<float4v*>(reinterpret_cast<float*>(a.gv) + goff);
        const float4v* iK = reinterpret_cast<const float4v*>(reinterpret_cast<const float*>(a.gk_in) + goff);
        const float4v* iV = reinterpret_cast<const float4v*>(reinterpret_cast<const float*>(a.gv_in) + goff);
        if (k < P) {
            if (a.accumulate_prefix) { vk += *iK; vv += *iV; }
            *gK = vk;
            *gV = vv;
        } else {
            if (a.has_incoming) { vk += *iK; vv += *iV; }
            float* dst = reinterpret_cast<float*>(a.dqkv) + ((long)(k - P) * a.B + b) * (3 * EE) + (long)h * 3 * DH + col;
            *reinterpret_cast<float4v*>(dst + DH) = vk;
            *reinterpret_cast<float4v*>(dst + 2 * DH) = vv;
            if (a.zero_slice_rows) {
                *gK = float4v{0.f, 0.f, 0.f, 0.f};
                *gV = float4v{0.f, 0.f, 0.f, 0.f};
            }
        }
    }
}

template <int DH> static void fwd_f32(const AttnArgs& a, hipStream_t s) {
    attn_f32_fwd_kernel<DH><<<dim3((a.T + 31) / 32, a.B * a.H), 256, 0, s>>>(a);
}
template <int DH> static void bwd_f32(const AttnArgs& a, hipStream_t s) {
    attn_f32_dq_kernel<DH><<<dim3((a.T + 31) / 32, a.B * a.H), 256, 0, s>>>(a);
    if (!a.dq_only) attn_f32_dkdv_kernel<DH><<<dim3((a.grad_rows + 31) / 32, a.B * a.H), 256, 0, s>>>(a);
}
void launch_attn_f32(bool backward, int head_dim, const AttnArgs& a, hipStream_t s) {
    switch (head_dim) {
    case 16: backward ? bwd_f32<16>(a, s) : fwd_f32<16>(a, s); break;
    case 32: backward ? bwd_f32<32>(a, s) : fwd_f32<32>(a, s); break;
    case 64: backward ? bwd_f32<64>(a, s) : fwd_f32<64>(a, s); break;
    case 80: backward ? bwd_f32<80>(a, s) : fwd_f32<80>(a, s); break;
    case 96: backward ? bwd_f32<96>(a, s) : fwd_f32<96>(a, s); break;
    default: backward ? bwd_f32<128>(a, s) : fwd_f32<128>(a, s); break;
    }
}

}  // namespace tp
