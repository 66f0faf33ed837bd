// Attention of whole sequences and long slices (16-bit): workgroups whose waves share the tiles they stream.
#include "attention_args.h"

namespace tp {

typedef float float8v __attribute__((ext_vector_type(8)));
template <typename T> using vec8_t = T __attribute__((ext_vector_type(8)));
template <typename T> __device__ __forceinline__ uint4 pack8v(float8v v) {
    return __builtin_bit_cast(uint4, __builtin_convertvector(v, vec8_t<T>));
}

template <typename T> using vec2_t = T __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
template <typename T> __device__ __forceinline__ unsigned pack2(float a, float b) {
    const float2v two = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(two, vec2_t<T>));
}

// As xcd_map, for nblocks blocks that start longest first: where all of an XCD's workgroups fit its 32 CUs in twos, the second of a
// CU is as short as the first is long.
__device__ __forceinline__ bool xcd_map_causal(int BH, int nblocks, int& bh, int& blk) {
    const int id = blockIdx.x, nbh8 = (BH + 7) >> 3, n = nbh8 * nblocks;
    int slot = id >> 3;
    if (n <= 64 && slot >= 32) slot = n + 31 - slot;
    bh = (id & 7) + 8 * (slot % nbh8);
    blk = slot / nbh8;
    return bh < BH;
}

// ------------------------------------------------------------------------------------------------
// Forward.  A workgroup of eight waves owns 128 queries of one (batch, head): four blocks of 32, each by two waves that
// take one half of every key tile and merge at the end.  A tile of 128 keys of K and V is loaded once for all of them, into
// a ring of two stages in which K runs one tile ahead of V.
//
// What bounds it: the vector ALU (16 exponentials at a quarter of its rate, and about as many cycles of the rest, per 32 x 32
// block) and the MFMAs (as long again), two waves a SIMD.  The forms that give every wave its own ring (attn_fwd2_kernel,
// attn_fwd3_kernel) take 128 KB of LDS for one wave a SIMD, which waits for memory a third of its time, and pull every K / V
// byte through the global -> LDS path once per 32 or 64 queries; here it is once per 128.
// Measured (fp16, causal, 2048 positions): 40 heads of 128 98 -> 70 us, 96 of 128 228 -> 152 (677 TFLOP/s), 32 of 80 69 -> 41;
// 64 heads of 64 at 1024 27 -> 23.  Raising one of a SIMD's waves over the other (s_setprio), and score MFMAs interleaved
// with the exponentials by the compiler (its LDS reads then sit in front of each MFMA), change nothing.
// ------------------------------------------------------------------------------------------------
template <typename T, int DH>
__global__ __launch_bounds__(512) void attn_fwd_long_kernel(AttnArgs a) {
    typedef Elem<T> E;
    constexpr int NDB = (DH + 31) / 32, NKS = DH / 16, PITCH = tile_pitch<DH>(), CPR = PITCH / 8;
    constexpr int NB = 2;                                   // 32-key blocks of a tile per wave
    constexpr int KT = 64 * NB, TILE = KT * PITCH, STAGE = 2 * TILE;
    constexpr int NLD = KT * CPR / 512;                     // loads per K or V tile and lane
    constexpr int NLOAD = 2 * NLD;
    constexpr int EPI_LD = NDB * 32 + 4;
    constexpr int RING_BYTES = 2 * STAGE * 2, EPI_BYTES = (4 * 2 * 32 + 4 * 32 * EPI_LD) * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[RING_BYTES > EPI_BYTES ? RING_BYTES : EPI_BYTES];
    T* ring = reinterpret_cast<T*>(smem);

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, li = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), qb = wave & 3, kh = wave >> 2;
    int bh, blk;
    if (!xcd_map(a.B * a.H, bh, blk)) return;
    const int b = bh / a.H, h = bh - b * a.H;
    const int T_ = a.T, P = a.P, S = a.P + a.T;
    const int q0 = ((T_ + 127) / 128 - 1 - blk) * 128;      // the blocks with the longest key range start first
    const int qw = q0 + 32 * qb, tq = qw + li;
    const bool qok = tq < T_;
    const int nt = (P + min(T_, q0 + 128) + KT - 1) / KT;   // tiles of the workgroup
    const int key_end = qw < T_ ? P + min(T_, qw + 32) : 0; // keys this wave's queries see

    unsigned koff[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int p = i * 512 + tid, r = p / CPR, lc = (p % CPR) ^ swz16<PITCH>(r);
        koff[i] = lc < DH / 8 ? (unsigned)(r * DH * 2 + lc * 16) : kNoChunk;
    }
    const char* Kb = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.kc) + (long)bh * a.cache_rows * DH));
    const char* Vb = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.vc) + (long)bh * a.cache_rows * DH));
    const unsigned lds0 = lds_addr(smem) + wave * 1024;
    // tile t of K (which = 0) or V (1) into its half of a stage; rows at or past S are clamped to row S - 1: finite data,
    // and every such key is masked
    auto issue = [&](int stage, int which, int tile) {
        const unsigned dst = lds0 + (unsigned)((stage * STAGE + which * TILE) * 2);
        const char* base = which ? Vb : Kb;
        const int row0 = tile * KT;
        if (row0 + KT <= S) {
            const char* sb = base + (long)row0 * (DH * 2);
#pragma unroll
            for (int i = 0; i < NLD; ++i) load_chunk_lds<DH>(koff[i], sb, dst + i * 8192);
        } else {
#pragma unroll
            for (int i = 0; i < NLD; ++i) {
                const int p = i * 512 + tid, r = p / CPR, lc = (p % CPR) ^ swz16<PITCH>(r);
                const unsigned off = lc < DH / 8 ? (unsigned)(min(row0 + r, S - 1) * DH * 2 + lc * 16) : kNoChunk;
                load_chunk_lds<DH>(off, base, dst + i * 8192);
            }
        }
    };
    issue(0, 0, 0);
    issue(0, 1, 0);
    if (nt > 1) issue(1, 0, 1);

    typename E::opnd_t qreg[NKS];
    load_row_operands<T, DH>(qreg, reinterpret_cast<const T*>(a.q) + (long)bh * a.q_bhs + (long)(qok ? tq : 0) * DH, qok, g);

    int okm[NKS], otr[NDB][2];          // element offsets of the lane's fetches inside a stage, its first block
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) okm[ks] = km_offset<T, PITCH>(kh * 32 * NB + li, ks * 16, lane);
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
        tr_offsets<T, PITCH, true>(kh * 32 * NB, db * 32, lane, otr[db][0], otr[db][1]);
        otr[db][0] += TILE;
        otr[db][1] += TILE;
    }

    float16v oacc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] = 0.f;
    float m = -INFINITY, lsum = 0.f;

    // the scores of the wave's keys of the tile in stage `so`
    auto scores = [&](int so, float16v* s) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[n][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int n = 0; n < NB; ++n) s[n] = E::mfma(load_km<T>(ring + so + okm[ks] + n * 32 * PITCH), qreg[ks], s[n]);
    };
    float16v s[NB];
    wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    scores(0, s);

    auto step = [&](auto sc, int t) __attribute__((always_inline)) {
        constexpr int st = decltype(sc)::value;
        // this wave's loads of K(t + 1) and V(t) have landed and its reads of K(t) and V(t - 1) are back
        wait_vmcnt<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (t + 1 < nt) issue(st ^ 1, 1, t + 1);
        if (t + 2 < nt) issue(st, 0, t + 2);
        const int key0 = t * KT + kh * NB * 32;
        if (key0 >= key_end) return;        // wave-uniform: this tile and all after it lie beyond the wave's queries
        if (key0 + 32 * NB - 1 > P + qw) {  // wave-uniform: the tile touches the causal boundary
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    if (key0 + n * 32 + acc_row(j, g) > P + tq) s[n][j] = -INFINITY;
        }
        float mt = -INFINITY;
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int j = 0; j < 16; ++j) mt = fmaxf(mt, s[n][j]);
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        // m is the row's REFERENCE value of the exponentials, not its running maximum (as in attn_fwd2_kernel): it moves
        // only when a row outgrows it by kSlack, exponentials stay below e^kSlack = 148.
        constexpr float kSlack = 5.0f;
        if (__builtin_amdgcn_ballot_w64(mt > m + kSlack) != 0) {
            const float m_new = fmaxf(m, mt);
            const float alpha = m_new == -INFINITY ? 1.0f : fast_exp2((m - m_new) * kLog2e);
            m = m_new;
            lsum *= alpha;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
        }
        const float mneg = m == -INFINITY ? 0.f : -m * kLog2e;
        // Block by block: the next tile's K and this tile's V fragments are asked for, the exponentials run while they come,
        // then the MFMAs, the next tile's scores in place of this one's.  (Behind the last tile the scores are those of
        // whatever the other stage holds: nothing reads them.)
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            typename E::opnd_t kf[NKS];
            uint4 vf[2][NDB];
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) kf[ks] = load_km<T>(ring + (st ^ 1) * STAGE + okm[ks] + n * 32 * PITCH);
#pragma unroll
            for (int hs = 0; hs < 2; ++hs)
#pragma unroll
                for (int db = 0; db < NDB; ++db) {
                    const int o = st * STAGE + (n * 32 + hs * 16) * PITCH;
                    vf[hs][db] = load_tr<T>(ring + o + otr[db][0], ring + o + otr[db][1]);
                }
            __builtin_amdgcn_sched_barrier(0);
            float8v e0, e1;
            float psum = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                e0[j] = fast_exp2(fmaf(s[n][j], kLog2e, mneg));        // -inf -> 0
                e1[j] = fast_exp2(fmaf(s[n][j + 8], kLog2e, mneg));
                psum += e0[j] + e1[j];
            }
            lsum += psum;
            const uint4 p[2] = {pack8v<T>(e0), pack8v<T>(e1)};
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 16; ++r) s[n][r] = 0.f;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) s[n] = E::mfma(kf[ks], qreg[ks], s[n]);
#pragma unroll
            for (int hs = 0; hs < 2; ++hs)
#pragma unroll
                for (int db = 0; db < NDB; ++db) oacc[db] = E::mfma(vf[hs][db], p[hs], oacc[db]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int t = 0; t < nt; t += 2) {
        step(std::integral_constant<int, 0>(), t);
        if (t + 1 < nt) step(std::integral_constant<int, 1>(), t + 1);
    }
    __syncthreads();            // every wave is done with the ring: the space is reused for the merge

    float* sM = reinterpret_cast<float*>(smem);         // [4][2][32]: the second halves' references and sums
    float* ebuf = sM + 4 * 2 * 32 + qb * 32 * EPI_LD;
    const float lw = lsum + __shfl_xor(lsum, 32, 64);
    if (kh == 1) {
        if (g == 0) { sM[qb * 64 + li] = m; sM[qb * 64 + 32 + li] = lw; }
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int jq = 0; jq < 4; ++jq)
                *reinterpret_cast<float4*>(ebuf + (db * 4 + jq) * 256 + lane * 4) =
                    make_float4(oacc[db][4 * jq], oacc[db][4 * jq + 1], oacc[db][4 * jq + 2], oacc[db][4 * jq + 3]);
    }
    __syncthreads();
    if (kh == 1) return;
    const float m1 = sM[qb * 64 + li], l1 = sM[qb * 64 + 32 + li];
    const float mt = fmaxf(m, m1), ms = mt == -INFINITY ? 0.f : mt;
    float f0 = fast_exp2((m - ms) * kLog2e), f1 = fast_exp2((m1 - ms) * kLog2e);
    const float L = lw * f0 + l1 * f1, inv = L > 0.f ? 1.0f / L : 0.f;
    f0 *= inv;
    f1 *= inv;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
            const float4 o = *reinterpret_cast<const float4*>(ebuf + (db * 4 + jq) * 256 + lane * 4);
            oacc[db][4 * jq] = oacc[db][4 * jq] * f0 + o.x * f1;
            oacc[db][4 * jq + 1] = oacc[db][4 * jq + 1] * f0 + o.y * f1;
            oacc[db][4 * jq + 2] = oacc[db][4 * jq + 2] * f0 + o.z * f1;
            oacc[db][4 * jq + 3] = oacc[db][4 * jq + 3] * f0 + o.w * f1;
        }
    if (g == 0 && qok) a.lse[(long)bh * a.st_bhs + tq] = L > 0.f ? mt + logf(L) : -INFINITY;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    acc_to_lds_rows<DH>(oacc, ebuf, lane);              // the wave's own block: LDS operations of one wave complete in order
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const long EE = (long)a.H * DH;
#pragma unroll
    for (int p = lane; p < 32 * DH / 8; p += 64) {
        const int row = p / (DH / 8), col = (p % (DH / 8)) * 8;
        if (qw + row >= T_) break;
        float v[8];
        *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(ebuf + row * EPI_LD + col);
        *reinterpret_cast<float4*>(v + 4) = *reinterpret_cast<const float4*>(ebuf + row * EPI_LD + col + 4);
        *reinterpret_cast<uint4*>(reinterpret_cast<T*>(a.o) + ((long)(qw + row) * a.B + b) * EE + (long)h * DH + col) = pack8<T>(v);
    }
}

// ------------------------------------------------------------------------------------------------
// dQ of 32 * QB queries, and their delta = rowsum(dO * O) for the dK / dV kernel that follows on the stream: blocks of 32
// queries, each by one of four waves (QB = 4) or by two that take one half of every key tile and add their sums at the end (QB = 2).
// K and V tiles lie in rings of 72 or 80 KB at most, so that two workgroups (three at head dimension 64) share a CU: the waves of a
// SIMD belong to different workgroups, and no barrier keeps them in step.
// A wave's work on a tile is one straight line of three rows of MFMAs, each beside the vector operations that it leaves the issue slots
// for and the LDS fetches of those a few MFMAs later: V dO^T | exponentials; the NEXT tile's K Q^T | dS; dQ += K^T dS.
// What bounds it: the waits between a tile's loads, LDS fetches and MFMAs that two waves a SIMD cover only in part (24 MFMAs of 32
// clocks and about 900 clocks of issue in 1750 per block of 32 x 32, 96 heads of 128); QB = 4 has three tiles of 32 keys under way where QB = 2
// has one of 64, and pulls half the bytes.
// Measured (fp16, causal, 2048 positions, us; before: eight waves on one ring of 128 KB, phases in step): 40 heads of 128 90 -> 76, 96 of
// 128 206 -> 168, 16 of 128 49 -> 41 (blocks of 64), 12 of 64 30 -> 25, 40 of 80 66 -> 58, 40 of 96 72 -> 63; 64 of 64 at 1024 24.1 -> 23.8, 300 of
// 64 at 256 22.2 -> 16.7; 40 of 128, 512 after 1536 60 -> 47 (32 queries a workgroup).  Two of the old workgroups on a CU at 64 (128 registers, spills): 24 -> 38.
// ------------------------------------------------------------------------------------------------
template <typename T, int DH, int QB>
__global__ __launch_bounds__(256, DH <= 64 ? 3 : 2) void attn_dq_long_kernel(AttnArgs a) {
    typedef Elem<T> E;
    constexpr int NDB = (DH + 31) / 32, NKS = DH / 16, NPV = 2 * NDB, PITCH = tile_pitch<DH>(), CPR = PITCH / 8;
    constexpr int KH = 4 / QB, KT = 32 * KH, TILE = KT * PITCH * 2;     // waves that share a query block's keys; (bytes)
    constexpr int AHEAD = QB == 4 ? 3 : 1, RK = AHEAD + 2, RV = AHEAD + 1, VRING = RK * TILE;      // tiles under way; slots
    constexpr int NLD = KT * CPR / 256;                     // loads per K or V tile and lane
    constexpr int W = DH == 128 || DH == 64 ? 6 : 9;        // fragments under way
    constexpr bool FOLD = DH > 64;                          // V dO^T starts at -delta (16 registers, which 64 does not have)
    constexpr int EPI_LD = NDB * 32 + 4;
    constexpr int RING_BYTES = (RK + RV) * TILE, EPI_BYTES = QB * 32 * EPI_LD * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[RING_BYTES > EPI_BYTES ? RING_BYTES : EPI_BYTES];

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, li = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), qb = wave % QB, kh = wave / QB;
    int bh, blk;
    if (!xcd_map_causal(a.B * a.H, (a.T + 32 * QB - 1) / (32 * QB), bh, blk)) return;
    const int b = bh / a.H, h = bh - b * a.H;
    const int T_ = a.T, P = a.P, S = a.P + a.T;
    const long EE = (long)a.H * DH;
    const int q0 = ((T_ + 32 * QB - 1) / (32 * QB) - 1 - blk) * (32 * QB);      // the blocks with the longest key range start first
    const int qw = q0 + 32 * qb, tq = qw + li, tr_row = min(tq, T_ - 1);
    const bool qok = tq < T_;
    const int nt = (P + min(T_, q0 + 32 * QB) + KT - 1) / KT;    // tiles of the workgroup
    // those in which the wave's block of 32 keys has one that its queries see: what lies beyond is not multiplied, not even by zero
    const int nw = qw < T_ ? max(0, P + min(T_, qw + 32) - kh * 32 + KT - 1) / KT : 0;

    // the lane's chunk of a tile's first rows and that of row S - 1 (the swizzle repeats every 16 rows: the same column in each load)
    const int lr = tid / CPR, lc = (tid % CPR) ^ swz16<PITCH>(lr);
    const unsigned koff = (unsigned)(lr * DH * 2 + lc * 16), klast = (unsigned)((S - 1) * DH * 2 + lc * 16);
    const bool chunk = DH == PITCH || lc < DH / 8;
    const char* Kb = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.kc) + (long)bh * a.cache_rows * DH));
    const char* Vb = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.vc) + (long)bh * a.cache_rows * DH));
    const unsigned lds0 = lds_addr(smem) + wave * 1024;
    // tile t of K or V to where it belongs; rows at or past S are clamped to row S - 1: finite data, and every such key is masked
    auto issue = [&](const char* base, unsigned dst, int tile) __attribute__((always_inline)) {
        const unsigned row = (unsigned)(tile * KT) * (DH * 2);
#pragma unroll
        for (int i = 0; i < NLD; ++i)
            if (chunk) dma16_saddr_lds(min(row + (unsigned)(i * (256 / CPR) * DH * 2) + koff, klast), base, lds0 + dst + i * 4096);
    };
    issue(Kb, 0, 0);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
        issue(Vb, VRING + i * TILE, i);
        issue(Kb, (i + 1) * TILE, i + 1);
    }

    typename E::opnd_t qreg[NKS], doreg[NKS];
    const long orow = ((long)tr_row * a.B + b) * EE + (long)h * DH;
    load_row_operands<T, DH>(qreg, reinterpret_cast<const T*>(a.q) + (long)bh * a.q_bhs + (long)tr_row * DH, qok, g);
    load_row_operands<T, DH>(doreg, reinterpret_cast<const T*>(a.d_o) + orow, qok, g);
    float delta = 0.f;
    {
        typename E::opnd_t oreg[NKS];
        load_row_operands<T, DH>(oreg, reinterpret_cast<const T*>(a.o) + orow, qok, g);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const float8v x = __builtin_convertvector(__builtin_bit_cast(vec8_t<T>, oreg[ks]), float8v) *
                              __builtin_convertvector(__builtin_bit_cast(vec8_t<T>, doreg[ks]), float8v);
#pragma unroll
            for (int e = 0; e < 8; ++e) delta += x[e];
        }
        delta += __shfl_xor(delta, 32, 64);
        if (kh == 0 && g == 0 && qok) a.delta[(long)bh * a.st_bhs + tq] = delta;
    }
    const float lneg = qok ? -a.lse[(long)bh * a.st_bhs + tq] * kLog2e : 0.f;

    // LDS addresses of the lane's fetches, which go round the rings: km in the next tile's K, vm in this one's V, tr in this one's K
    unsigned km[NKS], tr[NDB][2];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) km[ks] = lds_addr(smem) + km_offset<T, PITCH>(kh * 32 + li, ks * 16, lane) * 2;
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
        int o0, o1;
        tr_offsets<T, PITCH, true>(kh * 32, db * 32, lane, o0, o1);
        tr[db][0] = lds_addr(smem) + o0 * 2;
        tr[db][1] = lds_addr(smem) + o1 * 2;
    }
    auto km_from = [&](unsigned off, int ks) __attribute__((always_inline)) {
        typedef unsigned uint4v __attribute__((ext_vector_type(4)));
        return __builtin_bit_cast(uint4, *(__attribute__((address_space(3))) const uint4v*)(km[ks] + off));
    };
    auto transposed = [&](unsigned off, int i) __attribute__((always_inline)) {
        typedef __attribute__((address_space(3))) short4v* P3;
        const unsigned o = off + i / NDB * 16 * PITCH * 2;
        const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((P3)(tr[i % NDB][0] + o)));
        const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((P3)(tr[i % NDB][1] + o)));
        return make_uint4(lo.x, lo.y, hi.x, hi.y);
    };

    float16v dq[NDB], s, x, d, minus_delta;     // s: scores of the next tile; x: those of this one, then P and dS
#pragma unroll
    for (int r = 0; r < 16; ++r) minus_delta[r] = -delta;
    const float16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int db = 0; db < NDB; ++db) dq[db] = zero;
    auto barrier = [&](auto n) __attribute__((always_inline)) {
        wait_vmcnt<decltype(n)::value>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    barrier(std::integral_constant<int, 0>());
    s = zero;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) s = E::mfma(km_from(0, ks), qreg[ks], s);

    unsigned kslot = 0, vslot = 0;      // byte offsets of tile t's slots
    auto next_slot = [&](unsigned slot, unsigned n) __attribute__((always_inline)) { return slot == (n - 1) * TILE ? 0 : slot + TILE; };
    auto next_loads = [&](int t) __attribute__((always_inline)) {
        // this wave's loads of K(t + 1) and V(t) have landed, and its reads of the tiles before t are back
        if (t) barrier(std::integral_constant<int, (AHEAD - 1) * 2 * NLD>());
        issue(Vb, VRING + (vslot ? vslot : RV * TILE) - TILE, t + AHEAD);
        issue(Kb, (kslot ? kslot : RK * TILE) - TILE, t + AHEAD + 1);
    };
    for (int t = 0; t < nw; ++t) {
        next_loads(t);
        const unsigned knext = next_slot(kslot, RK);
        const int key0 = t * KT + kh * 32;
        x = s;
        if (key0 + 31 > P + qw) {       // wave-uniform: the block touches the causal boundary
            const int end = P + tq - key0 - acc_row(0, g);
#pragma unroll
            for (int j = 0; j < 16; ++j)
                if (acc_row(j, 0) > end) x[j] = -INFINITY;
        }
        // the fragments of the tile's NKS + NKS + NPV MFMAs in their order, W of them under way
        constexpr int NF = 2 * NKS + NPV;
        uint4 f[NF];
        auto fetch = [&](int i) __attribute__((always_inline)) {
            if (i < NKS) f[i] = km_from(VRING + vslot, i);
            else if (i < 2 * NKS) f[i] = km_from(knext, i - NKS);
            else if (i < NF) f[i] = transposed(kslot, i - 2 * NKS);
        };
#pragma unroll
        for (int i = 0; i < W; ++i) fetch(i);
        unsigned dw[8];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < NKS; ++k) {
            d = E::mfma(f[k], doreg[k], k == 0 ? (FOLD ? minus_delta : zero) : d);
            fetch(k + W);
#pragma unroll
            for (int j = k * 16 / NKS; j < (k + 1) * 16 / NKS; ++j) {
                x[j] = fast_exp2(fmaf(x[j], kLog2e, lneg));
                asm volatile("" : "+v"(x[j]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int k = 0; k < NKS; ++k) {
            s = E::mfma(f[NKS + k], qreg[k], k == 0 ? zero : s);
            fetch(NKS + k + W);
            if (k > 0) {                // (the last of V dO^T is under way beside the first)
#pragma unroll
                for (int j = (k - 1) * 16 / (NKS - 1); j < k * 16 / (NKS - 1); ++j) {
                    x[j] *= FOLD ? d[j] : d[j] - delta;
                    if (j & 1) {
                        dw[j / 2] = pack2<T>(x[j - 1], x[j]);
                        asm volatile("" : "+v"(dw[j / 2]));
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const uint4 ds[2] = {make_uint4(dw[0], dw[1], dw[2], dw[3]), make_uint4(dw[4], dw[5], dw[6], dw[7])};
#pragma unroll
        for (int i = 0; i < NPV; ++i) {
            dq[i % NDB] = E::mfma(f[2 * NKS + i], ds[i / NDB], dq[i % NDB]);
            fetch(2 * NKS + i + W);
            __builtin_amdgcn_sched_barrier(0);
        }
        kslot = knext;
        vslot = next_slot(vslot, RV);
    }
    for (int t = nw; t < nt; ++t) {     // the other waves' tiles: this one's share of their loads
        next_loads(t);
        kslot = next_slot(kslot, RK);
        vslot = next_slot(vslot, RV);
    }
    wait_vmcnt<0>();            // (the loads past the last tile)
    __syncthreads();            // every wave is done with the rings

    float* ebuf = reinterpret_cast<float*>(smem) + qb * 32 * EPI_LD;
    if constexpr (KH > 1) {
        if (kh == 1) {
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int jq = 0; jq < 4; ++jq)
                    *reinterpret_cast<float4*>(ebuf + (db * 4 + jq) * 256 + lane * 4) =
                        make_float4(dq[db][4 * jq], dq[db][4 * jq + 1], dq[db][4 * jq + 2], dq[db][4 * jq + 3]);
        }
        __syncthreads();
        if (kh == 1) return;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int jq = 0; jq < 4; ++jq) {
                const float4 o = *reinterpret_cast<const float4*>(ebuf + (db * 4 + jq) * 256 + lane * 4);
                dq[db][4 * jq] += o.x;
                dq[db][4 * jq + 1] += o.y;
                dq[db][4 * jq + 2] += o.z;
                dq[db][4 * jq + 3] += o.w;
            }
    }
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) dq[db][r] *= a.qscale;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    acc_to_lds_rows<DH>(dq, ebuf, lane);                // the wave's own block: LDS operations of one wave complete in order
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int p = lane; p < 32 * DH / 8; p += 64) {
        const int row = p / (DH / 8), col = (p % (DH / 8)) * 8;
        if (qw + row >= T_) break;
        float v[8];
        *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(ebuf + row * EPI_LD + col);
        *reinterpret_cast<float4*>(v + 4) = *reinterpret_cast<const float4*>(ebuf + row * EPI_LD + col + 4);
        *reinterpret_cast<uint4*>(reinterpret_cast<T*>(a.dqkv) + ((long)(qw + row) * a.B + b) * (3 * EE) + (long)h * 3 * DH + col) = pack8<T>(v);
    }
}

// ------------------------------------------------------------------------------------------------
// The same by eight waves for 128 queries: four blocks of 32, each by two waves that take one half of every key tile, tiles of 128
// keys, one workgroup to a CU above head dimension 64.  For 289 to 512 workgroups of long sequences (dq_form): the longest block then sets the
// time, and here two waves share its walk over the keys, with a CU to themselves.  us, this form / the better of the two above, causal,
// 2048 positions: 32 heads of 64 35.2 / 37.8, 25 of 80 44.6 / 46.1, 32 of 80 48.6 / 51.0, 32 of 96 51.6 / 54.1, 20 of 128 52.3 / 53.3;
// 24 of 96 at 1536 (288) 32.0 / 32.9; outside: 36 of 80 64.7 / 56.2, 16 of 128 48.7 / 40.9, 64 of 80 at 1024 33.5 / 31.6.
// ------------------------------------------------------------------------------------------------
template <typename T, int DH>
__global__ __launch_bounds__(512) void attn_dq_pairs_kernel(AttnArgs a) {
    typedef Elem<T> E;
    constexpr int NDB = (DH + 31) / 32, NKS = DH / 16, PITCH = tile_pitch<DH>(), CPR = PITCH / 8;
    constexpr int NB = 2;                                   // 32-key blocks of a tile per wave
    constexpr int KT = 64 * NB, TILE = KT * PITCH, STAGE = 2 * TILE;
    constexpr int NLD = KT * CPR / 512;                     // loads per K or V tile and lane
    constexpr int EPI_LD = NDB * 32 + 4;
    constexpr int RING_BYTES = 2 * STAGE * 2, EPI_BYTES = 4 * 32 * EPI_LD * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[RING_BYTES > EPI_BYTES ? RING_BYTES : EPI_BYTES];
    T* ring = reinterpret_cast<T*>(smem);

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, li = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), qb = wave & 3, kh = wave >> 2;
    int bh, blk;
    if (!xcd_map(a.B * a.H, bh, blk)) return;
    const int b = bh / a.H, h = bh - b * a.H;
    const int T_ = a.T, P = a.P, S = a.P + a.T;
    const long EE = (long)a.H * DH;
    const int q0 = ((T_ + 127) / 128 - 1 - blk) * 128;      // the blocks with the longest key range start first
    const int qw = q0 + 32 * qb, tq = qw + li, tr = min(tq, T_ - 1);
    const bool qok = tq < T_;
    const int nt = (P + min(T_, q0 + 128) + KT - 1) / KT;   // tiles of the workgroup
    const int key_end = qw < T_ ? P + min(T_, qw + 32) : 0; // keys this wave's queries see

    unsigned koff[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int p = i * 512 + tid, r = p / CPR, lc = (p % CPR) ^ swz16<PITCH>(r);
        koff[i] = lc < DH / 8 ? (unsigned)(r * DH * 2 + lc * 16) : kNoChunk;
    }
    const char* Kb = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.kc) + (long)bh * a.cache_rows * DH));
    const char* Vb = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.vc) + (long)bh * a.cache_rows * DH));
    const unsigned lds0 = lds_addr(smem) + wave * 1024;
    auto issue = [&](int stage, int tile) {                 // (rows at or past S as in the forward)
        const unsigned dst = lds0 + (unsigned)(stage * STAGE * 2);
        const int row0 = tile * KT;
#pragma unroll
        for (int which = 0; which < 2; ++which) {
            const char* base = which ? Vb : Kb;
            if (row0 + KT <= S) {
                const char* sb = base + (long)row0 * (DH * 2);
#pragma unroll
                for (int i = 0; i < NLD; ++i) load_chunk_lds<DH>(koff[i], sb, dst + which * TILE * 2 + i * 8192);
            } else {
#pragma unroll
                for (int i = 0; i < NLD; ++i) {
                    const int p = i * 512 + tid, r = p / CPR, lc = (p % CPR) ^ swz16<PITCH>(r);
                    const unsigned off = lc < DH / 8 ? (unsigned)(min(row0 + r, S - 1) * DH * 2 + lc * 16) : kNoChunk;
                    load_chunk_lds<DH>(off, base, dst + which * TILE * 2 + i * 8192);
                }
            }
        }
    };
    issue(0, 0);

    typename E::opnd_t qreg[NKS], doreg[NKS];
    const long orow = ((long)tr * a.B + b) * EE + (long)h * DH;
    load_row_operands<T, DH>(qreg, reinterpret_cast<const T*>(a.q) + (long)bh * a.q_bhs + (long)tr * DH, qok, g);
    load_row_operands<T, DH>(doreg, reinterpret_cast<const T*>(a.d_o) + orow, qok, g);
    float delta = 0.f;
    {
        typename E::opnd_t oreg[NKS];
        load_row_operands<T, DH>(oreg, reinterpret_cast<const T*>(a.o) + orow, qok, g);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const float8v x = __builtin_convertvector(__builtin_bit_cast(vec8_t<T>, oreg[ks]), float8v) *
                              __builtin_convertvector(__builtin_bit_cast(vec8_t<T>, doreg[ks]), float8v);
#pragma unroll
            for (int e = 0; e < 8; ++e) delta += x[e];
        }
        delta += __shfl_xor(delta, 32, 64);
        if (kh == 0 && g == 0 && qok) a.delta[(long)bh * a.st_bhs + tq] = delta;
    }
    const float lneg = qok ? -a.lse[(long)bh * a.st_bhs + tq] * kLog2e : 0.f;

    int okm[NKS], otr[NDB][2];          // element offsets of the lane's fetches inside a K tile, its first block
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) okm[ks] = km_offset<T, PITCH>(kh * 32 * NB + li, ks * 16, lane);
#pragma unroll
    for (int db = 0; db < NDB; ++db) tr_offsets<T, PITCH, true>(kh * 32 * NB, db * 32, lane, otr[db][0], otr[db][1]);

    float16v dq[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) dq[db][r] = 0.f;

    auto step = [&](auto sc, int t) __attribute__((always_inline)) {
        constexpr int st = decltype(sc)::value;
        wait_vmcnt<0>();                    // this wave's part of tile t has landed
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // and its reads of tile t - 1 are back
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (t + 1 < nt) issue(st ^ 1, t + 1);
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const int key0 = t * KT + (kh * NB + n) * 32, so = st * STAGE + n * 32 * PITCH;
            if (key0 >= key_end) break;     // wave-uniform
            typename E::opnd_t kf[NKS], vf[NKS];
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) kf[ks] = load_km<T>(ring + so + okm[ks]);
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) vf[ks] = load_km<T>(ring + so + TILE + okm[ks]);
            __builtin_amdgcn_sched_barrier(0);
            float16v s, d;
#pragma unroll
            for (int r = 0; r < 16; ++r) { s[r] = 0.f; d[r] = 0.f; }
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) s = E::mfma(kf[ks], qreg[ks], s);
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) d = E::mfma(vf[ks], doreg[ks], d);
            __builtin_amdgcn_sched_barrier(0);
            uint4 kt[2][NDB];
#pragma unroll
            for (int hs = 0; hs < 2; ++hs)
#pragma unroll
                for (int db = 0; db < NDB; ++db)
                    kt[hs][db] = load_tr<T>(ring + so + otr[db][0] + hs * 16 * PITCH, ring + so + otr[db][1] + hs * 16 * PITCH);
            __builtin_amdgcn_sched_barrier(0);
            if (key0 + 31 > P + qw) {       // wave-uniform: the block touches the causal boundary
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    if (key0 + acc_row(j, g) > P + tq) s[j] = -INFINITY;
            }
            float8v e0, e1;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                e0[j] = fast_exp2(fmaf(s[j], kLog2e, lneg)) * (d[j] - delta);
                e1[j] = fast_exp2(fmaf(s[j + 8], kLog2e, lneg)) * (d[j + 8] - delta);
            }
            const uint4 p[2] = {pack8v<T>(e0), pack8v<T>(e1)};
#pragma unroll
            for (int hs = 0; hs < 2; ++hs)
#pragma unroll
                for (int db = 0; db < NDB; ++db) dq[db] = E::mfma(kt[hs][db], p[hs], dq[db]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int t = 0; t < nt; t += 2) {
        step(std::integral_constant<int, 0>(), t);
        if (t + 1 < nt) step(std::integral_constant<int, 1>(), t + 1);
    }
    __syncthreads();            // every wave is done with the ring

    float* ebuf = reinterpret_cast<float*>(smem) + qb * 32 * EPI_LD;
    if (kh == 1) {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int jq = 0; jq < 4; ++jq)
                *reinterpret_cast<float4*>(ebuf + (db * 4 + jq) * 256 + lane * 4) =
                    make_float4(dq[db][4 * jq], dq[db][4 * jq + 1], dq[db][4 * jq + 2], dq[db][4 * jq + 3]);
    }
    __syncthreads();
    if (kh == 1) return;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
            const float4 o = *reinterpret_cast<const float4*>(ebuf + (db * 4 + jq) * 256 + lane * 4);
            dq[db][4 * jq] = (dq[db][4 * jq] + o.x) * a.qscale;
            dq[db][4 * jq + 1] = (dq[db][4 * jq + 1] + o.y) * a.qscale;
            dq[db][4 * jq + 2] = (dq[db][4 * jq + 2] + o.z) * a.qscale;
            dq[db][4 * jq + 3] = (dq[db][4 * jq + 3] + o.w) * a.qscale;
        }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    acc_to_lds_rows<DH>(dq, ebuf, lane);                // the wave's own block: LDS operations of one wave complete in order
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int p = lane; p < 32 * DH / 8; p += 64) {
        const int row = p / (DH / 8), col = (p % (DH / 8)) * 8;
        if (qw + row >= T_) break;
        float v[8];
        *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(ebuf + row * EPI_LD + col);
        *reinterpret_cast<float4*>(v + 4) = *reinterpret_cast<const float4*>(ebuf + row * EPI_LD + col + 4);
        *reinterpret_cast<uint4*>(reinterpret_cast<T*>(a.dqkv) + ((long)(qw + row) * a.B + b) * (3 * EE) + (long)h * 3 * DH + col) = pack8<T>(v);
    }
}

template <typename T> static void dq_pairs(int hd, const AttnArgs& a, hipStream_t s) {
    const unsigned grid = xcd_grid(a.B * a.H, (a.T + 127) / 128);
    switch (hd) {
    case 64: attn_dq_pairs_kernel<T, 64><<<grid, 512, 0, s>>>(a); break;
    case 80: attn_dq_pairs_kernel<T, 80><<<grid, 512, 0, s>>>(a); break;
    case 96: attn_dq_pairs_kernel<T, 96><<<grid, 512, 0, s>>>(a); break;
    default: attn_dq_pairs_kernel<T, 128><<<grid, 512, 0, s>>>(a); break;
    }
}
template <typename T, int QB> static void dq_long(int hd, const AttnArgs& a, hipStream_t s) {
    const unsigned grid = xcd_grid(a.B * a.H, (a.T + 32 * QB - 1) / (32 * QB));
    switch (hd) {
    case 64: attn_dq_long_kernel<T, 64, QB><<<grid, 256, 0, s>>>(a); break;
    case 80: attn_dq_long_kernel<T, 80, QB><<<grid, 256, 0, s>>>(a); break;
    case 96: attn_dq_long_kernel<T, 96, QB><<<grid, 256, 0, s>>>(a); break;
    default: attn_dq_long_kernel<T, 128, QB><<<grid, 256, 0, s>>>(a); break;
    }
}
// Blocks of 64 queries, of 128 or, eight waves each, of 128.  With w blocks of 128 that a chip of two (three at head dimension 64)
// to a CU runs at once, what counts is whether the longest one's walk over the keys ends after all others' work: then two waves to a
// block of 32 queries are better than one, by blocks of 64 or, for long sequences, by the eight-wave form.  Few heads, 512 to 3072 positions, 0
// to 1024 of context, 270 to 900 blocks: the form taken is within 0.7 % of the best of the three in the mean, 14 % at worst (120 of 64 at
// 512: 18.5 / 16.2); us, 64 / 128 / eight waves: 16 of 128 at 2048 (w = 256) 41 / 52 / 49, 20 of 80 (320) 39.5 / 45.5 / 39.0, 36 of 80
// (576) 62 / 56 / 65; 40 of 96 at 1024 (320) 26.0 / 29.0 / 26.4, 60 (480) 35.6 / 32.8 / 34.2, 40 after 512 43.5 / 41.0 / 41.9; 160 of 128 at 256 (320)
// 25.6 / 19.4 / 26.1; 48 of 64 at 2048 (768) 50.8 / 52.0 / 54.2, at 512 less to share: 120 (480) 18.5 / 16.2 / 18.8.
// Short calls of many heads take blocks of 128 that no second row fills: 600 of 128, 64 queries 20.9 / 19.2, 96 queries 33.4 / 25.0.
enum DqForm { kDq64, kDq128, kDqPairs };
static DqForm dq_form(int head_dim, long pairs, int T, int P) {
    const long w = pairs * ((T + 127) / 128);
    const bool uneven = T >= 1400 && 2L * P <= T;
    if (uneven && w > 288 && w <= (head_dim < 128 ? 512 : 384)) return kDqPairs;
    if (head_dim == 64) return w >= (uneven ? 800 : 512) ? kDq128 : kDq64;
    const bool longest = T >= 700 && w * (2L * P + T) <= (head_dim < 128 ? 384L : 340L) * ((long)P + T);
    return w > 256 && !longest ? kDq128 : kDq64;
}
void launch_attn_dq_long(int dtype, int head_dim, const AttnArgs& a, hipStream_t s) {
    switch (dq_form(head_dim, (long)a.B * a.H, a.T, a.P)) {
    case kDqPairs: dtype == TP_F16 ? dq_pairs<f16>(head_dim, a, s) : dq_pairs<bf16>(head_dim, a, s); break;
    case kDq128: dtype == TP_F16 ? dq_long<f16, 4>(head_dim, a, s) : dq_long<bf16, 4>(head_dim, a, s); break;
    default: dtype == TP_F16 ? dq_long<f16, 2>(head_dim, a, s) : dq_long<bf16, 2>(head_dim, a, s); break;
    }
}

// ------------------------------------------------------------------------------------------------
// dK / dV of 128 keys: four blocks of 32, each by two waves that take one half of every tile of 64 queries and exchange their
// sums at the end (one half finishes dK, the other dV).  Q, dO, lse and delta of a tile are loaded once for all eight waves.
// Accumulators of both (128 registers at head dimension 128) leave no room for the K and V rows beside the fragments: there
// they lie in LDS (64 KB beside the ring's 64) and are read again per block, below they stay in registers.
// SUFFIX: the keys of a slice against all later query positions (tp_attn_suffix_dkdv), everything indexed by position; else all
// keys of the cache against the slice's queries, with gradient caches of type T (tp_attn_prefix_bwd).
// Causal, 2048 positions: 40 heads of 128 167 -> 105 us, 96 of 128 411 -> 236; 40 of 128 at 512 25.6 -> 19.9; with gradient caches,
// 512 queries after 1536, dQ included 175 -> 118.
// ------------------------------------------------------------------------------------------------
template <typename T, int DH, bool SUFFIX>
__global__ __launch_bounds__(512) void attn_dkdv_long_kernel(AttnKeysArgs a) {
    typedef Elem<T> E;
    constexpr int NDB = (DH + 31) / 32, NKS = DH / 16, PITCH = tile_pitch<DH>(), CPR = PITCH / 8;
    constexpr bool KV_LDS = DH > 96;
    constexpr int QT = 64, TILE = QT * PITCH, STAGE = 2 * TILE, KV = 128 * PITCH;
    constexpr int NLD = QT * CPR / 512;                     // loads per Q or dO tile and lane
    constexpr int EPI_LD = NDB * 32 + 4, PART = 32 * EPI_LD;
    constexpr int RING_BYTES = 2 * STAGE * 2 + (KV_LDS ? 2 * KV * 2 : 0), EPI_BYTES = 8 * PART * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[RING_BYTES > EPI_BYTES ? RING_BYTES : EPI_BYTES];
    __shared__ __attribute__((aligned(16))) float stat[2][2][QT];       // [stage][lse, delta][query]
    T* ring = reinterpret_cast<T*>(smem);
    T* kv = ring + 2 * STAGE;

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, li = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kb = wave & 3, qh = wave >> 2;
    int bh, blk;
    if (!xcd_map(a.B * a.H, bh, blk)) return;
    const int b = bh / a.H, h = bh - b * a.H;
    const long EE = (long)a.H * DH;
    // the first keys, which the most queries see, start first
    if constexpr (!SUFFIX)
        if (a.grad_rows > a.key_end && !grad_rows_beyond<T, DH, 128, 512>(a, bh, a.key0 + blk * 128, a.key_end, tid)) return;
    const int key0 = a.key0 + blk * 128, kw = key0 + 32 * kb, key = kw + li, last_key = a.key_end - 1;
    const int q_beg = max(0, key0 - a.q_pos), nt = max(0, (a.nq - q_beg + QT - 1) / QT);

    unsigned qoff[NLD], dooff[NLD];
    const unsigned ldo = (unsigned)((long)a.B * EE * 2);
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int p = i * 512 + tid, r = p / CPR, lc = (p % CPR) ^ swz16<PITCH>(r);
        qoff[i] = lc < DH / 8 ? (unsigned)(r * DH * 2 + lc * 16) : kNoChunk;
        dooff[i] = lc < DH / 8 ? (unsigned)(r * ldo + lc * 16) : kNoChunk;
    }
    const char* Qb = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.q) + (long)bh * a.q_bhs));
    const char* dOb = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.d_o) + (long)b * EE + (long)h * DH));
    const float* stat_src = (wave & 1 ? a.delta : a.lse) + (long)bh * a.st_bhs;
    const unsigned lds0 = lds_addr(smem) + wave * 1024;
    auto issue = [&](int stage, int tile) {
        const unsigned dst = lds0 + (unsigned)(stage * STAGE * 2);
        const int row0 = q_beg + tile * QT;
        if (row0 + QT <= a.nq) {
            const char *sq = Qb + (long)row0 * (DH * 2), *so = dOb + (long)row0 * ldo;
#pragma unroll
            for (int i = 0; i < NLD; ++i) load_chunk_lds<DH>(qoff[i], sq, dst + i * 8192);
#pragma unroll
            for (int i = 0; i < NLD; ++i) load_chunk_lds<DH>(dooff[i], so, dst + TILE * 2 + i * 8192);
        } else {            // rows past the last query are clamped to it: finite data, and their P is zero
            const char *sq = Qb + (long)row0 * (DH * 2), *so = dOb + (long)row0 * ldo;
            const int last = a.nq - 1 - row0;
#pragma unroll
            for (int i = 0; i < NLD; ++i) {
                const int p = i * 512 + tid, r = p / CPR, lc = (p % CPR) ^ swz16<PITCH>(r);
                load_chunk_lds<DH>(lc < DH / 8 ? (unsigned)(min(r, last) * DH * 2 + lc * 16) : kNoChunk, sq, dst + i * 8192);
            }
#pragma unroll
            for (int i = 0; i < NLD; ++i) {
                const int p = i * 512 + tid, r = p / CPR, lc = (p % CPR) ^ swz16<PITCH>(r);
                load_chunk_lds<DH>(lc < DH / 8 ? (unsigned)(min(r, last) * ldo + lc * 16) : kNoChunk, so, dst + TILE * 2 + i * 8192);
            }
        }
        if (wave < 2) dma4(stat_src + min(row0 + lane, a.nq - 1), lds_addr(&stat[stage][wave][0]));
    };
    typename E::opnd_t kreg[KV_LDS ? 1 : NKS], vreg[KV_LDS ? 1 : NKS];
    const T* Kb = reinterpret_cast<const T*>(a.kc) + (long)bh * a.cache_rows * DH;
    const T* Vb = reinterpret_cast<const T*>(a.vc) + (long)bh * a.cache_rows * DH;
    if constexpr (KV_LDS) {
        const unsigned dst = lds_addr(kv) + wave * 1024;
#pragma unroll
        for (int i = 0; i < 128 * CPR / 512; ++i) {
            const int p = i * 512 + tid, r = p / CPR, lc = (p % CPR) ^ swz16<PITCH>(r);
            const unsigned off = (unsigned)(min(r, last_key - key0) * DH * 2 + lc * 16);
            dma16_saddr_lds(off, uniform_ptr(Kb + (long)key0 * DH), dst + i * 8192);
            dma16_saddr_lds(off, uniform_ptr(Vb + (long)key0 * DH), dst + KV * 2 + i * 8192);
        }
    } else {
        load_row_operands<T, DH>(kreg, Kb + (long)min(key, last_key) * DH, key <= last_key, g);
        load_row_operands<T, DH>(vreg, Vb + (long)min(key, last_key) * DH, key <= last_key, g);
    }
    if (nt > 0) issue(0, 0);

    int okm[NKS], otr[NDB][2];          // element offsets of the lane's fetches inside a Q tile
    const T* krows = kv + (kb - qh) * 32 * PITCH;           // the same of its keys' rows (the swizzle repeats every 16)
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) okm[ks] = km_offset<T, PITCH>(qh * 32 + li, ks * 16, lane);
#pragma unroll
    for (int db = 0; db < NDB; ++db) tr_offsets<T, PITCH, true>(qh * 32, db * 32, lane, otr[db][0], otr[db][1]);

    float16v dk[NDB], dv[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) { dk[db][r] = 0.f; dv[db][r] = 0.f; }

    auto step = [&](auto sc, int t) __attribute__((always_inline)) {
        constexpr int st = decltype(sc)::value, so = st * STAGE;
        wait_vmcnt<0>();                    // this wave's part of tile t has landed
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // and its reads of tile t - 1 are back
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (t + 1 < nt) issue(st ^ 1, t + 1);
        const int t0 = q_beg + t * QT + qh * 32;                // the wave's first query of the tile
        if (t0 >= a.nq || a.q_pos + t0 + 31 < kw) return;       // wave-uniform: none of them, or none that sees these keys
        // four k-steps' fragments at a time where both operands come out of LDS (registers)
        constexpr int KG = KV_LDS ? 4 : NKS;
        auto product = [&](int which) __attribute__((always_inline)) {      // 0: Q K^T, 1: dO V^T
            float16v x;
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = 0.f;
#pragma unroll
            for (int k0 = 0; k0 < NKS; k0 += KG) {
                typename E::opnd_t qf[KG], kf[KG];
#pragma unroll
                for (int ks = 0; ks < KG; ++ks) {
                    qf[ks] = load_km<T>(ring + so + which * TILE + okm[k0 + ks]);
                    if constexpr (KV_LDS) kf[ks] = load_km<T>(krows + which * KV + okm[k0 + ks]);
                    else kf[ks] = which ? vreg[k0 + ks] : kreg[k0 + ks];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int ks = 0; ks < KG; ++ks) x = E::mfma(qf[ks], kf[ks], x);
            }
            return x;
        };
        float16v s = product(0);
        const float16v d = product(1);
        __builtin_amdgcn_sched_barrier(0);
        if (a.q_pos + t0 < kw + 31 || t0 + 32 > a.nq) {         // wave-uniform: the causal boundary, or the last queries
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int q = t0 + acc_row(j, g);
                if (q >= a.nq || key > a.q_pos + q) s[j] = -INFINITY;
            }
        }
        float8v p0, p1, e0, e1;
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
            const float4v l4 = *reinterpret_cast<const float4v*>(&stat[st][0][qh * 32 + 8 * jq + 4 * g]);
            const float4v d4 = *reinterpret_cast<const float4v*>(&stat[st][1][qh * 32 + 8 * jq + 4 * g]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = 4 * jq + e;
                const float p = fast_exp2((s[j] - l4[e]) * kLog2e), ds = p * (d[j] - d4[e]);
                if (j < 8) { p0[j] = p; e0[j] = ds; } else { p1[j - 8] = p; e1[j - 8] = ds; }
            }
        }
        const uint4 pp[2] = {pack8v<T>(p0), pack8v<T>(p1)}, ds[2] = {pack8v<T>(e0), pack8v<T>(e1)};
        __builtin_amdgcn_sched_barrier(0);
        uint4 tf[2][NDB];
#pragma unroll
        for (int hs = 0; hs < 2; ++hs)
#pragma unroll
            for (int db = 0; db < NDB; ++db)
                tf[hs][db] = load_tr<T>(ring + so + TILE + otr[db][0] + hs * 16 * PITCH, ring + so + TILE + otr[db][1] + hs * 16 * PITCH);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int hs = 0; hs < 2; ++hs)
#pragma unroll
            for (int db = 0; db < NDB; ++db) dv[db] = E::mfma(tf[hs][db], pp[hs], dv[db]);
#pragma unroll
        for (int hs = 0; hs < 2; ++hs)
#pragma unroll
            for (int db = 0; db < NDB; ++db)
                tf[hs][db] = load_tr<T>(ring + so + otr[db][0] + hs * 16 * PITCH, ring + so + otr[db][1] + hs * 16 * PITCH);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int hs = 0; hs < 2; ++hs)
#pragma unroll
            for (int db = 0; db < NDB; ++db) dk[db] = E::mfma(tf[hs][db], ds[hs], dk[db]);
    };
    for (int t = 0; t < nt; t += 2) {
        step(std::integral_constant<int, 0>(), t);
        if (t + 1 < nt) step(std::integral_constant<int, 1>(), t + 1);
    }
    wait_vmcnt<0>();            // (K and V rows, where there was no tile)
    __syncthreads();            // every wave is done with the ring and the K and V rows

    // half 0 finishes dK with half 1's part, half 1 dV with half 0's
    float* part = reinterpret_cast<float*>(smem) + (kb * 2) * PART;
    auto give = [&](float* to, float16v (&x)[NDB]) __attribute__((always_inline)) {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int jq = 0; jq < 4; ++jq)
                *reinterpret_cast<float4*>(to + (db * 4 + jq) * 256 + lane * 4) =
                    make_float4(x[db][4 * jq], x[db][4 * jq + 1], x[db][4 * jq + 2], x[db][4 * jq + 3]);
    };
    if (qh == 0) give(part + PART, dv);
    else give(part, dk);
    __syncthreads();
    float* mine = part + qh * PART;
    auto finish = [&](float16v (&x)[NDB]) __attribute__((always_inline)) {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int jq = 0; jq < 4; ++jq) {
                const float4 o = *reinterpret_cast<const float4*>(mine + (db * 4 + jq) * 256 + lane * 4);
                x[db][4 * jq] += o.x;
                x[db][4 * jq + 1] += o.y;
                x[db][4 * jq + 2] += o.z;
                x[db][4 * jq + 3] += o.w;
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        acc_to_lds_rows<DH>(x, mine, lane);             // the wave's own block: LDS operations of one wave complete in order
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        T* gcache = reinterpret_cast<T*>(qh ? a.gv : a.gk);
        const T* gin = reinterpret_cast<const T*>(qh ? a.gv_in : a.gk_in);
#pragma unroll
        for (int p = lane; p < 32 * DH / 8; p += 64) {
            const int row = p / (DH / 8), col = (p % (DH / 8)) * 8, k = kw + row;
            if (k > last_key) break;
            float v[8];
            *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(mine + row * EPI_LD + col);
            *reinterpret_cast<float4*>(v + 4) = *reinterpret_cast<const float4*>(mine + row * EPI_LD + col + 4);
            uint4* dst = reinterpret_cast<uint4*>(reinterpret_cast<T*>(a.dqkv) + ((long)(k - a.slice0) * a.B + b) * (3 * EE) + (long)h * 3 * DH + (1 + qh) * DH + col);
            if constexpr (!SUFFIX) {
                const long at = ((long)bh * a.cache_rows + k) * DH + col;
                uint4* gp = reinterpret_cast<uint4*>(gcache + at);
                if (k < a.slice0 ? a.accumulate_prefix : a.has_incoming) {
                    const float8v old = __builtin_convertvector(__builtin_bit_cast(vec8_t<T>, *reinterpret_cast<const uint4*>(gin + at)), float8v);
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] += old[e];
                }
                if (k < a.slice0) dst = gp;
                else if (a.zero_slice_rows) *gp = make_uint4(0, 0, 0, 0);
            }
            *dst = pack8<T>(v);
        }
    };
    if (qh == 0) finish(dk);
    else finish(dv);
}

template <typename T, bool SUFFIX> static void dkdv_long(int hd, const AttnKeysArgs& a, hipStream_t s) {
    const unsigned grid = xcd_grid(a.B * a.H, (a.grad_rows - a.key0 + 127) / 128);
    switch (hd) {
    case 64: attn_dkdv_long_kernel<T, 64, SUFFIX><<<grid, 512, 0, s>>>(a); break;
    case 80: attn_dkdv_long_kernel<T, 80, SUFFIX><<<grid, 512, 0, s>>>(a); break;
    case 96: attn_dkdv_long_kernel<T, 96, SUFFIX><<<grid, 512, 0, s>>>(a); break;
    default: attn_dkdv_long_kernel<T, 128, SUFFIX><<<grid, 512, 0, s>>>(a); break;
    }
}
void launch_attn_dkdv_long(int dtype, int head_dim, bool suffix, const AttnKeysArgs& a, hipStream_t s) {
    if (dtype == TP_F16) suffix ? dkdv_long<f16, true>(head_dim, a, s) : dkdv_long<f16, false>(head_dim, a, s);
    else suffix ? dkdv_long<bf16, true>(head_dim, a, s) : dkdv_long<bf16, false>(head_dim, a, s);
}

template <typename T> static void fwd_long(int hd, const AttnArgs& a, hipStream_t s) {
    const unsigned grid = xcd_grid(a.B * a.H, (a.T + 127) / 128);
    switch (hd) {
    case 64: attn_fwd_long_kernel<T, 64><<<grid, 512, 0, s>>>(a); break;
    case 80: attn_fwd_long_kernel<T, 80><<<grid, 512, 0, s>>>(a); break;
    case 96: attn_fwd_long_kernel<T, 96><<<grid, 512, 0, s>>>(a); break;
    default: attn_fwd_long_kernel<T, 128><<<grid, 512, 0, s>>>(a); break;
    }
}
void launch_attn_fwd_long(int dtype, int head_dim, const AttnArgs& a, hipStream_t s) {
    if (dtype == TP_F16) fwd_long<f16>(head_dim, a, s);
    else fwd_long<bf16>(head_dim, a, s);
}

}  // namespace tp
