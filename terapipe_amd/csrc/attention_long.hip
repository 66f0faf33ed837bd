// Attention of whole sequences and long slices (16-bit): workgroups whose waves share the tiles they stream.
#include "attention_args.h"

namespace tp {

typedef float float8v __attribute__((ext_vector_type(8)));
template <typename T> using vec8_t = T __attribute__((ext_vector_type(8)));
template <typename T> __device__ __forceinline__ uint4 pack8v(float8v v) {
    return __builtin_bit_cast(uint4, __builtin_convertvector(v, vec8_t<T>));
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
// dQ of 128 queries, and their delta = rowsum(dO * O) for the dK / dV kernel that follows on the stream: the partition of the
// forward.  Per 32 x 32 block three products (K Q^T, V dO^T, K^T dS^T) and three fetches of 8 KB out of LDS against about 600
// cycles of vector ALU.  Causal, 2048 positions: 40 heads of 128 151 -> 95 us, 96 of 128 365 -> 212, 32 of 80 108 -> 54; 64 heads
// of 64 at 1024 39 -> 29.
// ------------------------------------------------------------------------------------------------
template <typename T, int DH>
__global__ __launch_bounds__(512) void attn_dq_long_kernel(AttnArgs a) {
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

template <typename T> static void dq_long(int hd, const AttnArgs& a, hipStream_t s) {
    const unsigned grid = xcd_grid(a.B * a.H, (a.T + 127) / 128);
    switch (hd) {
    case 64: attn_dq_long_kernel<T, 64><<<grid, 512, 0, s>>>(a); break;
    case 80: attn_dq_long_kernel<T, 80><<<grid, 512, 0, s>>>(a); break;
    case 96: attn_dq_long_kernel<T, 96><<<grid, 512, 0, s>>>(a); break;
    default: attn_dq_long_kernel<T, 128><<<grid, 512, 0, s>>>(a); break;
    }
}
void launch_attn_dq_long(int dtype, int head_dim, const AttnArgs& a, hipStream_t s) {
    if (dtype == TP_F16) dq_long<f16>(head_dim, a, s);
    else dq_long<bf16>(head_dim, a, s);
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
