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

// A [DH x 32] accumulator set (as in acc_to_lds_rows) rounded to T, turned to rows in the wave's own 32 x (DH + 8) elements of LDS
// and handed to store(row, column, 8 elements): the LDS operations of one wave complete in order.
template <typename T, int DH, typename F>
__device__ __forceinline__ void rows_out(const float16v* acc, T* buf, int lane, F store) {
    constexpr int NDB = (DH + 31) / 32, LD = NDB * 32 + 8;
    const int g = lane >> 5, li = lane & 31;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq)
            *reinterpret_cast<uint2*>(buf + li * LD + db * 32 + 8 * jq + 4 * g) =
                make_uint2(pack2<T>(acc[db][4 * jq], acc[db][4 * jq + 1]), pack2<T>(acc[db][4 * jq + 2], acc[db][4 * jq + 3]));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < 32 * DH / 512; ++i) {
        const int p = i * 64 + lane, row = p / (DH / 8), col = (p % (DH / 8)) * 8;
        store(row, col, *reinterpret_cast<const uint4*>(buf + row * LD + col));
    }
}

// ------------------------------------------------------------------------------------------------
// Forward.  A workgroup of four waves owns 32 * QB queries of one (batch, head): blocks of 32, each by one wave (QB = 4) or by
// two that take one half of every key tile and merge at the end (QB = 2).  K and V tiles are loaded once for all four waves, into
// rings of 64 KB at most, so that two workgroups (three at head dimension 64) share a CU: the two waves of a SIMD belong to
// different workgroups, and no barrier keeps them in step.  A wave works on three tiles at once, in one straight line: the
// exponentials of one tile stand between the score MFMAs of the next and the output MFMAs of the last.
//
// What bounds it: the vector ALU, whose issue slots an MFMA takes too (a 32 x 32 x 16 one about four): per 32 x 32 block 70
// operations, 16 of them exponentials, beside 8 to 16 MFMAs; MFMAs 0.41 and vector ALU 0.42 of the SIMD clocks at 96 heads of
// 128.  Without the LDS reads 10 to 17 % of the time would go, without the exponentials 9 %.
// Measured (fp16, causal, 2048 positions, us; before: eight waves on one ring of 128 KB, phases in step): 40 heads of 128
// 70 -> 56, 96 of 128 149 -> 118 (870 TFLOP/s), 16 of 128 41 -> 32 (blocks of 64), 32 of 80 39 -> 38; 64 of 64 at 1024 20.7 -> 19;
// 40 of 128, 512 after 1536 51 -> 32.  The tile's four slots with a barrier per tile instead of per two: 2 to 10 % slower at 64.
// ------------------------------------------------------------------------------------------------

template <typename T, int DH, int QB>
__global__ __launch_bounds__(256, 2) void attn_fwd_long_kernel(AttnArgs a) {
    typedef Elem<T> E;
    constexpr int KH = 4 / QB, SS = 2 / KH, R = 2 * SS;     // waves that share a query block's keys (a tile: 32 each); tiles between two barriers; slots of the rings
    constexpr int NDB = (DH + 31) / 32, NKS = DH / 16, PITCH = tile_pitch<DH>(), CPR = PITCH / 8;
    constexpr int KT = 32 * KH, TILE = KT * PITCH;
    constexpr int NLD = KT * CPR / 256;                     // loads per K or V tile and lane
    constexpr int EPI_LD = NDB * 32 + 4;
    constexpr int RING_BYTES = 2 * R * TILE * 2, EPI_BYTES = (KH > 1 ? QB * 64 * 4 : 0) + QB * 32 * EPI_LD * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[RING_BYTES > EPI_BYTES ? RING_BYTES : EPI_BYTES];
    T* ring = reinterpret_cast<T*>(smem);

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, li = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), qb = wave % QB, kh = wave / QB;
    int bh, blk;
    if (!xcd_map_causal(a.B * a.H, (a.T + 32 * QB - 1) / (32 * QB), bh, blk)) return;
    const int b = bh / a.H, h = bh - b * a.H;
    const int T_ = a.T, P = a.P, S = a.P + a.T;
    const int q0 = ((T_ + 32 * QB - 1) / (32 * QB) - 1 - blk) * (32 * QB);      // the blocks with the longest key range start first
    const int qw = q0 + 32 * qb, tq = qw + li;
    const bool qok = tq < T_;
    const int nt = (P + min(T_, q0 + 32 * QB) + KT - 1) / KT;   // tiles of the workgroup
    const int key_end = qw < T_ ? P + min(T_, qw + 32) : 0;     // keys this wave's queries see
    const int nt_w = max(0, (key_end - kh * 32 + KT - 1) / KT); // tiles that hold some of them for this wave

    // the lane's chunk of a tile's first rows and that of row S - 1 (the swizzle repeats every 16 rows: the same column in each load)
    const int lr = tid / CPR, lc = (tid % CPR) ^ swz16<PITCH>(lr);
    const unsigned koff = (unsigned)(lr * DH * 2 + lc * 16), klast = (unsigned)((S - 1) * DH * 2 + lc * 16);
    const bool chunk = DH == PITCH || lc < DH / 8;
    const char* Kb = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.kc) + (long)bh * a.cache_rows * DH));
    const char* Vb = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.vc) + (long)bh * a.cache_rows * DH));
    const unsigned lds0 = lds_addr(smem) + wave * 1024;
    // tile t of K (which = 0) or V (1) into a slot of its ring; rows at or past S are clamped to row S - 1: finite data, and
    // every such key is masked
    auto issue = [&](int slot, int which, int tile) __attribute__((always_inline)) {
        const unsigned dst = lds0 + (unsigned)((which * R + slot) * TILE * 2), row = (unsigned)(tile * KT) * (DH * 2);
#pragma unroll
        for (int i = 0; i < NLD; ++i)
            if (chunk) dma16_saddr_lds(min(row + (unsigned)(i * (256 / CPR) * DH * 2) + koff, klast), which ? Vb : Kb, dst + i * 4096);
    };
    typename E::opnd_t qreg[NKS];
    load_row_operands<T, DH>(qreg, reinterpret_cast<const T*>(a.q) + (long)bh * a.q_bhs + (long)(qok ? tq : 0) * DH, qok, g);

#pragma unroll
    for (int i = 0; i < R; ++i) issue(i, 0, i);
    if constexpr (SS == 2) issue(0, 1, 0);
#pragma unroll
    for (int i = 0; i < TILE / 2048; ++i)               // the V of the tile before the first, whose P is zero
        *reinterpret_cast<uint4*>(smem + (2 * R - 1) * TILE * 2 + (i * 256 + tid) * 16) = make_uint4(0, 0, 0, 0);

    int okm[NKS], otr[NDB][2];          // element offsets of the lane's fetches inside a tile
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) okm[ks] = km_offset<T, PITCH>(kh * 32 + li, ks * 16, lane);
#pragma unroll
    for (int db = 0; db < NDB; ++db) tr_offsets<T, PITCH, true>(kh * 32, db * 32, lane, otr[db][0], otr[db][1]);

    float16v oacc[NDB], s[2];
    const float16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int db = 0; db < NDB; ++db) oacc[db] = zero;
    float lsum = 0.f;
    typename E::opnd_t kf[NKS], vf[2 * NDB];
    uint4 p[2] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};

    auto barrier = [&]() __attribute__((always_inline)) {
        wait_vmcnt<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto row_max = [&](const float16v& x) __attribute__((always_inline)) {
        float v = x[0];
#pragma unroll
        for (int j = 1; j < 16; ++j) v = fmaxf(v, x[j]);
        return v;
    };
    barrier();
    s[0] = zero;
    s[1] = zero;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) s[0] = E::mfma(load_km<T>(ring + okm[ks]), qreg[ks], s[0]);
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) kf[ks] = load_km<T>(ring + TILE + okm[ks]);
    auto mask = [&](float16v& x, int key0) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (key0 + acc_row(j, g) > P + tq) x[j] = -INFINITY;
    };
    // The first reference is the maximum of two tiles: of one, the largest P of a row is less often exactly 1, and the result
    // 2 % further from fp64.
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) s[1] = E::mfma(kf[ks], qreg[ks], s[1]);
    mask(s[0], kh * 32);
    mask(s[1], KT + kh * 32);
    float smax = fmaxf(row_max(s[0]), row_max(s[1])), m = fmaxf(smax, __shfl_xor(smax, 32, 64));
    smax = m;
    if constexpr (SS == 1) {
        barrier();
        issue(0, 0, 2);
    }

    // Tile t: the exponentials of its scores (s[t & 1]) run between the MFMAs of its neighbours -- the scores of the next tile
    // (K fragments in kf), then the output of the one before (its P in p).  A fragment's registers are free when its MFMA has
    // gone: V fragments take the place of K's, and K's of the tile after next that of V's.
    auto stage = [&](auto slc, int t) __attribute__((always_inline)) {
        constexpr int sl = decltype(slc)::value, cur = sl & 1, nxt = cur ^ 1, NPV = 2 * NDB, NM = NKS + NPV;
        const int key0 = t * KT + kh * 32;
        const T* kafter = ring + (sl + 2) % R * TILE;
        const T* vbefore = ring + (R + (sl + R - 1) % R) * TILE;
        if (key0 + 31 > P + qw) {               // wave-uniform: the block touches the causal boundary
            mask(s[cur], key0);
            smax = row_max(s[cur]);
        }
        // m is the row's REFERENCE value of the exponentials, not its running maximum (as in attn_fwd2_kernel): it moves
        // only when a row outgrows it by kSlack, exponentials stay below e^kSlack = 148.
        constexpr float kSlack = 5.0f;
        float alpha = 1.f;
        unsigned long moved = __builtin_amdgcn_ballot_w64(smax > m + kSlack);
        if (moved) {
            const float m_new = fmaxf(m, fmaxf(smax, __shfl_xor(smax, 32, 64)));
            alpha = m_new == -INFINITY ? 1.0f : fast_exp2((m - m_new) * kLog2e);
            m = m_new;
            lsum *= alpha;
        }
        asm volatile("" : "+s"(moved));         // (one straight line between the two branches)
        const float mneg = m == -INFINITY ? 0.f : -m * kLog2e;
        __builtin_amdgcn_sched_barrier(0);
        unsigned pw[8];
        float e[16];
        float psum = 0.f;
#pragma unroll
        for (int k = 0; k < NM; ++k) {
            if (k < NKS) {
                s[nxt] = E::mfma(kf[k], qreg[k], k == 0 ? zero : s[nxt]);
#pragma unroll
                for (int i = k; i < (k == NKS - 1 ? NPV : k + 1); ++i) {
                    if (i >= NPV) break;
                    const T* v = vbefore + i / NDB * 16 * PITCH;
                    vf[i] = load_tr<T>(v + otr[i % NDB][0], v + otr[i % NDB][1]);
                }
            } else {
                const int i = k - NKS;
                oacc[i % NDB] = E::mfma(vf[i], p[i / NDB], oacc[i % NDB]);
#pragma unroll
                for (int ks = i; ks < (i == NPV - 1 ? NKS : i + 1); ++ks)
                    if (ks < NKS) kf[ks] = load_km<T>(kafter + okm[ks]);
            }
#pragma unroll
            for (int j = k * 16 / NM; j < (k + 1) * 16 / NM; ++j) {
                e[j] = fast_exp2(fmaf(s[cur][j], kLog2e, mneg));        // -inf -> 0
                psum += e[j];
                if (j & 1) {
                    pw[j / 2] = pack2<T>(e[j - 1], e[j]);
                    asm volatile("" : "+v"(pw[j / 2]), "+v"(psum)); // (here, not where the next tile wants them)
                }
            }
            if (k == NM - 2) {
                smax = row_max(s[nxt]);
                asm volatile("" : "+v"(smax));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (moved) {            // (what is added here was taken against the old reference)
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
        }
        lsum += psum;
        p[0] = make_uint4(pw[0], pw[1], pw[2], pw[3]);
        p[1] = make_uint4(pw[4], pw[5], pw[6], pw[7]);
    };
    // before the first of SS tiles: this wave's loads of V(t - 1 .. t + SS - 2) and K(t + 2 .. t + SS + 1) have landed, and its
    // reads of the tiles before them are back
    auto advance = [&](int sl, int t) __attribute__((always_inline)) {
        barrier();
#pragma unroll
        for (int i = 0; i < SS; ++i) {
            issue((sl + SS - 1 + i) % R, 1, t + SS - 1 + i);
            issue((sl + SS + 2 + i) % R, 0, t + SS + 2 + i);
        }
    };
    auto step = [&](auto slc, int t) __attribute__((always_inline)) {
        constexpr int sl = decltype(slc)::value;
        if constexpr (sl % SS == 0) advance(sl, t);
        stage(slc, t);
    };
    int t = 0;
    while (t < nt_w) {
        step(std::integral_constant<int, 0>(), t);
        if (++t >= nt_w) break;
        step(std::integral_constant<int, 1>(), t);
        if (++t >= nt_w) break;
        if constexpr (R == 4) {
            step(std::integral_constant<int, 2>(), t);
            if (++t >= nt_w) break;
            step(std::integral_constant<int, 3>(), t);
            ++t;
        }
    }
    // the output of the wave's last tile, then the tiles of the waves with later queries
    if (t % SS == 0) advance(t % R, t);
    {
        const T* vbefore = ring + (R + (t + R - 1) % R) * TILE;
#pragma unroll
        for (int i = 0; i < 2 * NDB; ++i) {
            const T* v = vbefore + i / NDB * 16 * PITCH;
            oacc[i % NDB] = E::mfma(load_tr<T>(v + otr[i % NDB][0], v + otr[i % NDB][1]), p[i / NDB], oacc[i % NDB]);
        }
    }
    for (++t; t <= nt; ++t)
        if (t % SS == 0) advance(t % R, t);
    wait_vmcnt<0>();
    __syncthreads();            // every wave is done with the ring: the space is reused

    float* sM = reinterpret_cast<float*>(smem);         // [QB][2][32]: the second halves' references and sums
    float* ebuf = sM + (KH > 1 ? QB * 64 : 0) + qb * 32 * EPI_LD;
    float lw = lsum + __shfl_xor(lsum, 32, 64);
    float f0 = 1.f;
    if constexpr (KH > 1) {
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
        f0 = fast_exp2((m - ms) * kLog2e);
        const float f1 = fast_exp2((m1 - ms) * kLog2e);
        lw = lw * f0 + l1 * f1;
        m = mt;
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
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    const float inv = lw > 0.f ? 1.0f / lw : 0.f;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] *= inv;
    if (g == 0 && qok) a.lse[(long)bh * a.st_bhs + tq] = lw > 0.f ? m + logf(lw) : -INFINITY;
    rows_out<T, DH>(oacc, reinterpret_cast<T*>(ebuf), lane, [&](int row, int col, uint4 v) __attribute__((always_inline)) {
        if (qw + row < T_) *reinterpret_cast<uint4*>(reinterpret_cast<T*>(a.o) + ((long)(qw + row) * a.B + b) * ((long)a.H * DH) + (long)h * DH + col) = v;
    });
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

template <typename T, int QB> static void fwd_long(int hd, const AttnArgs& a, hipStream_t s) {
    const unsigned grid = xcd_grid(a.B * a.H, (a.T + 32 * QB - 1) / (32 * QB));
    switch (hd) {
    case 64: attn_fwd_long_kernel<T, 64, QB><<<grid, 256, 0, s>>>(a); break;
    case 80: attn_fwd_long_kernel<T, 80, QB><<<grid, 256, 0, s>>>(a); break;
    case 96: attn_fwd_long_kernel<T, 96, QB><<<grid, 256, 0, s>>>(a); break;
    default: attn_fwd_long_kernel<T, 128, QB><<<grid, 256, 0, s>>>(a); break;
    }
}
void launch_attn_fwd_long(int dtype, int head_dim, int query_blocks, const AttnArgs& a, hipStream_t s) {
    if (dtype == TP_F16) query_blocks == 4 ? fwd_long<f16, 4>(head_dim, a, s) : fwd_long<f16, 2>(head_dim, a, s);
    else query_blocks == 4 ? fwd_long<bf16, 4>(head_dim, a, s) : fwd_long<bf16, 2>(head_dim, a, s);
}

}  // namespace tp
