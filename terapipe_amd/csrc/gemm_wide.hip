// The software-pipelined 256 x 256 GEMM tile of eight waves (16 x 16 x 32 MFMA blocks) and its launchers; a translation
// unit of its own so that it compiles beside gemm.hip.
#include "gemm_epilogue.h"

namespace tp {

// ---------------------------------------------------------------------------------------------
// 256 x 256 tile, k-tile 64 in two LDS stages (128 KB), eight waves (2 x 4, two per SIMD) of 128 x 64 each.
//
// What bounds a GEMM tile here is getting operands to the MFMAs: per k-tile the tile's bytes come through the global ->
// LDS path (a 256 x 256 tile needs half the bytes per flop of a 128 x 128 one) and the wave tiles' fragments out of LDS
// (192 KB per k-tile at 128 B/clk: three quarters of the MFMA time), so neither may stand still while MFMAs run.  A
// k-tile is two sub-steps of 32; in a sub-step a wave walks its eight row blocks.  As soon as the four MFMAs of row
// block i have gone out, the A fragment they used is dead and the NEXT sub-step's fragment i is fetched into the same
// registers: A is prefetched a whole sub-step ahead with a single register set, only the four B fragments (used to the
// end) have two.  That leaves a wave at 128 accumulators + 64 fragment registers of its 256, where two full sets (96)
// beside the addresses would spill.  The workgroup barrier sits after the first two row blocks of a k-tile's second
// sub-step: by then the fetches of this k-tile are long back, so no wave waits for LDS there; after it the buffer is
// free, and the loads of the k-tile two ahead go out behind the next row blocks' MFMAs.
// Measured against the 256 x 256 tile without this order (8192 x 8192 x 8192 fp16): NT 1092 -> 1330 TFLOP/s, NN 1135 ->
// 1362; taken apart (results garbage): without the tile loads 1584, without the fragment fetches 1574, without either
// 2200, without the barrier 1377 -- the LDS, which both go through, is what is left.  Four waves of 128 x 128 (two thirds of
// the fetches) reach 1276: nothing covers a wave's own stalls.  The TN form (both operands through transpose reads)
// is level with the 32-wide k-tile in four stages, which is kept for it.
// ---------------------------------------------------------------------------------------------
template <typename T, bool BKM>
__global__ __launch_bounds__(512)
void gemm_wide_kernel(GemmArgs a) {
    int tile_x, tile_y, tile_z;
    xcd_tile3((int)((blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x), (int)gridDim.x, (int)gridDim.y,
              (int)gridDim.z, tile_x, tile_y, tile_z);
    constexpr bool AKM = true;
    static_assert(sizeof(T) == 2, "16-bit only");
    constexpr int BM = 256, BN = 256, BK = 64, KS = 32, WM = 2, WN = 4, NT = 512;
    constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
    constexpr int AR = AKM ? BM : BK, AC = AKM ? BK : BM;
    constexpr int BR = BKM ? BN : BK, BC = BKM ? BK : BN;
    constexpr int A_ELEMS = AR * AC, STAGE_ELEMS = A_ELEMS + BR * BC;
    typedef ClampTileDma<T, AR, AC, NT, AKM, AKM> DA;
    typedef ClampTileDma<T, BR, BC, NT, BKM, BKM> DB;
    constexpr int NLOAD = DA::N + DB::N;
    static_assert(DA::N == 4 && DB::N == 4, "the load schedule below");
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * STAGE_ELEMS * 2];
    static_assert(WM * WN * 32 * 36 * 4 <= 2 * STAGE_ELEMS * 2, "the epilogue stages through the same memory");
    T* tiles = reinterpret_cast<T*>(smem);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave % WM, wn = wave / WM;
    const int m0 = tile_y * BM, n0 = tile_x * BN;
    const int kbeg = tile_z * a.kper;
    const int klen = min(a.K, kbeg + a.kper) - kbeg;
    const int nk = (klen + BK - 1) / BK, ragged = klen % BK;       // a ragged k has its short tile first (copy_ragged_tile)
    DA da;
    DB db;
    da.init(reinterpret_cast<const T*>(a.A), a.lda, m0, a.M, ragged ? kbeg - BK : kbeg, BK, tid);
    db.init(reinterpret_cast<const T*>(a.B), a.ldb, n0, a.N, ragged ? kbeg - BK : kbeg, BK, tid);
    const unsigned lds0 = lds_addr(smem);
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);

    float4v acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};

    // Element offsets of the lane's fragments inside stage 0.  k-major tiles: the swizzle repeats every 16 rows, so
    // block i is 16 rows of 64 further on and the second sub-step's offset is the one of the other half of the row.
    // Token-major tiles (rows of 256): the second sub-step is 32 rows further on; block i is an own offset.
    constexpr int NA = AKM ? 1 : TM, NB = BKM ? 1 : TN, PA = AKM ? 1 : 2, PB = BKM ? 1 : 2;
    constexpr int SA = AKM ? 2 : 1, SB = BKM ? 2 : 1;
    int oa[SA][NA][PA], ob[SB][NB][PB];
#pragma unroll
    for (int s = 0; s < SA; ++s)
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int mb = (wm * TM + i) * 16;
            if constexpr (AKM) oa[s][i][0] = TileLayout<T, AC, true>::off(mb + (lane & 15), s * KS + 8 * (lane >> 4));
            else tr_offsets16<T, AC>(0, mb, lane, oa[s][i][0], oa[s][i][PA - 1]);
        }
#pragma unroll
    for (int s = 0; s < SB; ++s)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int nb = (wn * TN + j) * 16;
            if constexpr (BKM) ob[s][j][0] = A_ELEMS + TileLayout<T, BC, true>::off(nb + (lane & 15), s * KS + 8 * (lane >> 4));
            else {
                tr_offsets16<T, BC>(0, nb, lane, ob[s][j][0], ob[s][j][PB - 1]);
                ob[s][j][0] += A_ELEMS;
                ob[s][j][PB - 1] += A_ELEMS;
            }
        }

    uint4 fa[TM], fb[2][TN];
    auto fetch_a = [&](auto ic, auto subc) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value, sub = decltype(subc)::value;
        if constexpr (AKM) fa[i] = load_km<T>(tiles + oa[sub][0][0] + i * 16 * AC);
        else fa[i] = load_tr<T>(tiles + oa[0][i][0] + sub * KS * AC, tiles + oa[0][i][PA - 1] + sub * KS * AC);
    };
    auto fetch_b = [&](auto jc, auto subc) __attribute__((always_inline)) {
        constexpr int j = decltype(jc)::value, sub = decltype(subc)::value;
        if constexpr (BKM) fb[sub][j] = load_km<T>(tiles + ob[sub][0][0] + j * 16 * BC);
        else fb[sub][j] = load_tr<T>(tiles + ob[0][j][0] + sub * KS * BC, tiles + ob[0][j][PB - 1] + sub * KS * BC);
    };
    // from one stage to the other: both lie on a power of two
    static_assert((STAGE_ELEMS & (STAGE_ELEMS - 1)) == 0, "stages are told apart by one bit of the offset");
    auto other_stage = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < SA; ++s)
#pragma unroll
            for (int i = 0; i < NA; ++i)
#pragma unroll
                for (int p = 0; p < PA; ++p) oa[s][i][p] ^= STAGE_ELEMS;
#pragma unroll
        for (int s = 0; s < SB; ++s)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int p = 0; p < PB; ++p) ob[s][j][p] ^= STAGE_ELEMS;
    };
    typedef std::integral_constant<int, 0> I0;
    typedef std::integral_constant<int, 1> I1;
    // the MFMAs of row block i on the sub-step's B set
    auto mfmas = [&](auto ic, auto subc) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value, sub = decltype(subc)::value;
        static_for<TN>([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            acc[i][j] = Mfma16x16x32<T>::run(fa[i], fb[sub][j], acc[i][j]);
        });
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load = [&](auto dc, unsigned sA) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value;
        if constexpr (d < DA::N) da.issue_one(d, sA, wave_u);
        else db.issue_one(d - DA::N, sA + (unsigned)(A_ELEMS * 2), wave_u);
    };

    // prologue: both buffers get a k-tile; k-tile 0 is waited for and its first sub-step fetched
    if (ragged) {
        copy_ragged_tile<T, AR, AC, NT, AKM, AKM>(tiles, reinterpret_cast<const T*>(a.A), a.lda, m0, a.M, kbeg + klen - ragged, ragged, tid);
        copy_ragged_tile<T, BR, BC, NT, BKM, BKM>(tiles + A_ELEMS, reinterpret_cast<const T*>(a.B), a.ldb, n0, a.N, kbeg + klen - ragged, ragged, tid);
        da.advance();
        db.advance();
    } else {
        da.issue(lds0, wave_u);
        db.issue(lds0 + (unsigned)(A_ELEMS * 2), wave_u);
    }
    if (nk > 1) {
        da.issue(lds0 + (unsigned)(STAGE_ELEMS * 2), wave_u);
        db.issue(lds0 + (unsigned)((STAGE_ELEMS + A_ELEMS) * 2), wave_u);
        wait_vmcnt<NLOAD>();
    } else {
        wait_vmcnt<0>();
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (a copied tile's stores)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    static_for<TN>([&](auto jc) __attribute__((always_inline)) { fetch_b(jc, I0{}); });
    static_for<TM>([&](auto ic) __attribute__((always_inline)) { fetch_a(ic, I0{}); });

    // The loop body is one straight line (a branch in it costs register copies): the last two k-tiles load the last
    // k-tile again into a buffer that nothing reads any more, and the last one's fetches for "the next" are not used.
    // (A single ragged k-tile loads the 64 positions before it: the plan gives this tile no k below 64.)
    unsigned stage = lds0;
    for (int kt = 0; kt < nk; ++kt) {
        if (kt + 2 >= nk) {
            da.origin -= da.step;
            db.origin -= db.step;
        }
        static_for<TM>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            mfmas(ic, I0{});
            fetch_a(ic, I1{});
            if constexpr (i < 2) {
                fetch_b(std::integral_constant<int, 2 * i>{}, I1{});
                fetch_b(std::integral_constant<int, 2 * i + 1>{}, I1{});
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        other_stage();
        mfmas(I0{}, I1{});
        mfmas(I1{}, I1{});
        // every fetch of this k-tile is back, and the next k-tile has landed once every wave says so
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        static_for<TM - 2>([&](auto ic2) __attribute__((always_inline)) {
            constexpr int i = decltype(ic2)::value + 2;
            if constexpr (i == 2) {
                fetch_a(I0{}, I0{});
                fetch_b(I0{}, I0{});
                fetch_b(I1{}, I0{});
            }
            if constexpr (i == 3) {
                fetch_a(I1{}, I0{});
                fetch_b(std::integral_constant<int, 2>{}, I0{});
                fetch_b(std::integral_constant<int, 3>{}, I0{});
            }
            __builtin_amdgcn_sched_barrier(0);
            mfmas(std::integral_constant<int, i>{}, I1{});
            fetch_a(std::integral_constant<int, i>{}, I0{});
            if constexpr (i < 6) {
                load(std::integral_constant<int, 2 * (i - 2)>{}, stage);
                load(std::integral_constant<int, 2 * (i - 2) + 1>{}, stage);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        da.advance();
        db.advance();
        stage = 2 * lds0 + (unsigned)(STAGE_ELEMS * 2) - stage;
    }
    wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    gemm_epilogue16<T, TM, TN, WM, WN>(a, acc, reinterpret_cast<float*>(smem), m0, n0, tile_z);
}

template <typename T>
static bool launch_wide_op(int op, dim3 grid, const GemmArgs& a, hipStream_t s) {
    if (op == TP_GEMM_NT) gemm_wide_kernel<T, true><<<grid, 512, 0, s>>>(a);
    else if (op == TP_GEMM_NN) gemm_wide_kernel<T, false><<<grid, 512, 0, s>>>(a);
    else return false;
    return true;
}

bool launch_gemm_wide(int op, int dtype, dim3 grid, const GemmArgs& a, hipStream_t s) {
    if (dtype == TP_F16) return launch_wide_op<f16>(op, grid, a, s);
    if (dtype == TP_BF16) return launch_wide_op<bf16>(op, grid, a, s);
    return false;
}

}  // namespace tp
