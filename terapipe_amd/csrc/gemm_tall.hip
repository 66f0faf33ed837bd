// The 256-row GEMM tiles for long activations and parameter gradients, all operand orders (16-bit).
#include "gemm_epilogue.h"
#include "vec_grads.h"

namespace tp {

// ---------------------------------------------------------------------------------------------
// Tall-tile variant for long activations (M >= 256): BM = 256 rows by four waves stacked in M, each
// holding a 64 x BN block of the output in accumulator registers (BN up to 192 -> 192 AGPRs; one wave per
// SIMD).  A 256 x 160 x 64 tile moves 52 KB for 5.2 MFLOP, 1.5 times the flops per byte of a 128 x 128 tile:
// the vector-memory path into LDS (64 B/clk per CU) stops being the limit.  BN is any multiple of 32, so
// the tile count can be matched to the 256 CUs (N = 20480: BN = 160 gives exactly 256 tiles for M = 512).
// Tiles are loaded with ClampTileDma (whole k-tiles only) and the operand fetches of k-step s+1 are issued
// before the MFMAs of k-step s.
// MI16: 16 x 16 x 32 MFMA blocks and ONE set of operand registers per wave (two waves share a SIMD: one computes
// while the other fetches; two sets of the twice as many operand registers do not fit beside the accumulators).
// GROUPED: behind the tiles, the blocks of the same rows' vector-parameter gradients: they run on the CUs that the last, part-filled round
// of tiles leaves, where in a launch of their own they wait for its end.
struct GemmTallGroupArgs : GemmGroupArgs { VecGradArgs vec; int tiles; };

template <typename T, bool AKM, bool BKM, int BM, int BN, int BK, int WM, int WN, int STAGES, bool GROUPED = false,
          bool MI16 = false>
__global__ __launch_bounds__(WM * WN * 64)
void gemm_tall_kernel(typename std::conditional<GROUPED, GemmTallGroupArgs, GemmArgs>::type args) {
    // which problem and which of its tiles (wave-uniform)
    int prob = 0, tile_x = blockIdx.x, tile_y = blockIdx.y;
    if constexpr (GROUPED) {
        static_assert(kGroupMax == 4, "the selects below are written out for four problems");
        int first = 0, tx = args.tiles_x[0], ty = args.tiles_y[0];
        if (1 < args.n && (int)blockIdx.x >= args.first_tile[1]) { prob = 1; first = args.first_tile[1]; tx = args.tiles_x[1]; ty = args.tiles_y[1]; }
        if (2 < args.n && (int)blockIdx.x >= args.first_tile[2]) { prob = 2; first = args.first_tile[2]; tx = args.tiles_x[2]; ty = args.tiles_y[2]; }
        if (3 < args.n && (int)blockIdx.x >= args.first_tile[3]) { prob = 3; first = args.first_tile[3]; tx = args.tiles_x[3]; ty = args.tiles_y[3]; }
        xcd_tile((int)blockIdx.x - first, tx, ty, tile_x, tile_y);
    } else if (gridDim.z == 1) {
        xcd_tile((int)(blockIdx.y * gridDim.x + blockIdx.x), (int)gridDim.x, (int)gridDim.y, tile_x, tile_y);
    }
    // (constant indices only: a dynamically indexed kernel argument would be copied to scratch memory)
    const GemmArgs a = [&]() -> GemmArgs {
        if constexpr (GROUPED) {
            if (prob == 1) return args.g[1];
            if (prob == 2) return args.g[2];
            if (prob == 3) return args.g[3];
            return args.g[0];
        } else {
            return args;
        }
    }();
    typedef Elem<T> E;
    static_assert(sizeof(T) == 2, "16-bit only");
    constexpr int NT = WM * WN * 64;
    constexpr int BLK = MI16 ? 16 : 32;                  // rows / columns of an MFMA block
    constexpr int KS = MI16 ? 32 : E::KSTEP;             // k of one MFMA
    static_assert(!MI16 || WM * WN == 8, "the 16 x 16 blocks are written for two waves per SIMD");
    constexpr int TM = BM / WM / BLK, TN = BN / WN / BLK;
    constexpr int AR = AKM ? BM : BK, AC = AKM ? BK : BM;
    constexpr int BR = BKM ? BN : BK, BC = BKM ? BK : BN;
    constexpr int A_ELEMS = AR * AC, B_ELEMS = BR * BC;
    constexpr int STAGE_ELEMS = A_ELEMS + B_ELEMS;
    typedef ClampTileDma<T, AR, AC, NT, AKM, MI16 && AKM> DA;
    typedef ClampTileDma<T, BR, BC, NT, BKM, MI16 && BKM> DB;
    constexpr int NLOAD = DA::N + DB::N;
    static_assert(NLOAD * (STAGES - 1) <= 63, "too many loads in flight for vmcnt");
    constexpr int TILE_BYTES = STAGES * STAGE_ELEMS * 2;
    constexpr int EPI_BYTES = WM * WN * 32 * 36 * 4;
    constexpr int SMEM_BYTES = TILE_BYTES > EPI_BYTES ? TILE_BYTES : EPI_BYTES;
    __shared__ __attribute__((aligned(16))) unsigned char smem[SMEM_BYTES];
    T* tiles = reinterpret_cast<T*>(smem);
    if constexpr (GROUPED) {
        static_assert(NT == kVecGradLanes * 32 && SMEM_BYTES >= kVecGradLds, "a block of vec_param_grads_block");
        if ((int)blockIdx.x >= args.tiles) {
            const int block = (int)blockIdx.x - args.tiles;
            VEC_GRAD_PICK(args.vec, block, pr, first)
            vec_param_grads_block<T, 8>(pr, block - first, smem);
            return;
        }
    }

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave % WM, wn = wave / WM;
    const int m0 = tile_y * BM, n0 = tile_x * BN;
    const int kbeg = blockIdx.z * a.kper;
    const int kend = min(a.K, kbeg + a.kper);
    DA da;
    DB db;
    const int nk = (kend - kbeg + BK - 1) / BK;
    const int ragged = (kend - kbeg) % BK;      // a ragged k has its short tile first (copy_ragged_tile)
    da.init(reinterpret_cast<const T*>(a.A), a.lda, m0, a.M, ragged ? kbeg - BK : kbeg, BK, tid);
    db.init(reinterpret_cast<const T*>(a.B), a.ldb, n0, a.N, ragged ? kbeg - BK : kbeg, BK, tid);
    const unsigned lds0 = lds_addr(smem);
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    auto issue = [&](int stage) {
        const unsigned sA = lds0 + (unsigned)(stage * STAGE_ELEMS * (int)sizeof(T));
        da.issue(sA, wave_u);
        db.issue(sA + (unsigned)(A_ELEMS * (int)sizeof(T)), wave_u);
    };

    typedef typename std::conditional<MI16, float4v, float16v>::type acc_t;
    acc_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < (MI16 ? 4 : 16); ++r) acc[i][j][r] = 0.f;

    constexpr int NKSTEP = BK / KS;
    constexpr int NPA = AKM ? 1 : 2, NPB = BKM ? 1 : 2;
    // lane's fetch offsets for k-step 0 of stage 0; k-steps and stages are compile-time byte offsets for
    // k-major operands (a k-step is two (four) chunks further along the row)
    int oa[NKSTEP][TM][NPA], ob[NKSTEP][TN][NPB];
    auto operand_offsets = [&](auto km_c, auto cols_c, int row0, int k0, int& o0, int& o1) {
        constexpr bool KM = decltype(km_c)::value;
        constexpr int COLS = decltype(cols_c)::value;
        if constexpr (MI16) {
            if constexpr (KM) o0 = o1 = TileLayout<T, COLS, true>::off(row0 + (lane & 15), k0 + 8 * (lane >> 4));
            else tr_offsets16<T, COLS>(k0, row0, lane, o0, o1);
        } else {
            if constexpr (KM) o0 = o1 = km_offset<T, COLS>(row0 + (lane & 31), k0, lane);
            else tr_offsets<T, COLS, false>(k0, row0, lane, o0, o1);
        }
    };
#pragma unroll
    for (int ks = 0; ks < NKSTEP; ++ks) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
            operand_offsets(std::integral_constant<bool, AKM>{}, std::integral_constant<int, AC>{}, (wm * TM + i) * BLK,
                            ks * KS, oa[ks][i][0], oa[ks][i][NPA - 1]);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            int o0, o1;
            operand_offsets(std::integral_constant<bool, BKM>{}, std::integral_constant<int, BC>{}, (wn * TN + j) * BLK,
                            ks * KS, o0, o1);
            ob[ks][j][0] = A_ELEMS + o0;
            ob[ks][j][NPB - 1] = A_ELEMS + o1;
        }
    }

    if (ragged) {
        copy_ragged_tile<T, AR, AC, NT, AKM, MI16 && AKM>(tiles, reinterpret_cast<const T*>(a.A), a.lda, m0, a.M, kend - ragged, ragged, tid);
        copy_ragged_tile<T, BR, BC, NT, BKM, MI16 && BKM>(tiles + A_ELEMS, reinterpret_cast<const T*>(a.B), a.ldb, n0, a.N, kend - ragged, ragged, tid);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        da.advance();
        db.advance();
    } else {
        issue(0);
    }
#pragma unroll
    for (int s = 1; s < STAGES - 1; ++s)
        if (s < nk) issue(s);

    constexpr int NSET = MI16 ? 1 : 2;
    typename E::opnd_t fa[NSET][TM], fb[NSET][TN];
    auto fetch = [&](auto ksc, auto sc, int buf) {
        constexpr int ks = decltype(ksc)::value, s = decltype(sc)::value;
        const T* st = tiles + s * STAGE_ELEMS;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if constexpr (AKM) fa[buf][i] = load_km<T>(st + oa[ks][i][0]);
            else fa[buf][i] = load_tr<T>(st + oa[ks][i][0], st + oa[ks][i][NPA - 1]);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if constexpr (BKM) fb[buf][j] = load_km<T>(st + ob[ks][j][0]);
            else fb[buf][j] = load_tr<T>(st + ob[ks][j][0], st + ob[ks][j][NPB - 1]);
        }
    };
    // No tile is loaded past the end of k (ClampTileDma does not bound the sliding axis): the last STAGES - 1
    // tiles issue nothing and wait for every outstanding load instead of all but the younger tiles'.
    auto tile = [&](auto sc, int kt) {
        constexpr int s = decltype(sc)::value;
        const bool more = kt + STAGES - 1 < nk;      // uniform
        if (more) wait_vmcnt<NLOAD * (STAGES - 2)>();
        else wait_vmcnt<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        fetch(std::integral_constant<int, 0>{}, sc, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue((s + STAGES - 1) % STAGES);   // issued while the fetch above is in flight
        auto step = [&](auto ksc) {
            constexpr int ks = decltype(ksc)::value;
            constexpr int set = MI16 ? 0 : (ks & 1);
            if constexpr (MI16) {
                if constexpr (ks > 0) fetch(ksc, sc, 0);
            } else if constexpr (ks + 1 < NKSTEP) {
                fetch(std::integral_constant<int, ks + 1>{}, sc, (ks + 1) & 1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if constexpr (MI16) acc[i][j] = Mfma16x16x32<T>::run(fa[set][i], fb[set][j], acc[i][j]);
                    else acc[i][j] = E::mfma(fa[set][i], fb[set][j], acc[i][j]);
                }
            if constexpr (MI16) __builtin_amdgcn_sched_barrier(0);
        };
        step(std::integral_constant<int, 0>{});
        if constexpr (NKSTEP > 1) step(std::integral_constant<int, 1>{});
        if constexpr (NKSTEP > 2) step(std::integral_constant<int, 2>{});
        if constexpr (NKSTEP > 3) step(std::integral_constant<int, 3>{});
        static_assert(NKSTEP <= 4, "k-tile of at most four k-steps");
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    for (int kt0 = 0; kt0 < nk; kt0 += STAGES) {
        if (kt0 + 0 < nk) tile(std::integral_constant<int, 0>{}, kt0);
        if constexpr (STAGES > 1) { if (kt0 + 1 < nk) tile(std::integral_constant<int, 1>{}, kt0 + 1); }
        if constexpr (STAGES > 2) { if (kt0 + 2 < nk) tile(std::integral_constant<int, 2>{}, kt0 + 2); }
        if constexpr (STAGES > 3) { if (kt0 + 3 < nk) tile(std::integral_constant<int, 3>{}, kt0 + 3); }
        static_assert(STAGES <= 4, "at most four stages");
    }
    wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if constexpr (MI16) gemm_epilogue16<T, TM, TN, WM, WN>(a, acc, reinterpret_cast<float*>(smem), m0, n0, (int)blockIdx.z);
    else gemm_epilogue<T, TM, TN, WM, WN>(a, acc, reinterpret_cast<float*>(smem), m0, n0, (int)blockIdx.z);
}

template <typename T, bool AKM, bool BKM>
static bool launch_tall_cfg(int cfg, dim3 grid, const GemmArgs& a, hipStream_t s) {
    switch (cfg) {
    case 2: gemm_tall_kernel<T, AKM, BKM, 256, 256, 32, 4, 2, 4, false, true><<<grid, 512, 0, s>>>(a); return true;
    case 17:
        if constexpr (BKM) { gemm_tall_kernel<T, AKM, BKM, 256, 160, 64, 4, 1, 3><<<grid, 256, 0, s>>>(a); return true; }
        return false;
    case 18: gemm_tall_kernel<T, AKM, BKM, 256, 128, 64, 4, 1, 3><<<grid, 256, 0, s>>>(a); return true;
    case 19: gemm_tall_kernel<T, AKM, BKM, 256, 256, 64, 4, 2, 2><<<grid, 512, 0, s>>>(a); return true;
    case 20: gemm_tall_kernel<T, AKM, BKM, 256, 256, 32, 4, 2, 4><<<grid, 512, 0, s>>>(a); return true;
    default: return false;
    }
}

template <typename T> static bool launch_tall_op(int cfg, int op, dim3 grid, const GemmArgs& a, hipStream_t s) {
    if (op == TP_GEMM_NT) return launch_tall_cfg<T, true, true>(cfg, grid, a, s);
    if (op == TP_GEMM_NN) return launch_tall_cfg<T, true, false>(cfg, grid, a, s);
    return launch_tall_cfg<T, false, false>(cfg, grid, a, s);
}

bool launch_gemm_tall(int cfg, int op, int dtype, dim3 grid, const GemmArgs& a, hipStream_t s) {
    if (dtype == TP_F16) return launch_tall_op<f16>(cfg, op, grid, a, s);
    if (dtype == TP_BF16) return launch_tall_op<bf16>(cfg, op, grid, a, s);
    return false;
}

template <typename T> static bool launch_tall_group(int cfg, int tiles, const GemmGroupArgs& group, const VecGradArgs* vec, hipStream_t s) {
    GemmTallGroupArgs ga = {};
    static_cast<GemmGroupArgs&>(ga) = group;
    ga.tiles = tiles;
    if (vec) {
        ga.vec = *vec;
        tiles += vec->first_block[kVecGradMax];
    }
    if (cfg == 2) gemm_tall_kernel<T, false, false, 256, 256, 32, 4, 2, 4, true, true><<<dim3(tiles), 512, 0, s>>>(ga);
    else if (cfg == 19) gemm_tall_kernel<T, false, false, 256, 256, 64, 4, 2, 2, true><<<dim3(tiles), 512, 0, s>>>(ga);
    else if (cfg == 20) gemm_tall_kernel<T, false, false, 256, 256, 32, 4, 2, 4, true><<<dim3(tiles), 512, 0, s>>>(ga);
    else return false;
    return true;
}

bool launch_gemm_tall_group(int cfg, int dtype, int tiles, const GemmGroupArgs& ga, const VecGradArgs* vec, hipStream_t s) {
    if (dtype == TP_F16) return launch_tall_group<f16>(cfg, tiles, ga, vec, s);
    if (dtype == TP_BF16) return launch_tall_group<bf16>(cfg, tiles, ga, vec, s);
    return false;
}

}  // namespace tp
