// Weight gradients over few rows: several TN products of one short k in one launch.
#include "gemm_epilogue.h"

namespace tp {

// ---------------------------------------------------------------------------------------------
// 128 x 128 tiles by four waves (2 x 2 of 64 x 64, 16 x 16 x 32 MFMA blocks), k-tile 32 in a ring of three stages (48 KB).
//
// What bounds these products is C: read, added to and written back, 4 bytes per output against 2 k / 128 of operands, mostly L2
// hits.  The 256 x 256 tile alone on a CU loads operands, multiplies, reads C and writes it one after the other, and a
// 1600-wide layer's 532 tiles are 2.08 rounds of them.  Here C (32 KB) is asked for right behind the first k-tiles and lands in
// LDS while the k loop runs, and two workgroups share a CU (80 KB each): one's stores go out under the other's loop.
// Four products of a 1600-wide layer added over 256 rows 51.3 -> 40.9 us (3.0 TB/s of C), over 64 37.4 -> 29.8; stored 36.5 -> 32.2.
// The smaller tile's operands eat the gain as k grows: added over 768 rows 86 -> 75, over 1024 level at best.
// ---------------------------------------------------------------------------------------------
template <typename T, bool ADD>
__global__ __launch_bounds__(256, 2)
void gemm_short_kernel(GemmGroupArgs args) {
    static_assert(sizeof(T) == 2 && kGroupMax == 4, "16-bit; the selects below are written out for four problems");
    int prob = 0, tile_x, tile_y, first = 0, tx = args.tiles_x[0], ty = args.tiles_y[0];
    if (1 < args.n && (int)blockIdx.x >= args.first_tile[1]) { prob = 1; first = args.first_tile[1]; tx = args.tiles_x[1]; ty = args.tiles_y[1]; }
    if (2 < args.n && (int)blockIdx.x >= args.first_tile[2]) { prob = 2; first = args.first_tile[2]; tx = args.tiles_x[2]; ty = args.tiles_y[2]; }
    if (3 < args.n && (int)blockIdx.x >= args.first_tile[3]) { prob = 3; first = args.first_tile[3]; tx = args.tiles_x[3]; ty = args.tiles_y[3]; }
    xcd_tile((int)blockIdx.x - first, tx, ty, tile_x, tile_y);
    const GemmArgs a = [&]() -> GemmArgs {
        if (prob == 1) return args.g[1];
        if (prob == 2) return args.g[2];
        if (prob == 3) return args.g[3];
        return args.g[0];
    }();
    constexpr int BT = 128, KS = 32, STAGES = 3, TILE = KS * BT, STAGE = 2 * TILE, WT = 64, TB = WT / 16, SPITCH = 36;
    constexpr int NC = ADD ? BT * BT / 8 / 256 : 0;         // loads of C per lane
    typedef ClampTileDma<T, KS, BT, 256, false, false> D;
    static_assert(2 * D::N == 4 && 4 * 32 * SPITCH * 4 <= STAGES * STAGE * 2, "the counts of the waits; the epilogue's staging");
    __shared__ __attribute__((aligned(16))) unsigned char smem[STAGES * STAGE * 2 + (ADD ? BT * BT * 2 : 16)];
    T* tiles = reinterpret_cast<T*>(smem);
    T* ctile = tiles + STAGES * STAGE;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
    const int m0 = tile_y * BT, n0 = tile_x * BT, nk = a.K / KS;
    D da, db;
    da.init(reinterpret_cast<const T*>(a.A), a.lda, m0, a.M, 0, KS, tid);
    db.init(reinterpret_cast<const T*>(a.B), a.ldb, n0, a.N, 0, KS, tid);
    const unsigned lds0 = lds_addr(smem);
    auto issue = [&](int stage) __attribute__((always_inline)) {
        da.issue(lds0 + (unsigned)(stage * STAGE * 2), wave);
        db.issue(lds0 + (unsigned)((stage * STAGE + TILE) * 2), wave);
    };
    issue(0);               // (k is a multiple of 64)
    issue(1);
    if (nk > 2) issue(2);
    if constexpr (ADD) {
        const char* C = uniform_ptr(reinterpret_cast<const char*>(reinterpret_cast<const T*>(a.C) + (long)m0 * a.ldc + n0));
        const int last_row = a.M - 1 - m0, last_col = a.N - 8 - n0;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int p = i * 256 + tid, row = min(p >> 4, last_row), col = min((p & 15) * 8, last_col);
            dma16_saddr_lds((unsigned)(((long)row * a.ldc + col) * 2), C, lds0 + (unsigned)(STAGES * STAGE * 2 + i * 4096 + wave * 1024));
        }
    }

    int oa[TB][2], ob[TB][2];
#pragma unroll
    for (int i = 0; i < TB; ++i) {
        tr_offsets16<T, BT>(0, wm * WT + 16 * i, lane, oa[i][0], oa[i][1]);
        tr_offsets16<T, BT>(0, wn * WT + 16 * i, lane, ob[i][0], ob[i][1]);
    }
    float4v acc[TB][TB];
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
        for (int j = 0; j < TB; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};

    int stage = 0;
    for (int kt = 0; kt < nk; ++kt) {
        // Loads in flight behind k-tile kt's: those of up to two further k-tiles, and C's, asked for behind the third
        const int later = min(2, nk - 1 - kt);
        if (ADD && kt < STAGES) {
            if (later == 2) wait_vmcnt<8 + NC>();
            else if (later == 1) wait_vmcnt<4 + NC>();
            else wait_vmcnt<NC>();
        } else {
            if (later == 2) wait_vmcnt<8>();
            else if (later == 1) wait_vmcnt<4>();
            else wait_vmcnt<0>();
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const T *ta = tiles + stage * STAGE, *tb = ta + TILE;
        uint4 fa[TB], fb[TB];
#pragma unroll
        for (int i = 0; i < TB; ++i) fa[i] = load_tr<T>(ta + oa[i][0], ta + oa[i][1]);
#pragma unroll
        for (int j = 0; j < TB; ++j) fb[j] = load_tr<T>(tb + ob[j][0], tb + ob[j][1]);
#pragma unroll
        for (int i = 0; i < TB; ++i)
#pragma unroll
            for (int j = 0; j < TB; ++j) acc[i][j] = Mfma16x16x32<T>::run(fa[i], fb[j], acc[i][j]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();           // every wave has read the stage
        asm volatile("" ::: "memory");
        if (kt + STAGES < nk) issue(stage);
        stage = stage == STAGES - 1 ? 0 : stage + 1;
    }
    wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();               // C is there
    asm volatile("" ::: "memory");

    float* st = reinterpret_cast<float*>(smem) + wave * 32 * SPITCH;
    const int q = lane >> 4, c = lane & 15, er = lane >> 2, ec = (lane & 3) * 8;
    static_for<4>([&](auto bc) __attribute__((always_inline)) {
        constexpr int bi = decltype(bc)::value & 1, bj = decltype(bc)::value >> 1;
        static_for<4>([&](auto dc) __attribute__((always_inline)) {
            constexpr int di = decltype(dc)::value >> 1, dj = decltype(dc)::value & 1;
#pragma unroll
            for (int r = 0; r < 4; ++r) st[(16 * di + 4 * q + r) * SPITCH + 16 * dj + c] = acc[2 * bi + di][2 * bj + dj][r];
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // the block is the wave's own
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
            const int lr = wm * WT + bi * 32 + er + 16 * pass, lc = wn * WT + bj * 32 + ec;
            const float4v v0 = *reinterpret_cast<const float4v*>(st + (er + 16 * pass) * SPITCH + ec);
            const float4v v1 = *reinterpret_cast<const float4v*>(st + (er + 16 * pass) * SPITCH + ec + 4);
            Raw8<T> old = {};
            if constexpr (ADD) old.r[0] = *reinterpret_cast<const uint4*>(ctile + lr * BT + lc);
            if (m0 + lr < a.M && n0 + lc < a.N)
                epilogue_apply8<T, ADD ? TP_EPI_ACCUMULATE : TP_EPI_STORE>(a, m0 + lr, n0 + lc, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7), old, old);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    });
}

template <typename T> static void short_group(bool add, int tiles, const GemmGroupArgs& ga, hipStream_t s) {
    if (add) gemm_short_kernel<T, true><<<dim3(tiles), 256, 0, s>>>(ga);
    else gemm_short_kernel<T, false><<<dim3(tiles), 256, 0, s>>>(ga);
}
bool launch_gemm_short_group(bool add, int dtype, int tiles, const GemmGroupArgs& ga, hipStream_t s) {
    if (dtype == TP_F16) short_group<f16>(add, tiles, ga, s);
    else if (dtype == TP_BF16) short_group<bf16>(add, tiles, ga, s);
    else return false;
    return true;
}

}  // namespace tp
