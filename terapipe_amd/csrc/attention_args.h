// Pieces shared by the attention translation units.
#pragma once
#include "common.h"

namespace tp {

struct AttnArgs {
    const void* q; const void* kc; const void* vc; void* o; float* lse;
    const void* d_o; float* delta; void* dqkv; void* gk; void* gv;
    int B, H, T, P;
    long cache_rows;
    int nsplit;
    float* part_o; float* part_lse;
    int accumulate_prefix, has_incoming, zero_slice_rows;
    const void* gk_in; const void* gv_in;   // where the incoming gradients lie: gk, gv, or caches of their own
    int grad_rows;                          // rows of the gradient caches that the call writes: P + T, or all
    int dq_only;
    int shared_queries, shared_keys;    // dQ / dK and dV by workgroups of 128 rows (attention_long.hip)
    float qscale;
    long q_bhs;      // elements between consecutive (batch, head) blocks of q
    long st_bhs;     // floats between consecutive (batch, head) blocks of lse / delta
};

static constexpr float kLog2e = 1.4426950408889634f;

// v_exp_f32: 2^x at hardware precision (about 1 ulp), results below the normal range flush to zero
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

template <typename T, int DH>
__device__ __forceinline__ void load_row_operands(typename Elem<T>::opnd_t* reg, const T* rowptr, bool valid, int g) {
    typedef Elem<T> E;
    constexpr int NKS = DH / E::KSTEP;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        if constexpr (sizeof(T) == 2) {
            reg[ks] = valid ? *reinterpret_cast<const uint4*>(rowptr + ks * 16 + 8 * g) : make_uint4(0, 0, 0, 0);
        } else {
            reg[ks] = valid ? rowptr[ks * 2 + g] : 0.f;
        }
    }
}

// Workgroups are dealt to the eight XCDs round-robin by linear id.  This maps the linear id to
// (batch*head, block) so that all blocks of one (batch, head) run on the same XCD and its K / V / Q / dO
// rows are fetched into one L2 only.  Launch with xcd_grid(BH, nblocks) workgroups; false = no work.
__device__ __forceinline__ bool xcd_map(int BH, int& bh, int& blk, int id = blockIdx.x) {
    const int xcd = id & 7, slot = id >> 3;
    const int nbh8 = (BH + 7) >> 3;
    bh = xcd + 8 * (slot % nbh8);
    blk = slot / nbh8;
    return bh < BH;
}
static inline unsigned xcd_grid(int BH, int nblocks) { return 8u * ((BH + 7) / 8) * nblocks; }

// ---- shared pieces of the second-generation 16-bit attention kernels -------------------------------

// LDS tiles of these kernels have rows of 64 or 128 elements (the swizzle's power of two).  Head dimensions between (80,
// 96) take rows of 128 whose last chunks are never loaded: their products run over the dimension's own k-steps of 16,
// and the output blocks of 32 columns may end past it (columns 80 to 95 of a head of 80 are computed on whatever the
// LDS holds there and not stored).
template <int DH> __host__ __device__ constexpr int tile_pitch() { return DH <= 64 ? 64 : 128; }
constexpr unsigned kNoChunk = 0xffffffffu;      // a lane whose chunk of the tile row lies past the head dimension
template <int DH> __device__ __forceinline__ void load_chunk_lds(unsigned off, const void* base, unsigned lds_wave_base) {
    if (DH == tile_pitch<DH>() || off != kNoChunk) dma16_saddr_lds(off, base, lds_wave_base);
}

// Wave-private transpose of a [DH x 32] fp32 accumulator set (register j of block db = row db*32 +
// acc_row(j, g), column lane & 31) into row-major [32][DH] through LDS, so that global memory is then
// touched in full rows.  `buf` is the wave's own 32 x (DH + 4) floats.  After the call lane l holds, for
// i in [0, DH / 8): row 2 * i' ... see rows_read.
template <int DH>
__device__ __forceinline__ void acc_to_lds_rows(const float16v* acc, float* buf, int lane) {
    constexpr int NDB = (DH + 31) / 32, LD = NDB * 32 + 4;
    const int g = lane >> 5, li = lane & 31;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq)
            *reinterpret_cast<float4*>(buf + li * LD + db * 32 + 8 * jq + 4 * g) =
                make_float4(acc[db][4 * jq], acc[db][4 * jq + 1], acc[db][4 * jq + 2], acc[db][4 * jq + 3]);
}

// The part of a key block's rows [first, first + BLK) that lies past the call's positions, in both gradient caches: the incoming
// gradient, or zeros.  False: the block has no other rows.  (uniform over the workgroup of NT threads)
// Copying both caches before the call read and wrote them once more than the call itself does, in two launches: 2 x 5.8 us for 25
// heads of 64 at 2048 positions, 2 x 9.8 for 40 of 128; here the rows below P cost nothing that the in-place form does not read.
template <typename GT, int DH, int BLK, int NT, typename Args>
__device__ __forceinline__ bool grad_rows_beyond(const Args& a, int bh, int first, int S, int tid) {
    const int lo = max(first, S), n = (min(first + BLK, a.grad_rows) - lo) * (DH * (int)sizeof(GT) / 16);
    const long off = ((long)bh * a.cache_rows + lo) * (DH * (int)sizeof(GT) / 16);
    uint4 *k = reinterpret_cast<uint4*>(a.gk) + off, *v = reinterpret_cast<uint4*>(a.gv) + off;
    if (a.gk_in) {
        const uint4 *ki = reinterpret_cast<const uint4*>(a.gk_in) + off, *vi = reinterpret_cast<const uint4*>(a.gv_in) + off;
        for (int i = tid; i < n; i += NT) {
            const uint4 x = ki[i], y = vi[i];
            k[i] = x;
            v[i] = y;
        }
    } else {
        for (int i = tid; i < n; i += NT) k[i] = v[i] = make_uint4(0, 0, 0, 0);
    }
    return first < S;
}

// piece i of the row-major read-back: row and first column of the four floats this lane gets
template <int DH> __device__ __forceinline__ void row_piece(int i, int lane, int& row, int& col) {
    constexpr int LPR = DH / 4;            // lanes per row
    const int idx = i * 64 + lane;
    row = idx / LPR;
    col = (idx % LPR) * 4;
}

// Calls of 128 queries and more against shared K / V tiles (attention_long.hip; 16-bit, head dimensions 64 to 128).
void launch_attn_fwd_long(int dtype, int head_dim, const AttnArgs& a, hipStream_t s);
void launch_attn_dq_long(int dtype, int head_dim, const AttnArgs& a, hipStream_t s);       // (leaves delta too)
// dK / dV of the keys [key0, key_end) against queries 0 .. nq - 1, which lie at the positions q_pos + i (attention_long.hip).  Row
// k - slice0 of dqkv takes key k from slice0 on; without `suffix` the gradient caches are as in AttnArgs.
struct AttnKeysArgs {
    const void* kc; const void* vc; const void* q; const void* d_o;
    const float* lse; const float* delta; void* dqkv; void* gk; void* gv;
    int B, H, key0, key_end, slice0, nq, q_pos;
    int accumulate_prefix, has_incoming, zero_slice_rows;
    const void* gk_in; const void* gv_in;
    int grad_rows;
    long cache_rows, q_bhs, st_bhs;
};
void launch_attn_dkdv_long(int dtype, int head_dim, bool suffix, const AttnKeysArgs& a, hipStream_t s);
// fp32, all head dimensions: 32 rows a workgroup, its waves sharing the other axis (attention_f32.hip); the backward's delta
// comes with its dQ launch.
void launch_attn_f32(bool backward, int head_dim, const AttnArgs& a, hipStream_t s);

}  // namespace tp
