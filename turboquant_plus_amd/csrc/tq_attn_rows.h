// k_decode_attn: split-K decode attention for one GQA group of 4 query heads.
//   One 64-lane wavefront owns one context split and walks it in tiles of 64
//   tokens.  Lane l holds packed row l of the tile (K: token l; V: dims l and
//   64+l of all 64 tokens), loaded as 16-byte chunks that are contiguous across
//   lanes.  Codes are turned into fp16 values through a table in LDS: for 2- and
//   3-bit codes a quad table (8-byte entries indexed by the 4*BITS bits of two
//   adjacent pair codes, one ds_read_b64 per four values = one MFMA operand), for
//   4-bit codes a pair table (4-byte entries).  They feed the 4x4x4 fp16 MFMA with
//   16 independent blocks: block b multiplies the 4 tokens 4b..4b+3 by the 4
//   query heads, so all 64 lanes and all 16 blocks do useful work.
//   The MFMA's A-matrix broadcast (cbsz = 4, abid = source block) lets one block's
//   A operand serve all 16 blocks:
//     QK: A = q[4 heads][4 dims] read from block g%16 (each lane keeps only two
//         4-dim slices of q), B_b = K^T[4 dims][tokens 4b..4b+3] -> lane l gets the 4
//         heads' logits of token l; a 4x4 transpose inside each lane quad turns that
//         into head l%4, tokens 4b..4b+3 for the softmax.
//     PV: V rows are dim-major inside the tile (lane l holds dims l and 64+l of the
//         64 tokens), so block b covers dims 4b..4b+3: A = P[4 heads][tokens 4T..4T+3],
//         the fp16 weights held by block T and broadcast, B_b = V[tokens 4T..4T+3][dims
//         4b..4b+3] -> D_b = out[4 heads][4 dims].  16 token groups x 2 dim halves = 32
//         MFMAs per tile into 16 accumulator registers; no cross-lane reduction at the
//         end of the split and no LDS traffic besides the LUT reads.
//   q8_0-style V (VBITS = 8): the same dim-major rows hold int8 values, and the four fp16 scales of a token
//   (one per 32 dims) go into the weights: block b covers dims of one 32-dim block per dim half, so the A
//   operand is broadcast inside each half of the wavefront (cbsz = 3) from weights that were multiplied by that
//   half's scales.
//   Online softmax in base 2 (log2(e) folded into the query scale).  The wavefronts
//   of a workgroup (up to 16 splits) merge their results in LDS and write one partial.
//   The last workgroup of a group to finish merges the group's partials (log-sum-exp), applies the transpose
//   of the V rotation and writes the output rows (merge_group): a step is one launch.  Queries are rotated and
//   scaled inside the kernel.
#pragma once
#include "tq_attn.h"

namespace tqattn {

// QK over the 32 dim groups: B = this lane's K row (4 dims per group), A = q from block G % 16
// (HG sets of four query heads share every dequantised operand: one table look-up, HG products)
template <int BITS, int HG, int... G>
__device__ __forceinline__ void qk_turbo(std::integer_sequence<int, G...>, const uint32_t (&kw)[4 * BITS],
                                         const char *lut, const half4_t (&qa)[HG][2], float4_t (&acc)[HG][4]) {
    (([&] {
         const half4_t kv = quad_values<BITS>(kw, lut, G);
#pragma unroll
         for (int hg = 0; hg < HG; ++hg) acc[hg][G & 3] = mfma4_bcast<(G & 15)>(qa[hg][G >> 4], kv, acc[hg][G & 3]);
     }()),
     ...);
}

// Heads of 256 dims: the lower half of the wavefront holds the rows of the tile's 32 tokens' first 128 dims, the
// upper half the rows of their second 128 dims, and each half takes its half of the query from its own blocks
// (A broadcast inside a half-wavefront, block G % 8; a lane keeps four dim groups)
template <int BITS, int... G>
__device__ __forceinline__ void qk_turbo_d256(std::integer_sequence<int, G...>, const uint32_t (&kw)[4 * BITS],
                                              const char *lut, const half4_t (&qa4)[4], float4_t (&acc)[4]) {
    (([&] {
         const half4_t kv = quad_values<BITS>(kw, lut, G);
         acc[G & 3] = mfma4_bcast8<(G & 7)>(qa4[G >> 3], kv, acc[G & 3]);
     }()),
     ...);
}

template <int... G>
__device__ __forceinline__ void qk_q8_d256(std::integer_sequence<int, G...>, const uint32_t (&kw)[32], const half4_t (&qa4)[4],
                                           float4_t (&acc)[4]) {
    (([&] {
         const half4_t kv = int8x4_to_half_0213(kw[G]);
         acc[G >> 3] = mfma4_bcast8<(G & 7)>(qa4[G >> 3], kv, acc[G >> 3]);
     }()),
     ...);
}

// ... and V rows whose 64 "tokens" are (token, half) pairs: quad T holds the rows of tokens 2T, 2T+1 in the order
// (2T, 0), (2T, 1), (2T+1, 0), (2T+1, 1).  The weights of tokens 4b..4b+3 sit in block b, so quad T takes them from
// block T / 2, with zeros in the places of the other half: one look-up feeds the output's two halves.
template <int BITS, int... T>
__device__ __forceinline__ void pv_all_d256(std::integer_sequence<int, T...>, const uint32_t (&vw)[4 * BITS], const char *lut,
                                            const half4_t (&pv_even)[2], const half4_t (&pv_odd)[2], float4_t (&acc_o)[2][2][2]) {
    (([&] {
         const half4_t v0 = quad_values<BITS>(vw, lut, 2 * T), v1 = quad_values<BITS>(vw, lut, 2 * T + 1);
#pragma unroll
         for (int dh = 0; dh < 2; ++dh) {
             const half4_t w = (T & 1) ? pv_odd[dh] : pv_even[dh];
             acc_o[dh][0][T & 1] = mfma4_bcast<(T >> 1)>(w, v0, acc_o[dh][0][T & 1]);
             acc_o[dh][1][T & 1] = mfma4_bcast<(T >> 1)>(w, v1, acc_o[dh][1][T & 1]);
         }
     }()),
     ...);
}

// q8_0-style K: one accumulator per 32-value block (dim groups 8*blk .. 8*blk+7), scaled afterwards
template <int HG, int... G>
__device__ __forceinline__ void qk_q8(std::integer_sequence<int, G...>, const uint32_t (&kw)[32],
                                      const half4_t (&qa)[HG][2], float4_t (&acc)[HG][4]) {
    // the values of a dim group come out in the order 0, 2, 1, 3; the kernel parks its queries in the same order
    (([&] {
         const half4_t kv = int8x4_to_half_0213(kw[G]);
#pragma unroll
         for (int hg = 0; hg < HG; ++hg) acc[hg][G >> 3] = mfma4_bcast<(G & 15)>(qa[hg][G >> 4], kv, acc[hg][G >> 3]);
     }()),
     ...);
}

// PV over the 16 token groups x 2 dim halves: A = weights of block T (broadcast), B = this lane's V row
template <int BITS, int HG, int... T>
__device__ __forceinline__ void pv_all(std::integer_sequence<int, T...>, const uint32_t (&vw)[4 * BITS],
                                       const char *lut, const half4_t (&pv)[HG], float4_t (&acc_o)[HG][2][2]) {
    // tokens 4T..4T+3 of dim half hf are quad 2T + hf of the row
    (([&] {
         const half4_t v0 = quad_values<BITS>(vw, lut, 2 * T), v1 = quad_values<BITS>(vw, lut, 2 * T + 1);
#pragma unroll
         for (int hg = 0; hg < HG; ++hg) {
             acc_o[hg][0][T & 1] = mfma4_bcast<T>(pv[hg], v0, acc_o[hg][0][T & 1]);
             acc_o[hg][1][T & 1] = mfma4_bcast<T>(pv[hg], v1, acc_o[hg][1][T & 1]);
         }
     }()),
     ...);
}

// q8_0-style V rows: dword 16*hf + T of the row = tokens 4T..4T+3 of dim half hf as int8.  a_lo / a_hi: the weights
// (times the scales of this half-wavefront's 32-dim block of dim half hf) that token groups T < 8 / T >= 8 take
// from block T % 8 of each half-wavefront.
template <int HG, int... T>
__device__ __forceinline__ void pv_all_q8(std::integer_sequence<int, T...>, const uint32_t (&vw)[32],
                                          const half4_t (&a_lo)[HG][2], const half4_t (&a_hi)[HG][2],
                                          float4_t (&acc_o)[HG][2][2]) {
    (([&] {
         const half4_t v0 = int8x4_to_half_0213(vw[T]), v1 = int8x4_to_half_0213(vw[16 + T]);
#pragma unroll
         for (int hg = 0; hg < HG; ++hg) {
             acc_o[hg][0][T & 1] = mfma4_bcast8<(T & 7)>(T < 8 ? a_lo[hg][0] : a_hi[hg][0], v0, acc_o[hg][0][T & 1]);
             acc_o[hg][1][T & 1] = mfma4_bcast8<(T & 7)>(T < 8 ? a_lo[hg][1] : a_hi[hg][1], v1, acc_o[hg][1][T & 1]);
         }
     }()),
     ...);
}

// q8_0-style V rows under heads of 256 dims: dword 16*hf + T = rows 4T..4T+3 = (token 2T, half 0), (2T, 1), (2T+1, 0),
// (2T+1, 1) of dim half hf, handed over in the order 0, 2, 1, 3.  a8[dh][hf][T & 1]: the weights of tokens 2T, 2T+1
// times the scales of their rows of half dh (for this half-wavefront's 32-dim block of dim half hf) in the places of
// that half's rows, zeros in the others; both half-wavefronts hold the same 32 tokens, so token pair T is served by
// block T / 2 of either half with its own scales.
template <int... T>
__device__ __forceinline__ void pv_all_q8_d256(std::integer_sequence<int, T...>, const uint32_t (&vw)[32],
                                               const half4_t (&a8)[2][2][2], float4_t (&acc_o)[2][2][2]) {
    (([&] {
         const half4_t v0 = int8x4_to_half_0213(vw[T]), v1 = int8x4_to_half_0213(vw[16 + T]);
#pragma unroll
         for (int dh = 0; dh < 2; ++dh) {
             acc_o[dh][0][T & 1] = mfma4_bcast8<(T >> 1)>(a8[dh][0][T & 1], v0, acc_o[dh][0][T & 1]);
             acc_o[dh][1][T & 1] = mfma4_bcast8<(T >> 1)>(a8[dh][1][T & 1], v1, acc_o[dh][1][T & 1]);
         }
     }()),
     ...);
}

// per-tile side data of the V rows: turbo = the fp16 norms of this lane's four tokens; q8_0-style = the fp16 scales
// [2 * dim half + swapped]: of this lane's four tokens (0) and of the four tokens of lane ^ 32 (1), for the 32-dim
// block that this lane's dims of that dim half lie in
// heads of 256 dims: the eight fp16 norms of the rows of this lane's four tokens (v[0], v[1]); q8_0-style: the eight
// scales of those rows for the 32-dim block of this lane's dims of dim half hf (v[2 hf], v[2 hf + 1])
template <int VBITS> struct VSide { uint2 v[VBITS == 8 ? 4 : 2]; };

constexpr float Q8V_PRESCALE = 64.0f;  // keeps weight * scale products out of fp16's subnormals; 65504 / 64 > any scale

// SHARE: K and V decode through one table (same width, same centroids); table positions are
// compile-time constants so that they fold into the LDS instructions' offset fields.
//
// Work distribution: a workgroup of W wavefronts (W = blockDim / 64 divides n_splits) owns W
// consecutive splits of one group, one split per wavefront (a fixed share, so results do not
// depend on timing).  The hardware favours the oldest wavefronts of a SIMD, and left alone
// the youngest finish late and alone on a memory system that needs every wavefront's loads
// in flight to stay busy.  So the wavefronts of a workgroup publish their progress in LDS and
// each sets its own issue priority to how many tiles it is behind the leader (at most 3):
// they finish within a tile or two of each other.
// int8 V rows take 32 registers instead of 8 to 16: those variants run with at most 8 wavefronts per workgroup,
// which leaves each more than the 128 registers of a 16-wavefront workgroup.
// Two sets of four query heads per pass (HG = 2: GQA groups of more than four heads read K/V once per eight heads)
// double the accumulators and the softmax state and run with at most 8 wavefronts too.
// Wavefronts per workgroup that a variant is compiled for (its register budget follows: 16 -> 128, 12 -> 168, 8 -> 256).
// wide12: eight heads per pass on turbo K and V rows of 128-dim heads without a bias list - 134-164 registers, so twelve
// wavefronts (three per SIMD) fit where two workgroups of eight do not.
__host__ __device__ constexpr int max_waves_per_workgroup(int vbits, int hg, bool wide12 = false) {
    return vbits == 8 ? 8 : hg == 2 ? (wide12 ? 12 : 8) : 16;
}

// BIAS: none, a sparse logit bias, dense rows, or both.  A template parameter and not branches: the list's cursor registers and
// per-tile test cost the eight-head variant 4 us per step when they were compiled in unconditionally (in the variant of dense rows:
// 8 to 68 bytes of scratch per lane with eight heads or 256 dims, and a wavefront per SIMD next to 8-bit rows; without them dense
// rows of 8 x 8 groups at 8192 tokens, eight heads: turbo3 23.3 -> 21.4 us, turbo3 K with turbo4 V 28.2 -> 23.8, 8-bit K with turbo3
// V 28.2 -> 25.6),
// and a dense row's load that may or may not have been issued makes the compiler wait for the youngest loads, i.e. the V rows
// just requested, at the top of every tile (4 x 20 000 tokens, turbo3, Sparse V: kernel 24.6 -> 22.6 us; 4 x 16 groups at 6000 tokens 15.1 ->
// 14.6; one user at 4000 10.8 -> 10.5).
constexpr int BIAS_NONE = 0, BIAS_LIST = 1, BIAS_DENSE = 2, BIAS_BOTH = BIAS_LIST | BIAS_DENSE;
// D256: heads of 256 dims.  A token is rows 2 token and 2 token + 1 of caches that are
// otherwise those of 128-dim heads with twice the tokens; a 64-row tile is 32 tokens.  The two sets of HG = 2 are
// then the output's two halves of one set of four heads: one softmax, two accumulator sets.
template <int KFMT, int KBITS, int VBITS, bool SPARSE, bool SHARE, int HG, int BIAS, bool D256 = false>
__global__ __launch_bounds__(64 * max_waves_per_workgroup(VBITS, HG, KFMT == KFMT_TURBO && !D256 && !(BIAS & BIAS_LIST)),
                             D256 && KFMT == KFMT_TURBO && VBITS != 8 ? 4 : 1) void k_decode_attn(AttnArgs a) {
    // (256-dim heads on turbo K rows: four wavefronts per SIMD = two workgroups of eight per CU, i.e. at most 128 registers - the
    // variant sits at 119-136 without the bound, and one register over 128 halves its occupancy)
    static_assert(!D256 || HG == 2, "256-dim heads: two accumulator sets, the output's halves");
    constexpr bool LIST = (BIAS & BIAS_LIST) != 0, DENSE = (BIAS & BIAS_DENSE) != 0;
    constexpr int HQ = D256 ? 1 : HG;   // sets of four heads whose logits and softmax state the wavefront keeps
    constexpr int KROW_DW = KFMT == KFMT_TURBO ? 4 * KBITS : 32;
    constexpr int KBLOCK = KFMT == KFMT_TURBO ? TQ_ROWS_PER_BLOCK * (16 * KBITS + 2) : TQ_ROWS_PER_BLOCK * 136;
    constexpr int VBLOCK = VBITS == 8 ? TQ_ROWS_PER_BLOCK * 136 : TQ_ROWS_PER_BLOCK * (16 * VBITS + 2);
    constexpr int KLUT_BYTES = KFMT == KFMT_TURBO ? lut_bytes(KBITS) : 0;
    static_assert(!SHARE || (KFMT == KFMT_TURBO && KBITS == VBITS), "a shared table needs equal code widths");
    // static LDS (its address is a compile-time constant, so table positions fold into the LDS
    // instructions): [K table][V table unless shared with K], and 1 KB per set of four heads that stages the
    // group's rotated queries (a region of its own: the tables are built while the queries are still on their way)
    constexpr int LUT_TOTAL = KLUT_BYTES + (SHARE ? 0 : lut_bytes(VBITS));
    __shared__ __attribute__((aligned(16))) char smem[LUT_TOTAL > 16 ? LUT_TOTAL : 16];
    __shared__ uint32_t lead;  // tiles finished by the wavefront that is furthest ahead
    __shared__ uint32_t skipped;  // Sparse V: (query, position) pairs skipped by this workgroup
    char *klut_s = smem;
    char *vlut_s = SHARE ? klut_s : klut_s + KLUT_BYTES;

    const int tid = threadIdx.x, lane = tid & 63;
    // workgroup-uniform values in scalar registers: tile loop, block addresses and bounds become scalar work
    const int n_waves = (int)(blockDim.x >> 6), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Wavefronts of this workgroup that work on one group: all of them, or - short contexts, a.gpw groups per
    // workgroup - as many as the group has splits; wave_g numbers them, tid_g their threads.
    // (shifts and masks prepared by the host: an integer division here is a few dozen instructions in front of the
    // first row request, which showed as half a microsecond per launch)
    const int gw = a.gpw > 1 ? a.n_splits : n_waves;
    const int wave_g = a.gpw > 1 ? (wave & (gw - 1)) : wave, wave0 = wave - wave_g;
    const int gidx = a.gpw > 1 ? (wave >> a.gw_shift) : 0;   // this wavefront's group among the workgroup's
    const int tid_g = tid - 64 * wave0;
    const int wgs_per_group = a.wgs_per_group;
    const int group = __builtin_amdgcn_readfirstlane(a.gpw > 1 ? (int)blockIdx.x * a.gpw + gidx : (int)(blockIdx.x / wgs_per_group));
    const int part = a.gpw > 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(blockIdx.x % wgs_per_group));
    const int pass_y = HG == 2 ? (int)blockIdx.y : 0;   // one set of four heads is always one pass
    const int head_off = a.head_off + pass_y * a.pass_heads, pgroup = pass_y * a.n_groups + group;
    const int split = part * n_waves + wave_g;  // index of this wavefront's partial
    // dynamic LDS: the wavefronts' merge space (end of the split), then 1 KB per group and set of four heads that
    // stages the rotated queries
    extern __shared__ __attribute__((aligned(16))) float merge_s[];
    char *q_stage = reinterpret_cast<char *>(merge_s) + (size_t)n_waves * HG * MERGE_FLOATS * sizeof(float) +
                    (size_t)gidx * (1024 * HG);
    // The context length: a kernel argument, or read from memory when the caller replays one captured launch at
    // changing lengths (the split geometry then follows the length; a.tokens stays the bias rows' stride).
    int tokens_now = (int)a.tokens, n_tiles = a.n_tiles, tiles_per_split = a.tiles_per_split;
    if (a.tokens_dev) {
        const int64_t t = *a.tokens_dev;
        tokens_now = __builtin_amdgcn_readfirstlane((int)(t < 0 ? 0 : (t < a.tokens ? t : a.tokens)));
        n_tiles = ((D256 ? 2 : 1) * tokens_now + 63) >> 6;
        tiles_per_split = (n_tiles + a.n_splits - 1) / a.n_splits;
    }
    const int rows_now = (D256 ? 2 : 1) * tokens_now;   // rows of the caches that hold the context
    const int t_begin = split * tiles_per_split;
    const int t_end = min(t_begin + tiles_per_split, n_tiles);
    const int b4 = lane & ~3;  // 4 * block index
    const int j = lane & 3;    // query head of the logits this lane holds; sub-row for V
    // K row of the tile that this lane owns, and the tile row of element i of its logits (e4 + es * i)
    const int krow = D256 ? 2 * (lane & 31) + (lane >> 5) : lane;
    const int e4 = D256 ? 2 * (b4 & 31) : b4, es = D256 ? 2 : 1;
    // tokens per tile, and the first of this lane's four tokens inside the tile
    constexpr int TT = D256 ? 32 : 64;
    const int t4 = D256 ? (b4 & 31) : b4;

    const uint8_t *kbase = a.k + (int64_t)group * a.blocks_per_seq * KBLOCK;
    const uint8_t *vbase = a.v + (int64_t)group * a.blocks_per_seq * VBLOCK;
    const char *klut_b = klut_s + (TQ_PAIRTAB3 && KFMT == KFMT_TURBO && KBITS == 3 ? 4 * lane : 0);
    const char *vlut_b = vlut_s + (TQ_PAIRTAB3 && VBITS == 3 ? 4 * lane : 0);

    // The first tile's rows are requested before anything else, so that the query rotation and
    // the table build overlap the first trip to memory.  Afterwards rows are fetched one tile
    // ahead into the same registers: the next K row right after QK has consumed the current
    // one, the next V row right after PV (with Sparse V only after a tile that used its V row).  After the split's last
    // tile the prefetch has every lane read row 0 of that tile's block (a handful of lines, never used): the rows are
    // read with the non-temporal hint, and a clamped re-read of the last tile's 64 rows went to memory again, one tile
    // in sixteen at 1024 tokens per split; a branch around the loads cost the eight-head variant 11 us.  The norms
    // travel with the rows, so no load is waited for in the tile that issued it.
    uint32_t kw[KROW_DW];
    uint32_t vw[4 * VBITS];
    // K: this lane's token's fp16 norm (turbo) or its four fp16 block scales (q8_0-style)
    auto load_knorm = [&](int tile) -> uint2 {
        const uint8_t *kb = kbase + (int64_t)(tile >> 1) * KBLOCK;
        const int r = (tile & 1) * 64 + krow;
        if constexpr (KFMT == KFMT_TURBO)
            return make_uint2(reinterpret_cast<const uint16_t *>(kb + TQ_ROWS_PER_BLOCK * 16 * KBITS)[r], 0u);
        else
            return *reinterpret_cast<const uint2 *>(kb + 8 * 2048 + 8 * r);
    };
    // V: fp16 norms of this lane's four tokens 4b..4b+3, or their q8_0-style scales ([tile][32-dim block][token])
    auto load_vnorm = [&](int tile) -> VSide<VBITS> {
        VSide<VBITS> r;
        const uint8_t *side = vbase + (int64_t)(tile >> 1) * VBLOCK + TQ_ROWS_PER_BLOCK * 16 * VBITS;
        if constexpr (VBITS == 8 && D256) {
            const int bh = lane >> 5;
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {   // rows e4 .. e4 + 7 of the tile: this lane's four tokens, both halves
                const uint4 s8 = *reinterpret_cast<const uint4 *>(side + 2 * ((((tile & 1) * 4 + 2 * hf + bh) * 64) + e4));
                r.v[2 * hf] = make_uint2(s8.x, s8.y);
                r.v[2 * hf + 1] = make_uint2(s8.z, s8.w);
            }
        } else if constexpr (VBITS == 8) {
            const int bh = lane >> 5;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                r.v[e] = *reinterpret_cast<const uint2 *>(side + 2 * ((((tile & 1) * 4 + 2 * (e >> 1) + bh) * 64) +
                                                                      (e & 1 ? b4 ^ 32 : b4)));
        } else if constexpr (D256) {
            const uint4 n8 = *reinterpret_cast<const uint4 *>(side + 2 * ((tile & 1) * 64 + e4));
            r.v[0] = make_uint2(n8.x, n8.y);
            r.v[1] = make_uint2(n8.z, n8.w);
        } else {
            r.v[0] = *reinterpret_cast<const uint2 *>(side + 2 * ((tile & 1) * 64 + b4));
            r.v[1] = make_uint2(0u, 0u);
        }
        return r;
    };
    unsigned long long arrivals_seen = 0ull;
    if (wgs_per_group > 1 && tid == 0) arrivals_seen = ld_dev(arrival_counter(a, pgroup, wgs_per_group));
    uint2 kn = make_uint2(0u, 0u);
    VSide<VBITS> gvu;
#pragma unroll
    for (auto &e : gvu.v) e = make_uint2(0u, 0u);
    int tile = t_begin;
    if (tile < t_end) {
        const int row0 = (tile & 1) * 64 + lane;
        const uint8_t *kb = kbase + (int64_t)(tile >> 1) * KBLOCK;
        if constexpr (KFMT == KFMT_TURBO) load_row<KBITS>(kb, (tile & 1) * 64 + krow, kw);
        else load_row<8>(kb, (tile & 1) * 64 + krow, kw);
        kn = load_knorm(tile);
        load_row<VBITS>(vbase + (int64_t)(tile >> 1) * VBLOCK, row0, vw);
        gvu = load_vnorm(tile);
    }
    if (tid == 0) {
        lead = 0;
        skipped = 0;
    }
    // pair-table entries for the table build below: requested now, needed after the query rotation
    uint32_t kpair = 0, vpair = 0;
    if constexpr (KFMT == KFMT_TURBO && KBITS == 3) kpair = a.klut[lane];
    if constexpr (!SHARE && VBITS == 3) vpair = a.vlut[lane];

    // A operand of QK, broadcast from one block per MFMA: lane (b, i) keeps q[head i] for the
    // dim groups g = b and g = b + 16 (4 dims each); MFMA g reads it from block g % 16.
    // The group's four queries are rotated by the first wavefronts (one 128-point butterfly per
    // head, two values per lane), scaled and parked as fp16 in 1 KB of LDS for everybody.
    auto load_q = [&](int h, float &x0, float &x1) {
        // heads past the group's last one repeat it (their results are not written)
        const int64_t e = D256 ? ((int64_t)group * a.q_group + min(head_off + (h & 3), a.q_group - 1)) * 256 + 128 * (h >> 2) + 2 * lane
                               : ((int64_t)group * a.q_group + min(head_off + h, a.q_group - 1)) * 128 + 2 * lane;
        if (a.q_dtype == TQ_F16) {
            const __half *qp = reinterpret_cast<const __half *>(a.q);
            x0 = __half2float(qp[e]);
            x1 = __half2float(qp[e + 1]);
        } else if (a.q_dtype == TQ_F32) {
            const float *qp = reinterpret_cast<const float *>(a.q);
            x0 = qp[e];
            x1 = qp[e + 1];
        } else {
            const double *qp = reinterpret_cast<const double *>(a.q);
            x0 = (float)qp[e];
            x1 = (float)qp[e + 1];
        }
    };
    // this wavefront's first head is requested now and rotated after the tables are built (the tables need only the
    // pair entries requested above, and nobody reads them before the barrier below)
    float xq0 = 0.0f, xq1 = 0.0f;
    if (wave_g < 4 * HG) load_q(wave_g, xq0, xq1);
    // (placed here, in front of the table build and the query rotation, so that its two dependent trips to memory - the
    // count of entries below the split, then the first window - pass while those run: behind them it delayed every
    // wavefront's first tile)
    // Sparse bias: a head's (position, value) list is walked as the tiles go by, sixteen entries at a time: lane (b, j)
    // holds entry sb_win + b of head j's list (b = lane / 4: the sixteen lanes that hold a head's logits hold a window
    // of its list), so a window is one load per lane, and a tile that has entries adds the window's sixteen to the
    // lanes that own their positions (an entry per dependent trip to memory made a list of 512 positions at the front
    // of the context double the step).  The window starts at the head's first entry inside this split: the number
    // of entries below the split's first token, counted with the whole wavefront (one entry per lane and round).
    int sb_win[HG], sb_pos[HG], sb_last[HG];   // sb_last: the window's last position (a cross-lane read per tile otherwise)
    float sb_val[HG];
#pragma unroll
    for (int hg = 0; hg < HG; ++hg) {
        sb_win[hg] = 0;
        sb_pos[hg] = sb_last[hg] = 0x7FFFFFFF;
        sb_val[hg] = 0.0f;
    }
    // entry e of the list of this lane's head in set hg (addresses are formed where they are needed: the path is rare)
    auto sb_entry = [&](int hg, int e) { return ((int64_t)group * a.q_group + min(head_off + 4 * hg + j, a.q_group - 1)) * a.sbias_n + e; };
    auto sb_load = [&](int hg) {   // this lane's entry of the window
        const int e = sb_win[hg] + (lane >> 2);
        const bool in = e < a.sbias_n;
        sb_pos[hg] = in ? a.sbias_pos[sb_entry(hg, in ? e : 0)] : 0x7FFFFFFF;
        sb_val[hg] = in ? a.sbias_val[sb_entry(hg, in ? e : 0)] : 0.0f;
        sb_last[hg] = __shfl(sb_pos[hg], 60 + j);   // the head's last lanes hold the window's last entry
    };
    if constexpr (LIST) {
        const int first_tok = t_begin * TT;
#pragma unroll
        for (int hg = 0; hg < HQ; ++hg) {
            int below[4];
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const int32_t *prow = a.sbias_pos + ((int64_t)group * a.q_group + min(head_off + 4 * hg + h, a.q_group - 1)) * a.sbias_n;
                int c = 0;
                for (int e0 = 0; e0 < a.sbias_n; e0 += 64) {
                    const int e = e0 + lane;
                    const int pe = e < a.sbias_n ? prow[e] : 0x7FFFFFFF;
                    c += __builtin_popcountll(__builtin_amdgcn_ballot_w64(pe < first_tok));
                }
                below[h] = c;
            }
            sb_win[hg] = j == 0 ? below[0] : j == 1 ? below[1] : j == 2 ? below[2] : below[3];
            sb_load(hg);
        }
    }
    if constexpr (KFMT == KFMT_TURBO) build_lut<KBITS>(klut_s, a.klut, kpair, tid, n_waves);
    if constexpr (!SHARE && VBITS != 8) build_lut<VBITS>(vlut_s, a.vlut, vpair, tid, n_waves);
    for (int h = wave_g; h < 4 * HG; h += gw) {
        _Float16 *qw = reinterpret_cast<_Float16 *>(q_stage) + h * 128;
        float x0 = xq0, x1 = xq1;
        if (h != wave_g) load_q(h, x0, x1);
        if (a.ks1) {
            x0 *= a.ks1[2 * lane];
            x1 *= a.ks1[2 * lane + 1];
            wht128_wave(x0, x1, lane);
            x0 *= a.ks2[2 * lane] * RSQRT128;
            x1 *= a.ks2[2 * lane + 1] * RSQRT128;
        }
        // q8_0-style K rows hand their four values of a dim group over in the order 0, 2, 1, 3 (qk_q8)
        const int d0 = 2 * lane, d1 = 2 * lane + 1;
        const int p0 = KFMT == KFMT_Q8 ? (d0 & ~3) | ((d0 & 1) << 1) | ((d0 >> 1) & 1) : d0;
        const int p1 = KFMT == KFMT_Q8 ? (d1 & ~3) | ((d1 & 1) << 1) | ((d1 >> 1) & 1) : d1;
        // turbo K: the rotated query is rounded to fp16 once, with the logit scale folded in.  q8_0-style K: an
        // fp16 query goes in as it is, so that its products with the int8 values are exact, and the logit scale
        // joins the rows' block scales in fp32 (rounding the scaled query would move logits of rows with large
        // channels by several 1e-3, which a peaked softmax over a long context turns into output error)
        const float qscale = KFMT == KFMT_Q8 ? 1.0f : a.scale_log2e;
        qw[p0] = (_Float16)(x0 * qscale);
        qw[p1] = (_Float16)(x1 * qscale);
    }
    if (wgs_per_group > 1 && tid == 0) install_tag(a, arrival_counter(a, pgroup, wgs_per_group), arrivals_seen);
    __syncthreads();
    half4_t qa[HG][2];
    half4_t qa4[4];   // 256-dim heads: dim groups b, b + 8, b + 16, b + 24 of this half-wavefront's half of the query
#pragma unroll
    for (int hg = 0; hg < HG; ++hg) {
        const uint2 *qp = reinterpret_cast<const uint2 *>(reinterpret_cast<const _Float16 *>(q_stage) + (4 * hg + j) * 128);
        qa[hg][0] = __builtin_bit_cast(half4_t, qp[lane >> 2]);
        qa[hg][1] = __builtin_bit_cast(half4_t, qp[(lane >> 2) + 16]);
    }
    if constexpr (D256) {
        const uint2 *qp = reinterpret_cast<const uint2 *>(reinterpret_cast<const _Float16 *>(q_stage) + (4 * (lane >> 5) + j) * 128);
#pragma unroll
        for (int k = 0; k < 4; ++k) qa4[k] = __builtin_bit_cast(half4_t, qp[((lane >> 2) & 7) + 8 * k]);
    }
    // out[head i][dim 64*hf + lane] partial sums; two chains per dim half for MFMA issue overlap
    float4_t acc_o[HG][2][2];
    float m_run[HG], l_run[HG];
#pragma unroll
    for (int hg = 0; hg < HG; ++hg) {
#pragma unroll
        for (int c = 0; c < 4; ++c) acc_o[hg][c >> 1][c & 1] = float4_t{0.f, 0.f, 0.f, 0.f};
        m_run[hg] = -INFINITY;
        l_run[hg] = 0.0f;
    }
    // additive logit bias of this lane's head and four tokens (natural-log units), one 16-byte load when the row
    // allows it; positions past the context read as 0 (they are masked anyway)
    const bool bias_vec = DENSE && (a.tokens & 3) == 0 && (reinterpret_cast<uintptr_t>(a.bias) & 15u) == 0;
    auto load_bias = [&](int t, int hg, float (&bv)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) bv[i] = 0.0f;
        const int tk = t * TT + t4;  // the launcher checks tokens < 2^31
        const float *row = a.bias + ((int64_t)group * a.q_group + min(head_off + 4 * hg + j, a.q_group - 1)) * a.tokens;
        if (bias_vec && tk + 3 < tokens_now) {
            const float4 v = *reinterpret_cast<const float4 *>(row + tk);
            bv[0] = v.x; bv[1] = v.y; bv[2] = v.z; bv[3] = v.w;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (tk + i < tokens_now) bv[i] = row[tk + i];
        }
    };
    float bias_next[HG][4];
#pragma unroll
    for (int hg = 0; hg < HQ; ++hg) {
        if constexpr (DENSE) load_bias(min(t_begin, max(t_end - 1, 0)), hg, bias_next[hg]);
    }
    unsigned nskip = 0;  // Sparse V: skipped (query, position) pairs of this wavefront (wave-uniform: counted from lane masks)
    bool v_ahead = true;  // Sparse V: this tile's V row was requested while the previous tile was processed

    unsigned long long head_ok[HG];  // lanes whose head (lane % 4 of each set) exists in this pass
#pragma unroll
    for (int hg = 0; hg < HG; ++hg) head_ok[hg] = __builtin_amdgcn_ballot_w64(head_off + 4 * hg + j < a.q_group);
#pragma unroll 1
    while (tile < t_end) {
        const int64_t blk = tile >> 1;
        const int half = tile & 1;
        const int row = half * 64 + lane;
        const uint8_t *vb = vbase + blk * VBLOCK;

        {   // issue priority = tiles behind the leader (wave-uniform, so the branches are scalar)
            const uint32_t done = (uint32_t)(tile - t_begin);
            const uint32_t behind = max(lead_progress(&lead, done, lane), done) - done;
            if (behind == 0) __builtin_amdgcn_s_setprio(0);
            else if (behind == 1) __builtin_amdgcn_s_setprio(1);
            else if (behind == 2) __builtin_amdgcn_s_setprio(2);
            else __builtin_amdgcn_s_setprio(3);
        }
        const int tile_next = tile + 1;
        const int tile_n = min(tile_next, t_end - 1);
        const int row_n = tile_next < t_end ? (tile_n & 1) * 64 + lane : 0;  // past the split: every lane the same row
        const int krow_n = tile_next < t_end ? (tile_n & 1) * 64 + krow : 0;
        const VSide<VBITS> gvu_next = load_vnorm(tile_n);
        const int n_valid = rows_now - tile * 64;   // >= 64 except in the sequence's last tile
        // the bias of this tile was requested a tile ago, like the rows; now the next tile's
        float bias4[HG][4];
#pragma unroll
        for (int hg = 0; hg < HQ; ++hg) {
#pragma unroll
            for (int i = 0; i < 4; ++i) bias4[hg][i] = DENSE ? bias_next[hg][i] * LOG2E : 0.0f;
            if constexpr (DENSE) load_bias(tile_n, hg, bias_next[hg]);
        }
        if constexpr (LIST) {
            // entries of this tile: positions ascend, so a window is done with once its last position lies below the
            // tile's end; a head then takes its next sixteen entries (wave-uniform loop, heads advance on their own)
            const int tile_lo = tile * TT, tile_hi = tile_lo + TT;
#pragma unroll
            for (int hg = 0; hg < HQ; ++hg) {
                bool fresh = true;   // this head's window has not been added to this tile yet
                while (true) {
                    const bool mine = fresh && sb_pos[hg] >= tile_lo && sb_pos[hg] < tile_hi;
                    // window slots (lane / 4) that hold an entry of this tile for any of the four heads
                    unsigned long long slots = __builtin_amdgcn_ballot_w64(mine);
                    slots = (slots | (slots >> 1) | (slots >> 2) | (slots >> 3)) & 0x1111111111111111ull;
                    auto add_slot = [&](int e4) {   // e4 = 4 * slot
                        const int pe = __shfl(sb_pos[hg], e4 + j);
                        const float ve = __shfl(sb_val[hg], e4 + j) * LOG2E;
                        const int d = pe - tile_lo - t4;   // positions outside this lane's four tokens (or this tile) match no i
                        if (fresh) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) bias4[hg][i] += d == i ? ve : 0.0f;
                        }
                    };
#pragma unroll 1
                    while (slots) {   // (unrolled over all sixteen slots this was faster for runs of positions and cost registers)
                        add_slot(__builtin_ctzll(slots));
                        slots &= slots - 1;
                    }
                    fresh = false;
                    const bool advance = sb_last[hg] < tile_hi;   // the whole window lies before the tile's end (padding never does)
                    if (__builtin_amdgcn_ballot_w64(advance) == 0ull) break;
                    if (advance) {
                        sb_win[hg] += 16;
                        fresh = true;
                    }
                    sb_load(hg);   // by every lane (the load ends in a cross-lane read); heads that stay reload what they hold
                }
            }
        }

        // ---- QK ------------------------------------------------------------------
        // D_b[head][token 4b + lane%4]: every lane gets the 4 heads' dot products of its own token
        float sc[HG][4];
        float4_t acc[HG][4];
#pragma unroll
        for (int hg = 0; hg < HG; ++hg)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[hg][c] = float4_t{0.f, 0.f, 0.f, 0.f};
        if constexpr (D256) {
            // each half-wavefront: its half of the query against its rows; a token's two halves meet across lane ^ 32
            float d[4];
            if constexpr (KFMT == KFMT_TURBO) {
                qk_turbo_d256<KBITS>(std::make_integer_sequence<int, 32>{}, kw, klut_b, qa4, acc[0]);
                d[0] = d[1] = d[2] = d[3] = __half2float(__ushort_as_half((unsigned short)kn.x));
            } else {
                qk_q8_d256(std::make_integer_sequence<int, 32>{}, kw, qa4, acc[0]);
                d[0] = __half2float(__ushort_as_half((unsigned short)(kn.x & 0xffff))) * a.scale_log2e;
                d[1] = __half2float(__ushort_as_half((unsigned short)(kn.x >> 16))) * a.scale_log2e;
                d[2] = __half2float(__ushort_as_half((unsigned short)(kn.y & 0xffff))) * a.scale_log2e;
                d[3] = __half2float(__ushort_as_half((unsigned short)(kn.y >> 16))) * a.scale_log2e;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float part = (acc[0][0][i] * d[0] + acc[0][1][i] * d[1]) + (acc[0][2][i] * d[2] + acc[0][3][i] * d[3]);
                sc[0][i] = part + xor_lane<32>(part);
            }
        } else if constexpr (KFMT == KFMT_TURBO) {
            qk_turbo<KBITS, HG>(std::make_integer_sequence<int, 32>{}, kw, klut_b, qa, acc);
            const float gk_own = __half2float(__ushort_as_half((unsigned short)kn.x));
#pragma unroll
            for (int hg = 0; hg < HG; ++hg)
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[hg][i] = ((acc[hg][0][i] + acc[hg][1][i]) + (acc[hg][2][i] + acc[hg][3][i])) * gk_own;
        } else {
            qk_q8<HG>(std::make_integer_sequence<int, 32>{}, kw, qa, acc);
            const uint2 su = kn;
            const float d0 = __half2float(__ushort_as_half((unsigned short)(su.x & 0xffff))) * a.scale_log2e;
            const float d1 = __half2float(__ushort_as_half((unsigned short)(su.x >> 16))) * a.scale_log2e;
            const float d2 = __half2float(__ushort_as_half((unsigned short)(su.y & 0xffff))) * a.scale_log2e;
            const float d3 = __half2float(__ushort_as_half((unsigned short)(su.y >> 16))) * a.scale_log2e;
#pragma unroll
            for (int hg = 0; hg < HG; ++hg)
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[hg][i] = (acc[hg][0][i] * d0 + acc[hg][1][i] * d1) + (acc[hg][2][i] * d2 + acc[hg][3][i] * d3);
        }
        {   // kw is dead now: fetch the next tile's K row into it
            const uint8_t *kbn = kbase + (int64_t)(tile_n >> 1) * KBLOCK;
            if constexpr (KFMT == KFMT_TURBO) load_row<KBITS>(kbn, krow_n, kw);
            else load_row<8>(kbn, krow_n, kw);
            kn = load_knorm(tile_n);
        }
        // -> lane (b, j): head j (of each set), tokens 4b..4b+3; then the online softmax in base 2
        float p[HG][4];
        // Sparse V bookkeeping on the scalar unit: a compare leaves a lane mask, and counting, the in-range test and
        // "does any lane keep anything" are mask arithmetic (the vector ALU only compares and zeroes the weight)
        unsigned long long any_keep = 0, token_ok[4] = {~0ull, ~0ull, ~0ull, ~0ull};
        if constexpr (SPARSE) {
            if (n_valid < 64) {
#pragma unroll
                for (int i = 0; i < 4; ++i) token_ok[i] = __builtin_amdgcn_ballot_w64(e4 + es * i < n_valid);
            }
        }
#pragma unroll
        for (int hg = 0; hg < HQ; ++hg) {
            quad_transpose(sc[hg], lane);
            float s[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] = BIAS ? sc[hg][i] + bias4[hg][i] : sc[hg][i];
            if (n_valid < 64) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (e4 + es * i >= n_valid) s[i] = -INFINITY;
            }
            const float mx = max_over_blocks(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])));
            const float m_new = fmaxf(m_run[hg], mx);
            // After the first tiles the running maximum rarely moves, and a correction factor of exactly 1 changes
            // nothing: the rescaling is skipped when no lane's maximum moved (a wave-uniform branch; same results).
            if (__builtin_amdgcn_ballot_w64(m_new != m_run[hg]) != 0ull) {
                // 0 on the first tile, 1 when the maximum stays (also while every position so far is masked with -inf)
                const float corr = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m_run[hg] - m_new);
                l_run[hg] *= corr;
                // accumulator register i belongs to head i; the factor of head i lives in lanes with lane%4 == i
                const float c0 = dpp<0x00>(corr), c1 = dpp<0x55>(corr), c2 = dpp<0xAA>(corr), c3 = dpp<0xFF>(corr);
#pragma unroll
                for (int ho = 0; ho < HG; ++ho) {
                    if (!D256 && ho != hg) continue;   // 256-dim heads: both halves of the output share the softmax
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        acc_o[ho][c >> 1][c & 1][0] *= c0;
                        acc_o[ho][c >> 1][c & 1][1] *= c1;
                        acc_o[ho][c >> 1][c & 1][2] *= c2;
                        acc_o[ho][c >> 1][c & 1][3] *= c3;
                    }
                }
                m_run[hg] = m_new;
            }
            const float m_ref = m_run[hg] == -INFINITY ? 0.0f : m_run[hg];  // all masked so far: weights are exp2(-inf) = 0, not NaN
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[hg][i] = __builtin_amdgcn_exp2f(s[i] - m_ref);  // results below 2^-126 flush to zero
                l_run[hg] += p[hg][i];
                if constexpr (SPARSE) {
                    const bool keep = p[hg][i] >= a.tau;
                    const unsigned long long keep_m = __builtin_amdgcn_ballot_w64(keep);
                    // 256-dim heads: both half-wavefronts hold the same 32 tokens; the lower one counts
                    const unsigned long long in_range = token_ok[i] & head_ok[hg] & (D256 ? 0xFFFFFFFFull : ~0ull);
                    nskip += (unsigned)__builtin_popcountll(in_range & ~keep_m);
                    if (!keep) p[hg][i] = 0.0f;
                    any_keep |= keep_m & in_range;
                }
            }
        }
        if constexpr (SPARSE) {
            // Every V row of the tile skipped: no dequant, and the next tile's V row is not requested in
            // advance (negligible weights come in runs); a tile that then does need its row fetches it here.
            if (any_keep == 0) {
                gvu = gvu_next;
                tile = tile_next;
                v_ahead = false;
                continue;
            }
            if (!v_ahead) load_row<VBITS>(vb, row, vw);
        }

        // ---- PV ------------------------------------------------------------------------
        // weights (times the stored V norm) as fp16: this lane is token group T = lane/4, head lane%4
        if constexpr (VBITS == 8 && D256) {
            half4_t a8[2][2][2];
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                // scales of rows 8b..8b+7 = (token 4b + i, half h) at 2 i + h
                const uint32_t sw[4] = {gvu.v[2 * hf].x, gvu.v[2 * hf].y, gvu.v[2 * hf + 1].x, gvu.v[2 * hf + 1].y};
#pragma unroll
                for (int dh = 0; dh < 2; ++dh) {
                    _Float16 w[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        w[i] = (_Float16)(p[0][i] * (__half2float(__ushort_as_half((unsigned short)(dh ? sw[i] >> 16 : sw[i] & 0xffff))) *
                                                     Q8V_PRESCALE));
                    const _Float16 z = (_Float16)0.0f;
                    a8[dh][hf][0] = dh ? half4_t{z, z, w[0], w[1]} : half4_t{w[0], w[1], z, z};
                    a8[dh][hf][1] = dh ? half4_t{z, z, w[2], w[3]} : half4_t{w[2], w[3], z, z};
                }
            }
            pv_all_q8_d256(std::make_integer_sequence<int, 16>{}, vw, a8, acc_o);
        } else if constexpr (VBITS == 8) {
            // The dims of block b lie in 32-dim block b / 8 (+ 2 for the upper dim half), so the weights carry that
            // block's scale and are broadcast inside each half of the wavefront: token group T is served by block
            // T % 8 of both halves, which therefore also needs the weights of the lane 32 away.
            auto weights = [&](const float (&w)[4], uint2 sc) {
                const float s0 = __half2float(__ushort_as_half((unsigned short)(sc.x & 0xffff))) * Q8V_PRESCALE;
                const float s1 = __half2float(__ushort_as_half((unsigned short)(sc.x >> 16))) * Q8V_PRESCALE;
                const float s2 = __half2float(__ushort_as_half((unsigned short)(sc.y & 0xffff))) * Q8V_PRESCALE;
                const float s3 = __half2float(__ushort_as_half((unsigned short)(sc.y >> 16))) * Q8V_PRESCALE;
                half4_t r;  // token order 0, 2, 1, 3, as int8x4_to_half_0213 hands the values over
                r[0] = (_Float16)(w[0] * s0);
                r[1] = (_Float16)(w[2] * s2);
                r[2] = (_Float16)(w[1] * s1);
                r[3] = (_Float16)(w[3] * s3);
                return r;
            };
            const bool upper = lane >= 32;
            half4_t a_lo[HG][2], a_hi[HG][2];
#pragma unroll
            for (int hg = 0; hg < HG; ++hg) {
                float ps[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) ps[i] = __shfl_xor(p[hg][i], 32);
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    const half4_t own = weights(p[hg], gvu.v[2 * hf]), swp = weights(ps, gvu.v[2 * hf + 1]);
                    a_lo[hg][hf] = upper ? swp : own;
                    a_hi[hg][hf] = upper ? own : swp;
                }
            }
            pv_all_q8<HG>(std::make_integer_sequence<int, 16>{}, vw, a_lo, a_hi, acc_o);
        } else if constexpr (D256) {
            // norms of rows 8b..8b+7 = (token 4b + i, half h) at 2 i + h
            const uint32_t nw[4] = {gvu.v[0].x, gvu.v[0].y, gvu.v[1].x, gvu.v[1].y};
            half4_t pv_even[2], pv_odd[2];
#pragma unroll
            for (int dh = 0; dh < 2; ++dh) {
                float g[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) g[i] = __half2float(__ushort_as_half((unsigned short)(dh ? nw[i] >> 16 : nw[i] & 0xffff)));
                const _Float16 z = (_Float16)0.0f;
                const _Float16 w0 = (_Float16)(p[0][0] * g[0]), w1 = (_Float16)(p[0][1] * g[1]);
                const _Float16 w2 = (_Float16)(p[0][2] * g[2]), w3 = (_Float16)(p[0][3] * g[3]);
                pv_even[dh] = dh ? half4_t{z, w0, z, w1} : half4_t{w0, z, w1, z};
                pv_odd[dh] = dh ? half4_t{z, w2, z, w3} : half4_t{w2, z, w3, z};
            }
            pv_all_d256<VBITS>(std::make_integer_sequence<int, 16>{}, vw, vlut_b, pv_even, pv_odd, acc_o);
        } else {
            const float g0 = __half2float(__ushort_as_half((unsigned short)(gvu.v[0].x & 0xffff)));
            const float g1 = __half2float(__ushort_as_half((unsigned short)(gvu.v[0].x >> 16)));
            const float g2 = __half2float(__ushort_as_half((unsigned short)(gvu.v[0].y & 0xffff)));
            const float g3 = __half2float(__ushort_as_half((unsigned short)(gvu.v[0].y >> 16)));
            half4_t pv[HG];
#pragma unroll
            for (int hg = 0; hg < HG; ++hg) {
                pv[hg][0] = (_Float16)(p[hg][0] * g0);
                pv[hg][1] = (_Float16)(p[hg][1] * g1);
                pv[hg][2] = (_Float16)(p[hg][2] * g2);
                pv[hg][3] = (_Float16)(p[hg][3] * g3);
            }
            // V row of this lane: dims lane and 64+lane for the tile's 64 tokens; quad 2T + hf =
            // tokens 4T..4T+3 of dim half hf.  Block b = lane/4 of the MFMA covers dims 4b..4b+3 (+64*hf); the
            // weights of token group T sit in block T and are broadcast to every block.
            pv_all<VBITS, HG>(std::make_integer_sequence<int, 16>{}, vw, vlut_b, pv, acc_o);
        }
        load_row<VBITS>(vbase + (int64_t)(tile_n >> 1) * VBLOCK, row_n, vw);
        v_ahead = true;
        gvu = gvu_next;
        tile = tile_next;
    }

    // ---- end of split: the workgroup's wavefronts merge their partials in LDS and write one ------
    if constexpr (VBITS == 8) {
#pragma unroll
        for (int hg = 0; hg < HG; ++hg)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc_o[hg][c >> 1][c & 1] *= 1.0f / Q8V_PRESCALE;
    }
    float l_tot[HG];
#pragma unroll
    for (int hg = 0; hg < HG; ++hg) l_tot[hg] = sum_over_blocks(l_run[hg]);
    if constexpr (D256) {
        // both half-wavefronts added the same 32 weights; the second accumulator set shares the softmax state
        l_tot[0] *= 0.5f;
        l_tot[1] = l_tot[0];
        m_run[1] = m_run[0];
    }
    auto slot = [&](int w) { return merge_s + w * (MERGE_FLOATS * HG); };
    float *mine = slot(wave);
#pragma unroll
    for (int hg = 0; hg < HG; ++hg) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int i = 0; i < 4; ++i) mine[hg * MERGE_FLOATS + i * 128 + 64 * hf + lane] = acc_o[hg][hf][0][i] + acc_o[hg][hf][1][i];
        if (lane < 4) *reinterpret_cast<float2 *>(mine + hg * MERGE_FLOATS + 512 + 2 * j) = make_float2(m_run[hg], l_tot[hg]);
    }
    if (SPARSE && lane == 0 && nskip) atomicAdd(&skipped, nskip);
    finish_group<HG, SPARSE>(a, slot, group, pgroup, head_off, wgs_per_group, part, tid, tid_g, gw, wave0, merge_s, &skipped);
}

// by the bias that the call carries
#define TQ_ATTN_LAUNCH(KF, KB, VB, SP, SH, HG, D256)                                                        \
    {                                                                                                      \
        if (a.bias && a.sbias_n) k_decode_attn<KF, KB, VB, SP, SH, HG, BIAS_BOTH, D256><<<grid, wg, lds, s>>>(a); \
        else if (a.bias) k_decode_attn<KF, KB, VB, SP, SH, HG, BIAS_DENSE, D256><<<grid, wg, lds, s>>>(a);  \
        else if (a.sbias_n) k_decode_attn<KF, KB, VB, SP, SH, HG, BIAS_LIST, D256><<<grid, wg, lds, s>>>(a); \
        else k_decode_attn<KF, KB, VB, SP, SH, HG, BIAS_NONE, D256><<<grid, wg, lds, s>>>(a);               \
    }
// ... one or two sets of four heads, and Sparse V
#define TQ_ATTN_PAIR(KF, KB, VB, SH)                                        \
    {                                                                      \
        if (hg == 2 && sparse) TQ_ATTN_LAUNCH(KF, KB, VB, true, SH, 2, false)   \
        else if (hg == 2) TQ_ATTN_LAUNCH(KF, KB, VB, false, SH, 2, false)       \
        else if (sparse) TQ_ATTN_LAUNCH(KF, KB, VB, true, SH, 1, false)         \
        else TQ_ATTN_LAUNCH(KF, KB, VB, false, SH, 1, false)                    \
        return true;                                                       \
    }
#define TQ_ATTN_256(KF, KB, VB, SH)                                         \
    {                                                                      \
        if (sparse) TQ_ATTN_LAUNCH(KF, KB, VB, true, SH, 2, true)               \
        else TQ_ATTN_LAUNCH(KF, KB, VB, false, SH, 2, true)                     \
        return true;                                                       \
    }

}  // namespace tqattn
