// Attention over packed KV and the prefill-shaped score tile.
//
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
// k_score_tile: TurboQuant inner-product estimate, 32x32x16 fp16 MFMA over a
//   K = 256 contraction ([R q | S q] against [g c[idx] | scale*rnorm*z]); key operands in registers, queries
//   through LDS, logit rows written 64 consecutive logits per store.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <cstring>
#include <type_traits>
#include <utility>

#include "tq_attn.h"

namespace {

using namespace tqattn;

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
// wide12: eight heads per pass on turbo K and V rows of 128-dim heads without a bias list - 145-165 registers, so twelve
// wavefronts (three per SIMD) fit where two workgroups of eight do not.
__host__ __device__ constexpr int max_waves_per_workgroup(int vbits, int hg, bool wide12 = false) {
    return vbits == 8 ? 8 : hg == 2 ? (wide12 ? 12 : 8) : 16;
}

// SBIAS: the call carries a sparse logit bias (a.sbias_n > 0).  A template parameter and not a branch: the cursor
// registers and the per-tile test cost the eight-head variant 4 us per step when they were compiled in unconditionally.
// D256: heads of 256 dims.  A token is rows 2 token and 2 token + 1 of caches that are
// otherwise those of 128-dim heads with twice the tokens; a 64-row tile is 32 tokens.  The two sets of HG = 2 are
// then the output's two halves of one set of four heads: one softmax, two accumulator sets.
template <int KFMT, int KBITS, int VBITS, bool SPARSE, bool SHARE, int HG, bool SBIAS, bool D256 = false>
__global__ __launch_bounds__(64 * max_waves_per_workgroup(VBITS, HG, KFMT == KFMT_TURBO && !D256 && !SBIAS),
                             D256 && KFMT == KFMT_TURBO && VBITS != 8 ? 4 : 1) void k_decode_attn(AttnArgs a) {
    // (256-dim heads on turbo K rows: four wavefronts per SIMD = two workgroups of eight per CU, i.e. at most 128 registers - the
    // variant sits at 119-136 without the bound, and one register over 128 halves its occupancy)
    static_assert(!D256 || HG == 2, "256-dim heads: two accumulator sets, the output's halves");
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
    if constexpr (SBIAS) {
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
    const bool bias_vec = a.bias && (a.tokens & 3) == 0 && (reinterpret_cast<uintptr_t>(a.bias) & 15u) == 0;
    auto load_bias = [&](int t, int hg, float (&bv)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) bv[i] = 0.0f;
        if (!a.bias) return;
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
    for (int hg = 0; hg < HQ; ++hg) load_bias(min(t_begin, max(t_end - 1, 0)), hg, bias_next[hg]);
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
            for (int i = 0; i < 4; ++i) bias4[hg][i] = bias_next[hg][i] * LOG2E;
            load_bias(tile_n, hg, bias_next[hg]);
        }
        if constexpr (SBIAS) {
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
            for (int i = 0; i < 4; ++i) s[i] = sc[hg][i] + bias4[hg][i];
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

// Sparse-V bookkeeping for launches with more groups than one workgroup polls (and for a caller that asks for the
// counts of a dense step): skip[0] = the sum of the decode workgroups' slots (plus the earlier passes'), skip[1] =
// all (query, position) pairs.  One workgroup.
__global__ __launch_bounds__(1024) void k_skip_sum(const unsigned long long *slots, int n_slots, unsigned long long *skip,
                                                   unsigned long long total_pairs, int accumulate) {
    __shared__ unsigned long long red;
    unsigned long long t = 0ull;
    for (int i = (int)threadIdx.x; i < n_slots; i += (int)blockDim.x) t += slots[i] & SKIP_COUNT_MASK;
    const unsigned long long sum = block_sum(t, &red, (int)threadIdx.x);
    if (threadIdx.x == 0) {
        skip[0] = (accumulate ? skip[0] : 0ull) + sum;
        skip[1] = total_pairs;
    }
}

constexpr int MAX_POLLED_SLOTS = 4096;  // workgroups of a launch whose Sparse-V slots the merging workgroups add up themselves
constexpr int MAX_PASSES = 64;           // four-head passes of one step (query heads per KV head <= 256)

inline int64_t align256(int64_t v) { return (v + 255) & ~(int64_t)255; }

// a value that no earlier call of this process used and that leftovers in a fresh workspace are unlikely to
// equal (splitmix64 of a process-wide counter; never 0, which is what a lowered flag holds)
std::atomic<unsigned long long> g_attn_seq{0};
unsigned long long next_nonce() {
    unsigned long long z = (g_attn_seq.fetch_add(1, std::memory_order_relaxed) + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (z >> 40) ? z : z | (1ull << 63);  // the upper 24 bits tag the Sparse-V words and must not be zero
}

struct WsLayout {
    int64_t part_o, part_ml, skip_slots, flags, pass_totals, total;
};
// How a parameter set is run: sets of four query heads per pass (2 when a KV head serves more than four query
// heads), wavefronts per workgroup (the largest power of two up to the variant's limit that divides the split
// count) and workgroups = partials per group.
struct AttnPlan {
    int hg, wpw, n_parts, gpw;
};
AttnPlan attn_plan(const tq_attn_params *p, bool bias_list) {
    AttnPlan pl;
    // 256-dim heads run as two accumulator sets (the output's halves) of one set of four heads
    pl.hg = p->head_dim == 256 || p->n_q_heads / p->n_kv_heads > 4 ? 2 : 1;
    const bool turbo_k = p->k_format == TQ_KFMT_TURBO, turbo_v = p->v_format == TQ_KFMT_TURBO;
    const bool wide12 = turbo_k && p->head_dim != 256 && !bias_list;
    pl.wpw = max_waves_per_workgroup(turbo_v ? 0 : 8, pl.hg, wide12);
    if (pl.wpw == 12 && p->n_splits % 12 != 0) pl.wpw = 8;
    while (p->n_splits % pl.wpw) pl.wpw >>= 1;
    // few groups (small batches): smaller workgroups, so that every CU gets one (a tile costs a wavefront the same
    // issue time however many share the SIMD)
    const int64_t groups = (int64_t)p->batch * p->n_kv_heads;
    // short contexts: a group has fewer splits than a workgroup has room for wavefronts.  Several groups then share a
    // workgroup (and its decode tables), provided that still makes a workgroup per CU
    const int wmax = max_waves_per_workgroup(turbo_v ? 0 : 8, pl.hg);   // groups share a workgroup in powers of two
    pl.gpw = 1;
    if (p->n_splits < wmax && wmax % p->n_splits == 0) {
        int g = wmax / p->n_splits;
        while (g > 1 && (groups % g != 0 || groups / g < 256)) g >>= 1;
        if (g > 1) {
            pl.gpw = g;
            pl.wpw = g * p->n_splits;
            pl.n_parts = 1;
            return pl;
        }
    }
    while (pl.wpw > 4 && pl.wpw % 2 == 0 && groups * (p->n_splits / pl.wpw) < 256) pl.wpw >>= 1;
    pl.n_parts = p->n_splits / pl.wpw;
    return pl;
}
int heads_per_pass(const tq_attn_params *p) { return p->head_dim == 256 || p->n_q_heads / p->n_kv_heads <= 4 ? 4 : 8; }
int passes_of(const tq_attn_params *p) { return (p->n_q_heads / p->n_kv_heads + heads_per_pass(p) - 1) / heads_per_pass(p); }
// passes: of a launch
WsLayout ws_layout(const tq_attn_params *p, int passes) {
    const int64_t groups = (int64_t)p->batch * p->n_kv_heads * passes;
    // a call with a bias list may run smaller workgroups (more partials per group) than one without: room for either
    const AttnPlan pl = attn_plan(p, false), pl_list = attn_plan(p, true);
    const int64_t parts = groups * (pl.n_parts > pl_list.n_parts ? pl.n_parts : pl_list.n_parts);
    WsLayout w;
    w.part_o = 0;
    w.part_ml = w.part_o + align256(parts * 4 * pl.hg * 128 * 4);
    w.skip_slots = w.part_ml + align256(parts * 4 * pl.hg * 2 * 4);
    w.flags = w.skip_slots + align256(parts * 8);
    w.pass_totals = w.flags + align256(parts * 8);
    w.total = w.pass_totals + align256(MAX_PASSES * 8);
    return w;
}

}  // namespace

int64_t tqk_attn_workspace_bytes(const tq_attn_params *p) { return ws_layout(p, p->sparse_v_tau > 0.0f ? 1 : passes_of(p)).total; }

int tqk_decode_attention(const tq_handle *hk, const tq_handle *hv, const tq_attn_params *p, const void *q, int q_dtype,
                         const void *k, const void *k_aux, const void *v, const float *bias, float *out,
                         unsigned long long *skip_count, void *ws, int64_t ws_bytes, hipStream_t s) {
    (void)k_aux;
    // All passes in one launch where the workspace has room: each is a chain of its own (launch, first rows, merge), one of few
    // groups leaves most of the chip idle, and they read the same rows.  Steps of two passes over 256-dim heads (us with the
    // append, one pass after the other / together): 2 x 8 KV heads x 259 tokens turbo4 35.0 / 19.6, 4 x 8 x 4000 turbo3 50.5 / 32.8,
    // 1 x 1 x 100 000 turbo2 169 / 95, 8 x 4 x 16 000 8-bit K with turbo3 V 86.2 / 82.4, 16 x 8 x 12 000 turbo4 180 / 174 to 178.
    // Sparse V counts pass by pass.
    int n_pass = p->sparse_v_tau > 0.0f ? 1 : passes_of(p);
    if (n_pass > 1 && ws_bytes < ws_layout(p, n_pass).total) n_pass = 1;
    const WsLayout w = ws_layout(p, n_pass);
    if (ws_bytes < w.total) {
        tq_set_error("tq_decode_attention: workspace %lld < %lld bytes", (long long)ws_bytes, (long long)w.total);
        return TQ_ERR_ARG;
    }
    const int64_t rows = (int64_t)p->batch * p->n_q_heads;
    const int groups = p->batch * p->n_kv_heads;
    const bool d256 = p->head_dim == 256;
    if (p->head_dim != 0 && p->head_dim != 128 && p->head_dim != 256) {
        tq_set_error("tq_decode_attention: head_dim %d (128 or 256)", (int)p->head_dim);
        return TQ_ERR_UNSUPPORTED;
    }
    const int64_t cache_rows = (d256 ? 2 : 1) * p->tokens;   // a 256-dim token is two rows of the caches
    float *part_o = reinterpret_cast<float *>((char *)ws + w.part_o);
    float *part_ml = reinterpret_cast<float *>((char *)ws + w.part_ml);
    const bool turbo_k = p->k_format == TQ_KFMT_TURBO;
    const float sc = p->scale * LOG2E;
    const unsigned long long total_pairs = (unsigned long long)rows * (unsigned long long)p->tokens;
    int rc = TQ_OK;
    if (q_dtype != TQ_F16 && q_dtype != TQ_F32 && q_dtype != TQ_F64) {
        tq_set_error("bad q dtype %d", q_dtype);
        return TQ_ERR_ARG;
    }

    AttnArgs a;
    a.q = q;
    a.q_dtype = q_dtype;
    a.ks1 = turbo_k ? hk->s1_32 : nullptr;
    a.ks2 = turbo_k ? hk->s2_32 : nullptr;
    a.scale_log2e = sc;
    a.k = (const uint8_t *)k;
    a.v = (const uint8_t *)v;
    a.klut = turbo_k ? (const uint32_t *)hk->pair_lut : nullptr;
    const bool turbo_v = p->v_format == TQ_KFMT_TURBO;
    a.vlut = turbo_v ? (const uint32_t *)hv->pair_lut : nullptr;
    const float *vs1 = turbo_v ? hv->s1_32 : nullptr, *vs2 = turbo_v ? hv->s2_32 : nullptr;
    const bool share = turbo_k && turbo_v && hk->bits == hv->bits &&
                       std::memcmp(hk->pair_lut_host, hv->pair_lut_host, sizeof(hk->pair_lut_host)) == 0;
    a.bias = bias;
    a.sbias_n = p->bias_entries;
    a.sbias_pos = p->bias_pos;
    a.sbias_val = p->bias_val;
    if (p->bias_entries < 0 || (p->bias_entries > 0 && (!p->bias_pos || !p->bias_val))) {
        tq_set_error("tq_decode_attention: bias_entries %d needs bias_pos and bias_val", (int)p->bias_entries);
        return TQ_ERR_ARG;
    }
    a.part_o = part_o;
    a.part_ml = part_ml;
    a.skip_slots = reinterpret_cast<unsigned long long *>((char *)ws + w.skip_slots);
    if (cache_rows >= ((int64_t)1 << 31)) {
        tq_set_error("tq_decode_attention: tokens %lld beyond 2^31 - 1", (long long)p->tokens);
        return TQ_ERR_UNSUPPORTED;
    }
    a.tokens = p->tokens;
    a.tokens_dev = p->tokens_dev;
    if (p->tokens_dev && skip_count) {
        tq_set_error("tq_decode_attention: the Sparse-V count is not kept for a context length read from memory (tokens_dev)");
        return TQ_ERR_UNSUPPORTED;
    }
    a.blocks_per_seq = ((d256 ? 2 : 1) * (p->capacity > 0 ? p->capacity : p->tokens) + TQ_ROWS_PER_BLOCK - 1) / TQ_ROWS_PER_BLOCK;
    a.n_groups = groups;
    a.n_splits = p->n_splits;
    a.n_tiles = (int)((cache_rows + 63) / 64);
    a.d256 = d256 ? 1 : 0;
    a.tiles_per_split = (a.n_tiles + p->n_splits - 1) / p->n_splits;
    a.tau = p->sparse_v_tau;
    const bool sparse = p->sparse_v_tau > 0.0f;
    if (sparse && !skip_count) {
        tq_set_error("tq_decode_attention: sparse_v_tau > 0 needs skip_count");
        return TQ_ERR_ARG;
    }
    // wavefronts per workgroup: the largest power of two up to 16 (8 for int8 V rows and for eight heads per pass)
    // that divides the split count
    const AttnPlan pl = attn_plan(p, p->bias_entries > 0);
    const int wpw = pl.wpw, hg = pl.hg;
    const unsigned pass_wgs = (unsigned)((int64_t)groups * pl.n_parts / pl.gpw);
    const dim3 grid(pass_wgs, n_pass);
    const unsigned wg = 64u * (unsigned)wpw;
    // dynamic LDS: the wavefronts' merge space, then the staged queries of the workgroup's groups
    const size_t merge_bytes = (size_t)wpw * hg * MERGE_FLOATS * sizeof(float) + (size_t)pl.gpw * 1024 * hg;
    a.gpw = pl.gpw;
    a.gw_shift = 0;
    while ((1 << a.gw_shift) < p->n_splits) ++a.gw_shift;
    a.wgs_per_group = pl.gpw > 1 ? 1 : p->n_splits / wpw;
    const int vb = turbo_v ? hv->bits : 8;
    const int kb = turbo_k ? hk->bits : 8;
    // The kernels work on four query heads of a KV head at a time (the 4-row MFMA block), or on eight (two sets
    // against the same dequantised rows) when a KV head serves more than four: a group of G heads takes
    // ceil(G / 8) passes over the same K/V; a last pass with fewer heads than it has rows repeats the group's
    // last head and does not write the repeats.
    a.q_group = p->n_q_heads / p->n_kv_heads;
    a.pass_heads = heads_per_pass(p);
    if (passes_of(p) > MAX_PASSES) {
        tq_set_error("tq_decode_attention: %d query heads per KV head (at most %d)", a.q_group, 4 * MAX_PASSES);
        return TQ_ERR_UNSUPPORTED;
    }
    a.out = out;
    a.vs1 = vs1;
    a.vs2 = vs2;
    a.flags = reinterpret_cast<unsigned long long *>((char *)ws + w.flags);
    a.poll_slots = sparse && pass_wgs <= (unsigned)MAX_POLLED_SLOTS;
    a.pass_totals = reinterpret_cast<unsigned long long *>((char *)ws + w.pass_totals);
    a.skip_count = skip_count;
    a.total_pairs = total_pairs;
    // A 4-bit side: k_decode_turbo, whose table of 64 KB has a copy per lane (16 x 8 groups at 32768 tokens, turbo4: 110 -> 97 us,
    // eight heads 121 -> 90; turbo4 K with turbo2 V 87 -> 77 and 100 -> 78).  It has to leave the workgroups that share a CU room
    // (25 x 8 groups at 3175 tokens in 1000 workgroups of four: 30.5 us against 28.4 here; turbo4 K with turbo3 V, 96 KB, 20 x 8
    // groups of eight heads at 2500 tokens in 320: 32.0 against 25.7), and building it has to pay: three tiles per wavefront and
    // four wavefronts (2 x 8 groups at 3000 tokens, three: 12.7 us against 13.2 here; 8 at 4000, two: 11.7 against 11.5; one at
    // 300, two wavefronts: 12.1 against 11.5).  Four heads with a bias list have no registers for it (16 x 9000 tokens with 64
    // entries: 41.4 against 38.8, with Sparse V 47.6 against 43.0), and dense bias rows keep the general variants.
    const int tables = tqk_decode_turbo_lds(kb, vb, share) + pl.gpw * 1024 * hg;
    const int per_cu = std::min((int)(((int64_t)pass_wgs * n_pass + 255) / 256), std::max(1, (hg == 2 ? 12 : 16) / wpw));
    const bool lane_tables = (kb == 4 || vb == 4) && per_cu * tables <= 160 * 1024 && a.tiles_per_split >= 3 && wpw >= 4 &&
                             !bias && (hg == 2 || !a.sbias_n);
    for (a.head_off = 0; a.head_off < a.q_group; a.head_off += n_pass * a.pass_heads) {
        a.pass = a.head_off / a.pass_heads;
        a.nonce = next_nonce();
        if (d256) {
#define TQ_ATTN_256_ONE(KF, KB, VB, SH)                                                                              \
    {                                                                                                                 \
        if (sparse && a.sbias_n) k_decode_attn<KF, KB, VB, true, SH, 2, true, true><<<grid, wg, merge_bytes, s>>>(a);  \
        else if (sparse) k_decode_attn<KF, KB, VB, true, SH, 2, false, true><<<grid, wg, merge_bytes, s>>>(a);         \
        else if (a.sbias_n) k_decode_attn<KF, KB, VB, false, SH, 2, true, true><<<grid, wg, merge_bytes, s>>>(a);      \
        else k_decode_attn<KF, KB, VB, false, SH, 2, false, true><<<grid, wg, merge_bytes, s>>>(a);                   \
    }
#define TQ_ATTN_256(B)                                   \
    if (share) TQ_ATTN_256_ONE(KFMT_TURBO, B, B, true)   \
    else TQ_ATTN_256_ONE(KFMT_TURBO, B, B, false)
#define TQ_ATTN_256X(KF, KB, VB) TQ_ATTN_256_ONE(KF, KB, VB, false)
            if (turbo_k && kb == vb && kb == 3) { TQ_ATTN_256(3); }
            else if (turbo_k && kb == vb && kb == 4) { TQ_ATTN_256(4); }
            else if (turbo_k && kb == vb && kb == 2) { TQ_ATTN_256(2); }
            else if (turbo_k && kb == 4 && vb == 2) { TQ_ATTN_256X(KFMT_TURBO, 4, 2); }
            else if (turbo_k && kb == 3 && vb == 2) { TQ_ATTN_256X(KFMT_TURBO, 3, 2); }
            else if (turbo_k && kb == 4 && vb == 3) { TQ_ATTN_256X(KFMT_TURBO, 4, 3); }
            else if (!turbo_k && vb == 2) { TQ_ATTN_256X(KFMT_Q8, 3, 2); }
            else if (!turbo_k && vb == 3) { TQ_ATTN_256X(KFMT_Q8, 3, 3); }
            else if (!turbo_k && vb == 4) { TQ_ATTN_256X(KFMT_Q8, 3, 4); }
            else if (!turbo_k && vb == 8) { TQ_ATTN_256X(KFMT_Q8, 3, 8); }
            else if (turbo_k && kb == 2 && vb == 8) { TQ_ATTN_256X(KFMT_TURBO, 2, 8); }
            else if (turbo_k && kb == 3 && vb == 8) { TQ_ATTN_256X(KFMT_TURBO, 3, 8); }
            else if (turbo_k && kb == 4 && vb == 8) { TQ_ATTN_256X(KFMT_TURBO, 4, 8); }
            else {
                tq_set_error("tq_decode_attention: head_dim 256 with K %d bits, V %d bits is not built", kb, vb);
                return TQ_ERR_UNSUPPORTED;
            }
#undef TQ_ATTN_256
#undef TQ_ATTN_256X
#undef TQ_ATTN_256_ONE
        } else {
#define TQ_ATTN_ONE(KF, KB, VB, SP, SH)                                            \
    {                                                                             \
        if (hg == 2 && a.sbias_n) k_decode_attn<KF, KB, VB, SP, SH, 2, true><<<grid, wg, merge_bytes, s>>>(a);   \
        else if (hg == 2) k_decode_attn<KF, KB, VB, SP, SH, 2, false><<<grid, wg, merge_bytes, s>>>(a);        \
        else if (a.sbias_n) k_decode_attn<KF, KB, VB, SP, SH, 1, true><<<grid, wg, merge_bytes, s>>>(a);        \
        else k_decode_attn<KF, KB, VB, SP, SH, 1, false><<<grid, wg, merge_bytes, s>>>(a);                      \
    }
#define TQ_ATTN(KF, KB, VB)                         \
    if (sparse) TQ_ATTN_ONE(KF, KB, VB, true, false)  \
    else TQ_ATTN_ONE(KF, KB, VB, false, false)
    // same width and same centroids: one table
#define TQ_ATTN_SAME(B)                                         \
    if (share && sparse) TQ_ATTN_ONE(KFMT_TURBO, B, B, true, true)    \
    else if (share) TQ_ATTN_ONE(KFMT_TURBO, B, B, false, true)        \
    else if (sparse) TQ_ATTN_ONE(KFMT_TURBO, B, B, true, false)       \
    else TQ_ATTN_ONE(KFMT_TURBO, B, B, false, false)
    if (turbo_k && turbo_v && lane_tables && tqk_launch_decode_turbo(a, kb, vb, share, 4 * hg, sparse, grid, wpw, s)) {}
    else if (turbo_k && kb == 3 && vb == 3) { TQ_ATTN_SAME(3); }
    else if (turbo_k && kb == 4 && vb == 4) { TQ_ATTN_SAME(4); }
    else if (turbo_k && kb == 2 && vb == 2) { TQ_ATTN_SAME(2); }
    else if (turbo_k && kb == 4 && vb == 2) { TQ_ATTN(KFMT_TURBO, 4, 2); }
    else if (turbo_k && kb == 3 && vb == 2) { TQ_ATTN(KFMT_TURBO, 3, 2); }
    else if (turbo_k && kb == 3 && vb == 4) { TQ_ATTN(KFMT_TURBO, 3, 4); }
    else if (turbo_k && kb == 4 && vb == 3) { TQ_ATTN(KFMT_TURBO, 4, 3); }
    else if (turbo_k && kb == 2 && vb == 3) { TQ_ATTN(KFMT_TURBO, 2, 3); }
    else if (turbo_k && kb == 2 && vb == 4) { TQ_ATTN(KFMT_TURBO, 2, 4); }
    else if (turbo_k && kb == 2 && vb == 8) { TQ_ATTN(KFMT_TURBO, 2, 8); }
    else if (!turbo_k && vb == 2) { TQ_ATTN(KFMT_Q8, 3, 2); }
    else if (!turbo_k && vb == 3) { TQ_ATTN(KFMT_Q8, 3, 3); }
    else if (!turbo_k && vb == 4) { TQ_ATTN(KFMT_Q8, 3, 4); }
    else if (!turbo_k && vb == 8) { TQ_ATTN(KFMT_Q8, 3, 8); }
    else if (turbo_k && kb == 3 && vb == 8) { TQ_ATTN(KFMT_TURBO, 3, 8); }
    else if (turbo_k && kb == 4 && vb == 8) { TQ_ATTN(KFMT_TURBO, 4, 8); }
    else {
        tq_set_error("tq_decode_attention: unsupported K/V format pair (k bits %d, v bits %d)", kb, vb);
        return TQ_ERR_UNSUPPORTED;
    }
        }
#undef TQ_ATTN
#undef TQ_ATTN_SAME
#undef TQ_ATTN_ONE
    rc = tq_check_launch("decode_attn");
    if (rc) return rc;
    if (skip_count && !a.poll_slots) {
        // more groups than the finishing workgroups poll (or a dense step whose caller wants the counts)
        k_skip_sum<<<1, 1024, 0, s>>>(a.skip_slots, sparse ? (int)pass_wgs : 0, skip_count, total_pairs, a.head_off > 0);
        rc = tq_check_launch("skip_sum");
        if (rc) return rc;
    }
    }
    return TQ_OK;
}

// ---- decode attention for callers that cannot allocate -----------------------------------
// The split partials live in a file-scope device array instead of a caller's workspace.  Every
// GPU the library runs on holds its own copy of the array, at its own address, until the process
// ends; the address is looked up once per device (with that device current) and kept.  In host
// code the array's name is only a handle for that lookup, never a device address.
namespace {
constexpr int64_t STATIC_WS_BYTES = TQ_STATIC_WORKSPACE_BYTES;
static __device__ __align__(256) unsigned char scratch[STATIC_WS_BYTES];
constexpr int MAX_DEVICES = 64;
void *g_scratch_ptr[MAX_DEVICES];  // per device: device address of that GPU's copy of `scratch`
std::mutex g_scratch_mutex;
}  // namespace

// Device address of the current device's scratch array (looked up on the first call per device).
int tqk_static_scratch(void **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
        tq_set_error("static workspace: hipGetDevice: %s (device %d)", hipGetErrorString(e), dev);
        return TQ_ERR_HIP;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            tq_set_error("static workspace: hipGetSymbolAddress: %s", hipGetErrorString(e));
            return TQ_ERR_HIP;
        }
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return TQ_OK;
}

int tqk_decode_attention_static(const tq_handle *hk, const tq_handle *hv, const tq_attn_params *p, const void *q,
                                int q_dtype, const void *k, const void *v, const float *bias, float *out,
                                unsigned long long *skip_count, hipStream_t s) {
    const int64_t need = ws_layout(p, 1).total;
    if (need > STATIC_WS_BYTES) {
        tq_set_error("tq_decode_attention_static: batch * n_kv_heads * n_splits = %lld needs %lld bytes of split "
                     "partials, the built-in workspace holds %lld; lower n_splits or use tq_decode_attention",
                     (long long)p->batch * p->n_kv_heads * p->n_splits, (long long)need, (long long)STATIC_WS_BYTES);
        return TQ_ERR_UNSUPPORTED;
    }
    void *ptr = nullptr;
    const int rc = tqk_static_scratch(&ptr);
    if (rc) return rc;
    // every partial and every skip slot that the merge kernel reads is written by this call's main kernel first,
    // so nothing of the previous call's contents needs clearing
    return tqk_decode_attention(hk, hv, p, q, q_dtype, k, nullptr, v, bias, out, skip_count, ptr, STATIC_WS_BYTES, s);
}

// ---- prefill-shaped TurboQuant inner-product estimator --------------------------------
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
constexpr int KT_STRIDE = 264;  // halves per staged key row (256 + 8: 16-byte reads of 16 rows hit 64 distinct banks)

// [R q | S q] as fp16 on the matrix cores: a workgroup of four wavefronts takes 32 queries, wavefront w the output
// rows 32w .. 32w+31 of the rotation and of the projection, as (W Q^T) with W's fragments prepared with the handle
// (rotation: +-1 entries, exact; projection: two fp16 terms) and the queries as the column side.  Queries that are
// not fp16 are split into two fp16 terms as well, so that every product is exact and the sums carry fp32 rounding
// only (as the scalar loop did).  Lane l ends up with query l % 32 and four consecutive outputs per register
// group: an 8-byte store, 512 contiguous bytes per wavefront.
template <typename TI>
__global__ __launch_bounds__(256) void k_prep_score_q(const TI *q, __half *qa, int64_t nq, const uint4 *wfrag) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 31, kb = lane >> 5;
    const int64_t blk = blockIdx.x;
    const int64_t v = min(blk * 32 + r, nq - 1);  // rows past the last query repeat it (their block is allocated)
    constexpr bool SPLIT = !std::is_same<TI, __half>::value;
    half8_t xh[8], xl[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const TI *src = q + v * 128 + 16 * t + 8 * kb;
        if constexpr (!SPLIT) {
            xh[t] = *reinterpret_cast<const half8_t *>(src);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = ldf(src + e);
                const _Float16 hi = (_Float16)x;
                xh[t][e] = hi;
                xl[t][e] = (_Float16)(x - (float)hi);
            }
        }
    }
    constexpr int SET = 4 * 8 * 64;  // fragments (16 bytes) per set
    const uint4 *fr = wfrag + (w * 8) * 64 + lane;
    float16_t rot, prj;
#pragma unroll
    for (int e = 0; e < 16; ++e) rot[e] = prj[e] = 0.0f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const half8_t wr = __builtin_bit_cast(half8_t, fr[t * 64]);
        const half8_t wh = __builtin_bit_cast(half8_t, fr[SET + t * 64]);
        const half8_t wl = __builtin_bit_cast(half8_t, fr[2 * SET + t * 64]);
        rot = __builtin_amdgcn_mfma_f32_32x32x16_f16(wr, xh[t], rot, 0, 0, 0);
        prj = __builtin_amdgcn_mfma_f32_32x32x16_f16(wl, xh[t], prj, 0, 0, 0);
        if constexpr (SPLIT) {
            rot = __builtin_amdgcn_mfma_f32_32x32x16_f16(wr, xl[t], rot, 0, 0, 0);
            prj = __builtin_amdgcn_mfma_f32_32x32x16_f16(wh, xl[t], prj, 0, 0, 0);
        }
        prj = __builtin_amdgcn_mfma_f32_32x32x16_f16(wh, xh[t], prj, 0, 0, 0);
    }
    // operand-major layout: the 16-byte chunk (row r of query block v / 32, K values 16t + 8kb .. + 7) that
    // lane r + 32kb of the score tile's MFMA reads in K step t sits at chunk index (block * 16 + t) * 64 + r + 32kb,
    // so one wave-wide operand load is 1 KB of contiguous memory.  Register group j of this lane holds outputs
    // 32w + 8j + 4kb + i, i = 0..3: elements 4kb .. 4kb+3 of the chunk of step (32w + 8j) / 16, half (j & 1).
#pragma unroll
    for (int part = 0; part < 2; ++part)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int o = 128 * part + 32 * w + 8 * j;  // first K value of the chunk
            const int t = o >> 4, half_sel = (o >> 3) & 1;
            const float sc = part == 0 ? RSQRT128 : 1.0f;
            const float16_t &a = part == 0 ? rot : prj;
            const __half2 lo2 = __halves2half2(__float2half_rn(a[4 * j] * sc), __float2half_rn(a[4 * j + 1] * sc));
            const __half2 hi2 = __halves2half2(__float2half_rn(a[4 * j + 2] * sc), __float2half_rn(a[4 * j + 3] * sc));
            uint2 u;
            u.x = *reinterpret_cast<const uint32_t *>(&lo2);
            u.y = *reinterpret_cast<const uint32_t *>(&hi2);
            *reinterpret_cast<uint2 *>(qa + (((blk * 16 + t) * 64 + r + 32 * half_sel) * 8 + 4 * kb)) = u;
        }
}

// One workgroup of eight wavefronts per 256 keys.  The keys are dequantised once into LDS as fp16
// [g*c[idx] | scale*rnorm*z]; every wavefront then takes the operands of its 64 keys into registers (128 of
// them) and the same LDS carries the queries instead, 128 at a time, double-buffered, brought in by loads that
// write LDS directly.  Matrix tiles are 32 x 32 x 16 with the queries on the M side and the keys on the N side.
// Wavefront w works on key group w % 4 (64 keys) and on the query half w / 4 of a tile, 32 queries at a time:
// per K step one query operand from LDS feeds two matrix instructions (the two 32-key halves of the group).
// The four wavefronts of a query half finish the same 32 logit rows at about the same time, each its own 64
// logits of them, so a row leaves the workgroup as 256 consecutive logits (1 KB in fp32) within a short time,
// not as 128-byte pieces spread over a sweep: the memory side takes that order markedly faster.
constexpr int SCORE_KEYS = 256;  // keys per workgroup (two 128-row blocks)
constexpr int SCORE_QT = 128;  // queries per LDS tile: four operand blocks of 16 KB
template <int BITS, typename TO, bool DRAIN>
__global__ __launch_bounds__(512, 1) void k_score_tile(const __half *qa, const uint8_t *packed, const uint8_t *sign_bits,
                                                      const __half *rnorms, int64_t nq, int64_t nk, TO *logits,
                                                      const uint32_t *pair_lut, float proj_scale, int tiles_per) {
    extern __shared__ __attribute__((aligned(16))) _Float16 kt[];  // keys [SCORE_KEYS][KT_STRIDE], then two query tiles
    __shared__ uint32_t ptab[1 << (2 * BITS)];                     // pair code -> (c[lo], c[hi]) as two halves
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t key0 = (int64_t)blockIdx.x * SCORE_KEYS;
    const int n_blocks = (int)((nq + 31) / 32);  // operand blocks the preparation wrote
    // the query tiles of this workgroup: all of them, or a share where few keys leave CUs without a workgroup
    const int t_begin = (int)blockIdx.y * tiles_per, t_end = min(t_begin + tiles_per, (int)((nq + SCORE_QT - 1) / SCORE_QT));
    typedef uint32_t chunk_t __attribute__((ext_vector_type(4)));   // 16 bytes: what a lane feeds to one matrix instruction
    const chunk_t *qchunks = reinterpret_cast<const chunk_t *>(qa);  // [block][K step][lane]
    // chunk group g (0..7) of a tile: lanes tid + 512 g of its 4096 chunks, i.e. half g % 2 of operand block g / 2
    auto tile_chunk = [&](int tile, int g) __attribute__((always_inline)) {
        const int blk = min(tile * (SCORE_QT / 32) + (g >> 1), n_blocks - 1);  // past the end: the last block again
        return qchunks + (int64_t)blk * 1024 + (g & 1) * 512 + tid;
    };
    // the first tile is requested before anything else and waits in registers until the keys have left LDS
    chunk_t first_tile[8];
#pragma unroll
    for (int g = 0; g < 8; ++g) first_tile[g] = *tile_chunk(t_begin, g);
    if (tid < (1 << (2 * BITS))) ptab[tid] = pair_lut[tid];
    __syncthreads();
    {
        // threads 0..255 dequantise the codes of one key each, threads 256..511 its sign bits; eight halves
        // (16 bytes) per LDS write
        typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
        const int key = tid & (SCORE_KEYS - 1), part = tid >> 8;
        uint4 *row = reinterpret_cast<uint4 *>(kt + key * KT_STRIDE) + part * 16;
        const bool valid = key0 + key < nk;
        if (part == 0) {
            if (valid) {
                const uint8_t *block = packed + (key0 + key) / TQ_ROWS_PER_BLOCK * (TQ_ROWS_PER_BLOCK * (16 * BITS + 2));
                uint32_t wv[4 * BITS];
                load_row<BITS>(block, key & (TQ_ROWS_PER_BLOCK - 1), wv);
                const _Float16 g = __builtin_bit_cast(
                    _Float16, reinterpret_cast<const unsigned short *>(block + TQ_ROWS_PER_BLOCK * 16 * BITS)[key & (TQ_ROWS_PER_BLOCK - 1)]);
                const half2_t g2 = {g, g};
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    uint32_t u[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t e = *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(ptab) +
                                                                               pair_off<BITS>(wv, 4 * c + i));
                        u[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, e) * g2);
                    }
                    row[c] = make_uint4(u[0], u[1], u[2], u[3]);
                }
            } else {
#pragma unroll
                for (int c = 0; c < 16; ++c) row[c] = make_uint4(0, 0, 0, 0);
            }
        } else {
            float rs = 0.f;
            uint4 sb = make_uint4(0, 0, 0, 0);
            if (valid) {
                rs = proj_scale * __half2float(rnorms[key0 + key]);
                sb = *reinterpret_cast<const uint4 *>(sign_bits + (key0 + key) * 16);
            }
            const uint32_t sw[4] = {sb.x, sb.y, sb.z, sb.w};
            // +rs where the bit is set, -rs where it is clear: two halves per word, the sign bits from the inverted bits
            const uint32_t mag = (uint32_t)__half_as_ushort(__float2half_rn(rs)) * 0x00010001u;
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                uint32_t u[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int jj = 8 * c + 2 * i;  // sign bits jj, jj + 1
                    const uint32_t nb = ~sw[jj >> 5] >> (jj & 31);
                    u[i] = mag ^ (((nb & 1u) << 15) | ((nb & 2u) << 30));
                }
                row[c] = make_uint4(u[0], u[1], u[2], u[3]);
            }
        }
    }
    __syncthreads();

    // lane l of a 32 x 32 result tile holds key column l % 32 for the query rows 8j + 4(l/32) + i
    const int kg = __builtin_amdgcn_readfirstlane(w & 3), qh = __builtin_amdgcn_readfirstlane(w >> 2);
    const int c32 = lane & 31, kb = lane >> 5;
    half8_t kf[2][16];  // [32-key half of the group][K step of 16]
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
        for (int t = 0; t < 16; ++t)
            kf[kh][t] = *reinterpret_cast<const half8_t *>(kt + (kg * 64 + kh * 32 + c32) * KT_STRIDE + t * 16 + 8 * kb);
    __syncthreads();  // every wavefront has its keys: the memory now holds query tiles
    chunk_t *qtile = reinterpret_cast<chunk_t *>(kt);  // [2][4096] chunks
#pragma unroll
    for (int g = 0; g < 8; ++g) qtile[g * 512 + tid] = first_tile[g];
    // (LDS only: a __syncthreads would also wait for the logit stores in flight)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // A finished (32 queries, 64 keys) block is written while the next one is being multiplied: one store
    // instruction after each matrix instruction, from a second set of accumulators.  One v_permlane32_swap per
    // accumulator pair puts the row 8j + i of both key halves into one register (lanes 0..31 the first half's 32
    // keys, lanes 32..63 the second's) and the row 8j + 4 + i into the other, so a store writes 64 consecutive
    // logits of one row.  The stores are buffer stores whose resource is that row's piece (scalar arithmetic): its
    // size is 0 for a row past the last query and ends at the last key, so the hardware drops what does not exist
    // and no store needs an address register or a branch.
    constexpr int NT_AUX = (TQ_STREAM_SITES & STREAM_LOGITS) ? 2 : 0;  // the non-temporal bit of a buffer instruction
    const int64_t key0w = key0 + kg * 64;
    const uint32_t piece_bytes = (uint32_t)max((int64_t)0, min((int64_t)64, nk - key0w)) * (uint32_t)sizeof(TO);
    const int lane_off = lane * (int)sizeof(TO);
    struct Pending {
        TO *base;  // first logit of the block's first row in this wavefront's key group
        int rows;  // rows of the block that exist (0: nothing is pending)
    };
    auto pend = [&](int row0) __attribute__((always_inline)) {
        Pending pb;
        pb.rows = __builtin_amdgcn_readfirstlane(max(0, min(32, (int)nq - row0)));
        const uint64_t b = reinterpret_cast<uint64_t>(logits + (int64_t)row0 * nk + key0w);
        // wave-uniform by construction; said explicitly so that the resources are built by scalar instructions
        pb.base = reinterpret_cast<TO *>(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32) |
                                         (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b));
        return pb;
    };
    auto store_row = [&](const Pending &pb, const uint32_t bits, const int row) __attribute__((always_inline)) {
        const uint32_t size = row < pb.rows ? piece_bytes : 0u;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(pb.base + (int64_t)row * nk, 0, (int)size, 0x00020000);
        if constexpr (sizeof(TO) == 4) {
            __builtin_amdgcn_raw_buffer_store_b32(bits, rs, lane_off, 0, NT_AUX);
        } else {
            __builtin_amdgcn_raw_buffer_store_b16(__half_as_ushort(__float2half_rn(__uint_as_float(bits))), rs, lane_off, 0, NT_AUX);
        }
    };

    float keep = 0.0f;  // measurement mode (no logits): the products stay live through a store that never happens
    // one block of 32 queries (operand block `b` of the tile in `cur`) against the 64 resident keys into acc, while
    // the pending block leaves from pacc; the first block of a tile also asks for the next tile (eight loads that
    // write LDS directly, one per step: no registers, no LDS write instructions, and a lead of at least 20 steps).
    // Query operands come from LDS AHEAD steps ahead, across blocks too: `pre` holds the first AHEAD operands of this
    // block on entry and those of the block that follows (operand block `b_after` of the buffer `after`) on exit.  The
    // second block of a tile therefore carries the tile's barrier, at the step in which its own last operand read has
    // been issued: behind it no wavefront reads `cur` any more, so the next tile may start filling it, and `next` is
    // complete.  Vector memory operations complete in issue order and 21 steps of two stores each lie between a
    // tile's last load and that step, so "at most 32 outstanding" covers the loads with a margin and leaves the
    // youngest logit stores in flight (a __syncthreads would wait for all of them).
    constexpr int AHEAD = 3;
    auto block = [&](const chunk_t *cur, chunk_t *next, const int b, const chunk_t *after, const int b_after, auto half,
                     const int tile_next, half8_t (&pre)[AHEAD], float16_t (&acc)[2], const float16_t (&pacc)[2],
                     const Pending &pb) __attribute__((always_inline)) {
        constexpr int HALF = decltype(half)::value;
        const float16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        const chunk_t *arow = cur + b * 1024 + lane;
        const chunk_t *arow_after = after + b_after * 1024 + lane;
        // the scheduling fence after every step keeps the compiler from hoisting all sixteen steps' reads to the top
        half8_t af[AHEAD + 1];
#pragma unroll
        for (int t = 0; t < AHEAD; ++t) af[t] = pre[t];
        uint32_t swapped = 0u;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            if (t + AHEAD < 16) af[(t + AHEAD) & AHEAD] = __builtin_bit_cast(half8_t, arow[(t + AHEAD) * 64]);
            if (HALF == 1 && t + AHEAD == 16) {
                if constexpr (DRAIN) asm volatile("s_waitcnt vmcnt(32) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
            if (t + AHEAD >= 16) pre[t + AHEAD - 16] = __builtin_bit_cast(half8_t, arow_after[(t + AHEAD - 16) * 64]);
            if (HALF == 0 && t < 8) {
                // lane l of the wavefront brings chunk l of the wavefront's 1 KB piece of chunk group g
                const int g = t;
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(tile_chunk(tile_next, g)),
                                                 (__attribute__((address_space(3))) void *)(next + g * 512 + w * 64), 16, 0, 0);
            }
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) {
                acc[kh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[t & AHEAD], kf[kh][t], t == 0 ? zero : acc[kh], 0, 0, 0);
                if constexpr (DRAIN) {
                    // accumulator element t = 4j + i: rows 8j + i (kh = 0 here) and 8j + 4 + i (kh = 1)
                    const int row = 8 * (t >> 2) + (t & 3);
                    if (kh == 0) {
                        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(pacc[0][t]), __float_as_uint(pacc[1][t]), false, false);
                        swapped = r[1];
                        store_row(pb, r[0], row);
                    } else {
                        store_row(pb, swapped, row + 4);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!DRAIN) {
#pragma unroll
            for (int kh = 0; kh < 2; ++kh)
#pragma unroll
                for (int e = 0; e < 16; ++e) keep += acc[kh][e];
        }
    };
    float16_t acc_a[2], acc_b[2];
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc_b[kh][e] = 0.0f;
    Pending pb = pend(0);
    pb.rows = 0;  // nothing is pending before the first block
    half8_t pre[AHEAD];
#pragma unroll
    for (int t = 0; t < AHEAD; ++t) pre[t] = __builtin_bit_cast(half8_t, qtile[(2 * qh) * 1024 + t * 64 + lane]);
#pragma unroll 1
    for (int tile = t_begin; tile < t_end; ++tile) {
        const chunk_t *cur = qtile + ((tile - t_begin) & 1) * 4096;
        chunk_t *next = qtile + ((tile - t_begin + 1) & 1) * 4096;
        const int row0 = tile * SCORE_QT + qh * 64;
        const int tile_next = min(tile + 1, t_end - 1);  // the last tile re-reads itself
        block(cur, next, 2 * qh, cur, 2 * qh + 1, std::integral_constant<int, 0>{}, tile_next, pre, acc_a, acc_b, pb);
        pb = pend(row0);
        block(cur, next, 2 * qh + 1, next, 2 * qh, std::integral_constant<int, 1>{}, tile_next, pre, acc_b, acc_a, pb);
        pb = pend(row0 + 32);
    }
    if constexpr (DRAIN) {  // the last block (in acc_b)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc_b[0][e]), __float_as_uint(acc_b[1][e]), false, false);
            const int row = 8 * (e >> 2) + (e & 3);
            store_row(pb, r[0], row);
            store_row(pb, r[1], row + 4);
        }
    } else {
        if (keep == 1.25e38f) reinterpret_cast<float *>(const_cast<__half *>(qa))[0] = keep;
    }
}

}  // namespace

int tqk_score_tile(const tq_handle *h, const void *q, int q_dtype, int64_t nq, const void *packed,
                   const uint8_t *sign_bits, const void *rnorms, int64_t nk, void *logits, int out_dtype, void *ws,
                   int64_t ws_bytes, hipStream_t s) {
    (void)ws_bytes;
    if (nq >= ((int64_t)1 << 31) / 128) {
        tq_set_error("tq_score_tile: %lld queries beyond 2^24 - 1", (long long)nq);
        return TQ_ERR_UNSUPPORTED;
    }
    __half *qa = reinterpret_cast<__half *>(ws);
    const unsigned qgrid = (unsigned)((nq + 31) / 32);
    const uint4 *wfrag = reinterpret_cast<const uint4 *>(h->score_wfrag);
    switch (q_dtype) {
    case TQ_F16: k_prep_score_q<__half><<<qgrid, 256, 0, s>>>((const __half *)q, qa, nq, wfrag); break;
    case TQ_F32: k_prep_score_q<float><<<qgrid, 256, 0, s>>>((const float *)q, qa, nq, wfrag); break;
    case TQ_F64: k_prep_score_q<double><<<qgrid, 256, 0, s>>>((const double *)q, qa, nq, wfrag); break;
    default: tq_set_error("bad q dtype %d", q_dtype); return TQ_ERR_ARG;
    }
    int rc = tq_check_launch("prep_score_q");
    if (rc) return rc;
    // A workgroup per 256 keys, one to a CU; fewer keys than fill the chip: the query tiles are shared out too, up to one round
    // of workgroups (each dequantises its keys again, side by side).  Scores and their preparation, us, not shared / shared: 11 835
    // keys x 962 queries 30 / 24, x 2048 51 / 42; 2000 x 2048 48 / 13.
    const int64_t key_wgs = (nk + SCORE_KEYS - 1) / SCORE_KEYS, tiles = (nq + SCORE_QT - 1) / SCORE_QT;
    const int64_t shares = std::max<int64_t>(1, std::min(tiles, 256 / key_wgs));
    const int tiles_per = (int)((tiles + shares - 1) / shares);
    const dim3 grid((unsigned)key_wgs, (unsigned)((tiles + tiles_per - 1) / tiles_per));
    const size_t lds = (size_t)SCORE_KEYS * KT_STRIDE * sizeof(_Float16);
#define TQ_SCORE(B, T, DR)                                                                                             \
    {                                                                                                                  \
        (void)hipFuncSetAttribute((const void *)k_score_tile<B, T, DR>, hipFuncAttributeMaxDynamicSharedMemorySize,   \
                                  (int)lds);                                                                           \
        k_score_tile<B, T, DR><<<grid, 512, lds, s>>>(qa, (const uint8_t *)packed, sign_bits, (const __half *)rnorms, \
                                                      nq, nk, (T *)logits, (const uint32_t *)h->pair_lut, (float)h->proj_scale, tiles_per); \
    }
#define TQ_SCORE_BITS(T, DR)                                                                              \
    if (h->bits == 2) TQ_SCORE(2, T, DR) else if (h->bits == 3) TQ_SCORE(3, T, DR) else TQ_SCORE(4, T, DR)
    if (!logits) {
        TQ_SCORE_BITS(float, false)  // measurement mode: everything but the stores
    } else if (out_dtype == TQ_F32) {
        TQ_SCORE_BITS(float, true)
    } else {
        TQ_SCORE_BITS(__half, true)
    }
#undef TQ_SCORE_BITS
#undef TQ_SCORE
    return tq_check_launch("score_tile");
}
