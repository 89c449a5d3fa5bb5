// Decode attention over turbo K and turbo V rows of 128-dim heads with 4-bit codes on a side: k_decode_turbo.
//
// What bounded the general kernel (k_decode_attn) on 4-bit rows was the LDS: two look-ups per four values in a 1 KB table, whose
// lanes meet in its banks (5 clocks and more per look-up for the 2 that 64 four-byte reads need), and with eight heads the 4x4x4
// matrix instructions.  Here the 256 pair entries lie once per lane (64 KB): no conflicts, and a position is one byte permute.
// 16 x 8 groups at 32768 tokens, turbo4: 110 -> 97 us (557 MB, 5.7 TB/s), eight heads 121 -> 90; 6 x 8 groups of eight heads at
// 10 007 tokens 27.5 -> 22.6.
// Pairs of 2- and 3-bit codes stay with the general kernel: their quad tables (one 8-byte read per four values, 6.4 clocks) have no
// room for copies, so only the matrix side would change, which is worth 8 us of 94 with eight heads, and costs 1 us of 80 with four
// (28 swaps and 16 permutes per tile for 41 instructions of transposing).  Eight heads alone are not moved here either: a head on 2- and
// 3-bit rows then has the same bits however many share its pass (where its splits are merged in one order), which it would lose.  (On rows with a 4-bit side it has them within
// either kernel, but which one runs may depend on the number of heads: the room for the tables, a list beside four heads.)
//
// One wavefront owns one context split and walks it in tiles of 64 tokens.  Both products run on the 16x16x32 fp16 matrix
// instructions with the packed side as the rows and the query heads as the columns:
//   QK: A = K[16 tokens][32 dims], B = q[32 dims][16 columns] -> lane (n = lane % 16, q = lane / 16) holds column n's
//       logits of tokens 4q..4q+3 of the 16.
//   PV: A = V^T[16 dims][32 tokens], B = P[32 tokens][16 columns] -> lane (n, q) holds dims 4q..4q+3 of column n.
// A matrix instruction does not mind in which order the contraction's positions come, as long as both sides agree, so
// every lane quarter q takes the part of a row that it can use without an exchange: of a K row 32 dims, of a V row (one
// dim, 64 tokens) the sixteen tokens whose weights that quarter's logits turn into.  A logit therefore becomes the weight
// operand of its own lane, the softmax state of a head is one register, and nothing is transposed.
//
// The 16 columns are NH = 4 or 8 query heads, R = 16 / NH times over: column r NH + h is head h.  All columns of the QK
// products are computed (the instruction has no smaller shape at this rate); of the four steps j (16 tokens each) copy r
// keeps steps r U .. r U + U - 1 (U = NH / 4), so a lane has 4 U logits of its own and no softmax work is done twice.
// Column h takes the weights of steps 0 and 1, column 8 + h those of steps 2 and 3 (zeros in the other's places, and in
// the remaining columns of four heads); the two are added once, at the end of the split.
//
// Why not the 4x4x4 instructions (16 blocks of 4 tokens x 4 heads), which waste no column: they run at a quarter of the
// rate, so eight heads cost twice the matrix time, and their results come out transposed to what the softmax wants.
#include <utility>

#include "tq_attn.h"

namespace {

using namespace tqattn;

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float4_t mfma16(half8_t a, half8_t b, float4_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// The part of a row that lane quarter q works on (tq_layout.h), as four elements of two quads each:
//   4 bits: 16-byte chunk q; element t = its dword t (group t's dword q)
//   3 bits, K: dword q of the three chunks = group q; element t < 3 = dword t, element 3 = the tail in the top bytes
//   3 bits, V: chunk q (element t = its dword t), and for quarter 3 the four groups' tails, put together by the lane that
//              loaded the row
//   2 bits: half q & 1 of chunk q / 2; element t = half t & 1 of dword t / 2
// 4-bit parts are loaded as such: 16 bytes of row n of each step.  Narrower ones would be loads of 4 and 8 bytes a lane, and an
// instruction takes its time by the lane and not by the byte (turbo3 K and V, 16 x 32768 tokens: 150 us against 80): those rows
// are loaded whole, lane 16 a + n row n of step a, and the parts change places across the lane quarters, two swaps per four
// registers.
// V rows: the four consecutive tokens (quad number inside the tile) of element j of quarter q; its two quads are those
// of dims r and 64 + r.  K rows are handed to the products so that step j's logits of quarter q are these tokens'.
template <int BITS> __device__ __forceinline__ int quad_of(int j, int q) {
    return BITS != 2 ? 4 * j + q : 8 * (q & 1) + 4 * (j >> 1) + 2 * (q >> 1) + (j & 1);
}
constexpr int parts_dwords(int bits, bool v_side) { return bits == 3 && v_side ? 4 : bits; }
template <int BITS, int VBITS, int PD>
__device__ __forceinline__ void load_parts(const uint8_t *rows, uint32_t offset, uint32_t (&w)[4][PD]) {
    if constexpr (BITS == 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint4 u = stream_load<STREAM_ATTN_ROWS>(reinterpret_cast<const uint4 *>(rows + offset + 64 * quad_of<VBITS>(j, 0)));
            w[j][0] = u.x; w[j][1] = u.y; w[j][2] = u.z; w[j][3] = u.w;
        }
    } else {
#pragma unroll
        for (int c = 0; c < BITS; ++c) {   // the row's part for quarter q in w[q]
            const uint4 u = stream_load<STREAM_ATTN_ROWS>(reinterpret_cast<const uint4 *>(rows + offset + 2048 * c));
            if constexpr (PD == 4) {
                w[c][0] = u.x; w[c][1] = u.y; w[c][2] = u.z; w[c][3] = u.w;
            } else if constexpr (BITS == 3) {
                w[0][c] = u.x; w[1][c] = u.y; w[2][c] = u.z; w[3][c] = u.w;
            } else {
                w[2 * c][0] = u.x; w[2 * c][1] = u.y; w[2 * c + 1][0] = u.z; w[2 * c + 1][1] = u.w;
            }
        }
    }
}
// the 24-bit tail that rides on the top bytes of a group's three dwords
__device__ __forceinline__ uint32_t tail_of(uint32_t d0, uint32_t d1, uint32_t d2) {
    return __builtin_amdgcn_perm(d2, __builtin_amdgcn_perm(d1, d0, 0x0c0c0703u), 0x0c070100u);
}
// w[q] of lane quarter j -> w[j] of lane quarter q
template <int BITS, int PD> __device__ __forceinline__ void exchange_parts(uint32_t (&w)[4][PD]) {
    if constexpr (BITS == 4) return;
#pragma unroll
    for (int d = 0; d < PD; ++d) {
        if constexpr (BITS == 3 && PD == 4) w[3][d] = tail_of(w[0][d], w[1][d], w[2][d]);
        auto s0 = __builtin_amdgcn_permlane32_swap(w[0][d], w[2][d], false, false);
        auto s1 = __builtin_amdgcn_permlane32_swap(w[1][d], w[3][d], false, false);
        auto t0 = __builtin_amdgcn_permlane16_swap(s0[0], s1[0], false, false);
        auto t1 = __builtin_amdgcn_permlane16_swap(s0[1], s1[1], false, false);
        w[0][d] = t0[0]; w[1][d] = t0[1]; w[2][d] = t1[0]; w[3][d] = t1[1];
    }
}
// K rows: first of the eight consecutive dims of element t of quarter q
template <int BITS> __device__ __forceinline__ int dim_of(int t, int q) {
    return BITS == 4 ? 32 * t + 8 * q : BITS == 3 ? 32 * q + 8 * t : 64 * (q & 1) + 32 * (t >> 1) + 16 * (q >> 1) + 8 * (t & 1);
}
// the four values of quad e of element t
template <int BITS, int PD> __device__ __forceinline__ uint2 quad_at(const uint32_t (&w)[PD], const char *lut, uint32_t own, int t, int e) {
    if constexpr (BITS == 4) {
        const uint32_t o0 = __builtin_amdgcn_perm(w[t], own, 0x0c020400u + 0x200u * e), o1 = __builtin_amdgcn_perm(w[t], own, 0x0c020500u + 0x200u * e);
        return make_uint2(*reinterpret_cast<const uint32_t *>(lut + o0), *reinterpret_cast<const uint32_t *>(lut + o1));
    } else if constexpr (BITS == 3) {
        const uint32_t x = PD == 3 && t == 3 ? tail_of(w[0], w[1], w[2]) : w[t];
        return *reinterpret_cast<const uint2 *>(lut + field_offset<3>(x, 12 * e, 12));
    } else {
        return *reinterpret_cast<const uint2 *>(lut + field_offset<3>(w[t >> 1], 16 * (t & 1) + 8 * e, 8));
    }
}
// Decode tables: quad entries for 2 and 3 bits (build_lut); for 4 bits the 256 pair entries once per lane, entry e of lane l at
// 256 e + 4 l: no two lanes meet in a bank, and a position is one byte permute of the row's dword and 4 l.
__host__ __device__ constexpr int table_bytes(int bits) { return bits == 4 ? 65536 : lut_bytes(bits); }
template <int BITS> __device__ __forceinline__ void build_table(char *dst, const uint32_t *pair_lut, uint4 four, int tid, int n_waves) {
    if constexpr (BITS == 4) {
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        // `four`: entries 4 l .. 4 l + 3 in lane l; four entries at a time, sixteen lanes a 256-byte row
        for (int i = wave; i < 64; i += n_waves) {
            const uint32_t e0 = __builtin_amdgcn_readlane(four.x, i), e1 = __builtin_amdgcn_readlane(four.y, i);
            const uint32_t e2 = __builtin_amdgcn_readlane(four.z, i), e3 = __builtin_amdgcn_readlane(four.w, i);
            const uint32_t lo = lane & 16 ? e1 : e0, hi = lane & 16 ? e3 : e2, e = lane & 32 ? hi : lo;
            *reinterpret_cast<uint4 *>(dst + 1024 * i + 16 * lane) = make_uint4(e, e, e, e);
        }
    } else {
        build_lut<BITS>(dst, pair_lut, four.x, tid, n_waves);
    }
}
__device__ __forceinline__ half8_t operand(uint2 a, uint2 b) { return __builtin_bit_cast(half8_t, make_uint4(a.x, a.y, b.x, b.y)); }

// sum / maximum over the lanes of one head (column copies r, quarters q)
template <int NH> __device__ __forceinline__ float sum_over_head(float v) {
    if constexpr (NH == 4) v += xor_lane<4>(v);
    v += xor_lane<8>(v);
    v += xor_lane<16>(v);
    v += xor_lane<32>(v);
    return v;
}
template <int NH> __device__ __forceinline__ float max_over_head(float v) {
    if constexpr (NH == 4) v = fmaxf(v, xor_lane<4>(v));
    v = fmaxf(v, xor_lane<8>(v));
    v = fmaxf(v, xor_lane<16>(v));
    v = fmaxf(v, xor_lane<32>(v));
    return v;
}

__device__ __forceinline__ float half_at(uint2 u, int i) {
    const uint32_t w = i < 2 ? u.x : u.y;
    return __half2float(__ushort_as_half((unsigned short)(i & 1 ? w >> 16 : w & 0xffffu)));
}

// NH: query heads per pass.  SHARE: K and V decode through one table (same width, same centroids).  LIST: the call carries
// a sparse logit bias (eight heads).  Work distribution, progress marks and the merge are those of k_decode_attn: a workgroup of W
// wavefronts owns W consecutive splits of one group (or a.gpw groups of fewer splits each).
template <int KBITS, int VBITS, bool SPARSE, bool SHARE, int NH, bool LIST>
__global__ __launch_bounds__(NH == 8 ? 768 : 1024) void k_decode_turbo(AttnArgs a) {
    static_assert(NH == 4 ? !LIST : NH == 8, "query heads per pass");
    static_assert(!SHARE || KBITS == VBITS, "a shared table needs equal code widths");
    constexpr int HG = NH / 4, U = NH / 4;
    constexpr int KBLOCK = TQ_ROWS_PER_BLOCK * (16 * KBITS + 2), VBLOCK = TQ_ROWS_PER_BLOCK * (16 * VBITS + 2);
    constexpr int LUT_TOTAL = table_bytes(KBITS) + (SHARE ? 0 : table_bytes(VBITS));
    // static LDS, so that table positions fold into the LDS instructions.  Behind the last tile the space takes the
    // wavefronts' slots, then merge_group's exchange.
    constexpr int MS = MERGE_FLOATS * HG;
    static_assert((NH == 8 ? 12 : 16) * MS * 4 <= LUT_TOTAL, "the slots of every wavefront fit where the tables were");
    __shared__ __attribute__((aligned(16))) char smem[LUT_TOTAL];
    __shared__ uint32_t lead;     // tiles finished by the wavefront that is furthest ahead
    __shared__ uint32_t skipped;  // Sparse V: (query, position) pairs skipped by this workgroup
    // (an LDS instruction's offset field holds 65535: a table of 64 KB comes second, the second of two goes into the position)
    constexpr int K_AT = KBITS == 4 && VBITS != 4 ? table_bytes(VBITS) : 0, V_AT = SHARE || KBITS == 4 ? 0 : table_bytes(KBITS);
    constexpr uint32_t V_HIGH = KBITS == 4 && VBITS == 4 && !SHARE ? 65536u : 0u;
    const char *const klut_s = smem + K_AT, *const vlut_s = smem + V_AT;

    const int tid = threadIdx.x, lane = tid & 63;
    const int n = lane & 15, q4 = lane >> 4, h = lane & (NH - 1), r = n / NH;
    const uint32_t kown = 4u * lane, vown = kown + V_HIGH;   // 4-bit codes: this lane's copy
    // workgroup-uniform values in scalar registers
    const int n_waves = (int)(blockDim.x >> 6), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gw = a.gpw > 1 ? a.n_splits : n_waves;   // wavefronts that work on one group
    const int wave_g = a.gpw > 1 ? (wave & (gw - 1)) : wave, wave0 = wave - wave_g;
    const int gidx = a.gpw > 1 ? (wave >> a.gw_shift) : 0;
    const int tid_g = tid - 64 * wave0;
    const int wgs_per_group = a.wgs_per_group;
    const int group = __builtin_amdgcn_readfirstlane(a.gpw > 1 ? (int)blockIdx.x * a.gpw + gidx : (int)(blockIdx.x / wgs_per_group));
    const int part = a.gpw > 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(blockIdx.x % wgs_per_group));
    const int pass_y = HG == 2 ? (int)blockIdx.y : 0;   // one set of four heads is always one pass
    const int head_off = a.head_off + pass_y * a.pass_heads, pgroup = pass_y * a.n_groups + group;
    const int split = part * n_waves + wave_g;
    // dynamic LDS: 1 KB per group and four heads that stages the rotated queries
    extern __shared__ __attribute__((aligned(16))) char q_all[];
    char *q_stage = q_all + (size_t)gidx * (1024 * HG);
    auto slot = [&](int w) { return reinterpret_cast<float *>(smem) + w * MS; };
    int tokens_now = (int)a.tokens, n_tiles = a.n_tiles, tiles_per_split = a.tiles_per_split;
    if (a.tokens_dev) {
        const int64_t t = *a.tokens_dev;
        tokens_now = __builtin_amdgcn_readfirstlane((int)(t < 0 ? 0 : (t < a.tokens ? t : a.tokens)));
        n_tiles = (tokens_now + 63) >> 6;
        tiles_per_split = (n_tiles + a.n_splits - 1) / a.n_splits;
    }
    const int t_begin = split * tiles_per_split;
    const int t_end = min(t_begin + tiles_per_split, n_tiles);
    // first of this lane's four tokens of its u-th step (tile-relative)
    int t4[U];
#pragma unroll
    for (int u = 0; u < U; ++u) t4[u] = 4 * quad_of<VBITS>(r * U + u, q4);

    const uint8_t *kbase = a.k + (int64_t)group * a.blocks_per_seq * KBLOCK;
    const uint8_t *vbase = a.v + (int64_t)group * a.blocks_per_seq * VBLOCK;
    // The first tile's rows are requested before anything else, so that the table build and the query rotation overlap
    // the first trip to memory; afterwards one tile ahead into the same registers, the norms with them.  Row n of step j is
    // token 4 quad_of(j, n / 4) + n % 4: the steps differ by constants.  After the split's last tile the prefetch has every
    // lane read the same address (a few lines, never used): a re-read of real rows would go to memory again.
    const uint32_t koff = KBITS == 4 ? 2048u * q4 + 16u * (4 * quad_of<VBITS>(0, n >> 2) + (n & 3)) : 16u * (4 * quad_of<VBITS>(q4, n >> 2) + (n & 3));
    const uint32_t voff = VBITS == 4 ? 16u * n + 2048u * q4 : 16u * lane;
    constexpr int KPD = parts_dwords(KBITS, false), VPD = parts_dwords(VBITS, true);
    uint32_t kw[4][KPD], vw[4][VPD];
    auto load_k = [&](int tile, bool any) {
        const uint8_t *p = kbase + (int64_t)(tile >> 1) * KBLOCK + (any ? (tile & 1) * 1024 : 0);
        load_parts<KBITS, VBITS>(p, any ? koff : 0u, kw);
    };
    auto load_v = [&](int tile, bool any) {
        const uint8_t *p = vbase + (int64_t)(tile >> 1) * VBLOCK + (any ? (tile & 1) * 1024 : 0);
        load_parts<VBITS, 4>(p, any ? voff : 0u, vw);   // row 16 j + n
    };
    auto load_norms = [&](const uint8_t *block_norms, int tile, uint2 (&g)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) g[u] = *reinterpret_cast<const uint2 *>(block_norms + (tile & 1) * 128 + 2u * (uint32_t)t4[u]);
    };
    auto k_norms = [&](int tile) { return kbase + (int64_t)(tile >> 1) * KBLOCK + TQ_ROWS_PER_BLOCK * 16 * KBITS; };
    auto v_norms = [&](int tile) { return vbase + (int64_t)(tile >> 1) * VBLOCK + TQ_ROWS_PER_BLOCK * 16 * VBITS; };
    unsigned long long arrivals_seen = 0ull;
    if (wgs_per_group > 1 && tid == 0) arrivals_seen = ld_dev(arrival_counter(a, pgroup, wgs_per_group));
    // pair-table entries for the table build
    uint4 kpair = make_uint4(0u, 0u, 0u, 0u), vpair = kpair;
    if constexpr (KBITS == 3) kpair.x = a.klut[lane];
    if constexpr (KBITS == 4) kpair = *reinterpret_cast<const uint4 *>(a.klut + 4 * lane);
    if constexpr (!SHARE && VBITS == 3) vpair.x = a.vlut[lane];
    if constexpr (!SHARE && VBITS == 4) vpair = *reinterpret_cast<const uint4 *>(a.vlut + 4 * lane);
    uint2 gk[U], gv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) gk[u] = gv[u] = make_uint2(0u, 0u);
    int tile = t_begin;
    if (tile < t_end) {
        load_k(tile, true);
        load_norms(k_norms(tile), tile, gk);
        load_v(tile, true);
        load_norms(v_norms(tile), tile, gv);
    }
    if (tid == 0) {
        lead = 0;
        skipped = 0;
    }

    auto load_q = [&](int head, float &x0, float &x1) {   // heads past the group's last one repeat it (their results are not written)
        const int64_t e = ((int64_t)group * a.q_group + min(head_off + head, a.q_group - 1)) * 128 + 2 * lane;
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
    // this wavefront's first head is requested now and rotated after the tables are built
    float xq0 = 0.0f, xq1 = 0.0f;
    if (wave_g < NH) load_q(wave_g, xq0, xq1);
    // Sparse bias: the 64 / NH lanes of a head hold a window of that many entries of its (position, value) list, lane's slot
    // lane / NH; the window starts at the head's first entry inside this split (entries below it counted with the whole
    // wavefront).  Requested in front of the table build, so that the two dependent trips to memory pass while it runs.
    constexpr int SLOTS = 64 / NH;
    int sb_win = 0, sb_pos = 0x7FFFFFFF, sb_last = 0x7FFFFFFF;   // sb_last: the window's last position
    float sb_val = 0.0f;
    auto sb_entry = [&](int e) { return ((int64_t)group * a.q_group + min(head_off + h, a.q_group - 1)) * a.sbias_n + e; };
    auto sb_load = [&] {
        const int e = sb_win + lane / NH;
        const bool in = e < a.sbias_n;
        sb_pos = in ? a.sbias_pos[sb_entry(in ? e : 0)] : 0x7FFFFFFF;
        sb_val = in ? a.sbias_val[sb_entry(in ? e : 0)] : 0.0f;
        sb_last = __shfl(sb_pos, 64 - NH + h);
    };
    if constexpr (LIST) {
        const int first_tok = t_begin * 64;
#pragma unroll
        for (int hh = 0; hh < NH; ++hh) {
            const int32_t *prow = a.sbias_pos + ((int64_t)group * a.q_group + min(head_off + hh, a.q_group - 1)) * a.sbias_n;
            int c = 0;
            for (int e0 = 0; e0 < a.sbias_n; e0 += 64) {
                const int e = e0 + lane;
                const int pe = e < a.sbias_n ? prow[e] : 0x7FFFFFFF;
                c += __builtin_popcountll(__builtin_amdgcn_ballot_w64(pe < first_tok));
            }
            if (h == hh) sb_win = c;
        }
        sb_load();
    }
    build_table<KBITS>(smem + K_AT, a.klut, kpair, tid, n_waves);
    if constexpr (!SHARE) build_table<VBITS>(smem + V_AT + V_HIGH, a.vlut, vpair, tid, n_waves);
    for (int head = wave_g; head < NH; head += gw) {
        _Float16 *qw = reinterpret_cast<_Float16 *>(q_stage) + head * 128;
        float x0 = xq0, x1 = xq1;
        if (head != wave_g) load_q(head, x0, x1);
        if (a.ks1) {
            x0 *= a.ks1[2 * lane];
            x1 *= a.ks1[2 * lane + 1];
            wht128_wave(x0, x1, lane);
            x0 *= a.ks2[2 * lane] * RSQRT128;
            x1 *= a.ks2[2 * lane + 1] * RSQRT128;
        }
        // the rotated query is rounded to fp16 once, with the logit scale (times log2 e) folded in
        qw[2 * lane] = (_Float16)(x0 * a.scale_log2e);
        qw[2 * lane + 1] = (_Float16)(x1 * a.scale_log2e);
    }
    if (wgs_per_group > 1 && tid == 0) install_tag(a, arrival_counter(a, pgroup, wgs_per_group), arrivals_seen);
    __syncthreads();
    half8_t qb[4];   // B operand of QK: head h, the dims of element t of this quarter
#pragma unroll
    for (int t = 0; t < 4; ++t)
        qb[t] = *reinterpret_cast<const half8_t *>(reinterpret_cast<const _Float16 *>(q_stage) + h * 128 + dim_of<KBITS>(t, q4));
    // out[head h][dims 64 hf + 16 c + 4 q4 + i], this column copy's tokens
    float4_t acc_o[4][2];
#pragma unroll
    for (int c = 0; c < 4; ++c) acc_o[c][0] = acc_o[c][1] = float4_t{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run[U];   // one sum per step: a head's arithmetic does not depend on how many share the pass
#pragma unroll
    for (int u = 0; u < U; ++u) l_run[u] = 0.0f;
    unsigned nskip = 0;   // Sparse V: skipped (query, position) pairs of this wavefront (wave-uniform)
    bool v_ahead = true;  // Sparse V: this tile's V row was requested while the previous tile was processed
    const unsigned long long head_ok = __builtin_amdgcn_ballot_w64(head_off + h < a.q_group);
#pragma unroll 1
    while (tile < t_end) {
        {   // issue priority = tiles behind the leader (wave-uniform, so the branches are scalar)
            const uint32_t done = (uint32_t)(tile - t_begin);
            const uint32_t behind = max(lead_progress(&lead, done, lane), done) - done;
            if (behind == 0) __builtin_amdgcn_s_setprio(0);
            else if (behind == 1) __builtin_amdgcn_s_setprio(1);
            else if (behind == 2) __builtin_amdgcn_s_setprio(2);
            else __builtin_amdgcn_s_setprio(3);
        }
        const bool more = tile + 1 < t_end;
        const int tile_n = more ? tile + 1 : tile;
        uint2 gv_next[U];
        load_norms(v_norms(tile_n), tile_n, gv_next);
        const int n_valid = tokens_now - tile * 64;   // >= 64 except in the sequence's last tile
        float bias4[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) bias4[u][i] = 0.0f;
        if constexpr (LIST) {
            // entries of this tile: positions ascend, so a window is done with once its last position lies below the
            // tile's end; a head then takes its next entries (wave-uniform loop, heads advance on their own)
            const int tile_lo = tile * 64, tile_hi = tile_lo + 64;
            bool fresh = true;   // this head's window has not been added to this tile yet
            while (true) {
                const bool mine = fresh && sb_pos >= tile_lo && sb_pos < tile_hi;
                // window slots (lane / NH) that hold an entry of this tile for any of the heads
                unsigned long long slots = __builtin_amdgcn_ballot_w64(mine);
                slots |= slots >> 1;
                slots |= slots >> 2;
                if constexpr (NH == 8) slots |= slots >> 4;
                slots &= NH == 8 ? 0x0101010101010101ull : 0x1111111111111111ull;
#pragma unroll 1
                while (slots) {
                    const int first = __builtin_ctzll(slots);   // NH * slot
                    const int pe = __shfl(sb_pos, first + h);
                    const float ve = __shfl(sb_val, first + h) * LOG2E;
                    if (fresh) {
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            const int d = pe - tile_lo - t4[u];   // positions outside these four tokens match no i
#pragma unroll
                            for (int i = 0; i < 4; ++i) bias4[u][i] += d == i ? ve : 0.0f;
                        }
                    }
                    slots &= slots - 1;
                }
                fresh = false;
                const bool advance = sb_last < tile_hi;   // the whole window lies before the tile's end (padding never does)
                if (__builtin_amdgcn_ballot_w64(advance) == 0ull) break;
                if (advance) {
                    sb_win += SLOTS;
                    fresh = true;
                }
                sb_load();   // by every lane (it ends in a cross-lane read); heads that stay reload what they hold
            }
        }

        // ---- QK: step j's 16 tokens against every column; this lane keeps its copy's steps ----------------
        exchange_parts<KBITS>(kw);
        float s[U][4];
        float4_t c[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) c[j] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 4; ++t)   // the four steps' chains side by side: one would wait for its own results
#pragma unroll
            for (int j = 0; j < 4; ++j) c[j] = mfma16(operand(quad_at<KBITS>(kw[j], klut_s, kown, t, 0), quad_at<KBITS>(kw[j], klut_s, kown, t, 1)), qb[t], c[j]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (U == 1) {
                const float lo = r & 1 ? c[1][i] : c[0][i], hi = r & 1 ? c[3][i] : c[2][i];
                s[0][i] = r & 2 ? hi : lo;
            } else {
                s[0][i] = r ? c[2][i] : c[0][i];
                s[U - 1][i] = r ? c[3][i] : c[1][i];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[u][i] = LIST ? fmaf(s[u][i], half_at(gk[u], i), bias4[u][i]) : s[u][i] * half_at(gk[u], i);
                if (n_valid < 64 && t4[u] + i >= n_valid) s[u][i] = -INFINITY;
            }
        load_k(tile_n, more);   // kw is dead now
        load_norms(k_norms(tile_n), tile_n, gk);

        // ---- online softmax in base 2; a head's state is the same in all of its lanes ----------------------
        float mx = fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3]));
        if constexpr (U == 2) mx = fmaxf(mx, fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
        const float m_new = fmaxf(m_run, max_over_head<NH>(mx));
        // after the first tiles the running maximum rarely moves, and a correction factor of exactly 1 changes nothing
        if (__builtin_amdgcn_ballot_w64(m_new != m_run) != 0ull) {
            // 0 on the first tile, 1 when the maximum stays (also while every position so far is masked with -inf)
            const float corr = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new);
#pragma unroll
            for (int u = 0; u < U; ++u) l_run[u] *= corr;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                acc_o[c][0] *= corr;
                acc_o[c][1] *= corr;
            }
            m_run = m_new;
        }
        const float m_ref = m_run == -INFINITY ? 0.0f : m_run;  // all masked so far: weights are exp2(-inf) = 0, not NaN
        float p[U][4];
        unsigned long long any_keep = 0;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[u][i] = __builtin_amdgcn_exp2f(s[u][i] - m_ref);  // results below 2^-126 flush to zero
                l_run[u] += p[u][i];
                if constexpr (SPARSE) {
                    // bookkeeping on the scalar unit: counting, the in-range test and "does any lane keep anything"
                    // are mask arithmetic
                    const bool keep = p[u][i] >= a.tau;
                    const unsigned long long keep_m = __builtin_amdgcn_ballot_w64(keep);
                    unsigned long long in_range = head_ok;
                    if (n_valid < 64) in_range &= __builtin_amdgcn_ballot_w64(t4[u] + i < n_valid);
                    nskip += (unsigned)__builtin_popcountll(in_range & ~keep_m);
                    if (!keep) p[u][i] = 0.0f;
                    any_keep |= keep_m & in_range;
                }
            }
        if constexpr (SPARSE) {
            // Every V row of the tile skipped: no dequant, and the next tile's V row is not requested in advance
            // (negligible weights come in runs); a tile that then does need its row fetches it here.
            if (any_keep == 0) {
#pragma unroll
                for (int u = 0; u < U; ++u) gv[u] = gv_next[u];
                ++tile;
                v_ahead = false;
                continue;
            }
            if (!v_ahead) load_v(tile, true);
        }

        exchange_parts<VBITS>(vw);
        // ---- PV: weights times the stored V norm as fp16, zero in the columns of the other copies ----------
        uint2 w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
            const half2_t lo = {(_Float16)(p[u][0] * half_at(gv[u], 0)), (_Float16)(p[u][1] * half_at(gv[u], 1))};
            const half2_t hi = {(_Float16)(p[u][2] * half_at(gv[u], 2)), (_Float16)(p[u][3] * half_at(gv[u], 3))};
            w[u] = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
        }
        // copies of four heads hold one step each: the even one takes its neighbour's as well, so that the products are the
        // same ones as with eight heads
        uint2 w_odd = w[U - 1];
        if constexpr (U == 1) w_odd = make_uint2(xor_lane<4>(w[0].x), xor_lane<4>(w[0].y));
        half8_t pb[2];   // steps 2 s, 2 s + 1
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            const uint2 z = make_uint2(0u, 0u);
            pb[st] = operand(n / 8 == st && (n & 7) < NH ? w[0] : z, n / 8 == st && (n & 7) < NH ? w_odd : z);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int st = 0; st < 2; ++st)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
                    acc_o[c][hf] = mfma16(operand(quad_at<VBITS>(vw[c], vlut_s, vown, 2 * st, hf), quad_at<VBITS>(vw[c], vlut_s, vown, 2 * st + 1, hf)),
                                          pb[st], acc_o[c][hf]);
        load_v(tile_n, more);
        v_ahead = true;
#pragma unroll
        for (int u = 0; u < U; ++u) gv[u] = gv_next[u];
        ++tile;
    }

    // ---- end of split: the column copies are added, the workgroup's wavefronts merge in LDS and write one partial ------
    const float l_tot = sum_over_head<NH>(U == 1 ? l_run[0] : l_run[0] + l_run[U - 1]);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float v = acc_o[c][hf][i];
                acc_o[c][hf][i] = v + xor_lane<8>(v);
            }
    __syncthreads();   // the tables' last readers are done: their space takes the slots
    float *mine = slot(wave) + (h >> 2) * MERGE_FLOATS;
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (n / 8 == (c & 1) && (n & 7) < NH) {   // the two columns of a head share the stores out
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) *reinterpret_cast<float4_t *>(mine + (h & 3) * 128 + 64 * hf + 16 * c + 4 * q4) = acc_o[c][hf];
        }
    if (lane < NH) *reinterpret_cast<float2 *>(mine + 512 + 2 * (h & 3)) = make_float2(m_run, l_tot);
    if (SPARSE && lane == 0 && nskip) atomicAdd(&skipped, nskip);
    finish_group<HG, SPARSE>(a, slot, group, pgroup, head_off, wgs_per_group, part, tid, tid_g, gw, wave0, reinterpret_cast<float *>(smem), &skipped);
}

template <int KB, int VB, bool SHARE> void launch_pair(const AttnArgs &a, int n_heads, bool sparse, dim3 grid, int waves, hipStream_t s) {
    const int hg = n_heads / 4;
    const size_t lds = (size_t)a.gpw * 1024 * hg;   // the staged queries
    const unsigned wg = 64u * (unsigned)waves;
#define TQ_ONE(SP, NH, LIST) k_decode_turbo<KB, VB, SP, SHARE, NH, LIST><<<grid, wg, lds, s>>>(a)
    if (n_heads == 8 && a.sbias_n) {
        if (sparse) TQ_ONE(true, 8, true);
        else TQ_ONE(false, 8, true);
    } else if (n_heads == 8) {
        if (sparse) TQ_ONE(true, 8, false);
        else TQ_ONE(false, 8, false);
    } else {
        if (sparse) TQ_ONE(true, 4, false);
        else TQ_ONE(false, 4, false);
    }
#undef TQ_ONE
}

}  // namespace

int tqk_decode_turbo_lds(int kb, int vb, bool share) { return table_bytes(kb) + (share ? 0 : table_bytes(vb)) + 1024; }

bool tqk_launch_decode_turbo(const AttnArgs &a, int kb, int vb, bool share, int n_heads, bool sparse, dim3 grid, int waves, hipStream_t s) {
#define TQ_PAIR(K, V) if (kb == K && vb == V) { launch_pair<K, V, false>(a, n_heads, sparse, grid, waves, s); return true; }
    if (kb == 4 && vb == 4 && share) {
        launch_pair<4, 4, true>(a, n_heads, sparse, grid, waves, s);
        return true;
    }
    TQ_PAIR(4, 4) TQ_PAIR(4, 2) TQ_PAIR(2, 4) TQ_PAIR(3, 4) TQ_PAIR(4, 3)
#undef TQ_PAIR
    return false;
}
