// Decode attention: a launch's plan, workspace and arguments (the kernels: tq_attn_rows.h, attn_turbo_kernels.hip), and the
// prefill-shaped score tile.
//
// k_score_tile: TurboQuant inner-product estimate, 32x32x16 fp16 MFMA over a
//   K = 256 contraction ([R q | S q] against [g c[idx] | scale*rnorm*z]); key operands in registers, queries
//   through LDS, logit rows written 64 consecutive logits per store.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <cstring>
#include <type_traits>
#include <utility>

#include "tq_attn_rows.h"

namespace {

using namespace tqattn;

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

// turbo K and V rows of 128-dim heads; kb, vb: code widths, hg: sets of four heads per pass; false: no such pair
bool launch_turbo(const AttnArgs &a, int kb, int vb, bool share, int hg, bool sparse, dim3 grid, unsigned wg, size_t lds, hipStream_t s) {
    // same width and same centroids: one table
#define TQ_SAME(B) if (kb == B && vb == B && share) TQ_ATTN_PAIR(KFMT_TURBO, B, B, true)
#define TQ_PAIR(K, V) if (kb == K && vb == V) TQ_ATTN_PAIR(KFMT_TURBO, K, V, false)
    TQ_SAME(3) TQ_SAME(4) TQ_SAME(2)
    TQ_PAIR(3, 3) TQ_PAIR(4, 4) TQ_PAIR(2, 2) TQ_PAIR(4, 2) TQ_PAIR(3, 2) TQ_PAIR(3, 4) TQ_PAIR(4, 3) TQ_PAIR(2, 3) TQ_PAIR(2, 4)
#undef TQ_SAME
#undef TQ_PAIR
    return false;
}

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

// What a call launches: workgroups, passes in one launch, and which kernel.  kb, vb: code widths, 8 for q8_0-style rows; share: K
// and V decode through one table; dense: the call carries dense bias rows.
struct StepPlan : AttnPlan {
    int n_pass;        // passes of one launch
    int64_t pass_wgs;  // workgroups of a pass
    bool lane_tables;  // k_decode_turbo
};
StepPlan step_plan(const tq_attn_params *p, int kb, int vb, bool share, bool dense, int64_t ws_bytes) {
    StepPlan pl;
    // wavefronts per workgroup: the largest power of two up to 16 (8 for int8 V rows and for eight heads per pass)
    // that divides the split count
    static_cast<AttnPlan &>(pl) = attn_plan(p, p->bias_entries > 0);
    // All passes in one launch where the workspace has room: each is a chain of its own (launch, first rows, merge), one of few
    // groups leaves most of the chip idle, and they read the same rows.  Steps of two passes over 256-dim heads (us with the
    // append, one pass after the other / together): 2 x 8 KV heads x 259 tokens turbo4 35.0 / 19.6, 4 x 8 x 4000 turbo3 50.5 / 32.8,
    // 1 x 1 x 100 000 turbo2 169 / 95, 8 x 4 x 16 000 8-bit K with turbo3 V 86.2 / 82.4, 16 x 8 x 12 000 turbo4 180 / 174 to 178.
    // Sparse V counts pass by pass.
    pl.n_pass = p->sparse_v_tau > 0.0f ? 1 : passes_of(p);
    if (pl.n_pass > 1 && ws_bytes < ws_layout(p, pl.n_pass).total) pl.n_pass = 1;
    pl.pass_wgs = (int64_t)p->batch * p->n_kv_heads * pl.n_parts / pl.gpw;
    // A 4-bit side: k_decode_turbo, whose table of 64 KB has a copy per lane (16 x 8 groups at 32768 tokens, turbo4: 110 -> 97 us,
    // eight heads 121 -> 90; turbo4 K with turbo2 V 87 -> 77 and 100 -> 78).  It has to leave the workgroups that share a CU room
    // (25 x 8 groups at 3175 tokens in 1000 workgroups of four: 30.5 us against 28.4 here; turbo4 K with turbo3 V, 96 KB, 20 x 8
    // groups of eight heads at 2500 tokens in 320: 32.0 against 25.7), and building it has to pay: three tiles per wavefront and
    // four wavefronts (2 x 8 groups at 3000 tokens, three: 12.7 us against 13.2 here; 8 at 4000, two: 11.7 against 11.5; one at
    // 300, two wavefronts: 12.1 against 11.5).  Four heads with a bias list have no registers for it (16 x 9000 tokens with 64
    // entries: 41.4 against 38.8, with Sparse V 47.6 against 43.0), and dense bias rows keep the general variants.
    // A context length read from memory is taken at its largest: at short ones the tables cost nothing that shows (16 x 8 groups,
    // turbo4, of 32 768 tokens 64 to 2048: 9.7 to 14.4 us, 10.1 to 19.0 in k_decode_attn; turbo3 K with turbo4 V 10.4 to 15.0, 10.3
    // to 17.3).
    const int tables = tqk_decode_turbo_lds(kb, vb, share) + pl.gpw * 1024 * pl.hg;
    const int64_t per_cu = std::min<int64_t>((pl.pass_wgs * pl.n_pass + 255) / 256, std::max(1, (pl.hg == 2 ? 12 : 16) / pl.wpw));
    const int64_t tiles = (p->tokens + 63) / 64, tiles_per_split = (tiles + p->n_splits - 1) / p->n_splits;
    pl.lane_tables = !TQ_PAIRTAB3 && p->head_dim != 256 && kb != 8 && vb != 8 && (kb == 4 || vb == 4) && per_cu * tables <= 160 * 1024 &&
                     tiles_per_split >= 3 && pl.wpw >= 4 && !dense && (pl.hg == 2 || !p->bias_entries);
    return pl;
}

}  // namespace

void tqk_attn_plan(const tq_attn_params *p, int kb, int vb, bool share, bool dense, int64_t ws_bytes, tq_attn_plan *out) {
    const StepPlan pl = step_plan(p, kb, vb, share, dense, ws_bytes);
    out->passes = pl.n_pass;
    out->heads_per_pass = heads_per_pass(p);
    out->wavefronts = pl.wpw;
    out->partials = pl.n_parts;
    out->groups_per_workgroup = pl.gpw;
    out->lane_tables = pl.lane_tables;
    out->workgroups = pl.pass_wgs * pl.n_pass;
}

int64_t tqk_attn_workspace_bytes(const tq_attn_params *p) { return ws_layout(p, p->sparse_v_tau > 0.0f ? 1 : passes_of(p)).total; }

int tqk_decode_attention(const tq_handle *hk, const tq_handle *hv, const tq_attn_params *p, const void *q, int q_dtype,
                         const void *k, const void *k_aux, const void *v, const float *bias, float *out,
                         unsigned long long *skip_count, void *ws, int64_t ws_bytes, hipStream_t s) {
    (void)k_aux;
    const bool turbo_k = p->k_format == TQ_KFMT_TURBO, turbo_v = p->v_format == TQ_KFMT_TURBO;
    const int kb = turbo_k ? hk->bits : 8, vb = turbo_v ? hv->bits : 8;
    const bool share = turbo_k && turbo_v && hk->bits == hv->bits &&
                       std::memcmp(hk->pair_lut_host, hv->pair_lut_host, sizeof(hk->pair_lut_host)) == 0;
    const StepPlan pl = step_plan(p, kb, vb, share, bias != nullptr, ws_bytes);
    const int n_pass = pl.n_pass, wpw = pl.wpw, hg = pl.hg;
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
    a.vlut = turbo_v ? (const uint32_t *)hv->pair_lut : nullptr;
    const float *vs1 = turbo_v ? hv->s1_32 : nullptr, *vs2 = turbo_v ? hv->s2_32 : nullptr;
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
    const unsigned pass_wgs = (unsigned)pl.pass_wgs;
    const dim3 grid(pass_wgs, n_pass);
    const unsigned wg = 64u * (unsigned)wpw;
    // dynamic LDS: the wavefronts' merge space, then the staged queries of the workgroup's groups
    const size_t merge_bytes = (size_t)wpw * hg * MERGE_FLOATS * sizeof(float) + (size_t)pl.gpw * 1024 * hg;
    a.gpw = pl.gpw;
    a.gw_shift = 0;
    while ((1 << a.gw_shift) < p->n_splits) ++a.gw_shift;
    a.wgs_per_group = pl.gpw > 1 ? 1 : p->n_splits / wpw;
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
    for (a.head_off = 0; a.head_off < a.q_group; a.head_off += n_pass * a.pass_heads) {
        a.pass = a.head_off / a.pass_heads;
        a.nonce = next_nonce();
        const bool launched = d256 ? tqk_launch_decode_256(a, kb, vb, share, sparse, grid, wg, merge_bytes, s)
                              : pl.lane_tables ? tqk_launch_decode_turbo(a, kb, vb, share, 4 * hg, sparse, grid, wpw, s)
                              : turbo_k && turbo_v ? launch_turbo(a, kb, vb, share, hg, sparse, grid, wg, merge_bytes, s)
                                                   : tqk_launch_decode_q8(a, kb, vb, hg, sparse, grid, wg, merge_bytes, s);
        if (!launched) {
            tq_set_error("tq_decode_attention: head_dim %d with K %d bits, V %d bits is not built", d256 ? 256 : 128, kb, vb);
            return TQ_ERR_UNSUPPORTED;
        }
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
