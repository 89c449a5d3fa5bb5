// What the decode attention kernels share: a step's arguments, decode tables in LDS, reductions over a wavefront, and the
// merge of the workgroups' partials inside the launch.
#pragma once
#include <type_traits>
#include <utility>

#include "tq_device.h"

namespace tqattn {

using namespace tqd;

constexpr float LOG2E = 1.4426950408889634f;
constexpr float RSQRT128 = 0.08838834764831845f;

template <typename T> __device__ inline float ldf(const T *p) { return (float)*p; }
template <> __device__ inline float ldf<__half>(const __half *p) { return __half2float(*p); }

template <int BITS> __device__ __forceinline__ uint32_t pair_off(const uint32_t (&w)[4 * BITS], int p) {
    return pair_lut_offset<BITS>(w, p);
}

// TQ_PAIRTAB3 (tq_measure.h; measurement builds only): 3-bit codes decode through a pair table with one copy
// per LDS bank (entry e of lane l at dword 64 e + l: no bank conflicts, two 4-byte reads per four values)
// instead of the 4096-entry quad table (one 8-byte read per four values, about 1.6 conflicts per read).
// bytes of the decode table of a codebook: quad entries for BITS <= 3, pair entries for 4
__host__ __device__ constexpr int lut_bytes(int bits) {
    if (TQ_PAIRTAB3 && bits == 3) return 64 * 64 * 4;
    return bits == 8 ? 0 : bits <= 3 ? 8 << (4 * bits) : 4 << (2 * bits);  // 8: int8 rows, no table
}

// the four values of quad Q (pairs 2Q, 2Q+1) of a row as an MFMA operand
template <int BITS> __device__ __forceinline__ half4_t quad_values(const uint32_t (&w)[4 * BITS], const char *lut, int Q) {
    if constexpr (TQ_PAIRTAB3 && BITS == 3) {
        // lut already points at this lane's bank (+ 4 * lane); a pair code selects the 256-byte row
        const uint32_t o0 = pair_lut_offset<BITS>(w, 2 * Q) << 6, o1 = pair_lut_offset<BITS>(w, 2 * Q + 1) << 6;
        const uint2 u = make_uint2(*reinterpret_cast<const uint32_t *>(lut + o0), *reinterpret_cast<const uint32_t *>(lut + o1));
        return __builtin_bit_cast(half4_t, u);
    } else if constexpr (BITS <= 3) {
        return __builtin_bit_cast(half4_t, *reinterpret_cast<const uint2 *>(lut + quad_lut_offset<BITS>(w, Q)));
    } else {
        const uint2 u = make_uint2(*reinterpret_cast<const uint32_t *>(lut + pair_lut_offset<BITS>(w, 2 * Q)),
                                   *reinterpret_cast<const uint32_t *>(lut + pair_lut_offset<BITS>(w, 2 * Q + 1)));
        return __builtin_bit_cast(half4_t, u);
    }
}

// build a codebook's decode table in LDS from its pair table (half2 per pair code) with n_waves wavefronts;
// `mine` is pair entry tid % 64, fetched by the caller ahead of time (used by the 3-bit table only)
template <int BITS>
__device__ __forceinline__ void build_lut(char *dst, const uint32_t *pair_lut, uint32_t mine, int tid, int n_waves) {
    constexpr int NP = 1 << (2 * BITS);
    if constexpr (TQ_PAIRTAB3 && BITS == 3) {
        uint32_t *t = reinterpret_cast<uint32_t *>(dst);
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        for (int e = wave; e < 64; e += n_waves) t[e * 64 + lane] = (uint32_t)__builtin_amdgcn_readlane((int)mine, e);
    } else if constexpr (BITS == 3) {
        // lane l holds pair entry l; wavefront w writes the rows hi = w, w + n_waves, ..
        uint2 *t = reinterpret_cast<uint2 *>(dst);
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        for (int hi = wave; hi < 64; hi += n_waves)
            t[hi * 64 + lane] = make_uint2(mine, (uint32_t)__builtin_amdgcn_readlane((int)mine, hi));
    } else if constexpr (BITS == 2) {
        for (int e = tid; e < 256; e += 64 * n_waves)
            reinterpret_cast<uint2 *>(dst)[e] = make_uint2(pair_lut[e & 15], pair_lut[e >> 4]);
    } else {
        static_assert(NP == 256, "pair table of 256 entries");
        for (int e = tid; e < 256; e += 64 * n_waves) reinterpret_cast<uint32_t *>(dst)[e] = pair_lut[e];
    }
}

// raise a progress mark in LDS to `mine` and return what it held before (one atomic per wavefront)
__device__ __forceinline__ uint32_t lead_progress(uint32_t *mark, uint32_t mine, int lane) {
    uint32_t t = 0;
    if (lane == 0) t = atomicMax(mark, mine);
    return __builtin_amdgcn_readfirstlane(t);
}

template <int BITS> __device__ __forceinline__ void load_row(const uint8_t *block, int row, uint32_t (&w)[4 * BITS]) {
#pragma unroll
    for (int c = 0; c < BITS; ++c) {
        const uint4 u = stream_load<STREAM_ATTN_ROWS>(reinterpret_cast<const uint4 *>(block + c * 2048 + row * 16));
        w[4 * c] = u.x; w[4 * c + 1] = u.y; w[4 * c + 2] = u.z; w[4 * c + 3] = u.w;
    }
}

__device__ __forceinline__ float4_t mfma4(half4_t a, half4_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_4x4x4f16(a, b, c, 0, 0, 0);
}

// 4x4x4 MFMA whose A operand is taken from block ABID and broadcast to all 16 blocks
template <int ABID> __device__ __forceinline__ float4_t mfma4_bcast(half4_t a, half4_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_4x4x4f16(a, b, c, 4, ABID, 0);
}

// the same with the A operand taken from block ABID of each group of 8 blocks (lanes 0..31 and 32..63 apart)
template <int ABID> __device__ __forceinline__ float4_t mfma4_bcast8(half4_t a, half4_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_4x4x4f16(a, b, c, 3, ABID, 0);
}

// four int8 of a dword as fp16, in the order 0, 2, 1, 3: 0x6400 | (x + 128) is the fp16 number 1024 + (x + 128),
// exactly, so a byte permute builds two of them at once and one packed fp16 subtraction of 1152 leaves (x0, x2)
// and (x1, x3)
__device__ __forceinline__ half4_t int8x4_to_half_0213(uint32_t w) {
    typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
    const uint32_t u = w ^ 0x80808080u;
    const half2_t bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    const half2_t h02 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x04020400u)) - bias;
    const half2_t h13 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x04030401u)) - bias;
    half4_t kv;
    kv[0] = h02[0];
    kv[1] = h02[1];
    kv[2] = h13[0];
    kv[3] = h13[1];
    return kv;
}

// transpose the 4x4 matrix held by a quad of lanes (element [lane%4][register]), two exchange stages
__device__ __forceinline__ void quad_transpose(float (&r)[4], int lane) {
    const bool b0 = lane & 1, b1 = lane & 2;
#pragma unroll
    for (int p = 0; p < 4; p += 2) {  // swap (even lane, odd reg) <-> (odd lane, even reg)
        const float give = b0 ? r[p] : r[p + 1];
        const float got = xor_lane<1>(give);
        if (b0) r[p] = got;
        else r[p + 1] = got;
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {     // swap (lane bit1 clear, reg p+2) <-> (lane bit1 set, reg p)
        const float give = b1 ? r[p] : r[p + 2];
        const float got = xor_lane<2>(give);
        if (b1) r[p] = got;
        else r[p + 2] = got;
    }
}

// sum over the 16 lanes that share lane%4 (blocks b = 0..15)
__device__ __forceinline__ float sum_over_blocks(float v) {
    v += xor_lane<4>(v);
    v += xor_lane<8>(v);
    v += xor_lane<16>(v);
    v += xor_lane<32>(v);
    return v;
}
__device__ __forceinline__ float max_over_blocks(float v) {
    v = fmaxf(v, xor_lane<4>(v));
    v = fmaxf(v, xor_lane<8>(v));
    v = fmaxf(v, xor_lane<16>(v));
    v = fmaxf(v, xor_lane<32>(v));
    return v;
}

struct AttnArgs {
    const void *q;       // [groups*4][128] queries in the original domain, q_dtype
    int q_dtype;
    const float *ks1, *ks2;  // K rotation signs (NULL: K is not rotated, q is only scaled)
    float scale_log2e;       // logit scale * log2(e), folded into the fp16 query
    const uint8_t *k, *v;
    const uint32_t *klut, *vlut;  // pair tables (half2 per pair code)
    const float *bias;            // [groups*4][tokens] natural-log units, or NULL
    const int32_t *sbias_pos;     // sparse bias: [groups*q_group][sbias_n] positions, ascending within a head (entries that
    const float *sbias_val;       // do not exist: any position >= tokens), and their values (natural-log units)
    int sbias_n;                  // entries per head, 0 = no sparse bias
    float *part_o;                // [groups][workgroups per group][4][128]
    float *part_ml;               // [groups][workgroups per group][4][2]  (m in log2 units, l)
    unsigned long long *skip_slots;  // Sparse V: [workgroup] nonce tag | (query, position) pairs it skipped; 0 after the count
    // merge of the workgroups' partials by the last workgroup of a group to finish (see merge_group)
    float *out;                      // [groups * q_group][128]
    const float *vs1, *vs2;          // V rotation signs (NULL: V rows are stored unrotated)
    unsigned long long *flags;       // [group][workgroups per group]; word 0 of a group is its arrival counter (tag | count), 0 after the merge
    unsigned long long nonce;        // differs from call to call (and from whatever the workspace held before)
    int poll_slots;                       // Sparse V: the merging workgroups add the slots up themselves
    unsigned long long *pass_totals;      // Sparse V: [pass] skipped pairs of each four-head pass of this step
    unsigned long long *skip_count;       // caller's {skipped, total} or NULL
    unsigned long long total_pairs;
    int pass;                             // head_off / pass_heads
    int64_t tokens, blocks_per_seq;
    const int64_t *tokens_dev;  // NULL, or where the step's context length is read from (<= tokens, which then is the maximum)
    int n_groups, n_splits, tiles_per_split, n_tiles;
    int q_group, head_off;  // query heads per KV head; first of the heads that this launch's first pass works on
    int d256;               // heads of 256 dims: a token is two 128-value rows (2 token + half) of the K and V caches
    int gpw;                // (batch, kv head) groups per workgroup: 1, or wavefronts per workgroup / n_splits when a group's
                            // splits are fewer than a workgroup's wavefronts (short contexts: the groups share the decode tables)
    int gw_shift;           // gpw > 1: log2(n_splits), a power of two then
    int wgs_per_group;      // gpw == 1: n_splits / wavefronts per workgroup
    float tau;
    int pass_heads;         // heads per pass; blockIdx.y numbers the passes of a launch, whose partials and counters follow each other
};

constexpr int KFMT_TURBO = 0, KFMT_Q8 = 1;
constexpr unsigned long long SKIP_COUNT_MASK = (1ull << 40) - 1ull;  // count bits of a Sparse-V slot; the rest is a nonce tag
constexpr int MERGE_FLOATS = 520;  // LDS floats per wavefront for the end-of-kernel merge: out[4][128], (m, l)[4]


constexpr unsigned long long ARRIVAL_COUNT_MASK = 0xFFFFFFull;  // workgroups of a group (the tag of the call sits above)

// ---- merging the workgroups' partials inside the launch -------------------------------------
// A group's partials are written by up to n_splits / wavefronts-per-workgroup workgroups that may run on
// different dies, whose L2 caches are not coherent with each other for ordinary accesses.  Everything the
// workgroups exchange therefore moves with device-scope atomic accesses (they go through to memory): a workgroup
// stores its partial, waits for the stores to complete, and then increments the group's arrival counter with one
// read-modify-write; the workgroup whose increment completes the count merges the group.  The counter carries a tag
// of the call, so what a fresh workspace happens to contain is not mistaken for arrivals, and the merging workgroup
// puts it back to zero, so a replay of a captured launch (same tag) starts clean.  No cache-wide write-back or
// invalidate is involved, which is what made a merge behind device-scope fences cost more than the second launch it
// saved.
// What the end of a step costs is its chain of waits, so every link keeps all of its loads in flight at once.  Timestamps of a
// step of 48 groups, eight heads, eight workgroups of four wavefronts each (6 x 10 007 tokens, turbo4; 33.1 us in all): the
// wavefronts' merge 3.4 us, its stores 0.3, the counter 0.8 (a look, then the increment), the partials' merge 4.7.  With
// the reads of all wavefronts in flight, the counter's tag installed at the start and two heads' loads side by side the step takes
// 27.3 us; one user's step at 4000 tokens 12.7 -> 10.6, 128 groups at 32K 78.1 -> 76.9, 256 groups with one partial 15.4 -> 12.7.
__device__ __forceinline__ void st_dev(float *p, float v) {
    __hip_atomic_store(reinterpret_cast<uint32_t *>(p), __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(unsigned long long *p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev2(float *p, float x, float y) {  // 8-byte aligned pair
    st_dev(reinterpret_cast<unsigned long long *>(p), ((unsigned long long)__float_as_uint(y) << 32) | __float_as_uint(x));
}
__device__ __forceinline__ unsigned long long ld_dev(const unsigned long long *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 ld_dev2(const float *p) {  // 8-byte aligned pair
    const unsigned long long u = ld_dev(reinterpret_cast<const unsigned long long *>(p));
    return make_float2(__uint_as_float((uint32_t)u), __uint_as_float((uint32_t)(u >> 32)));
}
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The partials [0, n) of NHD heads of a group, merged by one wavefront: running maximum M (log2 units), weight sum L and this
// lane's two output dims, all relative to M.  Up to 16 partials of a head have every load requested before the first is used, so
// the merge costs one trip to memory (in batches of four, sixteen partials took four trips at the very end of the launch).
struct MergedPart {
    float M, L, o0, o1;
};
template <int NP, int NHD>
__device__ __forceinline__ void merge_few(const float *ml0, const float *po0, int ML, int PO, const int (&head)[NHD], int p_lo, int n, int lane,
                                          MergedPart (&r)[NHD]) {
    float2 ml[NHD][NP], v[NHD][NP];
#pragma unroll
    for (int k = 0; k < NHD; ++k)
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int pc = p_lo + (p < n ? p : 0);
            ml[k][p] = ld_dev2(ml0 + pc * ML + head[k] * 2);
            v[k][p] = ld_dev2(po0 + (int64_t)pc * PO + head[k] * 128 + 2 * lane);
            if (p >= n) ml[k][p].y = 0.0f;
        }
#pragma unroll
    for (int k = 0; k < NHD; ++k) {
        r[k] = MergedPart{-INFINITY, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int p = 0; p < NP; ++p)
            if (ml[k][p].y > 0.0f) r[k].M = fmaxf(r[k].M, ml[k][p].x);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const float w = ml[k][p].y > 0.0f ? __builtin_amdgcn_exp2f(ml[k][p].x - r[k].M) : 0.0f;
            r[k].L = fmaf(ml[k][p].y, w, r[k].L);
            r[k].o0 = fmaf(v[k][p].x, w, r[k].o0);
            r[k].o1 = fmaf(v[k][p].y, w, r[k].o1);
        }
    }
}
__device__ __forceinline__ MergedPart merge_range(const float *ml0, const float *po0, int ML, int PO, int head, int p_lo, int p_hi,
                                                  int lane) {
    MergedPart r{-INFINITY, 0.0f, 0.0f, 0.0f};
    const int n = p_hi - p_lo;
    if (n <= 0) return r;
    if (n <= 16) {
        const int hd[1] = {head};
        MergedPart one[1];
        if (n <= 4) merge_few<4, 1>(ml0, po0, ML, PO, hd, p_lo, n, lane, one);
        else if (n <= 8) merge_few<8, 1>(ml0, po0, ML, PO, hd, p_lo, n, lane, one);
        else merge_few<16, 1>(ml0, po0, ML, PO, hd, p_lo, n, lane, one);
        return one[0];
    }
    {
        for (int p0 = p_lo; p0 < p_hi; p0 += 64) {  // lane <-> partial: maximum, then weights
            const int p = p0 + lane;
            float m = -INFINITY;
            if (p < p_hi) {
                const float2 e = ld_dev2(ml0 + p * ML + head * 2);
                if (e.y > 0.0f) m = e.x;
            }
            for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
            r.M = fmaxf(r.M, m);
        }
        for (int p0 = p_lo; p0 < p_hi; p0 += 64) {
            const int p = p0 + lane;
            float w = 0.0f, l = 0.0f;
            if (p < p_hi) {
                const float2 e = ld_dev2(ml0 + p * ML + head * 2);
                l = e.y;
                w = l > 0.0f ? __builtin_amdgcn_exp2f(e.x - r.M) : 0.0f;
            }
            float lw = l * w;
            for (int o = 32; o > 0; o >>= 1) lw += __shfl_xor(lw, o);
            r.L += lw;
            const int cnt = min(64, p_hi - p0);
            // eight partials per trip to memory (a lane exchange cannot sit in a loop that the compiler unrolls with
            // a remainder, so the batches are written out: past the count the last partial is read again with weight 0)
            for (int t0 = 0; t0 < cnt; t0 += 8) {
                float2 v[8];
                float wt[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const int t = min(t0 + k, cnt - 1);
                    v[k] = ld_dev2(po0 + (int64_t)(p0 + t) * PO + head * 128 + 2 * lane);
                    wt[k] = t0 + k < cnt ? __shfl(w, t) : 0.0f;
                }
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    r.o0 = fmaf(v[k].x, wt[k], r.o0);
                    r.o1 = fmaf(v[k].y, wt[k], r.o1);
                }
            }
        }
    }
    return r;
}

// A head's normalised output in the V rotation's domain (two dims per lane) -> its output row.  s1, s2: this lane's signs of the V
// rotation (unused where V rows are stored unrotated).
__device__ __forceinline__ void write_row(const AttnArgs &a, int group, int head_off, int head, float o0, float o1, float2 s1, float2 s2, int lane) {
    // heads of 256 dims: partial row 4 dh + i is dims 128 dh .. 128 dh + 127 of head i
    const int hq = a.d256 ? (head & 3) : head;
    if (head_off + hq >= a.q_group) return;   // a repeated head of a group with fewer left
    const int64_t row = a.d256 ? 2 * ((int64_t)group * a.q_group + head_off + hq) + (head >> 2) : (int64_t)group * a.q_group + head_off + head;
    if (a.vs1) {
        o0 *= s2.x;
        o1 *= s2.y;
        wht128_wave(o0, o1, lane);
        o0 *= s1.x * RSQRT128;
        o1 *= s1.y * RSQRT128;
    }
    *reinterpret_cast<float2 *>(a.out + row * 128 + 2 * lane) = make_float2(o0, o1);
}

// The group's partials -> output rows (log-sum-exp merge, then the V rotation's transpose).  A workgroup with at least
// twice as many wavefronts as the pass has heads gives every head several wavefronts, each merging a share of the
// partials, and joins their results through `lds` (free LDS of 132 floats per wavefront; unused otherwise); one with fewer
// wavefronts than heads has the loads of two heads in flight together: the merge runs at the very end of the launch, so its
// trips to memory are the launch's tail.
template <int HG>
__device__ __forceinline__ void merge_group(const AttnArgs &a, int group, int pgroup, int head_off, int n_parts, int tid, int n_waves,
                                            float *lds, float2 s1, float2 s2) {
    constexpr int NH = 4 * HG, ML = 2 * NH, PO = 128 * NH;  // heads, (m, l) floats and output floats of one partial
    const int lane = tid & 63, wave = tid >> 6;
    const float *ml0 = a.part_ml + (int64_t)pgroup * n_parts * ML;
    const float *po0 = a.part_o + (int64_t)pgroup * n_parts * PO;
    auto finish = [&](int head, MergedPart r) {
        const float invL = r.L > 0.0f ? 1.0f / r.L : 0.0f;
        write_row(a, group, head_off, head, r.o0 * invL, r.o1 * invL, s1, s2, lane);
    };
    auto head_exists = [&](int head) { return head_off + (a.d256 ? (head & 3) : head) < a.q_group; };
    const int n_sub = n_waves >= 2 * NH && n_parts > 4 ? n_waves / NH : 1;
    if (n_sub == 1) {
        if (n_waves < NH && n_parts <= 8) {
            for (int head = wave; head < NH; head += 2 * n_waves) {
                const int hd[2] = {head, min(head + n_waves, NH - 1)};
                MergedPart two[2];
                merge_few<8, 2>(ml0, po0, ML, PO, hd, 0, n_parts, lane, two);
                finish(head, two[0]);
                if (head + n_waves < NH) finish(head + n_waves, two[1]);
            }
            return;
        }
        for (int head = wave; head < NH; head += n_waves)
            if (head_exists(head)) finish(head, merge_range(ml0, po0, ML, PO, head, 0, n_parts, lane));
        return;
    }
    const int head = wave % NH, sub = wave / NH;
    const int per = (n_parts + n_sub - 1) / n_sub;
    const bool mine = sub < n_sub && head_exists(head);
    MergedPart r{-INFINITY, 0.0f, 0.0f, 0.0f};
    if (mine) r = merge_range(ml0, po0, ML, PO, head, min(sub * per, n_parts), min(sub * per + per, n_parts), lane);
    float *slot = lds + (head * n_sub + (sub < n_sub ? sub : 0)) * 132;
    if (mine) {
        *reinterpret_cast<float2 *>(slot + 2 * lane) = make_float2(r.o0, r.o1);
        if (lane == 0) {
            slot[128] = r.M;
            slot[129] = r.L;
        }
    }
    __syncthreads();
    if (mine && sub == 0) {
        const float *s0 = lds + head * n_sub * 132;
        float M = -INFINITY;
        for (int k = 0; k < n_sub; ++k)
            if (s0[k * 132 + 129] > 0.0f) M = fmaxf(M, s0[k * 132 + 128]);
        MergedPart t{M, 0.0f, 0.0f, 0.0f};
        for (int k = 0; k < n_sub; ++k) {
            const float l = s0[k * 132 + 129];
            const float w = l > 0.0f ? __builtin_amdgcn_exp2f(s0[k * 132 + 128] - M) : 0.0f;
            const float2 o = *reinterpret_cast<const float2 *>(s0 + k * 132 + 2 * lane);
            t.L = fmaf(l, w, t.L);
            t.o0 = fmaf(o.x, w, t.o0);
            t.o1 = fmaf(o.y, w, t.o1);
        }
        finish(head, t);
    }
}

// A group's wavefronts -> one partial (in memory, or where the group has only this one, normalised, in the first wavefront's
// slot).  A wavefront's slot: per set of four heads out[4][128] relative to its own maximum, then (m, l)[4].  Every thread takes
// 1 to 4 neighbouring values and has the reads of all W slots in flight before it uses the first: a loop of LDS round trips per
// value made this 2.2 us of a step of four wavefronts and 3.4 us with eight heads.
template <int HG, int W, class Slot>
__device__ __forceinline__ void combine_waves_of(Slot slot, int wave0, int tid_g, float *po, float *pml, bool only) {
    constexpr int E = 512 * HG, PER = E / (64 * W), VW = PER >= 4 ? 4 : PER >= 2 ? 2 : 1;
    typedef float vec_t __attribute__((ext_vector_type(VW)));
    for (int e = VW * tid_g; e < E; e += VW * 64 * W) {
        const int src = (e >> 9) * MERGE_FLOATS + (e & 511), ml_at = (e >> 9) * MERGE_FLOATS + 512 + 2 * ((e >> 7) & 3);
        float2 ml[W];
        vec_t v[W];
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float *s = slot(wave0 + w);
            ml[w] = *reinterpret_cast<const float2 *>(s + ml_at);
            v[w] = *reinterpret_cast<const vec_t *>(s + src);
        }
        float M = -INFINITY, L = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w)
            if (ml[w].y > 0.0f) M = fmaxf(M, ml[w].x);   // wavefronts that saw an unmasked position
        vec_t sum = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const bool seen = ml[w].y > 0.0f;   // false for a sum that is not a number, too: it stays out of the others'
            const float f = seen ? __builtin_amdgcn_exp2f(ml[w].x - M) : 0.0f;
            L = seen ? fmaf(ml[w].y, f, L) : L;
#pragma unroll
            for (int i = 0; i < VW; ++i) sum[i] = fmaf(v[w][i], f, sum[i]);
        }
        if (only) {
            *reinterpret_cast<vec_t *>(slot(wave0) + src) = sum * (L > 0.0f ? 1.0f / L : 0.0f);   // no other thread reads this place
        } else {
            if constexpr (VW == 1) st_dev(po + e, sum[0]);
            else
#pragma unroll
                for (int i = 0; i < VW; i += 2) st_dev2(po + e + i, sum[i], sum[i + 1]);
            if ((e & 127) == 0) st_dev2(pml + 2 * (e >> 7), M, L);
        }
    }
}
template <int HG, class Slot>
__device__ __forceinline__ void combine_waves(Slot slot, int gw, int wave0, int tid_g, float *po, float *pml, bool only) {
    switch (gw) {   // the counts that attn_plan makes: powers of two, with eight heads also twelve and its halves
        case 1: combine_waves_of<HG, 1>(slot, wave0, tid_g, po, pml, only); break;
        case 2: combine_waves_of<HG, 2>(slot, wave0, tid_g, po, pml, only); break;
        case 4: combine_waves_of<HG, 4>(slot, wave0, tid_g, po, pml, only); break;
        case 8: combine_waves_of<HG, 8>(slot, wave0, tid_g, po, pml, only); break;
        default:
            if constexpr (HG == 1) {
                combine_waves_of<HG, 16>(slot, wave0, tid_g, po, pml, only);
            } else {
                if (gw == 3) combine_waves_of<HG, 3>(slot, wave0, tid_g, po, pml, only);
                else if (gw == 6) combine_waves_of<HG, 6>(slot, wave0, tid_g, po, pml, only);
                else combine_waves_of<HG, 12>(slot, wave0, tid_g, po, pml, only);
            }
    }
}

// sum over the workgroup of one 64-bit value per thread (every thread gets the total); red: one shared word
__device__ __forceinline__ unsigned long long block_sum(unsigned long long t, unsigned long long *red, int tid) {
    if (tid == 0) *red = 0ull;
    __syncthreads();
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o);
    if ((tid & 63) == 0 && t) atomicAdd(red, t);
    __syncthreads();
    return *red;
}
// The arrival counter of a group: the call's tag in the upper 40 bits, the number of workgroups whose partial is in memory in the
// lower 24.  A word that does not carry the tag (whatever a fresh workspace held, or the zero a finished call leaves) gets it
// from the first workgroup to look, with a count of zero; workgroups do so at their start, so that one read-modify-write per
// workgroup remains at their end.
__device__ __forceinline__ unsigned long long *arrival_counter(const AttnArgs &a, int pgroup, int n_parts) { return a.flags + (int64_t)pgroup * n_parts; }
__device__ __forceinline__ void install_tag(const AttnArgs &a, unsigned long long *ctr, unsigned long long seen) {
    const unsigned long long tag = a.nonce & ~ARRIVAL_COUNT_MASK;
    // a failed exchange means that another workgroup of this call was first: nobody else writes the word meanwhile
    if ((seen & ~ARRIVAL_COUNT_MASK) != tag)
        __hip_atomic_compare_exchange_strong(ctr, &seen, tag, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The end of a workgroup's part: its wavefronts' results (in their slots) become one partial, the group's last workgroup to
// arrive merges the partials and writes the output rows.  gw wavefronts from wave0 on work on the group (tid_g numbers their
// threads); lds: 132 floats of LDS per wavefront for merge_group, free once the slots have been read; skipped: Sparse V, the
// workgroup's count in LDS.
template <int HG, bool SPARSE, class Slot>
__device__ __forceinline__ void finish_group(const AttnArgs &a, Slot slot, int group, int pgroup, int head_off, int n_parts, int part, int tid,
                                             int tid_g, int gw, int wave0, float *lds, const uint32_t *skipped) {
    constexpr int NH = 4 * HG;
    const int lane = tid & 63;
    // the V rotation's signs, requested before the waits below
    float2 s1 = make_float2(1.0f, 1.0f), s2 = s1;
    if (a.vs1) {
        s1 = *reinterpret_cast<const float2 *>(a.vs1 + 2 * lane);
        s2 = *reinterpret_cast<const float2 *>(a.vs2 + 2 * lane);
    }
    __syncthreads();   // every slot (and the skipped count) is written
    const int64_t at = (int64_t)pgroup * n_parts + part;
    combine_waves<HG>(slot, gw, wave0, tid_g, a.part_o + at * NH * 128, a.part_ml + at * NH * 2, n_parts == 1);
    if constexpr (SPARSE) {
        // one slot per workgroup, added up by the merging workgroups: thousands of wavefronts finishing together
        // on one atomic would queue for longer than the kernel's own tail, and nothing needs clearing
        if (tid == 0) st_dev(a.skip_slots + blockIdx.x, (a.nonce & ~SKIP_COUNT_MASK) | (unsigned long long)*skipped);
    }
    if (n_parts > 1 || SPARSE) wait_stores();  // this lane's part of the partial (and the skip slot) is in memory
    __syncthreads();
    if (n_parts > 1) {
        // Read-modify-writes on one word happen one after the other, so exactly one workgroup brings the count to n_parts: it
        // merges, and every other partial was complete in memory before its owner's increment, hence before this one's.
        __shared__ int i_am_last;
        if (tid == 0) {
            const unsigned long long before = __hip_atomic_fetch_add(arrival_counter(a, pgroup, n_parts), 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            i_am_last = (int)(before & ARRIVAL_COUNT_MASK) + 1 == n_parts;
        }
        __syncthreads();
        if (!i_am_last) return;
    }
    // Sparse V: every workgroup's slot carries its count (40 bits: at most 4 heads x 2^31 positions) under 24 bits
    // of the nonce.  A merging workgroup reads all slots of the launch now, so that the trip to memory overlaps
    // the merge; the one that finds them all tagged (the merging workgroup of the group that finishes last does)
    // writes the step's total.  Launches with more workgroups than one can poll are added up by a launch of their
    // own (poll_slots == 0).
    int all_in = 1;
    unsigned long long counted = 0ull;
    if constexpr (SPARSE) {
        if (a.poll_slots) {
            const unsigned long long tag = a.nonce & ~SKIP_COUNT_MASK;
            for (int g = tid; g < (int)gridDim.x; g += (int)blockDim.x) {
                const unsigned long long word = ld_dev(a.skip_slots + g);
                all_in &= (word & ~SKIP_COUNT_MASK) == tag;
                counted += word & SKIP_COUNT_MASK;
            }
        }
    }
    if (n_parts > 1) {
        merge_group<HG>(a, group, pgroup, head_off, n_parts, tid, gw, lds, s1, s2);   // one group per workgroup then
    } else {
        const float *rows = slot(wave0);
        for (int head = tid_g >> 6; head < NH; head += gw) {
            const float2 o = *reinterpret_cast<const float2 *>(rows + (head >> 2) * MERGE_FLOATS + (head & 3) * 128 + 2 * lane);
            write_row(a, group, head_off, head, o.x, o.y, s1, s2, lane);
        }
    }
    if (n_parts > 1 && tid == 0) st_dev(arrival_counter(a, pgroup, n_parts), 0ull);  // a replay of a captured launch (same tag) starts from zero
    if constexpr (SPARSE) {
        if (a.poll_slots) {
            if (!__syncthreads_and(all_in)) return;
            __shared__ unsigned long long red;
            const unsigned long long pass_total = block_sum(counted, &red, tid);
            for (int g = tid; g < (int)gridDim.x; g += (int)blockDim.x) st_dev(a.skip_slots + g, 0ull);
            if (tid == 0) {
                // this pass's total is kept apart so that writing the step's total twice (two groups finishing
                // together) gives the same value both times
                st_dev(a.pass_totals + a.pass, pass_total);
                unsigned long long sum = pass_total;
                for (int k = 0; k < a.pass; ++k) sum += ld_dev(a.pass_totals + k);
                a.skip_count[0] = sum;
                a.skip_count[1] = a.total_pairs;
            }
        }
    }
}

}  // namespace tqattn

// Launchers of the kernel files; kb, vb: code widths (8: q8_0-style rows), hg: sets of four heads per pass; false: no such pair.
// attn_turbo_kernels.hip: 128-dim heads, turbo rows, 4-bit on one side or both; n_heads 4 or 8; and a workgroup's static LDS
bool tqk_launch_decode_turbo(const tqattn::AttnArgs &a, int kb, int vb, bool share, int n_heads, bool sparse, dim3 grid, int waves,
                             hipStream_t s);
int tqk_decode_turbo_lds(int kb, int vb, bool share);
bool tqk_launch_decode_q8(const tqattn::AttnArgs &a, int kb, int vb, int hg, bool sparse, dim3 grid, unsigned wg, size_t lds, hipStream_t s);
bool tqk_launch_decode_256(const tqattn::AttnArgs &a, int kb, int vb, bool share, bool sparse, dim3 grid, unsigned wg, size_t lds,
                           hipStream_t s);
