// Reference-API kernels: float64 arithmetic, any dimension up to 4096.
//
// These back the Python classes that keep the reference's signatures
// (PolarQuant, QJL, the rotation and codebook free functions, pack helpers).
// Dense rotations and projections run as one float64 matrix-core product per
// call with the per-vector work in its prologue and epilogue (k_dense64).  The
// sign-diagonal Walsh-Hadamard rotation is a butterfly in LDS, one workgroup of
// 128 threads per VB = 8 vectors (4 or 2 for dimensions above 1024 / 2048), in
// the reference's stage order, which makes the float64 WHT results
// bit-identical to NumPy's.
#include <algorithm>

#include "tq_internal.h"
#include "tq_device64.h"

namespace {

using namespace tq64;

// number of midpoints strictly below v: nb = 2^bits - 1 of them, ascending (NaN: 0)
__device__ __forceinline__ int level_of(double v, const double *bounds, int bits) {
    int c = 0;
    for (int b = bits - 1; b >= 0; --b) {
        const int t = c + (1 << b);
        if (bounds[t - 1] < v) c = t;
    }
    return c;
}

// ---- dense products: out[row][j] = sum_k f(in[row][k]) M[k][j], float64 matrix cores -----------------------------
// One thread per (output, vector) read the whole matrix from L2 once per VB vectors and an LDS operand per multiply:
// 1.56 ms per product for 256 vectors of 1536 (0.8 of 75 TFLOP/s), 92 us for 32 768 of 128.  Here a wavefront owns RT x
// CT tiles of 16 x 16 outputs of v_mfma_f64_16x16x4_f64 and a slice of the contraction or all of it: 28 to 32 and 34 to 43 us
// by what is folded in (back to back and traced).  What
// bounds it is the matrix instruction (64 clocks; 22 and 20 us of them at the 1.7 GHz the part holds here), then the
// uneven last round of workgroups.  The order of the contraction is free, so in a chunk of 16 values lane quarter q takes
// values 4q .. 4q+3 for the chunk's four steps: the A operand of four steps is one vector load, the B operand of a step
// four runs of 128 bytes.  Nothing is staged in LDS during the product.
// The contraction is summed in `slices` slices (the chunks in turn), as many as the dimension alone says, and the slices are
// added in their order, so that a vector's results do not depend on the batch it comes in.  SPLIT: a wavefront per slice, the
// tiles added in LDS at the end, wavefronts past the slices on further rows.  Else a wavefront goes through the slices of its
// tiles one after the other and keeps their sum beside the running one.  Column blocks are dealt to the XCDs in turn, so that
// each XCD's L2 holds only its eighth of the matrix (an 18.9 MB matrix at d = 1536 against 4 MB of L2).
// The vectors' norms are row properties that the contraction's own operands give, a lane quarter's squares summed over the
// slices and then over the quarters (one multiply-add per operand
// beside the tiles' matrix instructions) and divide the finished sums, so nothing passes over the input twice.
enum DenseOp { DENSE_ROTATE, DENSE_QUANTIZE, DENSE_DEQUANTIZE, DENSE_QJL_QUANTIZE, DENSE_QJL_DEQUANTIZE };

struct DenseArgs {
    int d;
    int64_t n;
    const double *mat;        // M, row-major [d][d]
    const void *in;           // [n][d]: vectors, indices or signs
    int slices;               // of the contraction; SPLIT: wavefronts that share a tile's
    unsigned n_row, n_col;    // row and column blocks of the launch
    // quantize: bounds, bits; dequantize: centroids, norm_correction
    const double *bounds, *centroids;
    int bits, norm_correction;
    const double *norms_in;   // dequantize, QJL dequantize
    double *norms_out;        // quantize, QJL quantize
    void *out;                // ROTATE: values; QUANTIZE: indices; (QJL_)DEQUANTIZE: float64; QJL_QUANTIZE: int8 signs
    double *rotated;          // quantize: rotated unit vectors or NULL
    const void *x;            // dequantize: the vectors that `residual` is taken against
    double *residual;
    double proj_scale, shrinkage;
    int accumulate;           // QJL dequantize: add to out
};

typedef double double4_t __attribute__((ext_vector_type(4)));

// OP, element type of the input, and of the output (of x: DEQUANTIZE)
template <DenseOp OP, typename TI, typename TO, int RT, int CT, int NW, bool SPLIT>
__global__ __launch_bounds__(64 * NW) void k_dense64(DenseArgs a) {
    constexpr bool NORMS = OP == DENSE_QUANTIZE || OP == DENSE_QJL_QUANTIZE || OP == DENSE_DEQUANTIZE;
    constexpr int NT_ = RT * CT;
    extern __shared__ double sm[];   // SPLIT: [NW][NT_][4][64] tiles of one slice
    __shared__ double table[OP == DENSE_DEQUANTIZE || OP == DENSE_QUANTIZE ? 256 : 1];
    __shared__ double sq_s[NORMS && SPLIT ? NW : 1][4][RT * 16];   // squares of a slice's rows by lane quarter
    __shared__ double norm_s[NORMS ? NW : 1][RT * 16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, q = lane >> 4;
    const int ks = SPLIT ? a.slices : 1;   // wavefronts per tile
    const int kslice = wave % ks, rgroup = wave / ks, rgs = NW / ks;
    unsigned row_b, col_b;
    if (a.n_col >= 8) {   // column block % 8 = blockIdx % 8 = the XCD
        const unsigned i = blockIdx.x >> 3;
        row_b = i % a.n_row;
        col_b = (i / a.n_row) * 8 + (blockIdx.x & 7);
        if (col_b >= a.n_col) return;
    } else {
        col_b = blockIdx.x % a.n_col;
        row_b = blockIdx.x / a.n_col;
    }
    const int d = a.d;
    const int64_t row0 = ((int64_t)row_b * rgs + rgroup) * (RT * 16);
    const int col0 = (int)col_b * (CT * 16);
    if constexpr (OP == DENSE_DEQUANTIZE) {
        for (int e = tid; e < 256; e += 64 * NW) table[e] = a.centroids[min(e, (1 << a.bits) - 1)];
        __syncthreads();
    }
    if constexpr (OP == DENSE_QUANTIZE)
        for (int e = tid; e < (1 << a.bits) - 1; e += 64 * NW) table[e] = a.bounds[e];

    // Addresses are a wave-uniform part, which moves with the chunk, and a lane's own offset.  Rows and columns past the
    // end repeat the last one; their sums are not stored.
    const int64_t rbase = row0 < a.n ? row0 : a.n - 1;
    const TI *in = reinterpret_cast<const TI *>(a.in) + rbase * d;
    uint32_t aoff[RT], boff[CT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) aoff[rt] = (uint32_t)min((int64_t)(16 * rt + c16), a.n - 1 - rbase) * d + 4 * q;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) boff[ct] = 4 * q * d + min(col0 + 16 * ct + c16, d - 1);

    struct Operands {
        TI x[RT][4];
        double b[CT][4];
    };
    auto load = [&](int chunk, Operands &o) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) __builtin_memcpy(o.x[rt], in + 16 * chunk + aoff[rt], 4 * sizeof(TI));
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const double *mrow = a.mat + (int64_t)(16 * chunk + s) * d;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) o.b[ct][s] = mrow[boff[ct]];
        }
    };
    double4_t acc[RT][CT];
    double sq[RT][2];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        sq[rt][0] = sq[rt][1] = 0.0;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = double4_t{0.0, 0.0, 0.0, 0.0};
    }
    auto value = [&](TI e) {
        if constexpr (OP == DENSE_DEQUANTIZE) return table[e];   // 256 entries, those past the codebook its last
        else return ldd(&e, 0);
    };
    auto multiply = [&](const Operands &o) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const double v = value(o.x[rt][s]);
                if constexpr (NORMS) sq[rt][s & 1] = fma(v, v, sq[rt][s & 1]);
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, o.b[ct][s], acc[rt][ct], 0, 0, 0);
            }
        }
    };
    const int full = d >> 4;
    if ((d & 15) && kslice == 0) {   // what is past the whole chunks opens the first slice, value by value
        const int k0 = 16 * full + 4 * q;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const bool in_row = k0 + s < d;
            double bv[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) bv[ct] = a.mat[(int64_t)min(k0 + s, d - 1) * d + min(col0 + 16 * ct + c16, d - 1)];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const double v = in_row ? value(in[aoff[rt] - 4 * q + min(k0 + s, d - 1)]) : 0.0;
                if constexpr (NORMS) sq[rt][s & 1] = fma(v, v, sq[rt][s & 1]);
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, bv[ct], acc[rt][ct], 0, 0, 0);
            }
        }
    }
    // whole chunks; the request past this wavefront's last one repeats it, so that what has to be waited for is the same on
    // every path (a branch around the request made the compiler wait for the newest one everywhere: 59 against 32 us for
    // 256 vectors of 1536; holding the request in front of the products with scheduling barriers changed nothing)
    int left = SPLIT ? (full - kslice + ks - 1) / ks : full;
    double4_t sum[SPLIT ? 1 : RT][SPLIT ? 1 : CT];   // the finished slices
    double sq_sum[RT];
    if constexpr (!SPLIT) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            sq_sum[rt] = 0.0;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) sum[rt][ct] = double4_t{0.0, 0.0, 0.0, 0.0};
        }
    }
    auto after = [&](int c) {   // the chunk after c
        c += a.slices;
        return SPLIT || c < full ? c : c % a.slices + 1;
    };
    auto finish = [&](int c) {   // c: the chunk just multiplied; the last one of its slice?
        if constexpr (!SPLIT) {
            if (c + a.slices < full) return;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                if constexpr (NORMS) {
                    sq_sum[rt] += sq[rt][0] + sq[rt][1];
                    sq[rt][0] = sq[rt][1] = 0.0;
                }
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    sum[rt][ct] += acc[rt][ct];
                    acc[rt][ct] = double4_t{0.0, 0.0, 0.0, 0.0};
                }
            }
        }
    };
    if (left > 0) {
        Operands o0, o1;
        int c = kslice, next;
        load(c, o0);
        while (true) {
            next = left > 1 ? after(c) : c;
            load(next, o1);
            multiply(o0);
            finish(c);
            c = next;
            if (--left == 0) break;
            next = left > 1 ? after(c) : c;
            load(next, o0);
            multiply(o1);
            finish(c);
            c = next;
            if (--left == 0) break;
        }
    }
    // norms: a lane quarter's squares, summed over the slices, then over the quarters
    if constexpr (NORMS) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            double s = SPLIT ? sq[rt][0] + sq[rt][1] : sq_sum[rt];
            if (SPLIT && ks > 1) {
                sq_s[wave][q][16 * rt + c16] = s;
            } else {
                s += __shfl_xor(s, 16);
                s += __shfl_xor(s, 32);
                if (q == 0) norm_s[rgroup][16 * rt + c16] = sqrt(s);
            }
        }
    }
    if (SPLIT && ks > 1) {
        double *mine = sm + (size_t)wave * NT_ * 256 + lane;
#pragma unroll
        for (int t = 0; t < NT_; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) mine[(t * 4 + i) * 64] = acc[t / CT][t % CT][i];
    }
    __syncthreads();
    if constexpr (NORMS && SPLIT) {
        if (ks > 1) {
            for (int e = tid; e < rgs * RT * 16; e += 64 * NW) {
                const int g = e / (RT * 16), r = e % (RT * 16);
                double t[4] = {0.0, 0.0, 0.0, 0.0};
                for (int w = 0; w < ks; ++w)
#pragma unroll
                    for (int k = 0; k < 4; ++k) t[k] += sq_s[g * ks + w][k][r];
                norm_s[g][r] = sqrt((t[0] + t[1]) + (t[2] + t[3]));
            }
            __syncthreads();
        }
    }
    if constexpr (OP == DENSE_QUANTIZE || OP == DENSE_QJL_QUANTIZE) {
        if (col_b == 0 && kslice == 0)
            for (int r = lane; r < RT * 16; r += 64)
                if (row0 + r < a.n) a.norms_out[row0 + r] = norm_s[rgroup][r];
    }
#pragma unroll
    for (int t = 0; t < NT_; ++t) {
        if (t % ks != kslice) continue;   // the tile's wavefronts share out its tiles
        const int rt = t / CT, ct = t % CT, col = col0 + 16 * ct + c16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 16 * rt + 4 * i + q;
            const int64_t row = row0 + r;
            double y;
            if constexpr (!SPLIT) {
                y = sum[rt][ct][i];
            } else if (ks > 1) {
                y = 0.0;
                const double *part = sm + (size_t)(rgroup * ks) * NT_ * 256 + (t * 4 + i) * 64 + lane;
                for (int w = 0; w < ks; ++w) y += part[(size_t)w * NT_ * 256];
            } else {
                y = acc[rt][ct][i];
            }
            if (row >= a.n || col >= d) continue;
            const int64_t at = row * d + col;
            if constexpr (OP == DENSE_ROTATE) {
                std_(reinterpret_cast<TO *>(a.out), at, y);
            } else if constexpr (OP == DENSE_QUANTIZE) {
                const double nv = norm_s[rgroup][r];
                y /= nv > 0.0 ? nv : 1.0;
                // a norm past the type's range: finite entries over it are zeros, whatever their sums came to
                if (sizeof(TI) == 8 && nv == INFINITY) {
                    y = 0.0;
                    for (int k = 0; k < d; ++k) y += value(reinterpret_cast<const TI *>(a.in)[row * d + k]) * 0.0;
                }
                reinterpret_cast<uint8_t *>(a.out)[at] = (uint8_t)level_of(y, table, a.bits);
                if (a.rotated) a.rotated[at] = y;
            } else if constexpr (OP == DENSE_DEQUANTIZE) {
                if (a.norm_correction) {
                    const double cn = norm_s[rgroup][r];
                    y /= cn > 1e-10 ? cn : 1.0;
                }
                const double v = y * a.norms_in[row];
                if (a.out) reinterpret_cast<double *>(a.out)[at] = v;
                if (a.residual) a.residual[at] = ldd(reinterpret_cast<const TO *>(a.x), at) - v;
            } else if constexpr (OP == DENSE_QJL_QUANTIZE) {
                reinterpret_cast<int8_t *>(a.out)[at] = y < 0.0 ? (int8_t)-1 : (int8_t)1;
            } else {
                const double v = y * ((a.proj_scale * a.norms_in[row]) * a.shrinkage);
                double *o = reinterpret_cast<double *>(a.out) + at;
                *o = a.accumulate ? *o + v : v;
            }
        }
    }
}

template <DenseOp OP, typename TI, typename TO, int RT, int CT, bool SPLIT>
void launch_dense_tiles(DenseArgs a, int slices, hipStream_t s) {
    constexpr int NW = 8;
    a.slices = slices;
    const int ks = SPLIT ? slices : 1;
    const int rows = NW / ks * RT * 16;
    a.n_row = (unsigned)((a.n + rows - 1) / rows);
    a.n_col = (unsigned)((a.d + CT * 16 - 1) / (CT * 16));
    const unsigned grid = a.n_col >= 8 ? a.n_row * ((a.n_col + 7) / 8 * 8) : a.n_row * a.n_col;
    const size_t lds = ks > 1 ? (size_t)NW * RT * CT * 256 * sizeof(double) : 0;
    if (lds > 48 * 1024)
        (void)hipFuncSetAttribute((const void *)k_dense64<OP, TI, TO, RT, CT, NW, SPLIT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    k_dense64<OP, TI, TO, RT, CT, NW, SPLIT><<<grid, 64 * NW, lds, s>>>(a);
}

// Slices: eight, or as many as there are chunks of 16 values; by the dimension alone (see k_dense64).
// Tiles and wavefronts per tile, by the amount of work (us per product; SPLIT / not):
//   not SPLIT where whole tiles fill the chip - from 1536 tiles of 2 x 2 below 512 dimensions, where a slice is short beside
//   the exchange of its tiles (32 768 vectors of 128: 55 / 39; 4096 of 384: 50 / 43; 8192 of 128, 1024 tiles: 17 / 22), from
//   4096 above (4096 of 768, 3072 tiles: 117 / 141; 4096 of 1536, 6144 tiles: equal);
//   up to 16 vectors: single tiles (one vector of 1536: 8.0 against 11.5; sixteen: 12.7 against 15.3);
//   else the tiles of 1 x 1, 1 x 2, 2 x 2 or 2 x 3 whose workgroups are done first, where the launch takes as long as the CU
//   with the most of them and a workgroup as long as split_cost's last argument, to scale (a matrix operand is loaded per row
//   tile and a vector's per column tile, so small tiles cost more than their share).  256 of 1536, 1.5 workgroups of 2 x 2 per
//   CU or one of 2 x 3: 33.5 to 34.1 / 27.7 to 28.4 back to back; 200 of 1536 the same; 1000 of 384: 12.6 to 13.3 / 10.6 to 11.9; 325 of 768,
//   2 x 2 / 1 x 2: 18.2 / 13.9; 100 of 1536, 1 x 2 / 2 x 2: 21.9 to 25.1 / 19.5 to 20.6; 20 of 1536, 1 x 2 / 1 x 1: 13.6 / 10.6.
//   Not 1 x 1 or 1 x 2 from the fourth workgroup of a CU on (325 of 1536, 2 x 2 / 1 x 2: 47 / 38 to 49), nor 2 x 3 for less than a
//   tenth (2300 of 1536: 204 to 235 / 230) or where fewer than eight slices leave a workgroup short (5000 of 100: 12.2 / 12.8).
// A count of slices that follows the work as well (16 / 8 / 4 / 2 / none) is up to a tenth faster for many vectors (32 768 of
// 128: 37.9 us, of 256: 106 for 116, 1000 of 1536: 102 for 114) and differs in the last place between a batch and its vectors
// one by one.
// Workgroups of rt x ct tiles, shared by `slices` wavefronts each, on the busiest of the 256 CUs (of the 32 of an XCD where the
// columns are dealt to those), times the time of one; none if they are more than `most`.
inline int64_t split_cost(const DenseArgs &a, int slices, int rt, int ct, int64_t most, int cost) {
    const int64_t rows = 8 / slices * rt * 16, n_row = (a.n + rows - 1) / rows, n_col = (a.d + 16 * ct - 1) / (16 * ct);
    const int64_t wgs = n_col >= 8 ? (n_row * ((n_col + 7) / 8) + 31) / 32 : (n_row * n_col + 255) / 256;
    return wgs > most ? INT64_MAX : wgs * cost;
}

template <DenseOp OP, typename TI, typename TO>
int launch_dense(const DenseArgs &a, const char *what, hipStream_t s) {
    const int64_t tiles = ((a.n + 31) / 32) * ((a.d + 31) / 32);
    int slices = 8;
    while (slices > 1 && 16 * slices > a.d) slices >>= 1;
    if (slices > 1 && tiles >= (a.d < 512 ? 1536 : 4096)) {
        launch_dense_tiles<OP, TI, TO, 2, 2, false>(a, slices, s);
        return tq_check_launch(what);
    }
    const int64_t c11 = split_cost(a, slices, 1, 1, 3, 63), c12 = split_cost(a, slices, 1, 2, 3, 88),
                  c22 = split_cost(a, slices, 2, 2, INT64_MAX, 145), c23 = split_cost(a, slices, 2, 3, slices == 8 ? INT64_MAX : 0, 245);
    if (a.n <= 16 || c11 < std::min({c12, c22, c23})) launch_dense_tiles<OP, TI, TO, 1, 1, true>(a, slices, s);
    else if (c12 < std::min(c22, c23)) launch_dense_tiles<OP, TI, TO, 1, 2, true>(a, slices, s);
    else if (c22 <= c23) launch_dense_tiles<OP, TI, TO, 2, 2, true>(a, slices, s);
    else launch_dense_tiles<OP, TI, TO, 2, 3, true>(a, slices, s);
    return tq_check_launch(what);
}

template <int VB, typename TI, typename TO>
__global__ __launch_bounds__(NT) void k_rotate64(const TI *x, TO *y, int64_t n, RotArgs r) {
    extern __shared__ double sm[];
    double *xs = sm, *ys = sm + VB * r.pd;
    const int64_t v0 = (int64_t)blockIdx.x * VB;
    load_block<VB>(x, n, v0, r.d, r.pd, xs);
    rotate_block<VB>(r, xs, ys);
    for (int i = threadIdx.x; i < VB * r.d; i += NT) {
        const int v = i / r.d, j = i % r.d;
        if (v0 + v < n) std_(y, (v0 + v) * r.d + j, ys[v * r.pd + j]);
    }
}

template <int VB, typename T>
__global__ __launch_bounds__(NT) void k_quantize64(const T *x, int64_t n, RotArgs r, const double *bounds, int bits,
                                                  uint8_t *idx, double *norms, double *rotated) {
    extern __shared__ double sm[];
    __shared__ double nrm[VB];
    double *xs = sm, *ys = sm + VB * r.pd;
    const int64_t v0 = (int64_t)blockIdx.x * VB;
    load_block<VB>(x, n, v0, r.d, r.pd, xs);
    norms_block<VB>(xs, r.d, r.pd, nrm);
    for (int i = threadIdx.x; i < VB * r.pd; i += NT) {
        const double nv = nrm[i / r.pd];
        xs[i] = xs[i] / (nv > 0.0 ? nv : 1.0);
    }
    __syncthreads();
    rotate_block<VB>(r, xs, ys);
    for (int i = threadIdx.x; i < VB * r.d; i += NT) {
        const int v = i / r.d, j = i % r.d;
        if (v0 + v >= n) continue;
        const double yv = ys[v * r.pd + j];
        idx[(v0 + v) * r.d + j] = (uint8_t)level_of(yv, bounds, bits);
        if (rotated) rotated[(v0 + v) * r.d + j] = yv;
    }
    if (threadIdx.x < VB && v0 + threadIdx.x < n) norms[v0 + threadIdx.x] = nrm[threadIdx.x];
}

template <int VB, typename T>
__global__ __launch_bounds__(NT) void k_dequantize64(const uint8_t *idx, const double *norms, int64_t n, RotArgs r,
                                                    const double *centroids, int n_centroids, int norm_correction, double *out,
                                                    const T *x, double *residual) {
    extern __shared__ double sm[];
    __shared__ double nrm[VB];
    double *xs = sm, *ys = sm + VB * r.pd;
    const int64_t v0 = (int64_t)blockIdx.x * VB;
    for (int i = threadIdx.x; i < VB * r.pd; i += NT) {
        const int v = i / r.pd, j = i % r.pd;
        xs[i] = (v0 + v < n && j < r.d) ? centroids[min((int)idx[(v0 + v) * r.d + j], n_centroids - 1)] : 0.0;
    }
    __syncthreads();
    if (norm_correction) {
        norms_block<VB>(xs, r.d, r.pd, nrm);
        for (int i = threadIdx.x; i < VB * r.pd; i += NT) {
            const double nv = nrm[i / r.pd];
            xs[i] = xs[i] / (nv > 1e-10 ? nv : 1.0);
        }
        __syncthreads();
    }
    rotate_block<VB>(r, xs, ys);
    for (int i = threadIdx.x; i < VB * r.d; i += NT) {
        const int v = i / r.d, j = i % r.d;
        if (v0 + v >= n) continue;
        const double o = ys[v * r.pd + j] * norms[v0 + v];
        if (out) out[(v0 + v) * r.d + j] = o;
        if (residual) residual[(v0 + v) * r.d + j] = ldd(x, (v0 + v) * r.d + j) - o;
    }
}

struct Bounds {
    double b[255];
};

__global__ void k_nearest(const double *values, int64_t n, Bounds bd, int nb, int32_t *idx) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double v = values[i];
    int c = 0;
    for (int k = 0; k < nb; ++k) c += (bd.b[k] < v) ? 1 : 0;
    idx[i] = c;
}

// signs [n,d] int8 -> packed [n, ceil(d/8)], first element in the MSB.
__global__ void k_pack_bits(const int8_t *signs, int64_t n, int d, uint8_t *packed) {
    const int nbytes = (d + 7) / 8;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * nbytes) return;
    const int64_t row = i / nbytes;
    const int byte = (int)(i % nbytes);
    unsigned v = 0;
    for (int b = 0; b < 8; ++b) {
        const int j = byte * 8 + b;
        if (j < d && signs[row * d + j] > 0) v |= 0x80u >> b;
    }
    packed[i] = (uint8_t)v;
}

__global__ void k_unpack_bits(const uint8_t *packed, int64_t n, int d, int8_t *signs) {
    const int nbytes = (d + 7) / 8;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * d) return;
    const int64_t row = i / d;
    const int j = (int)(i % d);
    const unsigned bit = (packed[row * nbytes + j / 8] >> (7 - (j % 8))) & 1u;
    signs[i] = bit ? (int8_t)1 : (int8_t)-1;
}

// One MSB-first bit stream: bit t of the stream is bit (bits-1 - t%bits) of idx[t/bits].
__global__ void k_pack_indices(const uint8_t *idx, int64_t count, int bits, uint8_t *packed) {
    const int64_t nbytes = (count * bits + 7) / 8;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nbytes) return;
    unsigned v = 0;
    for (int b = 0; b < 8; ++b) {
        const int64_t t = i * 8 + b;
        const int64_t e = t / bits;
        if (e < count && ((idx[e] >> (bits - 1 - (int)(t % bits))) & 1u)) v |= 0x80u >> b;
    }
    packed[i] = (uint8_t)v;
}

inline size_t lds_bytes(int pd) { return (size_t)2 * vectors_per_workgroup(pd) * pd * sizeof(double); }

// Workgroups that stage more than 48 KB need the limit raised per kernel.
template <typename K> inline void allow_lds(K kernel, size_t bytes) {
    if (bytes > 48 * 1024)
        (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}
inline unsigned nblocks(int64_t n, int pd) {
    const int vb = vectors_per_workgroup(pd);
    return (unsigned)((n + vb - 1) / vb);
}
// F uses VB as a compile-time constant
#define DISPATCH_VB(pd, F)                                         \
    switch (vectors_per_workgroup(pd)) {                           \
    case 8: { constexpr int VB = 8; F; } break;                    \
    case 4: { constexpr int VB = 4; F; } break;                    \
    default: { constexpr int VB = 2; F; } break; }

RotArgs rot_args(const tq_handle *h, int transpose) {
    RotArgs r;
    r.d = h->d;
    r.pd = h->pd;
    r.mat = nullptr;
    r.sa = transpose ? h->s2_64 : h->s1_64;
    r.sb = transpose ? h->s1_64 : h->s2_64;
    return r;
}

// dense rotation: forward out[j] = sum_k Pi[j][k] in[k], i.e. M = Pi^T row-major
DenseArgs dense_args(const tq_handle *h, const double *mat, const void *in, int64_t n) {
    DenseArgs a = {};
    a.d = h->d;
    a.n = n;
    a.mat = mat;
    a.in = in;
    a.bits = h->bits;
    a.bounds = h->bounds64;
    a.centroids = h->centroids64;
    a.norm_correction = h->norm_correction;
    return a;
}
inline const double *rotation_matrix(const tq_handle *h, int transpose) { return transpose ? h->rot64 : h->rot64_t; }

// Outputs that lie in the input's memory: the column blocks of a product each read whole rows, so none may store before all
// have read.  Such calls take the kernels below, which stage a workgroup's rows in LDS before they store (one thread per
// output, the whole matrix per VB vectors: 2.8 times the time of k_dense64 for 32 768 vectors of 128).
RotArgs dense_rows_args(const tq_handle *h, int transpose) {
    RotArgs r = {};
    r.d = r.pd = h->d;
    r.mat = rotation_matrix(h, transpose);
    return r;
}
inline bool overlap(const void *a, int64_t a_bytes, const void *b, int64_t b_bytes) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return a && b && x < y + (uintptr_t)b_bytes && y < x + (uintptr_t)a_bytes;
}
inline int64_t size_of(int dtype) { return dtype == TQ_F16 ? 2 : dtype == TQ_F32 ? 4 : 8; }

#define DISPATCH_IN(dt, F)          \
    switch (dt) {                   \
    case TQ_F16: { using TI = __half; F; } break; \
    case TQ_F32: { using TI = float; F; } break;  \
    case TQ_F64: { using TI = double; F; } break; \
    default: tq_set_error("bad dtype %d", dt); return TQ_ERR_ARG; }

template <typename TI, typename TO>
int launch_rotate_to(const void *x, void *y, int64_t n, const RotArgs &r, hipStream_t s) {
    const size_t lds = lds_bytes(r.pd);
    DISPATCH_VB(r.pd, (allow_lds(k_rotate64<VB, TI, TO>, lds),
                       k_rotate64<VB, TI, TO><<<nblocks(n, r.pd), NT, lds, s>>>((const TI *)x, (TO *)y, n, r)));
    return tq_check_launch("rotate64");
}

template <typename TI>
int launch_rotate(const void *x, void *y, int64_t n, int out_dtype, const RotArgs &r, hipStream_t s) {
    switch (out_dtype) {
    case TQ_F16: return launch_rotate_to<TI, __half>(x, y, n, r, s);
    case TQ_F32: return launch_rotate_to<TI, float>(x, y, n, r, s);
    case TQ_F64: return launch_rotate_to<TI, double>(x, y, n, r, s);
    default: tq_set_error("bad dtype %d", out_dtype); return TQ_ERR_ARG;
    }
}

template <typename TI> int launch_rotate_dense(const DenseArgs &a, int out_dtype, hipStream_t s) {
    switch (out_dtype) {
    case TQ_F16: return launch_dense<DENSE_ROTATE, TI, __half>(a, "rotate64", s);
    case TQ_F32: return launch_dense<DENSE_ROTATE, TI, float>(a, "rotate64", s);
    case TQ_F64: return launch_dense<DENSE_ROTATE, TI, double>(a, "rotate64", s);
    default: tq_set_error("bad dtype %d", out_dtype); return TQ_ERR_ARG;
    }
}

}  // namespace

int tqk_fwht(const void *x, void *y, int64_t n, int len, int in_dtype, int out_dtype, hipStream_t s) {
    RotArgs r;
    r.d = r.pd = len;
    r.mat = r.sa = r.sb = nullptr;
    DISPATCH_IN(in_dtype, return launch_rotate<TI>(x, y, n, out_dtype, r, s));
}

int tqk_rotate64(const tq_handle *h, const void *x, void *y, int64_t n, int in_dtype, int out_dtype, int transpose,
                 hipStream_t s) {
    const int64_t count = n * h->d;
    const bool in_place = overlap(x, count * size_of(in_dtype), y, count * size_of(out_dtype));
    if (h->rotation == TQ_ROT_WHT || in_place) {
        const RotArgs r = h->rotation == TQ_ROT_WHT ? rot_args(h, transpose) : dense_rows_args(h, transpose);
        DISPATCH_IN(in_dtype, return launch_rotate<TI>(x, y, n, out_dtype, r, s));
    }
    DenseArgs a = dense_args(h, rotation_matrix(h, transpose), x, n);
    a.out = y;
    DISPATCH_IN(in_dtype, return launch_rotate_dense<TI>(a, out_dtype, s));
}

int tqk_nearest(const double *values, int64_t n, const double *bounds_host, int nb, int32_t *idx, hipStream_t s) {
    Bounds bd;
    for (int k = 0; k < nb; ++k) bd.b[k] = bounds_host[k];
    k_nearest<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(values, n, bd, nb, idx);
    return tq_check_launch("nearest");
}

template <typename TI>
static int quantize_from(const tq_handle *h, const void *x, int64_t n, uint8_t *idx, double *norms, double *rotated, hipStream_t s) {
    const int64_t count = n * h->d, bytes = count * (int64_t)sizeof(TI);
    const bool in_place = overlap(x, bytes, rotated, count * 8) || overlap(x, bytes, idx, count) || overlap(x, bytes, norms, n * 8);
    if (h->rotation == TQ_ROT_WHT || in_place) {
        const RotArgs r = h->rotation == TQ_ROT_WHT ? rot_args(h, 0) : dense_rows_args(h, 0);
        DISPATCH_VB(r.pd, (allow_lds(k_quantize64<VB, TI>, lds_bytes(r.pd)),
                           k_quantize64<VB, TI><<<nblocks(n, r.pd), NT, lds_bytes(r.pd), s>>>((const TI *)x, n, r, h->bounds64, h->bits,
                                                                                            idx, norms, rotated)));
        return tq_check_launch("quantize64");
    }
    DenseArgs a = dense_args(h, rotation_matrix(h, 0), x, n);
    a.out = idx;
    a.norms_out = norms;
    a.rotated = rotated;
    return launch_dense<DENSE_QUANTIZE, TI, uint8_t>(a, "quantize64", s);
}

int tqk_quantize_indices(const tq_handle *h, const void *x, int64_t n, int in_dtype, uint8_t *idx, double *norms,
                         double *rotated, hipStream_t s) {
    DISPATCH_IN(in_dtype, return quantize_from<TI>(h, x, n, idx, norms, rotated, s));
}

template <typename TX>
static int dequantize_to(const tq_handle *h, const uint8_t *idx, const double *norms, int64_t n, double *out, const void *x,
                         double *residual, hipStream_t s) {
    if (h->rotation == TQ_ROT_WHT) {
        const RotArgs r = rot_args(h, 1);
        DISPATCH_VB(r.pd, (allow_lds(k_dequantize64<VB, TX>, lds_bytes(r.pd)),
                           k_dequantize64<VB, TX><<<nblocks(n, r.pd), NT, lds_bytes(r.pd), s>>>(
                               idx, norms, n, r, h->centroids64, h->n_centroids, h->norm_correction, out, (const TX *)x, residual)));
        return tq_check_launch("dequantize64");
    }
    DenseArgs a = dense_args(h, rotation_matrix(h, 1), idx, n);
    a.norms_in = norms;
    a.out = out;
    a.x = x;
    a.residual = residual;
    return launch_dense<DENSE_DEQUANTIZE, uint8_t, TX>(a, "dequantize64", s);
}

int tqk_dequantize_indices(const tq_handle *h, const uint8_t *idx, const double *norms, int64_t n, double *out,
                           const void *x, int x_dtype, double *residual, hipStream_t s) {
    if (!residual) x_dtype = TQ_F64;
    DISPATCH_IN(x_dtype, return dequantize_to<TI>(h, idx, norms, n, out, x, residual, s));
}

// projections: out[j] = sum_k S[j][k] in[k] with M = S^T, and sum_k S[k][j] z[k] with M = S
int tqk_qjl_quantize(const tq_handle *h, const void *rr, int64_t n, int in_dtype, int8_t *signs, double *norms,
                     hipStream_t s) {
    DenseArgs a = dense_args(h, h->proj64_t, rr, n);
    a.out = signs;
    a.norms_out = norms;
    DISPATCH_IN(in_dtype, return (launch_dense<DENSE_QJL_QUANTIZE, TI, int8_t>(a, "qjl_quantize64", s)));
}

int tqk_qjl_dequantize(const tq_handle *h, const int8_t *signs, const double *norms, double shrinkage, int64_t n,
                       double *out, int accumulate, hipStream_t s) {
    DenseArgs a = dense_args(h, h->proj64, signs, n);
    a.norms_in = norms;
    a.out = out;
    a.proj_scale = h->proj_scale;
    a.shrinkage = shrinkage;
    a.accumulate = accumulate;
    return launch_dense<DENSE_QJL_DEQUANTIZE, int8_t, double>(a, "qjl_dequantize64", s);
}

int tqk_pack_bits(const int8_t *signs, int64_t n, int d, uint8_t *packed, hipStream_t s) {
    const int64_t total = n * ((d + 7) / 8);
    k_pack_bits<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(signs, n, d, packed);
    return tq_check_launch("pack_bits");
}

int tqk_unpack_bits(const uint8_t *packed, int64_t n, int d, int8_t *signs, hipStream_t s) {
    const int64_t total = n * d;
    k_unpack_bits<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(packed, n, d, signs);
    return tq_check_launch("unpack_bits");
}

int tqk_pack_indices(const uint8_t *idx, int64_t count, int bits, uint8_t *packed, hipStream_t s) {
    const int64_t nbytes = (count * bits + 7) / 8;
    k_pack_indices<<<(unsigned)((nbytes + 255) / 256), 256, 0, s>>>(idx, count, bits, packed);
    return tq_check_launch("pack_indices");
}
