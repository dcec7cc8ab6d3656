// Device kernels of the Llama decode executor around the paged attention
// path: weight dequantisation at load, RMSNorm, matrix-vector products,
// rotary embedding and the SwiGLU gate (core/include/tvara/model.hpp:47-126,
// core/include/tvara/quant.hpp:14-71,178-184).
//
// Rounding follows the reference's: products and sums the reference rounds to
// float one at a time are written with __fmul_rn / __fsub_rn / __fadd_rn so
// the compiler does not contract them into FMAs; dot products and the RMS sum
// accumulate in double and round once, as quant::dot_f32 and rms_norm do.
#include <algorithm>

#include "model.hpp"
#include "q8.hpp"
#include "q8_pipe.hpp"
#include "device_util.hpp"

namespace tvara_amd {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ void flag_bad(int* bad, float v) {
    if (!__builtin_isfinite(v)) atomicOr(bad, 1);
}

// ------------------------------------------------------------ dequantisation

__global__ void check_f32_kernel(const float* w, size_t n, int* bad) {
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x)
        flag_bad(bad, w[i]);
}

__global__ void f16_kernel(const uint8_t* raw, size_t n, float* out, int* bad) {
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const uint16_t h = static_cast<uint16_t>(raw[2 * i] | (raw[2 * i + 1] << 8));
        const float v = half_bits_to_float(h);
        out[i] = v;
        flag_bad(bad, v);
    }
}

// Q8_0: 34-byte groups, x = d * q (quant.hpp:39-49)
__global__ void q8_0_kernel(const uint8_t* raw, size_t n, float* out, int* bad) {
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const uint8_t* g = raw + (i / 32) * 34;
        const float d = half_bits_to_float(static_cast<uint16_t>(g[0] | (g[1] << 8)));
        const float v = __fmul_rn(d, static_cast<float>(static_cast<int8_t>(g[2 + i % 32])));
        out[i] = v;
        flag_bad(bad, v);
    }
}

// Q4_0: 18-byte groups; byte j holds elements j (low nibble) and j+16 (high),
// x = d * (q - 8) (quant.hpp:50-60)
__global__ void q4_0_kernel(const uint8_t* raw, size_t n, float* out, int* bad) {
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const uint8_t* g = raw + (i / 32) * 18;
        const int e = static_cast<int>(i % 32);
        const float d = half_bits_to_float(static_cast<uint16_t>(g[0] | (g[1] << 8)));
        const unsigned q = e < 16 ? (g[2 + e] & 15u) : (g[2 + e - 16] >> 4);
        const float v = __fmul_rn(d, static_cast<float>(static_cast<int>(q) - 8));
        out[i] = v;
        flag_bad(bad, v);
    }
}

// Q4_K: 144-byte super-blocks of 256: fp16 d, fp16 dmin, 12 bytes of 6-bit
// (scale, min) pairs for eight groups of 32, then 128 bytes of nibbles
// (group g reads byte 16 + (g/2)*32 + i, high nibble for odd g);
// x = d*scale*q - dmin*min (quant.hpp:62-85)
__global__ void q4_k_kernel(const uint8_t* raw, size_t n, float* out, int* bad) {
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const uint8_t* b = raw + (i / 256) * 144;
        const int e = static_cast<int>(i % 256), g = e / 32, k = e % 32;
        const float d = half_bits_to_float(static_cast<uint16_t>(b[0] | (b[1] << 8)));
        const float dmin = half_bits_to_float(static_cast<uint16_t>(b[2] | (b[3] << 8)));
        const uint8_t* s = b + 4;
        unsigned sc, mn;
        if (g < 4) {
            sc = s[g] & 63u;
            mn = s[g + 4] & 63u;
        } else {
            sc = (s[g + 4] & 15u) | ((s[g - 4] >> 6) << 4);
            mn = (s[g + 4] >> 4) | ((s[g] >> 6) << 4);
        }
        const unsigned packed = b[16 + (g / 2) * 32 + k];
        const unsigned q = (g & 1) ? (packed >> 4) : (packed & 15u);
        const float v = __fsub_rn(__fmul_rn(__fmul_rn(d, static_cast<float>(sc)), static_cast<float>(q)),
                                  __fmul_rn(dmin, static_cast<float>(mn)));
        out[i] = v;
        flag_bad(bad, v);
    }
}

// ------------------------------------------------------------------- RMSNorm

// out = x * float(1/sqrt(sum(x^2)/n + eps)) * w, the sum in double
// (model.hpp:54-61); one workgroup
__global__ __launch_bounds__(1024) void rmsnorm_kernel(const float* x, const float* w, float* out, int n, float eps) {
    __shared__ double part[1024 / 64];
    __shared__ float inv;
    x += static_cast<size_t>(blockIdx.x) * n;  // one workgroup per row of a batch
    out += static_cast<size_t>(blockIdx.x) * n;
    double sum = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) sum += static_cast<double>(x[i]) * x[i];
    for (int o = 32; o >= 1; o >>= 1) sum += __shfl_xor(sum, o);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int k = 0; k < static_cast<int>(blockDim.x >> 6); ++k) t += part[k];
        inv = static_cast<float>(1.0 / sqrt(t / static_cast<double>(n) + static_cast<double>(eps)));
    }
    __syncthreads();
    const float iv = inv;
    for (int i = threadIdx.x; i < n; i += blockDim.x) out[i] = __fmul_rn(__fmul_rn(x[i], iv), w[i]);
}

// ------------------------------------------------------------- matvec

// y = W v for row-major W [rows][cols]: one wave per row, double accumulation
// rounded once (quant::dot_f32); output rows are cut into up to three
// segments, each written to its own buffer, optionally as residual + y (the
// reference's x[j] += residual[j]).
struct MatvecArgs {
    const float* w;
    const float* v;
    int rows, cols;
    MatvecSegment seg[3];
    int nseg;
};

template <bool VEC>
__global__ __launch_bounds__(kThreads) void matvec_kernel(const MatvecArgs a) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
    if (row >= a.rows) return;
    const float* wr = a.w + static_cast<size_t>(row) * a.cols;
    double acc = 0;
    if constexpr (VEC) {
        const int c4 = a.cols / 4;
        for (int k = lane; k < c4; k += 64) {
            const float4 w4 = reinterpret_cast<const float4*>(wr)[k];
            const float4 v4 = reinterpret_cast<const float4*>(a.v)[k];
            acc = fma(static_cast<double>(w4.x), static_cast<double>(v4.x), acc);
            acc = fma(static_cast<double>(w4.y), static_cast<double>(v4.y), acc);
            acc = fma(static_cast<double>(w4.z), static_cast<double>(v4.z), acc);
            acc = fma(static_cast<double>(w4.w), static_cast<double>(v4.w), acc);
        }
    } else {
        for (int k = lane; k < a.cols; k += 64) acc = fma(static_cast<double>(wr[k]), static_cast<double>(a.v[k]), acc);
    }
    for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane) return;
    int r = row, s = 0;
    while (s + 1 < a.nseg && r >= a.seg[s].rows) r -= a.seg[s++].rows;
    const float y = static_cast<float>(acc);
    float* out = a.seg[s].out;
    out[r] = a.seg[s].residual ? __fadd_rn(a.seg[s].residual[r], y) : y;
}

// Y[j] = W X[j] for a batch of vectors (one per sequence), as a skinny GEMM:
// a workgroup owns 64 rows of W and up to 64 vectors; K advances in chunks
// of 32 columns staged in LDS (W tile [64][32], X tile [64][32], double
// buffered), and each thread accumulates a 4-row x 4-vector micro-tile in
// f32.  Every weight is read from HBM once per launch; the X tile comes from
// L2.
constexpr int kTileRows = 64, kTileVecs = 64, kTileK = 32;

struct BatchMatvecArgs {
    const float* w;
    const float* x;  // [n][cols]
    int rows, cols, n;
    MatvecSegment seg[3];  // output j of segment s: seg.out[j * seg.rows + r]
    int nseg;
    int chunks_per_split;  // K chunks of kTileK per blockIdx.y
    float* partial;        // split-K: [gridDim.y][n_total][rows] partial sums, else null
    int n_total, j0;       // partial layout: vector stride and this launch's first vector
};

__global__ __launch_bounds__(256) void batch_matvec_kernel(const BatchMatvecArgs a) {
    __shared__ float ws[2][kTileRows][kTileK + 4];
    __shared__ float xs[2][kTileVecs][kTileK + 4];
    const int t = threadIdx.x;
    const int row0 = blockIdx.x * kTileRows;
    // staging map: thread t copies float4 (t % 8) of rows t/8 and t/8 + 32
    const int sc = (t % 8) * 4, sr = t / 8;
    // micro-tile: rows 4*(t%16) .. +3, vectors 4*(t/16) .. +3
    const int mr = (t % 16) * 4, mv = (t / 16) * 4;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
    auto stage = [&](int buf, int k0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = sr + 32 * h;
            float4 w = make_float4(0.f, 0.f, 0.f, 0.f), x = w;
            if (row0 + r < a.rows) w = *reinterpret_cast<const float4*>(a.w + static_cast<size_t>(row0 + r) * a.cols + k0 + sc);
            if (r < a.n) x = *reinterpret_cast<const float4*>(a.x + static_cast<size_t>(r) * a.cols + k0 + sc);
            *reinterpret_cast<float4*>(&ws[buf][r][sc]) = w;
            *reinterpret_cast<float4*>(&xs[buf][r][sc]) = x;
        }
    };
    const int kbeg = blockIdx.y * a.chunks_per_split;
    const int nk = min(a.cols / kTileK - kbeg, a.chunks_per_split);
    stage(0, kbeg * kTileK);
    __syncthreads();
    for (int kc = 0; kc < nk; ++kc) {
        const int buf = kc & 1;
        if (kc + 1 < nk) stage(buf ^ 1, (kbeg + kc + 1) * kTileK);
#pragma unroll
        for (int k = 0; k < kTileK; k += 4) {
            float4 w4[4], x4[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) w4[i] = *reinterpret_cast<const float4*>(&ws[buf][mr + i][k]);
#pragma unroll
            for (int j = 0; j < 4; ++j) x4[j] = *reinterpret_cast<const float4*>(&xs[buf][mv + j][k]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc[i][j] = fmaf(w4[i].x, x4[j].x, acc[i][j]);
                    acc[i][j] = fmaf(w4[i].y, x4[j].y, acc[i][j]);
                    acc[i][j] = fmaf(w4[i].z, x4[j].z, acc[i][j]);
                    acc[i][j] = fmaf(w4[i].w, x4[j].w, acc[i][j]);
                }
        }
        __syncthreads();
    }
    if (a.partial) {  // split-K: the fixed-order sum happens afterwards
        float* p = a.partial + static_cast<size_t>(blockIdx.y) * a.n_total * a.rows;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (row0 + mr + i < a.rows && mv + j < a.n)
                    p[static_cast<size_t>(a.j0 + mv + j) * a.rows + row0 + mr + i] = acc[i][j];
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = row0 + mr + i;
        if (row >= a.rows) break;
        int rr = row, sg = 0;
        while (sg + 1 < a.nseg && rr >= a.seg[sg].rows) rr -= a.seg[sg++].rows;
        const MatvecSegment& S = a.seg[sg];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (mv + j >= a.n) break;
            const size_t at = static_cast<size_t>(mv + j) * S.rows + rr;
            S.out[at] = S.residual ? __fadd_rn(S.residual[at], acc[i][j]) : acc[i][j];
        }
    }
}

// y[j][r] = sum over splits s (in order) of partial[s][j][r], to the segments
__global__ void split_sum_kernel(const BatchMatvecArgs a, int splits) {
    const size_t total = static_cast<size_t>(a.n) * a.rows;
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < total;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        float sum = 0.f;
        for (int sp = 0; sp < splits; ++sp) sum += a.partial[static_cast<size_t>(sp) * total + i];
        const int j = static_cast<int>(i / a.rows);
        int rr = static_cast<int>(i % a.rows), sg = 0;
        while (sg + 1 < a.nseg && rr >= a.seg[sg].rows) rr -= a.seg[sg++].rows;
        const MatvecSegment& S = a.seg[sg];
        const size_t at = static_cast<size_t>(j) * S.rows + rr;
        S.out[at] = S.residual ? __fadd_rn(S.residual[at], sum) : sum;
    }
}

// out[j] = table[idx[j]] (embedding rows of a batch)
__global__ void gather_embedding_kernel(const float* table, const uint32_t* idx, int n, int h, float* out) {
    const size_t total = static_cast<size_t>(n) * h;
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < total;
         i += static_cast<size_t>(gridDim.x) * blockDim.x)
        out[i] = table[static_cast<size_t>(idx[i / h]) * h + i % h];
}

// [layers][n][kv] -> [n][layers][kv] (one token row per sequence for the append)
__global__ void interleave_layers_kernel(const float* src, float* dst, int layers, int n, int kv) {
    const size_t total = static_cast<size_t>(layers) * n * kv;
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < total;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const size_t e = i % kv, j = (i / kv) % n, l = i / (static_cast<size_t>(kv) * n);
        dst[(j * layers + l) * kv + e] = src[i];
    }
}

// ------------------------------------------------------------- RoPE

// rotate pair i of every head of q and k by the (cos, sin) of this position
// (model.hpp:63-72): interleaved pairs (2i, 2i+1) or split (i, i+dim/2)
__global__ void rope_kernel(float* q, int qheads, float* k, int kheads, int dim, const float* cs, int interleaved) {
    const int half = dim / 2;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (qheads + kheads) * half) return;
    // row blockIdx.y of a batch: its own position's (cos, sin)
    q += static_cast<size_t>(blockIdx.y) * qheads * dim;
    k += static_cast<size_t>(blockIdx.y) * kheads * dim;
    cs += static_cast<size_t>(blockIdx.y) * dim;
    const int h = t / half, i = t % half;
    float* x = h < qheads ? q + static_cast<size_t>(h) * dim : k + static_cast<size_t>(h - qheads) * dim;
    const int ia = interleaved ? 2 * i : i, ib = interleaved ? 2 * i + 1 : i + half;
    const float c = cs[2 * i], s = cs[2 * i + 1];
    const float left = x[ia], right = x[ib];
    x[ia] = __fsub_rn(__fmul_rn(left, c), __fmul_rn(right, s));
    x[ib] = __fadd_rn(__fmul_rn(right, c), __fmul_rn(left, s));
}

// ------------------------------------------------------------- SwiGLU

// gate = gate * (sigmoid(gate) * up), the sigmoid in the overflow-free form
// of model.hpp:111-116
__global__ void swiglu_kernel(float* gate, const float* up, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = gate[i];
    const float small = expf(-fabsf(g));
    const float one = __fadd_rn(1.f, small);
    const float sig = g >= 0 ? __fdiv_rn(1.f, one) : __fdiv_rn(small, one);
    gate[i] = __fmul_rn(g, __fmul_rn(sig, up[i]));
}

// ------------------------------------------------------------- Q8_0 weights

// one thread per (row, group): the 34-byte GGUF group to its tile slots
__global__ void q8_repack_kernel(const uint8_t* raw, int rows, int groups, int row0, int stride, uint8_t* q,
                                 uint16_t* d, int* bad) {
    const int pairs = (groups + 1) / 2;
    const size_t total = static_cast<size_t>(rows) * groups;
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < total;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const int r = static_cast<int>(i / groups), g = static_cast<int>(i % groups);
        const uint8_t* src = raw + i * 34;
        const int row = row0 + r * stride, rr = row % 16;
        const size_t block = static_cast<size_t>(row / 16) * pairs + g / 2;
        const uint16_t h = static_cast<uint16_t>(src[0] | (src[1] << 8));
        d[(block * 16 + rr) * 2 + g % 2] = h;
        if (!__builtin_isfinite(half_bits_to_float(h))) atomicOr(bad, 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint8_t* dst = q + (block * 64 + rr + 16 * j) * 16 + (g % 2) * 8;
#pragma unroll
            for (int b = 0; b < 8; ++b) dst[b] = src[2 + 8 * j + b];
        }
    }
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct Q8MatvecArgs {
    const uint4* q;
    const uint32_t* d;  // the two groups' fp16 scales of a row, per (tile, pair)
    const float* v;     // the input, or x when norm_w is set
    const float* norm_w;  // RMSNorm weight: the input is rms_norm(x) * norm_w
    float eps;
    int rows, tiles, groups, pairs, cols;
    MatvecSegment seg[3];
    int nseg;
    // epilogue on adjacent row pairs (2i, 2i+1): rotate the first rope_rows
    // rows by rope_cs (interleaved RoPE over rope_dim-wide heads), or, with
    // swiglu, write gate * (sigmoid(gate) * up) of rows (gate i, up i) to
    // seg[0].out[i]
    const float* rope_cs;
    int rope_dim, rope_rows;
    int swiglu;
};

// sum of 8 int8 (two dwords) times 8 floats, in f32
__device__ __forceinline__ float dot8(uint32_t lo, uint32_t hi, float4 a, float4 b) {
    float s = sbyte_to_float<0>(lo) * a.x;
    s = fmaf(sbyte_to_float<1>(lo), a.y, s);
    s = fmaf(sbyte_to_float<2>(lo), a.z, s);
    s = fmaf(sbyte_to_float<3>(lo), a.w, s);
    s = fmaf(sbyte_to_float<0>(hi), b.x, s);
    s = fmaf(sbyte_to_float<1>(hi), b.y, s);
    s = fmaf(sbyte_to_float<2>(hi), b.z, s);
    return fmaf(sbyte_to_float<3>(hi), b.w, s);
}

__device__ __forceinline__ void write_segment(const MatvecSegment* seg, int nseg, int row, size_t col_offset_rows,
                                              float y) {
    int r = row, s = 0;
    while (s + 1 < nseg && r >= seg[s].rows) r -= seg[s++].rows;
    const size_t at = col_offset_rows * seg[s].rows + r;
    seg[s].out[at] = seg[s].residual ? __fadd_rn(seg[s].residual[at], y) : y;
}

// y = W v over Q8_0 tiles: a workgroup per RT 16-row tiles, its W waves
// taking contiguous shares of the group pairs, U pairs a step with every
// load issued first (16 bytes of weights per lane per tile and pair).  The
// input vector is staged in LDS first -- normalised there when the product
// follows an RMSNorm (model.hpp:54-61: sum of squares in double, the scale
// rounded to float, (x * s) * w), which each workgroup computes for itself.
// Lane l accumulates row l%16 of each tile over its eight columns of each
// group: the eight products in f32, times the group's d, added in double;
// lanes and waves are then summed in double and each row rounds to float
// once.  Pairs past the share, and the zero group that completes an odd
// count, are selected away rather than multiplied (their loads stay in
// bounds).
template <int W, int RT, bool kStream>
__global__ __launch_bounds__(W * 64) void matvec_q8_kernel(const Q8MatvecArgs a) {
    constexpr int U = 2;
    extern __shared__ float vs[];  // cols floats
    __shared__ double red[W][RT][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int P = a.pairs, G = a.groups, C = a.cols;
    const int per = (P + W - 1) / W;
    const int p0 = min(P, wave * per), p1 = min(P, p0 + per);
    int tl[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) tl[r] = min(static_cast<int>(blockIdx.x) * RT + r, a.tiles - 1);
    // U pairs of every tile from pair p on, clamped to the wave's last pair
    // (a wave without pairs reads pair P - 1 and adds nothing).  The weights
    // are read once a token.  Those of a model that outgrows the 256 MB
    // memory-side cache pass through the caches non-temporally, or each layer's
    // 65 MB would evict the next kernels' code and inputs (Llama-3.2-1B, one
    // token: the layers' attention kernel 13.2 -> 10.7 us, the call 850 ->
    // 799; their scales, half a line a read, stay cached: streamed too, the
    // gate|up product takes 12.3 against 11.9 us).  A smaller model's are still
    // there at the next token and stay.  Kernel time a token, kept against
    // streamed: SmolLM2-135M's shape, 143 MB, 747 against 800 us; three layers of
    // TinyLlama's, 200 MB, 119 against 125; six, 335 MB, 239 against 235.
    auto load = [&](int p, uint4 (&qq)[RT][U], uint32_t (&dd)[RT][U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int pc = min(p + u, p1 - 1);
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const size_t blk = static_cast<size_t>(tl[r]) * P + pc;
                const u32x4* at = reinterpret_cast<const u32x4*>(a.q) + blk * 64 + lane;
                qq[r][u] = __builtin_bit_cast(uint4, kStream ? __builtin_nontemporal_load(at) : *at);
                dd[r][u] = a.d[blk * 16 + (lane & 15)];
            }
        }
    };
    // the first step's weights are requested before the input is staged
    uint4 qq[RT][U];
    uint32_t dd[RT][U];
    load(p0, qq, dd);
    if (a.norm_w) {
        // one pass over the input and the norm weights, both staged in LDS as
        // float4s (two per thread a step, all four loads requested first);
        // each thread then rescales the elements it staged
        float* ws = vs + C;
        constexpr int S = 4 * W * 64;
        double sq = 0;
        for (int k0 = 4 * static_cast<int>(threadIdx.x); k0 < C; k0 += 2 * S) {
            const int k1 = min(k0 + S, C - 4);
            const float4 x0 = *reinterpret_cast<const float4*>(a.v + k0);
            const float4 w0 = *reinterpret_cast<const float4*>(a.norm_w + k0);
            const float4 x1 = *reinterpret_cast<const float4*>(a.v + k1);
            const float4 w1 = *reinterpret_cast<const float4*>(a.norm_w + k1);
            sq += static_cast<double>(x0.x) * x0.x + static_cast<double>(x0.y) * x0.y +
                  static_cast<double>(x0.z) * x0.z + static_cast<double>(x0.w) * x0.w;
            *reinterpret_cast<float4*>(vs + k0) = x0;
            *reinterpret_cast<float4*>(ws + k0) = w0;
            if (k0 + S < C) {
                sq += static_cast<double>(x1.x) * x1.x + static_cast<double>(x1.y) * x1.y +
                      static_cast<double>(x1.z) * x1.z + static_cast<double>(x1.w) * x1.w;
                *reinterpret_cast<float4*>(vs + k1) = x1;
                *reinterpret_cast<float4*>(ws + k1) = w1;
            }
        }
        for (int o = 32; o >= 1; o >>= 1) sq += __shfl_xor(sq, o);
        if (lane == 0) red[wave][0][0] = sq;
        __syncthreads();
        double t = 0;
        for (int w = 0; w < W; ++w) t += red[w][0][0];
        const float inv = static_cast<float>(1.0 / sqrt(t / static_cast<double>(C) + static_cast<double>(a.eps)));
        for (int k = 4 * static_cast<int>(threadIdx.x); k < C; k += S) {
            float4 x = *reinterpret_cast<const float4*>(vs + k);
            const float4 w = *reinterpret_cast<const float4*>(ws + k);
            x.x = __fmul_rn(__fmul_rn(x.x, inv), w.x);
            x.y = __fmul_rn(__fmul_rn(x.y, inv), w.y);
            x.z = __fmul_rn(__fmul_rn(x.z, inv), w.z);
            x.w = __fmul_rn(__fmul_rn(x.w, inv), w.w);
            *reinterpret_cast<float4*>(vs + k) = x;
        }
        __syncthreads();  // red is reused below
    } else {
        for (int k = 4 * threadIdx.x; k < C; k += 4 * W * 64)
            *reinterpret_cast<float4*>(vs + k) = *reinterpret_cast<const float4*>(a.v + k);
    }
    __syncthreads();
    const float* vp = vs + 8 * (lane >> 4);
    double acc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r] = 0;
    for (int p = p0; p < p1; p += U) {
        // the next step's weights are in flight while this step is summed
        // (unconditional, clamped: the last step re-reads its own pairs)
        uint4 nq[RT][U];
        uint32_t nd[RT][U];
        load(min(p + U, p1 - 1), nq, nd);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int pc = min(p + u, p1 - 1);
            const bool live = p + u < p1, second = 2 * pc + 1 < G;
            const int c0 = 64 * pc, c1 = second ? c0 + 32 : c0;
            const float4 v0 = *reinterpret_cast<const float4*>(vp + c0);
            const float4 v1 = *reinterpret_cast<const float4*>(vp + c0 + 4);
            const float4 v2 = *reinterpret_cast<const float4*>(vp + c1);
            const float4 v3 = *reinterpret_cast<const float4*>(vp + c1 + 4);
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const double s0 = static_cast<double>(half_bits_to_float(static_cast<uint16_t>(dd[r][u] & 0xffff))) *
                                  dot8(qq[r][u].x, qq[r][u].y, v0, v1);
                const double s1 = static_cast<double>(half_bits_to_float(static_cast<uint16_t>(dd[r][u] >> 16))) *
                                  dot8(qq[r][u].z, qq[r][u].w, v2, v3);
                const double t = second ? s0 + s1 : s0;
                acc[r] += live ? t : 0.0;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                qq[r][u] = nq[r][u];
                dd[r][u] = nd[r][u];
            }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        acc[r] += __shfl_xor(acc[r], 16);
        acc[r] += __shfl_xor(acc[r], 32);
        if (lane < 16) red[wave][r][lane] = acc[r];
    }
    __syncthreads();
    if (wave || lane >= 16) return;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        double t = red[0][r][lane];
#pragma unroll
        for (int w = 1; w < W; ++w) t += red[w][r][lane];
        const int tile = static_cast<int>(blockIdx.x) * RT + r, row = tile * 16 + lane;
        float y = static_cast<float>(t);
        const float other = __shfl_xor(y, 1);  // the row-pair partner (lanes 0..15 all take part)
        if (a.swiglu) {
            // model.hpp:111-116, with the overflow-free sigmoid
            if (!(lane & 1) && tile < a.tiles && row + 1 < a.rows) {
                const float small = expf(-fabsf(y));
                const float one = __fadd_rn(1.f, small);
                const float sig = y >= 0 ? __fdiv_rn(1.f, one) : __fdiv_rn(small, one);
                a.seg[0].out[row / 2] = __fmul_rn(y, __fmul_rn(sig, other));
            }
            continue;
        }
        if (a.rope_cs && row < a.rope_rows) {  // model.hpp:63-72
            const int i = (row % a.rope_dim) / 2;
            const float c = a.rope_cs[2 * i], sn = a.rope_cs[2 * i + 1];
            y = lane & 1 ? __fadd_rn(__fmul_rn(y, c), __fmul_rn(other, sn))
                         : __fsub_rn(__fmul_rn(y, c), __fmul_rn(other, sn));
        }
        if (tile < a.tiles && row < a.rows) write_segment(a.seg, a.nseg, row, 0, y);
    }
}

// The batched product runs on fp16 MFMAs.  int8 weights are exact in fp16;
// each activation vector is scaled by a power of two (max |x| into
// [2^13, 2^14), exact) and split as x = hi + lo with hi = fp16(x) and
// lo = fp16(x - hi), which keeps 22 of its 24 bits.  One 16x16x32 MFMA then
// covers exactly one Q8_0 group: C = A*Bhi + A*Blo in f32, and the
// accumulator takes d * C.  A lane l of a product reads 16 bytes, columns
// 8(l/16) .. +7 of vector l%16 of a tile.  Two orders:
//  by lane, where the chunked kernel reads them straight into registers:
//    halves[((vt*groups + k/32)*2 + part)*64 + lane][k%8], part 0 = hi, 1 = lo
//    (in the other order its reads touch sixteen lines an instruction: 10.6
//    against 15.9 us for 64 vectors of the 2,048-column products);
//  by line, where the tiled GEMM stages them: a vector's halves of a group are
//    128 contiguous bytes, halves[((vt*groups + k/32)*16 + j%16)*2 + part][k%32],
//    so that an epilogue, a workgroup per vector, writes whole lines (by lane
//    every line is written in pieces by eight workgroups: the SwiGLU of 2,048
//    vectors of 8,192 takes 87 us against 49, the norms 24 against 16).
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));

// Elements k0 .. k0 + 7 of vector j (k0 % 8 == 0, already scaled): one
// 16-byte store each for the hi and the lo halves
template <bool kByLine>
__device__ __forceinline__ void put_halves8(_Float16* halves, int groups, int j, int k0, const float (&v)[8]) {
    half8 hi, lo;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        hi[i] = static_cast<_Float16>(v[i]);
        lo[i] = static_cast<_Float16>(v[i] - static_cast<float>(hi[i]));
    }
    const size_t block = (static_cast<size_t>(j / 16) * groups + k0 / 32) * 1024;  // of a vector tile and group
    const size_t at = block + (kByLine ? (j % 16) * 64 + k0 % 32 : ((j % 16) + 16 * ((k0 % 32) / 8)) * 8);
    *reinterpret_cast<half8*>(halves + at) = hi;
    *reinterpret_cast<half8*>(halves + at + (kByLine ? 32 : 512)) = lo;
}

__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

__device__ __forceinline__ void store8(float* p, const float (&v)[8]) {
    reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
}

// the power of two that brings max |x| into [2^13, 2^14) (1 for 0 or a
// non-finite maximum, which then propagates)
__device__ __forceinline__ int halves_shift(float m) {
    int e = 0;
    if (m > 0.f && __builtin_isfinite(m)) {
        frexpf(m, &e);
        return 14 - e;
    }
    return 0;
}

// max over the workgroup (every thread gets it); scratch holds a float per wave
__device__ __forceinline__ float block_max(float m, float* scratch) {
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = m;
    __syncthreads();
    float r = scratch[0];
    for (int w = 1; w < static_cast<int>(blockDim.x >> 6); ++w) r = fmaxf(r, scratch[w]);
    return r;
}

// The per-vector epilogues run a workgroup per vector; a thread takes
// eight consecutive elements a chunk (float4 loads, 16-byte halves stores),
// at most kEpiChunks chunks: rows of up to 16,384 at 1,024 threads.
constexpr int kEpiChunks = 2;

// threads for a row of h elements: one chunk each up to 1,024 threads
inline int epi_threads(int h) { return std::min(1024, std::max(64, ((h / 8 + 63) / 64) * 64)); }

// halves of vector j = blockIdx.x (a row of cols floats)
template <bool kByLine>
__global__ __launch_bounds__(1024) void split_halves_kernel(const float* x, int cols, int groups, _Float16* halves,
                                                             float* unscale) {
    __shared__ float part[16];
    const int j = blockIdx.x, T = blockDim.x;
    const float* xr = x + static_cast<size_t>(j) * cols;
    float v[kEpiChunks][8];
    float m = 0.f;
#pragma unroll
    for (int c = 0; c < kEpiChunks; ++c) {
        const int e0 = 8 * (static_cast<int>(threadIdx.x) + T * c);
        if (e0 < cols) {
            load8(xr + e0, v[c]);
#pragma unroll
            for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(v[c][i]));
        }
    }
    const int shift = halves_shift(block_max(m, part));
    const float up = ldexpf(1.f, shift);
    if (threadIdx.x == 0) unscale[j] = ldexpf(1.f, -shift);
#pragma unroll
    for (int c = 0; c < kEpiChunks; ++c) {
        const int e0 = 8 * (static_cast<int>(threadIdx.x) + T * c);
        if (e0 < cols) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[c][i] *= up;
            put_halves8<kByLine>(halves, groups, j, e0, v[c]);
        }
    }
}

// eight int8 (two dwords) to eight fp16: each byte b, offset by 128, becomes
// the fp16 1024 + (b ^ 0x80) (0x64 above the byte), from which 1152 is
// subtracted exactly
__device__ __forceinline__ half8 i8x8_to_half8(uint2 q) {
    const uint32_t x = q.x ^ 0x80808080u, y = q.y ^ 0x80808080u;
    const uint32_t w[4] = {__builtin_amdgcn_perm(0x64646464u, x, 0x04010400u),
                           __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u),
                           __builtin_amdgcn_perm(0x64646464u, y, 0x04010400u),
                           __builtin_amdgcn_perm(0x64646464u, y, 0x04030402u)};
    const half2v bias = {static_cast<_Float16>(1152.f), static_cast<_Float16>(1152.f)};
    half8 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const half2v h = __builtin_bit_cast(half2v, w[i]) - bias;
        r[2 * i] = h[0];
        r[2 * i + 1] = h[1];
    }
    return r;
}

struct Q8BatchArgs {
    const uint4* q;
    const uint16_t* d;
    const uint4* halves;  // 8 fp16 per lane, see put_halves8
    const float* unscale;
    int rows, tiles, groups, pairs;  // tiles: one past the last row tile of this launch
    int tile0;                       // its first row tile (blockIdx.x counts from it)
    int n;              // vectors
    int n_total_tiles;  // vector tiles the halves hold
    int groups_per_split;
    float* out;  // [gridDim.y][n][rows]
};

// A workgroup of NT waves covers RT row tiles (RT x 16 rows) over a share of
// the groups; wave w owns vector tile w (16 vectors).  The operands are taken as
// C^T = X W^T: A = the wave's fp16 activation halves (registers, straight
// from global memory), B = the row tiles' int8 weights, converted to fp16 once
// per workgroup and shared through LDS, so lane l accumulates weight row l%16
// of each tile for vectors 4(l/16) + i and needs one scale per tile and
// group.  K advances in chunks of two group pairs: the int8 tiles and scales
// of chunk c + 2 are requested while chunk c is multiplied (two register
// sets), staged into the other LDS buffer after it (one barrier per chunk);
// the activations of chunk c + 1 are requested after chunk c's barrier.
// Prefetches are unconditional (clamped to the last chunk) so that the
// compiler keeps them ahead of the arithmetic.
//
// Every operand is read through a buffer descriptor: a thread keeps a fixed
// byte offset per load slot and a chunk adds one scalar offset, so the loads
// cost no vector address arithmetic.  The weight and scale views cover this
// workgroup's row tiles only and the activation view this wave's vector
// tile; reads past a view return zero.  The groups past the split's end (a
// last chunk of fewer than four) read their activations past the view, so
// they multiply zeros and add exactly nothing.
constexpr int kBufferWord3 = 0x00020000;  // gfx9 buffer descriptor, dword 3

__device__ __forceinline__ __amdgpu_buffer_rsrc_t view(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), kBufferWord3);
}

template <int NT, int RT>
__global__ __launch_bounds__(256) void batch_q8_kernel(const Q8BatchArgs a) {
    constexpr int P = 2, CG = 2 * P;                 // pairs and groups per chunk
    constexpr int NTH = 64 * NT;
    constexpr int RAW = RT * P * 64;                 // uint4 of int8 per chunk
    constexpr int WPT = (RAW + NTH - 1) / NTH;       // per thread
    constexpr int DW = RT * P * 16;                  // scale dwords per chunk (16 rows x 2 groups each)
    constexpr int DPT = (DW + NTH - 1) / NTH;        // per thread
    __shared__ half8 ws[2][CG][RT][64];
    __shared__ uint32_t wd[2][RT][P][16];
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gbeg = static_cast<int>(blockIdx.y) * a.groups_per_split;
    const int gend = min(a.groups, gbeg + a.groups_per_split);
    const int pbeg = gbeg / 2;
    const int nchunks = (gend - gbeg + CG - 1) / CG;
    const int t0 = a.tile0 + static_cast<int>(blockIdx.x) * RT;
    const int tiles_here = min(RT, a.tiles - t0);
    const __amdgpu_buffer_rsrc_t qv =
        view(a.q + static_cast<size_t>(t0) * a.pairs * 64, static_cast<uint32_t>(tiles_here * a.pairs) * 1024u);
    const __amdgpu_buffer_rsrc_t dv = view(reinterpret_cast<const uint32_t*>(a.d) + static_cast<size_t>(t0) * a.pairs * 16,
                                           static_cast<uint32_t>(tiles_here * a.pairs) * 64u);
    const uint32_t xbytes = static_cast<uint32_t>(a.groups) * 2048u;
    const int vt = min(static_cast<int>(blockIdx.z) * NT + wave, a.n_total_tiles - 1);  // (past the batch: not stored)
    const __amdgpu_buffer_rsrc_t xv = view(a.halves + static_cast<size_t>(vt) * a.groups * 2 * 64, xbytes);
    // byte offsets of this thread's load slots within a chunk
    uint32_t qoff[WPT], doff[DPT];
#pragma unroll
    for (int i = 0; i < WPT; ++i) {
        const int e = min(tid + NTH * i, RAW - 1);
        const int r = (e >> 6) / P, p = (e >> 6) % P;
        qoff[i] = static_cast<uint32_t>(((r * a.pairs + p) * 64 + (e & 63)) * 16);
    }
#pragma unroll
    for (int i = 0; i < DPT; ++i) {
        const int e = min(tid + NTH * i, DW - 1);
        const int r = e / (P * 16), p = (e / 16) % P;
        doff[i] = static_cast<uint32_t>(((r * a.pairs + p) * 16 + (e & 15)) * 4);
    }
    const uint32_t xoff = static_cast<uint32_t>(lane) * 16u;

    auto load_raw = [&](int chunk, uint4 (&raw)[WPT], uint32_t (&dr)[DPT]) {
        const int pc = pbeg + chunk * P;
#pragma unroll
        for (int i = 0; i < WPT; ++i)
            raw[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(qv, qoff[i], pc * 1024, 0));
#pragma unroll
        for (int i = 0; i < DPT; ++i) dr[i] = __builtin_amdgcn_raw_buffer_load_b32(dv, doff[i], pc * 64, 0);
    };
    auto stage = [&](int buf, const uint4 (&raw)[WPT], const uint32_t (&dr)[DPT]) {
#pragma unroll
        for (int i = 0; i < WPT; ++i) {
            const int e = tid + NTH * i;
            if (RAW % NTH && e >= RAW) break;
            const int r = (e >> 6) / P, p = (e >> 6) % P, l = e & 63;
            ws[buf][2 * p][r][l] = i8x8_to_half8(make_uint2(raw[i].x, raw[i].y));
            ws[buf][2 * p + 1][r][l] = i8x8_to_half8(make_uint2(raw[i].z, raw[i].w));
        }
#pragma unroll
        for (int i = 0; i < DPT; ++i) {
            const int e = tid + NTH * i;
            if (e < DW) wd[buf][e / (P * 16)][(e / 16) % P][e & 15] = dr[i];
        }
    };
    auto load_x = [&](int chunk, u32x4 (&x)[CG][2]) {
#pragma unroll
        for (int c = 0; c < CG; ++c) {
            const int g = gbeg + chunk * CG + c;
            const int so = g < gend ? g * 2048 : static_cast<int>(xbytes);  // past the split: zeros
            x[c][0] = __builtin_amdgcn_raw_buffer_load_b128(xv, xoff, so, 0);
            x[c][1] = __builtin_amdgcn_raw_buffer_load_b128(xv, xoff + 1024u, so, 0);
        }
    };
    float4v acc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r] = float4v{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](int buf, const u32x4 (&x)[CG][2]) {
        uint32_t dd[RT][P];
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int p = 0; p < P; ++p) dd[r][p] = wd[buf][r][p][lane & 15];
#pragma unroll
        for (int c = 0; c < CG; ++c) {
            const half8 xh = __builtin_bit_cast(half8, x[c][0]), xl = __builtin_bit_cast(half8, x[c][1]);
            half8 w[RT];
#pragma unroll
            for (int r = 0; r < RT; ++r) w[r] = ws[buf][c][r][lane];
            float4v cc[RT];
#pragma unroll
            for (int r = 0; r < RT; ++r)
                cc[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, w[r], float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < RT; ++r) cc[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, w[r], cc[r], 0, 0, 0);
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const float d = half_bits_to_float(static_cast<uint16_t>(dd[r][c / 2] >> (c % 2 ? 16 : 0)));
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[r][i] = fmaf(d, cc[r][i], acc[r][i]);
            }
        }
    };

    uint4 rA[WPT], rB[WPT];
    uint32_t dA[DPT], dB[DPT];
    u32x4 xA[CG][2], xB[CG][2];
    const int c1 = min(1, nchunks - 1);
    load_raw(0, rA, dA);
    load_x(0, xA);
    load_raw(c1, rB, dB);
    stage(0, rA, dA);
    load_x(c1, xB);
    __syncthreads();
    for (int k = 0;; k += 2) {
        load_raw(min(k + 2, nchunks - 1), rA, dA);
        compute(0, xA);
        stage(1, rB, dB);
        __syncthreads();
        if (k + 1 >= nchunks) break;
        load_x(min(k + 2, nchunks - 1), xA);
        load_raw(min(k + 3, nchunks - 1), rB, dB);
        compute(1, xB);
        stage(0, rA, dA);
        __syncthreads();
        if (k + 2 >= nchunks) break;
        load_x(min(k + 3, nchunks - 1), xB);
    }
    // lane l holds row l%16 of each tile for vectors 4(l/16) + i of its tile
    float* out = a.out + static_cast<size_t>(blockIdx.y) * a.n * a.rows;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int j = (static_cast<int>(blockIdx.z) * NT + wave) * 16 + 4 * (lane >> 4) + i;
        if (j >= a.n) continue;
        const float us = a.unscale[j];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int row = (t0 + r) * 16 + (lane & 15);
            if (t0 + r < a.tiles && row < a.rows) out[static_cast<size_t>(j) * a.rows + row] = acc[r][i] * us;
        }
    }
}

// The same product as a tiled GEMM, for many vectors.  A workgroup of eight
// waves (two by four) owns 2*VT vector tiles by sixteen row tiles over one K
// split, a wave VT by four of them, so that the operands a wave reads from LDS
// per group, (2*VT + 4) KiB, feed 8*VT MFMAs.  K advances a group pair a step,
// two steps ahead of the products: the activation halves go from memory
// straight into one of three LDS buffers (16 bytes a lane, in operand order),
// the int8 weights into one of two register sets and from there, converted
// once for the workgroup, into one of two LDS buffers; the scales a lane needs
// stay in registers.  A step has one barrier.
// With VT = 4 the buffers take all 160 KB of LDS: one workgroup a CU, two
// waves a SIMD.
// Workgroups are numbered so that each XCD takes a contiguous run of tiles
// (eight row blocks by the vector blocks), whose operands its L2 then shares.
// Row tiles past the matrix and vector tiles past the batch read the last tile
// again and are not stored; the group that completes an odd count has weights
// and scales of zero (as the matrix was laid out) and multiplies the last one's
// halves (q8_pipe.hpp).
//
// Bound: issue on the SIMDs.  At 2,048 vectors of the 16,384 x 2,048 gate|up
// MFMAs take 43% of the cycles and the vector instructions (two thirds of them
// the four scale FMAs a product) 32-43%, and the two add up rather than
// overlap; LDS is busy 22%, without a bank conflict.
// MI355X, 3,072 / 2,048 / 16,384 x 2,048 and 2,048 x 8,192, against the kernel
// it replaced (weights kept in LDS, activations read through L1 by every
// wave), which took four times its time at 512: 78.6 / 45.3 / 330 / 161 us at
// 2,048 vectors against 137 / 112 / 530 / 264 (834 TFLOP/s of fp16 products on
// the third), and 28.5 / 25.9 / 89 / 45 us at 512 against 34 / 28 / 133 / 66.
template <int VT>
__global__ __launch_bounds__(512, 2) void batch_q8_pipe_kernel(const Q8BatchArgs a) {
    constexpr int BV = 2 * VT, BR = kPipeRowTiles;  // vector and row tiles of a workgroup
    constexpr int XL = BV * 4 / 8;       // KiB of halves a wave loads per pair
    // separate arrays, so that the compiler sees that a step's reads do not
    // touch the buffers in flight and does not wait for them
    __shared__ u32x4 x0[BV][4][64], x1[BV][4][64], x2[BV][4][64];  // [vector tile][group * 2 + part][lane]
    __shared__ half8 w0[2][BR][64], w1[2][BR][64];                 // [group][row tile][lane]
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int vh = wave & 1, rh = wave >> 1;
    // logical tile of this workgroup
    const int nrb = (a.tiles - a.tile0 + BR - 1) / BR, nvb = (a.n_total_tiles + BV - 1) / BV;
    int vb, rb;
    {
        const int total = nrb * nvb, b = static_cast<int>(blockIdx.x);
        const int per = total / 8, extra = total % 8, xcd = b % 8;
        const int id = xcd * per + min(xcd, extra) + b / 8;
        const int band = id / (8 * nvb), rows_here = min(8, nrb - band * 8), in = id - band * 8 * nvb;
        vb = in / rows_here;
        rb = band * 8 + in - vb * rows_here;
    }
    const int t0 = a.tile0 + rb * BR;
    const int tiles_here = min(BR, a.tiles - t0);
    const int pbeg = static_cast<int>(blockIdx.y) * (a.groups_per_split / 2);
    const int np = min(a.pairs, pbeg + a.groups_per_split / 2) - pbeg;
    const __amdgpu_buffer_rsrc_t qv =
        view(a.q + static_cast<size_t>(t0) * a.pairs * 64, static_cast<uint32_t>(tiles_here * a.pairs) * 1024u);
    const __amdgpu_buffer_rsrc_t dv = view(reinterpret_cast<const uint32_t*>(a.d) + static_cast<size_t>(t0) * a.pairs * 16,
                                           static_cast<uint32_t>(tiles_here * a.pairs) * 64u);
    const __amdgpu_buffer_rsrc_t xv =
        view(a.halves, static_cast<uint32_t>(a.n_total_tiles) * static_cast<uint32_t>(a.groups) * 2048u);
    const uint32_t xoff = static_cast<uint32_t>((lane & 15) * 128 + (lane >> 4) * 16);
    const uint32_t qoff = static_cast<uint32_t>(lane * 16), doff = static_cast<uint32_t>((lane & 15) * 4);

    uint4 ra[2], rb2[2];
    uint32_t da[4], db[4], dc[4];
    auto load_w = [&](int p, uint4 (&raw)[2], uint32_t (&dn)[4]) {
#pragma unroll
        for (int i = 0; i < 2; ++i)  // row tiles wave and wave + 8 to convert
            raw[i] = __builtin_bit_cast(
                uint4, __builtin_amdgcn_raw_buffer_load_b128(
                           qv, qoff, pipe_weight_offset(wave + 8 * i, tiles_here, a.pairs, pbeg + p), 0));
#pragma unroll
        for (int r = 0; r < 4; ++r)
            dn[r] = __builtin_amdgcn_raw_buffer_load_b32(
                dv, doff, pipe_scale_offset(rh * 4 + r, tiles_here, a.pairs, pbeg + p), 0);
    };
    auto load_x = [&](int p, u32x4 (&x)[BV][4][64]) {
#pragma unroll
        for (int i = 0; i < XL; ++i) {
            const int t = (wave * XL + i) / 4, part = (wave * XL + i) % 4;
            const int vt = min(vb * BV + t, a.n_total_tiles - 1);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xv, (__attribute__((address_space(3))) void*)&x[t][part][0], 16, xoff,
                                                     pipe_vector_offset(vt, a.groups, 2 * (pbeg + p) + part / 2, part % 2), 0,
                                                     0);
        }
    };
    auto stage = [&](const uint4 (&raw)[2], half8 (&ws)[2][BR][64]) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            ws[0][wave + 8 * i][lane] = i8x8_to_half8(make_uint2(raw[i].x, raw[i].y));
            ws[1][wave + 8 * i][lane] = i8x8_to_half8(make_uint2(raw[i].z, raw[i].w));
        }
    };
    float4v acc[VT][4];
#pragma unroll
    for (int v = 0; v < VT; ++v)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[v][r] = float4v{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const u32x4 (&x)[BV][4][64], const half8 (&ws)[2][BR][64], const uint32_t (&dd)[4]) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            half8 w[4];
            float d[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                w[r] = ws[g][rh * 4 + r][lane];
                d[r] = half_bits_to_float(static_cast<uint16_t>(dd[r] >> (16 * g)));
            }
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                const half8 xh = __builtin_bit_cast(half8, x[vh * VT + v][2 * g][lane]);
                const half8 xl = __builtin_bit_cast(half8, x[vh * VT + v][2 * g + 1][lane]);
                float4v cc[4];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    cc[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, w[r], float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) cc[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, w[r], cc[r], 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[v][r][i] = fmaf(d[r], cc[r][i], acc[v][r][i]);
            }
        }
    };
    // Step p: wait for this wave's part of pair p (requested two steps ago; the
    // newest step's loads stay in flight) and for its LDS writes, meet the
    // others, request pair p + 2 into the buffer read in step p - 1, multiply
    // pair p, convert pair p + 1.  Loads past the split repeat its last pair,
    // so that every step issues the same number and the count below holds.
    constexpr int kPerStep = 2 + 4 + XL;
    auto step = [&](int p, const u32x4 (&xc)[BV][4][64], u32x4 (&xn)[BV][4][64], const half8 (&wc)[2][BR][64],
                    half8 (&wn)[2][BR][64], const uint32_t (&dcur)[4], uint32_t (&dnxt)[4], uint4 (&rload)[2],
                    const uint4 (&rstage)[2]) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kPerStep) : "memory");
        const int pn = min(p + 2, np - 1);
        load_w(pn, rload, dnxt);
        load_x(pn, xn);
        compute(xc, wc, dcur);
        __builtin_amdgcn_sched_barrier(0);  // the conversion waits for loads: not ahead of the products
        stage(rstage, wn);
    };
    load_w(0, ra, da);
    load_x(0, x0);
    __builtin_amdgcn_sched_barrier(0);  // the first step's wait counts on pair 0 being requested first
    load_w(min(1, np - 1), rb2, db);
    load_x(min(1, np - 1), x1);
    stage(ra, w0);
    for (int p = 0;; p += 6) {
        step(p, x0, x2, w0, w1, da, dc, ra, rb2);
        if (p + 1 >= np) break;
        step(p + 1, x1, x0, w1, w0, db, da, rb2, ra);
        if (p + 2 >= np) break;
        step(p + 2, x2, x1, w0, w1, dc, db, ra, rb2);
        if (p + 3 >= np) break;
        step(p + 3, x0, x2, w1, w0, da, dc, rb2, ra);
        if (p + 4 >= np) break;
        step(p + 4, x1, x0, w0, w1, db, da, ra, rb2);
        if (p + 5 >= np) break;
        step(p + 5, x2, x1, w1, w0, dc, db, rb2, ra);
        if (p + 6 >= np) break;
    }
    // no load may be in flight into this workgroup's LDS when it ends
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // lane l holds row l%16 of each row tile for vectors 4(l/16) + i
    float* out = a.out + static_cast<size_t>(blockIdx.y) * a.n * a.rows;
#pragma unroll
    for (int v = 0; v < VT; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = (vb * BV + vh * VT + v) * 16 + 4 * (lane >> 4) + i;
            if (j >= a.n) continue;
            const float us = a.unscale[j];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int tile = t0 + rh * 4 + r, row = tile * 16 + (lane & 15);
                if (tile < a.tiles && row < a.rows) out[static_cast<size_t>(j) * a.rows + row] = acc[v][r][i] * us;
            }
        }
}

// ---------------------------------------------------------- batch epilogues
//
// The batched products write f32 sums per K split, [splits][n][rows]; these
// kernels add the splits in order (from 0.f, as one split's value is itself)
// and apply what follows the product in the layer.

// The sum runs in split order.  The partials are read N at a time (N = 1, 2
// or 4 when that covers every split, else 8), all N requested before the
// first add; clamped indices keep the loads unconditional, and a select (not
// an add of 0.f) skips the surplus ones.
template <int N>
__device__ __forceinline__ float split_sum(const float* p, int splits, size_t stride, size_t at) {
    float s = 0.f;
    for (int k0 = 0; k0 < splits; k0 += N) {
        float v[N];
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = p[static_cast<size_t>(min(k0 + k, splits - 1)) * stride + at];
#pragma unroll
        for (int k = 0; k < N; ++k) s = k0 + k < splits ? s + v[k] : s;
    }
    return s;
}

__device__ __forceinline__ float split_total(const float* p, int splits, size_t stride, size_t at) {
    if (splits == 1) return split_sum<1>(p, splits, stride, at);
    if (splits == 2) return split_sum<2>(p, splits, stride, at);
    if (splits <= 4) return split_sum<4>(p, splits, stride, at);
    return split_sum<8>(p, splits, stride, at);
}

// the split sums of eight consecutive elements at p + at (16-byte aligned),
// in split order from 0.f, four splits' loads requested at a time
__device__ __forceinline__ void split_total8(const float* p, int splits, size_t stride, size_t at, float (&s)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = 0.f;
    for (int k0 = 0; k0 < splits; k0 += 4) {
        float v[4][8];
#pragma unroll
        for (int k = 0; k < 4; ++k) load8(p + static_cast<size_t>(min(k0 + k, splits - 1)) * stride + at, v[k]);
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int i = 0; i < 8; ++i) s[i] = k0 + k < splits ? s[i] + v[k][i] : s[i];
    }
}

// Q|K|V rows of vector j: q and k rotated by row j's (cos, sin)
// (model.hpp:63-72), v copied; one thread per rotation pair or v element
__global__ void qkv_epilogue_kernel(const float* p, int splits, int n, int qheads, int kheads, int dim, int interleaved,
                                    const float* cs, float* q, float* k, float* v) {
    const int half = dim / 2, rows = (qheads + 2 * kheads) * dim, kw = kheads * dim;
    const int pairs = (qheads + kheads) * half, per = pairs + kw;
    const size_t stride = static_cast<size_t>(n) * rows;
    const size_t total = static_cast<size_t>(n) * per;
    for (size_t t = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; t < total;
         t += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const int j = static_cast<int>(t / per), e = static_cast<int>(t % per);
        const size_t base = static_cast<size_t>(j) * rows;
        if (e >= pairs) {
            const int c = e - pairs;
            v[static_cast<size_t>(j) * kw + c] = split_total(p, splits, stride, base + qheads * dim + kw + c);
            continue;
        }
        const int h = e / half, i = e % half;
        const int ia = interleaved ? 2 * i : i, ib = interleaved ? 2 * i + 1 : i + half;
        const float left = split_total(p, splits, stride, base + h * dim + ia);
        const float right = split_total(p, splits, stride, base + h * dim + ib);
        const float c = cs[static_cast<size_t>(j) * dim + 2 * i], s = cs[static_cast<size_t>(j) * dim + 2 * i + 1];
        float* x = h < qheads ? q + (static_cast<size_t>(j) * qheads + h) * dim
                              : k + (static_cast<size_t>(j) * kheads + (h - qheads)) * dim;
        x[ia] = __fsub_rn(__fmul_rn(left, c), __fmul_rn(right, s));
        x[ib] = __fadd_rn(__fmul_rn(right, c), __fmul_rn(left, s));
    }
}

// Vector j = blockIdx.x: x += the product's sum (the residual add, when p is
// given), then RMSNorm with w (model.hpp:54-61: sum of squares in double,
// scale rounded to float, (x * s) * w) into `norm` (when given) and, when
// `halves` is given, into the next product's fp16 halves.  A thread keeps
// its chunks in registers between the passes.
template <bool kByLine>
__global__ __launch_bounds__(1024) void resid_norm_kernel(const float* p, int splits, float* x, const float* w, int n,
                                                          int h, float eps, float* norm, _Float16* halves, int groups,
                                                          float* unscale) {
    __shared__ double part[16];
    __shared__ float mpart[16];
    const int j = blockIdx.x, T = blockDim.x;
    float* xr = x + static_cast<size_t>(j) * h;
    const size_t stride = static_cast<size_t>(n) * h;
    float y[kEpiChunks][8], wv[kEpiChunks][8];
    double sq = 0;
#pragma unroll
    for (int c = 0; c < kEpiChunks; ++c) {
        const int e0 = 8 * (static_cast<int>(threadIdx.x) + T * c);
        if (e0 < h) {
            load8(xr + e0, y[c]);
            load8(w + e0, wv[c]);
            if (p) {
                float t[8];
                split_total8(p, splits, stride, static_cast<size_t>(j) * h + e0, t);
#pragma unroll
                for (int i = 0; i < 8; ++i) y[c][i] = __fadd_rn(y[c][i], t[i]);
                store8(xr + e0, y[c]);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) sq += static_cast<double>(y[c][i]) * y[c][i];
        }
    }
    for (int o = 32; o >= 1; o >>= 1) sq += __shfl_xor(sq, o);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sq;
    __syncthreads();
    double t = 0;
    for (int wave = 0; wave < T / 64; ++wave) t += part[wave];
    const float inv = static_cast<float>(1.0 / sqrt(t / static_cast<double>(h) + static_cast<double>(eps)));
    float mx = 0.f;
#pragma unroll
    for (int c = 0; c < kEpiChunks; ++c) {
        const int e0 = 8 * (static_cast<int>(threadIdx.x) + T * c);
        if (e0 < h) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                y[c][i] = __fmul_rn(__fmul_rn(y[c][i], inv), wv[c][i]);
                mx = fmaxf(mx, fabsf(y[c][i]));
            }
            if (norm) store8(norm + static_cast<size_t>(j) * h + e0, y[c]);
        }
    }
    if (!halves) return;
    const int shift = halves_shift(block_max(mx, mpart));
    const float up = ldexpf(1.f, shift);
    if (threadIdx.x == 0) unscale[j] = ldexpf(1.f, -shift);
#pragma unroll
    for (int c = 0; c < kEpiChunks; ++c) {
        const int e0 = 8 * (static_cast<int>(threadIdx.x) + T * c);
        if (e0 < h) {
#pragma unroll
            for (int i = 0; i < 8; ++i) y[c][i] *= up;
            put_halves8<kByLine>(halves, groups, j, e0, y[c]);
        }
    }
}

// Vector j = blockIdx.x of the fused gate|up product: gate * (sigmoid(gate)
// * up) (model.hpp:111-116) into `out` (when given) and, when given, the next
// product's halves
template <bool kByLine>
__global__ __launch_bounds__(1024) void swiglu_epilogue_kernel(const float* p, int splits, int n, int inter, float* out,
                                                               _Float16* halves, int groups, float* unscale,
                                                               int interleaved) {
    __shared__ float mpart[16];
    const int j = blockIdx.x, T = blockDim.x;
    const size_t stride = static_cast<size_t>(n) * 2 * inter, base = static_cast<size_t>(j) * 2 * inter;
    float val[kEpiChunks][8];
    float mx = 0.f;
#pragma unroll
    for (int c = 0; c < kEpiChunks; ++c) {
        const int e0 = 8 * (static_cast<int>(threadIdx.x) + T * c);
        if (e0 < inter) {
            float g[8], u[8];
            if (interleaved) {  // rows 2e (gate), 2e + 1 (up)
                float a[8], b[8];
                split_total8(p, splits, stride, base + 2 * static_cast<size_t>(e0), a);
                split_total8(p, splits, stride, base + 2 * static_cast<size_t>(e0) + 8, b);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    g[i] = a[2 * i], u[i] = a[2 * i + 1];
                    g[4 + i] = b[2 * i], u[4 + i] = b[2 * i + 1];
                }
            } else {
                split_total8(p, splits, stride, base + e0, g);
                split_total8(p, splits, stride, base + inter + e0, u);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float small = expf(-fabsf(g[i]));
                const float one = __fadd_rn(1.f, small);
                const float sig = g[i] >= 0 ? __fdiv_rn(1.f, one) : __fdiv_rn(small, one);
                val[c][i] = __fmul_rn(g[i], __fmul_rn(sig, u[i]));
                mx = fmaxf(mx, fabsf(val[c][i]));
            }
            if (out) store8(out + static_cast<size_t>(j) * inter + e0, val[c]);
        }
    }
    if (!halves) return;
    const int shift = halves_shift(block_max(mx, mpart));
    const float up = ldexpf(1.f, shift);
    if (threadIdx.x == 0) unscale[j] = ldexpf(1.f, -shift);
#pragma unroll
    for (int c = 0; c < kEpiChunks; ++c) {
        const int e0 = 8 * (static_cast<int>(threadIdx.x) + T * c);
        if (e0 < inter) {
#pragma unroll
            for (int i = 0; i < 8; ++i) val[c][i] *= up;
            put_halves8<kByLine>(halves, groups, j, e0, val[c]);
        }
    }
}

// element (j, c) of row idx[j] (or `row`) of a Q8_0 table
__global__ void gather_embedding_q8_kernel(const uint8_t* q, const uint16_t* d, int pairs, const uint32_t* idx,
                                           uint32_t row, int n, int h, float* out) {
    const size_t total = static_cast<size_t>(n) * h;
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < total;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const int j = static_cast<int>(i / h), c = static_cast<int>(i % h);
        const uint32_t r = idx ? idx[j] : row;
        const int g = c / 32;
        const size_t blk = static_cast<size_t>(r / 16) * pairs + g / 2;
        const int lane = static_cast<int>(r % 16) + 16 * ((c % 32) / 8);
        const float dv = half_bits_to_float(d[(blk * 16 + r % 16) * 2 + g % 2]);
        out[i] = __fmul_rn(dv, static_cast<float>(static_cast<int8_t>(q[(blk * 64 + lane) * 16 + (g % 2) * 8 + c % 8])));
    }
}

unsigned grid_for(size_t n) {
    return static_cast<unsigned>(std::min<size_t>((n + kThreads - 1) / kThreads, 8192));
}

}  // namespace

void launch_dequant(uint32_t type, const uint8_t* raw, size_t n, float* out, int* bad, hipStream_t s) {
    if (!n) return;
    switch (type) {
        case 0:  // f32 payloads are copied in place; only checked here
            launch("model_dequant", check_f32_kernel, dim3(grid_for(n)), dim3(kThreads), 0, s,
                   static_cast<const float*>(out), n, bad);
            break;
        case 1: launch("model_dequant", f16_kernel, dim3(grid_for(n)), dim3(kThreads), 0, s, raw, n, out, bad); break;
        case 2: launch("model_dequant", q4_0_kernel, dim3(grid_for(n)), dim3(kThreads), 0, s, raw, n, out, bad); break;
        case 8: launch("model_dequant", q8_0_kernel, dim3(grid_for(n)), dim3(kThreads), 0, s, raw, n, out, bad); break;
        case 12: launch("model_dequant", q4_k_kernel, dim3(grid_for(n)), dim3(kThreads), 0, s, raw, n, out, bad); break;
        default: throw std::invalid_argument("unsupported native weight type");
    }
    TVARA_HIP(hipGetLastError());
}

void launch_rmsnorm(const float* x, const float* w, float* out, int n, float eps, hipStream_t s, int rows) {
    launch("model_rmsnorm", rmsnorm_kernel, dim3(rows), dim3(1024), 0, s, x, w, out, n, eps);
    TVARA_HIP(hipGetLastError());
}

void launch_split_sum(const float* p, int splits, int n, int rows, float* out, hipStream_t s) {
    BatchMatvecArgs b{};
    b.rows = rows;
    b.n = n;
    b.nseg = 1;
    b.seg[0] = MatvecSegment{out, rows, nullptr};
    b.partial = const_cast<float*>(p);
    launch("model_matvec_sum", split_sum_kernel, dim3(grid_for(static_cast<size_t>(n) * rows)), dim3(kThreads), 0, s, b,
           splits);
    TVARA_HIP(hipGetLastError());
}

void launch_gather_embedding(const float* table, const uint32_t* idx, int n, int h, float* out, hipStream_t s) {
    launch("model_embedding", gather_embedding_kernel, dim3(grid_for(static_cast<size_t>(n) * h)), dim3(kThreads), 0, s,
           table, idx, n, h, out);
    TVARA_HIP(hipGetLastError());
}

void launch_interleave_layers(const float* src, float* dst, int layers, int n, int kv, hipStream_t s) {
    const size_t total = static_cast<size_t>(layers) * n * kv;
    launch("model_interleave", interleave_layers_kernel, dim3(grid_for(total)), dim3(kThreads), 0, s, src, dst, layers,
           n, kv);
    TVARA_HIP(hipGetLastError());
}

void launch_matvec(const float* w, int rows, int cols, const float* v, const MatvecSegment* seg, int nseg,
                   hipStream_t s) {
    MatvecArgs a{};
    a.w = w;
    a.v = v;
    a.rows = rows;
    a.cols = cols;
    a.nseg = nseg;
    for (int i = 0; i < nseg; ++i) a.seg[i] = seg[i];
    const dim3 grid((rows + kThreads / 64 - 1) / (kThreads / 64));
    if (cols % 4 == 0)
        launch("model_matvec", matvec_kernel<true>, grid, dim3(kThreads), 0, s, a);
    else
        launch("model_matvec", matvec_kernel<false>, grid, dim3(kThreads), 0, s, a);
    TVARA_HIP(hipGetLastError());
}

void launch_rope(float* q, int qheads, float* k, int kheads, int dim, const float* cs, bool interleaved,
                 hipStream_t s, int rows) {
    const int n = (qheads + kheads) * (dim / 2);
    launch("model_rope", rope_kernel, dim3((n + kThreads - 1) / kThreads, rows), dim3(kThreads), 0, s, q, qheads, k,
           kheads, dim, cs, interleaved ? 1 : 0);
    TVARA_HIP(hipGetLastError());
}

void launch_swiglu(float* gate, const float* up, int n, hipStream_t s) {
    launch("model_swiglu", swiglu_kernel, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, s, gate, up, n);
    TVARA_HIP(hipGetLastError());
}

void launch_q8_repack(const uint8_t* raw, int rows, int cols, int row0, int stride, Weight& w, int* bad,
                      hipStream_t s) {
    const size_t total = static_cast<size_t>(rows) * (cols / 32);
    if (!total) return;
    launch("model_q8_repack", q8_repack_kernel, dim3(grid_for(total)), dim3(kThreads), 0, s, raw, rows, cols / 32, row0,
           stride, static_cast<uint8_t*>(w.q.ptr), static_cast<uint16_t*>(w.d.ptr), bad);
    TVARA_HIP(hipGetLastError());
}

void launch_matvec_q8(const Weight& w, const float* v, const MatvecSegment* seg, int nseg, hipStream_t s,
                      const float* norm_w, float eps, const float* rope_cs, int rope_dim, int rope_rows) {
    if (w.cols > 15360) throw std::invalid_argument("Q8_0 matrix wider than 15,360 columns");
    Q8MatvecArgs a{};
    a.q = static_cast<const uint4*>(w.q.ptr);
    a.d = static_cast<const uint32_t*>(w.d.ptr);
    a.v = v;
    a.norm_w = norm_w;
    a.eps = eps;
    a.rows = w.rows;
    a.tiles = w.tiles();
    a.groups = w.groups();
    a.pairs = w.pairs();
    a.cols = w.cols;
    a.nseg = nseg;
    for (int i = 0; i < nseg; ++i) a.seg[i] = seg[i];
    a.rope_cs = rope_cs;
    a.rope_dim = rope_dim;
    a.rope_rows = rope_rows;
    a.swiglu = w.interleaved ? 1 : 0;
    // two tiles per workgroup (sharing the staged input) for the largest
    // matrices.  Waves per workgroup: up to about sixteen waves per CU over
    // the launch (4,096), at most sixteen, at least two when there is work
    // for two, and at least two group pairs a wave (MI355X, Llama-3.2-1B shapes, two pairs a step:
    // 16,384 x 2,048 gate|up in 11.2 us at one tile and four waves against
    // 12.3 at two tiles and eight; 2,048 x 8,192 down 8.6 us at sixteen;
    // 3,072 x 2,048 QKV 6.1-6.2 us at eight or sixteen; the 128,256-row
    // logits in 58 us at two waves against 65 at one)
    const int rt = a.tiles >= 4096 ? 2 : 1;
    const int wgs = (a.tiles + rt - 1) / rt;
    int want = 1;
    while (want < 16 && 2 * want * 2 <= a.pairs && (want < 2 || wgs * want * 2 <= 4096)) want *= 2;
    const dim3 grid(wgs);
    // the input, and the norm weights beside it when the product normalises
    const size_t lds = static_cast<size_t>(w.cols) * sizeof(float) * (norm_w ? 2 : 1);
    auto go = [&](auto kernel, auto streaming, int waves) {
        launch("model_matvec_q8", w.streamed ? streaming : kernel, grid, dim3(64 * waves), lds, s, a);
    };
    if (rt == 2) {
        if (want >= 8) go(matvec_q8_kernel<8, 2, false>, matvec_q8_kernel<8, 2, true>, 8);
        else if (want >= 4) go(matvec_q8_kernel<4, 2, false>, matvec_q8_kernel<4, 2, true>, 4);
        else if (want >= 2) go(matvec_q8_kernel<2, 2, false>, matvec_q8_kernel<2, 2, true>, 2);
        else go(matvec_q8_kernel<1, 2, false>, matvec_q8_kernel<1, 2, true>, 1);
    } else {
        if (want >= 16) go(matvec_q8_kernel<16, 1, false>, matvec_q8_kernel<16, 1, true>, 16);
        else if (want >= 8) go(matvec_q8_kernel<8, 1, false>, matvec_q8_kernel<8, 1, true>, 8);
        else if (want >= 4) go(matvec_q8_kernel<4, 1, false>, matvec_q8_kernel<4, 1, true>, 4);
        else if (want >= 2) go(matvec_q8_kernel<2, 1, false>, matvec_q8_kernel<2, 1, true>, 2);
        else go(matvec_q8_kernel<1, 1, false>, matvec_q8_kernel<1, 1, true>, 1);
    }
    TVARA_HIP(hipGetLastError());
}

namespace {
// one wave per vector tile
template <int RT>
void launch_batch_q8(int nt, dim3 grid, hipStream_t s, const Q8BatchArgs& a) {
    switch (nt) {
        case 1: launch("model_matvec_q8", batch_q8_kernel<1, RT>, grid, dim3(64), 0, s, a); break;
        case 2: launch("model_matvec_q8", batch_q8_kernel<2, RT>, grid, dim3(128), 0, s, a); break;
        case 3: launch("model_matvec_q8", batch_q8_kernel<3, RT>, grid, dim3(192), 0, s, a); break;
        default: launch("model_matvec_q8", batch_q8_kernel<4, RT>, grid, dim3(256), 0, s, a); break;
    }
}

struct F32Plan {
    int tiles, per, splits;
};
F32Plan f32_plan(int rows, int cols) {
    F32Plan p{};
    p.tiles = (rows + kTileRows - 1) / kTileRows;
    const int chunks = cols / kTileK;
    const int want = std::max(1, std::min(chunks, (512 + p.tiles - 1) / p.tiles));
    p.per = (chunks + want - 1) / want;
    p.splits = (chunks + p.per - 1) / p.per;
    return p;
}

int pipe_for(const Weight& w, int n) { return w.q8 ? pipe_choice(w.tiles(), w.groups(), n) : 0; }

// row tiles [tile0, tile1), K in `per` groups a split
Q8BatchArgs batch_args(const Weight& w, int per, int tile0, int tile1, const _Float16* halves, const float* unscale,
                       int n, float* out) {
    Q8BatchArgs a{};
    a.q = static_cast<const uint4*>(w.q.ptr);
    a.d = static_cast<const uint16_t*>(w.d.ptr);
    a.halves = reinterpret_cast<const uint4*>(halves);
    a.unscale = unscale;
    a.rows = w.rows;
    a.tiles = tile1;
    a.tile0 = tile0;
    a.groups = w.groups();
    a.pairs = w.pairs();
    a.n = n;
    a.n_total_tiles = (n + 15) / 16;
    a.groups_per_split = per;
    a.out = out;
    return a;
}

// the chunked kernel over every block of up to four vector tiles
void launch_chunked(const Weight& w, int rt, int splits, int per, int tile0, int tile1, const _Float16* halves,
                    const float* unscale, int n, float* out, hipStream_t s) {
    const Q8BatchArgs a = batch_args(w, per, tile0, tile1, halves, unscale, n, out);
    const int nt = std::min(4, a.n_total_tiles);
    const dim3 grid((tile1 - tile0 + rt - 1) / rt, splits, (a.n_total_tiles + 3) / 4);
    if (rt == 4)
        launch_batch_q8<4>(nt, grid, s, a);
    else
        launch_batch_q8<2>(nt, grid, s, a);
}

void launch_pipe(const Weight& w, const PipePlan& p, int tile0, int tile1, const _Float16* halves,
                 const float* unscale, int n, float* out, hipStream_t s) {
    const Q8BatchArgs a = batch_args(w, p.per, tile0, tile1, halves, unscale, n, out);
    if (static_cast<double>(a.n_total_tiles) * a.groups * 2048 >= 2147483648.0)
        throw std::invalid_argument("batched product input above 2 GiB");
    const dim3 grid(p.gx, p.splits);
    if (p.vt == 4)
        launch("model_matvec_q8", batch_q8_pipe_kernel<4>, grid, dim3(512), 0, s, a);
    else
        launch("model_matvec_q8", batch_q8_pipe_kernel<2>, grid, dim3(512), 0, s, a);
}
}  // namespace

bool halves_by_line(const Weight& w, int n) { return pipe_for(w, n) != 0; }

int batch_splits(const Weight& w, int n) {
    if (!w.q8) return f32_plan(w.rows, w.cols).splits;
    const int vt = pipe_for(w, n);
    return vt ? pipe_plan(w.tiles(), w.groups(), n, vt).splits : q8_plan(w.tiles(), w.groups()).splits;
}

size_t batch_part_floats(const Weight& w, int n) {
    // the splits depend on the count of 16-vector tiles
    size_t most = 0;
    for (int j = std::min(n, 16); j; j = j < n ? std::min(n, j + 16) : 0)
        most = std::max(most, static_cast<size_t>(batch_splits(w, j)) * j * w.rows);
    return most;
}

void launch_batch_product(const Weight& w, const float* x, const _Float16* halves, const float* unscale, int n,
                          float* out, hipStream_t s) {
    if (const int vt = pipe_for(w, n)) {
        launch_pipe(w, pipe_plan(w.tiles(), w.groups(), n, vt), 0, w.tiles(), halves, unscale, n, out, s);
    } else if (w.q8) {
        const Q8Plan p = q8_plan(w.tiles(), w.groups());
        launch_chunked(w, p.rt, p.splits, p.per, 0, w.tiles(), halves, unscale, n, out, s);
    } else {
        if (w.cols % kTileK) throw std::invalid_argument("batched matvec needs a row width divisible by 32");
        const F32Plan p = f32_plan(w.rows, w.cols);
        for (int j0 = 0; j0 < n; j0 += kTileVecs) {
            BatchMatvecArgs a{};
            a.w = static_cast<const float*>(w.f32.ptr);
            a.x = x + static_cast<size_t>(j0) * w.cols;
            a.rows = w.rows;
            a.cols = w.cols;
            a.n = std::min(kTileVecs, n - j0);
            a.chunks_per_split = p.per;
            a.partial = out;
            a.n_total = n;
            a.j0 = j0;
            launch("model_matvec", batch_matvec_kernel, dim3(p.tiles, p.splits), dim3(256), 0, s, a);
        }
    }
    TVARA_HIP(hipGetLastError());
}

void launch_batch_product_tiles(const Weight& w, int tile0, int tile1, const _Float16* halves, const float* unscale,
                                int n, float* out, hipStream_t s) {
    if (!w.q8 || batch_splits(w, n) != 1 || tile0 < 0 || tile0 >= tile1 || tile1 > w.tiles())
        throw std::invalid_argument("row-tile range of a batched product needs an unsplit Q8_0 matrix");
    if (const int vt = pipe_for(w, n)) {
        launch_pipe(w, pipe_plan(tile1 - tile0, w.groups(), n, vt, 1), tile0, tile1, halves, unscale, n, out, s);
        TVARA_HIP(hipGetLastError());
        return;
    }
    const Q8Plan p = q8_plan(w.tiles(), w.groups());
    launch_chunked(w, p.rt, 1, p.per, tile0, tile1, halves, unscale, n, out, s);
    TVARA_HIP(hipGetLastError());
}

void launch_split_halves(const float* x, int n, int cols, _Float16* halves, float* unscale, bool by_line,
                         hipStream_t s) {
    if (cols % 32 || cols > 1024 * 8 * kEpiChunks) throw std::invalid_argument("batched decode width above 16384");
    launch("model_split_halves", by_line ? split_halves_kernel<true> : split_halves_kernel<false>, dim3(n),
           dim3(epi_threads(cols)), 0, s, x, cols, cols / 32, halves, unscale);
    TVARA_HIP(hipGetLastError());
}

void launch_qkv_epilogue(const float* p, int splits, int n, int qheads, int kheads, int dim, bool interleaved,
                         const float* cs, float* q, float* k, float* v, hipStream_t s) {
    const size_t total = static_cast<size_t>(n) * ((qheads + kheads) * (dim / 2) + kheads * dim);
    launch("model_qkv_epilogue", qkv_epilogue_kernel, dim3(grid_for(total)), dim3(kThreads), 0, s, p, splits, n, qheads,
           kheads, dim, interleaved ? 1 : 0, cs, q, k, v);
    TVARA_HIP(hipGetLastError());
}

void launch_resid_norm(const float* p, int splits, float* x, const float* w, int n, int h, float eps, float* norm,
                       _Float16* halves, float* unscale, bool by_line, hipStream_t s) {
    if (h % 32 || h > 1024 * 8 * kEpiChunks) throw std::invalid_argument("batched decode width above 16384");
    launch("model_resid_norm", by_line ? resid_norm_kernel<true> : resid_norm_kernel<false>, dim3(n),
           dim3(epi_threads(h)), 0, s, p, splits, x, w, n, h, eps, norm, halves, h / 32, unscale);
    TVARA_HIP(hipGetLastError());
}

void launch_swiglu_epilogue(const float* p, int splits, int n, int inter, float* out, _Float16* halves,
                            float* unscale, bool by_line, hipStream_t s, bool interleaved) {
    if (inter % 32 || inter > 1024 * 8 * kEpiChunks) throw std::invalid_argument("batched decode width above 16384");
    launch("model_swiglu_epilogue", by_line ? swiglu_epilogue_kernel<true> : swiglu_epilogue_kernel<false>, dim3(n),
           dim3(epi_threads(inter)), 0, s, p, splits, n, inter, out, halves, inter / 32, unscale, interleaved ? 1 : 0);
    TVARA_HIP(hipGetLastError());
}

void launch_gather_embedding_q8(const Weight& w, const uint32_t* idx, uint32_t row, int n, float* out,
                                hipStream_t s) {
    const size_t total = static_cast<size_t>(n) * w.cols;
    launch("model_embedding", gather_embedding_q8_kernel, dim3(grid_for(total)), dim3(kThreads), 0, s,
           static_cast<const uint8_t*>(w.q.ptr), static_cast<const uint16_t*>(w.d.ptr), w.pairs(), idx, row, n,
           w.cols, out);
    TVARA_HIP(hipGetLastError());
}

}  // namespace tvara_amd
