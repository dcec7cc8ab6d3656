// Causal chunk attention in f32 (fused_prompt_attention,
// core/include/tvara/attention.hpp:85-89) as tiles on the f32 matrix cores
// (v_mfma_f32_16x16x4_f32: f32 operands, products and sums).
//
// A workgroup takes 128 query rows of one (sequence, KV head), a row being one
// (chunk position, query head of the GQA slice), 16 * NT rows a wave; all its
// waves share the key tiles, 64 keys each, read from the paged pool (f32, or
// Q8_0 dequantised on the way) a tile ahead into registers and from there into
// the other of two LDS buffers.
//
// Both contractions take their operands four at a time from one 16-byte LDS
// read, by the freedom to number a contraction's terms and the output's rows:
//  S^T = K Q^T: step (c, i) covers columns 16c + 4g + i of lane group g = l/16,
//    so a lane reads K[key l%16][16c + 4g ..+3] for four steps, and holds the
//    same columns of its query row.
//  O^T = V^T P^T: step (mt, i) covers keys 16mt + 4g + i, whose probabilities
//    are exactly the lane's own results of the first product; output row r of
//    tile (h, j) is column 64h + 4r + j, so a lane reads V[key][64h + 4(l%16)
//    ..+3] for four tiles and ends up with runs of 16 output columns.
//
// Sums.  A score is D/16 chains of four steps, summed pairwise; 32 keys'
// contribution to the output is a chain of eight steps from zero, added to the
// running output: chains as short as the decode kernels', where one over all
// keys would round more the longer the context (relative error in the 2-norm
// against 64 bits, six chunks of 33-700 tokens after 300-1,600, decode kernels
// then tiles: 3.8e-7 and 3.1e-7 at 32 x 8 heads of 64, 3.6e-7 and 3.1e-7 of
// 128).  Softmax in log2 units with the lazy rescale of the decode
// kernels.  A score that is not finite sets *err (OnlineAttention::update's
// rejection, attention.hpp:11), whether or not it would have mattered.
//
// Bound: the f32 matrix rate (157 TFLOP/s), plus the softmax's vector work,
// which adds to it.  MI355X, against the same rows through the decode kernels
// (which read every key once per row from L2 and multiply on the vector ALU):
// those six chunks 715 -> 328 us (87 TFLOP/s) and 1,337 -> 641 us; 8 x 512 after
// 2,000 tokens 2,610 -> 735 us (103 TFLOP/s); 400 rows of four sequences after
// 2,000 over Q8_0 blocks 470 -> 328 us.
#include <algorithm>

#include "common.hpp"
#include "device_util.hpp"
#include "q8.hpp"

namespace tvara_amd {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr float kThreshold = 8.0f;
constexpr int kKeys = 64;
constexpr int kRowsPerGroup = 128;  // query rows of a workgroup
constexpr int kBufferWord3 = 0x00020000;  // gfx9 buffer descriptor, dword 3

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

template <int D, int NT, bool kQ8>
__global__ __launch_bounds__(64 * kRowsPerGroup / (16 * NT), 2) void prefill_f32_kernel(const PrefillArgs a) {
    constexpr int W = kRowsPerGroup / (16 * NT);  // waves
    constexpr int C = D / 16, H = D / 64;         // 16-column chunks, 64-column halves
    constexpr int P = D + 4;                      // LDS pitch in floats: 16 rows' 16-byte reads hit every bank once
    constexpr int LPR = D / 4;                    // staging lanes per key row
    constexpr int KPP = 64 * W / LPR;             // keys per staging pass
    constexpr int SP = kKeys / KPP;               // staging passes per tile
    static_assert(D == 64 || D == 128, "head_dim 64 or 128");
    static_assert(SP * KPP == kKeys && KPP <= 16, "a pass lies within one block");
    __shared__ __attribute__((aligned(16))) float klds[2][kKeys * P];
    __shared__ __attribute__((aligned(16))) float vlds[2][kKeys * P];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, r16 = lane & 15;
    const int G = a.group, PW = 16 * NT / G, QT = W * PW;  // positions per wave and workgroup
    // the plan's work list (heaviest first within each XCD)
    const int4 sd = a.work[2 * blockIdx.x], wk = a.work[2 * blockIdx.x + 1];
    const int start = sd.y, nrows = sd.z, kh = wk.x & 0xffff, split = wk.x >> 16, q0 = wk.y, kt0 = wk.z;
    if (!nrows) return;  // the list's padding
    const int kmax = start + min(q0 + QT, nrows);
    const int ntiles = wk.w;
    const int pw0 = q0 + wave * PW;
    const int wave_kmax = pw0 < nrows ? start + min(pw0 + PW, nrows) : 0;
    const int kvw = a.lay.kv_width;
    const int32_t* tab = a.tables + sd.x;

    // this lane's row of each row tile: position, head, last visible key
    int pos[NT], head[NT], lim[NT];
    bool live[NT];
    f32x4 q[NT][C];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int r = 16 * nt + r16;
        pos[nt] = pw0 + r / G;
        head[nt] = kh * G + r % G;
        live[nt] = r < PW * G && pos[nt] < nrows;
        lim[nt] = live[nt] ? start + pos[nt] : start;  // (padding rows meet no key that may be stale)
        const float* qp = a.q + (static_cast<size_t>(sd.w + pos[nt]) * a.heads + head[nt]) * D + 4 * g;
#pragma unroll
        for (int c = 0; c < C; ++c)
            q[nt][c] = live[nt] ? *reinterpret_cast<const f32x4*>(qp + 16 * c) : f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // ---- staging, as in the bf16 tiles: a wave's rows of a pass lie in one
    // block, whose id is wave-uniform; ids are loaded a tile ahead of the rows
    const int skey = tid / LPR, col = 4 * (tid % LPR);
    const int wkey = __builtin_amdgcn_readfirstlane(skey);
    const int tpb = a.lay.tpb, tsh = __builtin_ctz(static_cast<unsigned>(tpb));
    const unsigned roff =
        static_cast<unsigned>(kQ8 ? skey * D + col : (skey * kvw + col) * static_cast<int>(sizeof(float)));
    const unsigned soff = static_cast<unsigned>(tpb * D + (skey * (D / 32) + col / 32) * 2);
    const int kvh = kh / a.kv_share;
    const size_t kbytes = kQ8 ? static_cast<size_t>(a.layer) * 2 * a.lay.section + static_cast<size_t>(kvh) * a.lay.head_bytes
                              : (static_cast<size_t>(a.layer) * 2 * tpb * kvw + static_cast<size_t>(kvh) * D) * sizeof(float);
    const int vsec = static_cast<int>(kQ8 ? a.lay.section : static_cast<size_t>(tpb) * kvw * sizeof(float));
    const int brange = static_cast<int>(a.lay.stride - kbytes);
    f32x4 kreg[SP], vreg[SP];
    int bid[SP];
    // keys past the workgroup's reach read the last reachable block (in
    // bounds, possibly stale): their scores are masked and their V zeroed
    auto tabload = [&](int kt) {
#pragma unroll
        for (int p = 0; p < SP; ++p) bid[p] = tab[min(kt * kKeys + KPP * p + wkey, kmax - 1) >> tsh];
    };
    auto gload = [&](int kt) {
#pragma unroll
        for (int p = 0; p < SP; ++p) {
            const int base = (kt * kKeys + KPP * p) & (tpb - 1);  // the pass's first slot in its block
            const int rso = base * (kQ8 ? D : kvw * static_cast<int>(sizeof(float))), sso = base * (D / 32) * 2;
            const char* blk =
                a.pool + static_cast<size_t>(__builtin_amdgcn_readfirstlane(bid[p])) * a.lay.stride + kbytes;
            const __amdgpu_buffer_rsrc_t r =
                __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(blk), 0, brange, kBufferWord3);
            if constexpr (kQ8) {  // four int8 and their scale's bits, dequantised when staged
                const unsigned kq = __builtin_amdgcn_raw_buffer_load_b32(r, roff, rso, 0);
                const unsigned ks = __builtin_amdgcn_raw_buffer_load_b16(r, soff, sso, 0);
                const unsigned vq = __builtin_amdgcn_raw_buffer_load_b32(r, roff, vsec + rso, 0);
                const unsigned vs = __builtin_amdgcn_raw_buffer_load_b16(r, soff, vsec + sso, 0);
                kreg[p] = f32x4{__builtin_bit_cast(float, kq), __builtin_bit_cast(float, ks), 0.f, 0.f};
                vreg[p] = f32x4{__builtin_bit_cast(float, vq), __builtin_bit_cast(float, vs), 0.f, 0.f};
            } else {
                kreg[p] = __builtin_amdgcn_raw_buffer_load_b128(r, roff, rso, 0);
                vreg[p] = __builtin_amdgcn_raw_buffer_load_b128(r, roff, vsec + rso, 0);
            }
        }
    };
    auto values = [](f32x4 x) {  // Q8_0: d * q, as dequantize_q8_0
        if constexpr (kQ8) {
            const float x0 = x[0], x1 = x[1];  // (a bit cast of a vector element reads element 0)
            const uint32_t w = __builtin_bit_cast(uint32_t, x0);
            const float d = half_bits_to_float(static_cast<uint16_t>(__builtin_bit_cast(uint32_t, x1)));
            return f32x4{sbyte_to_float<0>(w) * d, sbyte_to_float<1>(w) * d, sbyte_to_float<2>(w) * d,
                         sbyte_to_float<3>(w) * d};
        } else {
            return x;
        }
    };
    auto lstore = [&](int kt, int buf) {
#pragma unroll
        for (int p = 0; p < SP; ++p) {
            const int at = (KPP * p + skey) * P + col;
            f32x4 v = values(vreg[p]);
            if (kt * kKeys + KPP * p + skey >= kmax) v = f32x4{0.f, 0.f, 0.f, 0.f};
            *reinterpret_cast<f32x4*>(&klds[buf][at]) = values(kreg[p]);
            *reinterpret_cast<f32x4*>(&vlds[buf][at]) = v;
        }
    };

    f32x4 acc[4 * H][NT];  // output tile (h, j) at 4h + j
#pragma unroll
    for (int dt = 0; dt < 4 * H; ++dt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[dt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m[NT], l[NT], nonfinite = 0.f;  // nonfinite: 0, or NaN once a score is not finite
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        m[nt] = -INFINITY;
        l[nt] = 0.f;
    }

    auto compute = [&](int kt, int buf) {
        const int kbase = kt * kKeys;
        if (kbase >= wave_kmax) return;
        const float* kl = klds[buf] + r16 * P + 4 * g;
        const float* vl = vlds[buf] + 4 * g * P + 4 * r16;
        f32x4 s[4][NT];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            f32x4 t[C][NT];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const f32x4 kk = *reinterpret_cast<const f32x4*>(kl + 16 * mt * P + 16 * c);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) t[c][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        t[c][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[i], q[nt][c][i], t[c][nt], 0, 0, 0);
            }
#pragma unroll
            for (int w = C / 2; w >= 1; w /= 2)
#pragma unroll
                for (int c = 0; c < w; ++c)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) t[c][nt] += t[c + w][nt];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) s[mt][nt] = t[0][nt];
        }
        const bool diagonal = kbase + kKeys - 1 > start + pw0;  // some row's limit lies in the tile
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float mx = -INFINITY;
#pragma unroll
            for (int mt = 0; mt < 4; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float x = s[mt][nt][i];
                    const bool seen = !diagonal || kbase + 16 * mt + 4 * g + i <= lim[nt];
                    nonfinite = fmaf(seen ? x : 0.f, 0.f, nonfinite);
                    s[mt][nt][i] = seen ? x : -INFINITY;
                    mx = fmaxf(mx, s[mt][nt][i]);
                }
            mx *= a.qscale;
            // raise the running maximum on the first tile with keys that a row
            // sees and where a tile exceeds it by more than the threshold
            if (__any(mx > m[nt] + kThreshold)) {
                const float mn = fmaxf(m[nt], cross_row_max(mx));
                const float alpha = m[nt] == -INFINITY ? 0.f : fast_exp2(m[nt] - mn);
                m[nt] = mn;
                l[nt] *= alpha;
#pragma unroll
                for (int dt = 0; dt < 4 * H; ++dt) acc[dt][nt] *= alpha;
            }
            const float base = m[nt] == -INFINITY ? 0.f : m[nt];  // (no key seen yet: probabilities 0)
            float sum = 0.f;
#pragma unroll
            for (int mt = 0; mt < 4; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float p = fast_exp2(fmaf(s[mt][nt][i], a.qscale, -base));
                    s[mt][nt][i] = p;
                    sum += p;
                }
            l[nt] += sum;
        }
        // A row must not meet the values of keys it does not see: 0 times a
        // value that is not finite would reach it as NaN.  Tiles on the
        // diagonal look for such values and, if there are any, add the tile's
        // keys one by one.
        bool plain = true;
        if (diagonal) {
            float t = 0.f;
#pragma unroll 1
            for (int key = 0; key < 16; ++key)
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const f32x4 v = *reinterpret_cast<const f32x4*>(vlds[buf] + (16 * g + key) * P + 64 * h + 4 * r16);
#pragma unroll
                    for (int j = 0; j < 4; ++j) t = fmaf(v[j], 0.f, t);
                }
            plain = !__any(t != 0.f);  // t is 0 or NaN
        }
#pragma unroll
        for (int hh = 0; hh < 2 * H; ++hh) {
            const int h = hh / 2, m0 = hh % 2 * 2;  // output half, key half
            f32x4 part[4][NT];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) part[j][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (plain) {
#pragma unroll
                for (int mt = m0; mt < m0 + 2; ++mt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const f32x4 v = *reinterpret_cast<const f32x4*>(vl + (16 * mt + i) * P + 64 * h);
#pragma unroll
                        for (int j = 0; j < 4; ++j)
#pragma unroll
                            for (int nt = 0; nt < NT; ++nt)
                                part[j][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j], s[mt][nt][i], part[j][nt], 0, 0, 0);
                    }
            } else {
#pragma unroll
                for (int mt = m0; mt < m0 + 2; ++mt)
#pragma unroll 1
                    for (int e = 0; e < 16; ++e) {  // key 16mt + e: lane group e/4, element e%4
                        const int i = e & 3;
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt) {
                            const float own = i == 0 ? s[mt][nt][0] : i == 1 ? s[mt][nt][1] : i == 2 ? s[mt][nt][2] : s[mt][nt][3];
                            const float p = __shfl(own, r16 + 16 * (e >> 2));
                            const bool seen = kbase + 16 * mt + e <= lim[nt];
#pragma unroll
                            for (int o = 0; o < 4; ++o) {
                                const f32x4 v =
                                    *reinterpret_cast<const f32x4*>(vlds[buf] + (16 * mt + e) * P + 64 * h + 4 * (4 * g + o));
#pragma unroll
                                for (int j = 0; j < 4; ++j)
                                    part[j][nt][o] = seen ? fmaf(p, v[j], part[j][nt][o]) : part[j][nt][o];
                            }
                        }
                    }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) acc[4 * h + j][nt] += part[j][nt];
        }
    };

    auto tile = [&](int t) { return min(t, ntiles - 1); };
    tabload(kt0);
    gload(kt0);
    tabload(tile(kt0 + 1));
    lstore(kt0, 0);
    __syncthreads();
    for (int kt = kt0; kt < ntiles; ++kt) {
        const int buf = (kt - kt0) & 1;
        gload(tile(kt + 1));
        tabload(tile(kt + 2));
        compute(kt, buf);
        lstore(tile(kt + 1), buf ^ 1);
        __syncthreads();
    }

    if (__any(nonfinite != 0.f) && lane == 0) *a.err = 1;
    // the workgroup's first row's (its rows have as many runs, in slots that follow)
    const int2 runs = a.row_runs ? a.row_runs[sd.w + q0] : make_int2(0, 1);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const float total = cross_row_sum(l[nt]);
        if (!live[nt]) continue;
        // lane group g, element i of tile (h, j): column 64h + 16g + 4i + j
        size_t at = static_cast<size_t>(sd.w + pos[nt]) * a.heads + head[nt];
        float* o = a.out + at * D + 16 * g;
        float inv = total;
        if (runs.y > 1) {
            at = static_cast<size_t>(runs.x + (pos[nt] - q0) * runs.y + split) * a.heads + head[nt];
            if (g == 0) *reinterpret_cast<float2*>(a.part_ml + 2 * at) = make_float2(m[nt], total);
            if (m[nt] == -INFINITY) continue;  // no key of this run: not used either
            o = a.part_acc + at * D + 16 * g;
            inv = 1.f;
        }
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<float4*>(o + 64 * h + 4 * i) =
                    make_float4(acc[4 * h][nt][i] / inv, acc[4 * h + 1][nt][i] / inv, acc[4 * h + 2][nt][i] / inv,
                                acc[4 * h + 3][nt][i] / inv);
    }
}

// The runs of a (row, head) combined by log-sum-exp in order; a thread per
// four columns, all loads of a round of runs requested together.  Runs in which
// the row sees no key (maximum -inf) are left out; a row of one run was written
// by its workgroup.
template <int D>
__global__ __launch_bounds__(256) void prefill_merge_kernel(const PrefillArgs a) {
    constexpr int U = 8;
    const size_t n = static_cast<size_t>(a.total_rows) * a.heads;
    const size_t t = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x, at = t / (D / 4);
    if (at >= n) return;
    const int c = 4 * static_cast<int>(t % (D / 4));
    const int2 runs = a.row_runs[at / a.heads];
    const int splits = runs.y;
    if (splits == 1) return;
    float M = -INFINITY, L = 0.f;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < splits; s0 += U) {
        float2 ml[U];
        f32x4 x[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const size_t p = static_cast<size_t>(runs.x + min(s0 + k, splits - 1)) * a.heads + at % a.heads;
            ml[k] = *reinterpret_cast<const float2*>(a.part_ml + 2 * p);
            x[k] = *reinterpret_cast<const f32x4*>(a.part_acc + p * D + c);
        }
        float mc = M;
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (s0 + k < splits) mc = fmaxf(mc, ml[k].x);
        if (mc == -INFINITY) continue;
        const float scale = fast_exp2(M - mc);  // 0 while M is -inf
        L *= scale;
        sum *= scale;
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const bool some = s0 + k < splits && ml[k].x != -INFINITY;
            const float w = some ? fast_exp2(ml[k].x - mc) : 0.f;
            L = fmaf(w, some ? ml[k].y : 0.f, L);
#pragma unroll
            for (int i = 0; i < 4; ++i) sum[i] = some ? fmaf(w, x[k][i], sum[i]) : sum[i];
        }
        M = mc;
    }
    const f32x4 out = sum / L;
    // (a.err null: the f32 tiles, whose values may be anything)
    if (a.err && !(__builtin_isfinite(out[0]) && __builtin_isfinite(out[1]) && __builtin_isfinite(out[2]) &&
                   __builtin_isfinite(out[3])))
        *a.err = 1;
    *reinterpret_cast<f32x4*>(a.out + at * D + c) = out;
}

}  // namespace

void launch_prefill_f32(const PrefillArgs& a, hipStream_t s) {
    if (!prefill_bf16_supported(a.lay, a.group))
        throw std::invalid_argument(
            "f32 prefill tiles need f32 or Q8_0 blocks of 16 to 1,024 tokens (a power of two, under 2 GiB), head_dim 64 "
            "or 128, and a GQA slice of 1-8 heads");
    if (a.workgroups <= 0) return;
    const bool q8 = a.lay.format == kQ8, wide = a.lay.head_dim == 128;
    const dim3 grid(a.workgroups);
    // 32 rows a wave at head_dim 64; 16 at 128, where the accumulators of 32
    // would not leave two waves a SIMD
    if (wide)
        launch("paged_prefill_f32", q8 ? prefill_f32_kernel<128, 1, true> : prefill_f32_kernel<128, 1, false>, grid,
               dim3(512), 0, s, a);
    else
        launch("paged_prefill_f32", q8 ? prefill_f32_kernel<64, 2, true> : prefill_f32_kernel<64, 2, false>, grid,
               dim3(256), 0, s, a);
    TVARA_HIP(hipGetLastError());
    if (a.row_runs) {
        PrefillArgs m = a;
        m.err = nullptr;
        launch_prefill_merge(m, s);
    }
}

void launch_prefill_merge(const PrefillArgs& a, hipStream_t s) {
    const size_t threads = static_cast<size_t>(a.total_rows) * a.heads * (a.lay.head_dim / 4);
    launch("paged_prefill_merge", a.lay.head_dim == 128 ? prefill_merge_kernel<128> : prefill_merge_kernel<64>,
           dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, s, a);
    TVARA_HIP(hipGetLastError());
}

int prefill_f32_positions(const BlockLayout& lay, int group) {
    return lay.head_dim == 128 ? 8 * (16 / group) : 4 * (32 / group);
}

// Tiles or rows: whichever the rates below put ahead.  A tile launch costs 10 us
// and 6.4 us of a CU per workgroup and key tile (5 where two workgroups share
// it, at head_dim 64), for however few of its 128 rows are there.  The decode
// kernels pay for every row, whose keys they read again, from L2: at 8 TFLOP/s
// per query head of the group up to 26 (Q8_0 16 up to 55; 10-40 and 12-60
// measured, as the rows' splits happen to share an XCD's L2), and at 0.7 of that
// once a sequence's keys are past the caches.  MI355X, tiles against rows, us, 32 x
// 8 heads of 64 in f32: one row after 130,000 tokens 421 against 106, 16 rows 429
// against 1,233; 64 sequences after 4,000, one row each 444 against 174, 8 rows
// 450 against 652; 8 after 16,000, 4 rows 413 against 326, 16 rows 420 against
// 431.  Over 1,163 chunks of 1-1,000 rows in both formats the rule's choice is within
// 0.4% of the faster one in the geometric mean and 1.41 times as long at worst,
// always tiles 6.3% and 4.9 times.  Chunks under 0.7 GFLOP, 3 over Q8_0, are rows: tiles
// against rows 25 against 26 us at 0.54, 32 against 31.5 at 0.66, 31 against 44
// at 1.0; over Q8_0 70 against 72 at 3.2.
//
// Key splits: one workgroup per CU where the chunk alone gives fewer (64 rows
// after 4,000 tokens, head_dim 64: 40 us in 256 units of work, 44 in 512;
// 256 rows after 1,000 at 128: 72, 89, 103 in 1,024), and units of a quarter of
// a CU's share up to 1,024 workgroups, where whole rounds of unequal
// workgroups leave a tail (six chunks of 33-700 tokens: 328 us against 431
// unsplit).  At least two tiles a split.  Even batches of more workgroups are
// faster unsplit, so they are split only where the longest would outlast a CU's
// whole share: 33 rows after 130,000 tokens beside 40 prompts of 128 take 2,598
// us row by row, 12,738 unsplit and 862 split, 16 after 16,000 beside ten of 512
// 374, 1,491 and 200.
F32TileShape prefill_f32_shape(const BlockLayout& lay, int group, size_t n, const size_t* start, const size_t* rows) {
    const bool q8 = lay.format == kQ8;
    const size_t qt = prefill_f32_positions(lay, group);
    size_t wgs = 0, work = 0, read = 0, longest = 0;  // read: key tiles, as the causal mask leaves them
    double flops = 0, row_us = 5;
    const double rate = 1e6 * (q8 ? std::min(55, 16 * group) : std::min(26, 8 * group));  // flops per us
    const double token_bytes = 2.0 * lay.kv_heads * lay.head_dim * (q8 ? 34.0 / 32.0 : 4.0);
    for (size_t i = 0; i < n; ++i) {
        const size_t tiles = (start[i] + rows[i] + kKeys - 1) / kKeys, w = (rows[i] + qt - 1) / qt;
        wgs += w;
        work += w * tiles;
        longest = std::max(longest, tiles);
        for (size_t q = qt; q < rows[i] + qt; q += qt) read += (start[i] + std::min(q, rows[i]) + kKeys - 1) / kKeys;
        const double f = 4.0 * lay.kv_heads * group * lay.head_dim * rows[i] * (start[i] + 0.5 * rows[i]);
        flops += f;
        row_us += f / (token_bytes * start[i] > 100e6 ? 0.7 * rate : rate);
    }
    work *= lay.kv_heads;
    wgs *= lay.kv_heads;
    const double tile_us = 10 + (lay.head_dim == 64 && wgs >= 256 ? 5 : 6.4) / 256 * read * lay.kv_heads;
    F32TileShape f{};
    f.use = flops >= (q8 ? 3e9 : 0.7e9) && tile_us < row_us;
    f.splits = 1;
    f.split_tiles = static_cast<int>(longest);
    if (wgs < 1024 || longest * 256 > work) {
        const size_t units = wgs < 256 ? 256 : 1024;
        const size_t per = std::max<size_t>(2, (work + units - 1) / units);
        f.split_tiles = static_cast<int>(std::min(per, longest));
        f.splits = static_cast<int>((longest + f.split_tiles - 1) / f.split_tiles);
    }
    return f;
}

}  // namespace tvara_amd
