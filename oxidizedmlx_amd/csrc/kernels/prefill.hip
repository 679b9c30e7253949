// prefill.hip — the kernels that run many prompt positions of a decoder-only
// model at once (the caller is csrc/decoder.cpp). A pass takes cp consecutive
// positions t0 .. t0+cp-1 of every sequence; row r = b*cp + p is position
// t0 + p of sequence b. Per layer:
//   prefill_rms      rms of every row of the residual stream
//   gemm<QKV,norm>   q; k and v into the KV cache
//   prefill_attn     attention of every row over the cache (positions 0..t)
//   gemm<RESID>      x += o·Wo^T + bo
//   prefill_rms, gemm<SILU,norm>, gemm<RESID>   the MLP
// and, where the caller wants them, gemm<LOGITS,norm> with the rows' argmax.
//
// Every result has the bits that the one-position step (decode.hip) gives:
// the same f32 activations as three bf16 planes against the same bf16
// weights on the same MFMA, the same k-slices with each plane's accumulator
// of its own, added as hi + (mid + lo) and in slice order, the same order of
// every sum of squares, score, softmax and P·V. A prompt position therefore
// costs a share of one pass over the weights instead of a step of its own
// (62 dependent launches for 12 layers, ~330 us), and which of the two ran
// cannot be told from the results.
#include <algorithm>

#include "../common.hpp"
#include "../kernels.hpp"
#include "decode_common.hpp"
#include "device_math.hpp"

#pragma clang fp contract(off)

namespace mlxhip {
namespace {

using namespace dec;
using dev::div_by;
using dev::shared_divisor;
using dev::sigmoid_ref;
using dev::wave_max;
using dev::wave_sum;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Rows' planes in the MFMA B operand's fragment order, as the weights are in
// the A operand's: 16-row tiles, each a run of 32-k steps of 64 lanes x 8
// bf16, lane = row % 16 + 16 * ((k % 32) / 8). Element (row, k) of a plane:
__device__ inline int64_t frag_index(int64_t row, int k, int K) {
    return (((row / 16) * (K / KSTEP) + k / KSTEP) * WAVE + (row % 16) + 16 * ((k % KSTEP) / 8)) * 8 + k % 8;
}

// Four consecutive values (k a multiple of 4) into the planes.
__device__ inline void store_split4(uint16_t* xs, int64_t plane, int64_t row, int k, int K, const f32x4& v) {
    uint16_t t[4][3];
#pragma unroll
    for (int j = 0; j < 4; ++j) split_terms(v[j], t[j]);
    uint16_t* at = xs + frag_index(row, k, K);
#pragma unroll
    for (int q = 0; q < 3; ++q)
        *reinterpret_cast<uint2*>(at + q * plane) = make_uint2((uint32_t)t[0][q] | ((uint32_t)t[1][q] << 16),
                                                               (uint32_t)t[2][q] | ((uint32_t)t[3][q] << 16));
}

// ── embeddings of the pass's tokens: x and its planes ──────────────────────
__global__ __launch_bounds__(256) void prefill_embed_kernel(const uint16_t* __restrict__ emb,
                                                            const int* __restrict__ tokens, float* __restrict__ x,
                                                            uint16_t* __restrict__ xs, int64_t plane, int d, int vocab,
                                                            int batch, int cp, int t0) {
    const int row = blockIdx.x, b = row / cp, t = t0 + row % cp;
    int tok = tokens[(int64_t)t * batch + b];
    tok = tok < 0 ? 0 : (tok > vocab - 1 ? vocab - 1 : tok);
    const uint16_t* src = emb + (int64_t)tok * d;
    for (int k = 4 * threadIdx.x; k < d; k += 4 * blockDim.x) {
        const uint2 e = *reinterpret_cast<const uint2*>(src + k);
        const f32x4 v = {bf16_f32(e.x & 0xFFFFu), bf16_f32(e.x >> 16), bf16_f32(e.y & 0xFFFFu), bf16_f32(e.y >> 16)};
        *reinterpret_cast<f32x4*>(x + (int64_t)row * d + k) = v;
        store_split4(xs, plane, row, k, d, v);
    }
}

// ── sqrt(mean(x^2) + eps) of every row, and its reciprocal ─────────────────
// One wave per row. The step's order (gemv_kernel): units of 8 values, lane
// l the units l, l + 64, ..., then the butterfly.
constexpr int RMS_ROWS = 4;
__global__ __launch_bounds__(RMS_ROWS* WAVE) void prefill_rms_kernel(const float* __restrict__ x,
                                                                     float2* __restrict__ rms, int rows, int d,
                                                                     float eps) {
    const int row = blockIdx.x * RMS_ROWS + threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    if (row >= rows) return;
    const float* xr = x + (int64_t)row * d;
    float ss = 0.0f;
    for (int c = lane; c < d / 8; c += WAVE) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(xr + 8 * c);
        const f32x4 b = *reinterpret_cast<const f32x4*>(xr + 8 * c + 4);
        float u = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) u += a[j] * a[j];
#pragma unroll
        for (int j = 0; j < 4; ++j) u += b[j] * b[j];
        ss += u;
    }
    ss = wave_sum(ss);
    if (lane == 0) {
        float v = sqrtf(ss / (float)d + eps), r;
        shared_divisor(v, r);
        rms[row] = make_float2(v, r);
    }
}

// ── Y[rows, N] = X[rows, K] · W[N, K]^T ────────────────────────────────────
//
// One wave computes FT feature tiles x RT row tiles (16 x 16 each) over all
// of K; the waves of a workgroup take neighbouring feature tiles of the same
// rows. Both operands are stored in fragment order, so a wave loads its
// fragments (1 KB of consecutive memory each) straight into registers, PD
// steps ahead: no LDS and no barrier in the loop. K is not split over waves:
// the step's k-slices are summed one after another, which fixes their order.
// Bound by the fragments' way from L2: (FT + 3 RT) KB per step against
// 3 FT RT MFMAs, so the wide shape is taken as soon as its waves fill the
// chip, and a narrow one spreads few rows over more SIMDs.
template <int EPI, int FT, int RT, int PD>
__global__ __launch_bounds__(256) void prefill_gemm_kernel(PrefillGemm p, int slice_steps, int row_groups) {
    const int K = p.k, N = p.n, S = K / KSTEP;
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, nw = blockDim.x / WAVE;
    // Consecutive workgroups run on different XCDs: each XCD takes a
    // contiguous range, the rows of one feature group first, so a weight
    // comes into one XCD's L2.
    const unsigned L = blockIdx.x, G = gridDim.x;
    const unsigned wg = G % 8 == 0 ? (L % 8) * (G / 8) + L / 8 : L;
    const int rg = (int)(wg % (unsigned)row_groups), fg = (int)(wg / (unsigned)row_groups);
    const int ntiles = (N + TILE_N - 1) / TILE_N;
    const int ft0 = (fg * nw + wave) * FT;
    if (ft0 >= ntiles) return;
    const int rt0 = rg * RT, rtiles = (p.rows + 15) / 16;
    // Tiles past the end load the last one's fragments and store nothing.
    const u32x4* wp[FT];
    const u32x4* xp[RT][3];
#pragma unroll
    for (int f = 0; f < FT; ++f)
        wp[f] = reinterpret_cast<const u32x4*>(p.w) + (int64_t)min(ft0 + f, ntiles - 1) * S * WAVE + lane;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int q = 0; q < 3; ++q)
            xp[r][q] = reinterpret_cast<const u32x4*>(p.xs + q * p.plane) + (int64_t)min(rt0 + r, rtiles - 1) * S * WAVE +
                       lane;
    u32x4 a[PD][FT], b[PD][RT][3];
    auto load = [&](int u, int s) {
        const int64_t o = (int64_t)min(s, S - 1) * WAVE;
#pragma unroll
        for (int f = 0; f < FT; ++f) a[u][f] = wp[f][o];
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int q = 0; q < 3; ++q) b[u][r][q] = xp[r][q][o];
    };
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc[FT][RT][3], sum[FT][RT];
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            sum[f][r] = f32x4{-0.0f, -0.0f, -0.0f, -0.0f};  // -0 + v is v: the first slice as it is
#pragma unroll
            for (int q = 0; q < 3; ++q) acc[f][r][q] = zero;
        }
    auto end_slice = [&]() {
#pragma unroll
        for (int f = 0; f < FT; ++f)
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                f32x4(&c)[3] = acc[f][r];
#pragma unroll
                for (int j = 0; j < 4; ++j) sum[f][r][j] = sum[f][r][j] + (c[0][j] + (c[1][j] + c[2][j]));
                c[0] = c[1] = c[2] = zero;
            }
    };
#pragma unroll
    for (int u = 0; u < PD; ++u) load(u, u);
    int left = slice_steps;
    for (int s0 = 0; s0 < S; s0 += PD) {
#pragma unroll
        for (int u = 0; u < PD; ++u) {
            if (s0 + u < S) {
#pragma unroll
                for (int f = 0; f < FT; ++f)
#pragma unroll
                    for (int r = 0; r < RT; ++r)
#pragma unroll
                        for (int q = 0; q < 3; ++q)
                            acc[f][r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                __builtin_bit_cast(bf16x8, a[u][f]), __builtin_bit_cast(bf16x8, b[u][r][q]),
                                acc[f][r][q], 0, 0, 0);
                load(u, s0 + u + PD);
                if (--left == 0) {
                    end_slice();
                    left = slice_steps;
                }
            }
        }
    }
    if (left != slice_steps) end_slice();  // a last slice that is shorter

    // Lane l holds row l % 16 and the features 4 * (l / 16) + j, j < 4, of each tile.
    const int kg = lane / 16;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int row = (rt0 + r) * 16 + lane % 16;
        const bool live = row < p.rows;
        const int rc = live ? row : 0, bi = rc / p.cp, t = p.t0 + rc % p.cp;
        float2 rms = make_float2(1.0f, 1.0f);
        if (EPI != PREFILL_RESID) rms = p.rms[rc];
        uint64_t key = 0;
#pragma unroll
        for (int f = 0; f < FT; ++f) {
            const int n = (ft0 + f) * TILE_N + 4 * kg;
            f32x4 v = sum[f][r];
            if constexpr (EPI != PREFILL_RESID)
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = div_by(v[j], rms.x, rms.y);
            if constexpr (EPI == PREFILL_LOGITS) {
                const bool on = live && t < p.t_end;
                float* lo = p.out ? p.out + (int64_t)bi * p.ldo + (int64_t)t * N + n : nullptr;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (on && n + j < N) {
                        if (lo) lo[j] = v[j];
                        key = max_u64(key, logit_key(v[j], n + j));
                    }
                }
            } else {
                if (!live || ft0 + f >= ntiles) continue;  // N is a multiple of 16 here
                const uint2 bb = *reinterpret_cast<const uint2*>(p.bias + n);
                const f32x4 bv = {bf16_f32(bb.x & 0xFFFFu), bf16_f32(bb.x >> 16), bf16_f32(bb.y & 0xFFFFu),
                                  bf16_f32(bb.y >> 16)};
                v = v + bv;
                if constexpr (EPI == PREFILL_SILU) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = v[j] * sigmoid_ref(v[j]);
                    store_split4(p.outs, p.oplane, row, n, N, v);
                } else if constexpr (EPI == PREFILL_RESID) {
                    f32x4* o = reinterpret_cast<f32x4*>(p.out + (int64_t)row * p.ldo + n);
                    v = *o + v;
                    *o = v;
                    store_split4(p.outs, p.oplane, row, n, N, v);
                } else {  // PREFILL_QKV
                    const int seg = n / p.dmodel, nn = n - seg * p.dmodel;
                    const int h = nn / p.head_dim, dd = nn - h * p.head_dim;
                    const int64_t bh = (int64_t)bi * p.heads + h;
                    if (seg == 0)
                        *reinterpret_cast<f32x4*>(p.out + (int64_t)row * p.ldo + nn) = v;
                    else if (seg == 1)
#pragma unroll
                        for (int j = 0; j < 4; ++j) p.kc[(bh * p.head_dim + dd + j) * p.tmax + t] = v[j];
                    else
                        *reinterpret_cast<f32x4*>(p.vc + (bh * p.tmax + t) * p.head_dim + dd) = v;
                }
            }
        }
        if constexpr (EPI == PREFILL_LOGITS) {
            key = max_u64(key, shfl_xor_u64(key, 16));
            key = max_u64(key, shfl_xor_u64(key, 32));
            if (lane < 16 && live) p.part[(int64_t)(ft0 / FT) * p.rows + row] = key;
        }
    }
}

// The rows' argmax over the LM head's partial maxima: a workgroup takes 16
// rows, 16 threads a row.
__global__ __launch_bounds__(256) void prefill_argmax_kernel(const uint64_t* __restrict__ part, int groups, int rows,
                                                             int* __restrict__ argmax_out, int batch, int cp, int t0,
                                                             int t_end) {
    __shared__ uint64_t sm[16][16];
    const int rl = threadIdx.x % 16, gl = threadIdx.x / 16;
    const int row = blockIdx.x * 16 + rl;
    uint64_t m = 0;
    if (row < rows)
        for (int g = gl; g < groups; g += 16) m = max_u64(m, part[(int64_t)g * rows + row]);
    sm[gl][rl] = m;
    __syncthreads();
    if (gl == 0 && row < rows) {
        for (int g = 1; g < 16; ++g) m = max_u64(m, sm[g][rl]);
        const int b = row / cp, t = t0 + row % cp;
        if (t < t_end) argmax_out[(int64_t)t * batch + b] = (int)(0xFFFFFFFFu - (uint32_t)m);
    }
}

// ── attention of the pass's rows over the KV cache ─────────────────────────
// One 256-thread workgroup per (sequence, head) and Q consecutive queries.
// Per query this is decode_attn_kernel's arithmetic, step for step (position
// j's score on thread j % 256, each wave's maximum and sum of exp over its
// positions, P·V over position groups added in order); the K column and the V
// rows that a thread loads serve all Q queries.
constexpr int ATT_BLOCK = 256;
constexpr int ATT_WAVES = ATT_BLOCK / WAVE;

template <int HD, int Q>
__global__ __launch_bounds__(ATT_BLOCK) void prefill_attn_kernel(const float* __restrict__ q,
                                                                 const float* __restrict__ kc,
                                                                 const float* __restrict__ vc, uint16_t* __restrict__ os,
                                                                 int64_t plane, int heads, int tmax, float scale, int t0,
                                                                 int cp, int sld) {
    constexpr int C4 = HD / 4, G = ATT_BLOCK / C4, VCH = 16;
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float* s = sm;                 // [Q][sld] scores
    float* part = s + Q * sld;     // [Q][G][HD] P·V partials
    __shared__ float slot[Q][2 * ATT_WAVES];  // (max, sum) of each wave
    const int bh = blockIdx.x, b = bh / heads, h = bh % heads, d = heads * HD;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    const float* kT = kc + (int64_t)bh * HD * tmax;
    const float* vv = vc + (int64_t)bh * tmax * HD;
    // The longest queries first: the last round is then the shortest.
    const int p0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * Q;
    const int nq = min(Q, cp - p0);
    const int T = t0 + p0 + nq;       // positions the last query sees; query i sees T - nq + 1 + i
    const int T0 = t0 + p0 + 1;       // and all of them see these
    int Ti[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i) Ti[i] = t0 + p0 + min(i, nq - 1) + 1;
    // The queries go through LDS, where every lane reads the same address
    // (through the scalar cache their 4 x 64 values spilled the SGPRs); the
    // partials of P·V take the place later.
    float* ql = part;  // [Q][HD]
    for (int e = tid; e < Q * HD; e += ATT_BLOCK)
        ql[e] = q[((int64_t)b * cp + p0 + min(e / HD, nq - 1)) * d + h * HD + e % HD];

    const int c = tid % C4, g = tid / C4;
    float4 vr[VCH];
    auto load_v = [&](int j0) {
#pragma unroll
        for (int u = 0; u < VCH; ++u) {
            const int j = min(j0 + u * G, T0 - 1);
            vr[u] = *reinterpret_cast<const float4*>(vv + (int64_t)j * HD + 4 * c);
        }
    };
    load_v(g);
    // A row past T0 is some of the queries' only: not 0 times a V that may have
    // overflowed for the others. At most one of them is this thread's.
    static_assert(Q - 1 <= G, "one row past T0 per position group");
    const int jt = T0 + (g + G - T0 % G) % G;
    float4 vt;
    if constexpr (Q > 1) vt = *reinterpret_cast<const float4*>(vv + (int64_t)min(jt, T - 1) * HD + 4 * c);
    __syncthreads();  // the queries

    constexpr int KCH = HD < 32 ? HD : 32;
    float mloc[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i) mloc[i] = -INFINITY;
    for (int j = tid; j < T; j += ATT_BLOCK) {
        float acc[Q];
#pragma unroll
        for (int i = 0; i < Q; ++i) acc[i] = 0.0f;
        // Not unrolled: the queries of all of HD in registers would spill.
#pragma unroll 1
        for (int d0 = 0; d0 < HD; d0 += KCH) {
            float kv[KCH];
#pragma unroll
            for (int u = 0; u < KCH; ++u) kv[u] = kT[(int64_t)(d0 + u) * tmax + j];
#pragma unroll
            for (int i = 0; i < Q; ++i)
#pragma unroll
                for (int u = 0; u < KCH; u += 4) {
                    const float4 q4 = *reinterpret_cast<const float4*>(ql + i * HD + d0 + u);
                    acc[i] += q4.x * kv[u];
                    acc[i] += q4.y * kv[u + 1];
                    acc[i] += q4.z * kv[u + 2];
                    acc[i] += q4.w * kv[u + 3];
                }
        }
#pragma unroll
        for (int i = 0; i < Q; ++i) {
            if (j < Ti[i]) {
                const float sc = acc[i] * scale;
                s[i * sld + j] = sc;
                mloc[i] = fmaxf(mloc[i], sc);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        const float mw = wave_max(mloc[i]);
        float lloc = 0.0f;
        for (int j = tid; j < Ti[i]; j += ATT_BLOCK) {
            const float e = expf(s[i * sld + j] - mw);
            s[i * sld + j] = e;
            lloc += e;
        }
        const float lw = wave_sum(lloc);
        if (lane == 0) {
            slot[i][2 * wave] = mw;
            slot[i][2 * wave + 1] = lw;
        }
    }
    __syncthreads();
    static_assert(ATT_WAVES == 4, "four wave factors");
    float f[Q][4], l[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        float m = slot[i][0];
#pragma unroll
        for (int w = 1; w < ATT_WAVES; ++w) m = fmaxf(m, slot[i][2 * w]);
#pragma unroll
        for (int w = 0; w < ATT_WAVES; ++w) f[i][w] = slot[i][2 * w] == -INFINITY ? 0.0f : expf(slot[i][2 * w] - m);
        l[i] = ((slot[i][1] * f[i][0] + slot[i][3] * f[i][1]) + slot[i][5] * f[i][2]) + slot[i][7] * f[i][3];
    }
    float4 acc[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i) acc[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int j0 = g; j0 < T0; j0 += G * VCH) {
        if (j0 != g) load_v(j0);
#pragma unroll
        for (int u = 0; u < VCH; ++u) {
            const int j = j0 + u * G;
#pragma unroll
            for (int i = 0; i < Q; ++i) {
                const float pj =
                    j < T0 ? s[i * sld + j] * pick4((j >> 6) & 3, f[i][0], f[i][1], f[i][2], f[i][3]) : 0.0f;
                acc[i].x += pj * vr[u].x;
                acc[i].y += pj * vr[u].y;
                acc[i].z += pj * vr[u].z;
                acc[i].w += pj * vr[u].w;
            }
        }
    }
#pragma unroll
    for (int i = 1; i < Q; ++i) {
        if (jt < Ti[i]) {
            const float pj = s[i * sld + jt] * pick4((jt >> 6) & 3, f[i][0], f[i][1], f[i][2], f[i][3]);
            acc[i].x += pj * vt.x;
            acc[i].y += pj * vt.y;
            acc[i].z += pj * vt.z;
            acc[i].w += pj * vt.w;
        }
    }
#pragma unroll
    for (int i = 0; i < Q; ++i) *reinterpret_cast<float4*>(part + (i * G + g) * HD + 4 * c) = acc[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        if (i < nq && tid < HD) {
            float r = part[i * G * HD + tid];
            for (int gg = 1; gg < G; ++gg) r += part[(i * G + gg) * HD + tid];
            uint16_t t[3];
            split_terms(r / l[i], t);
            uint16_t* at = os + frag_index((int64_t)b * cp + p0 + i, h * HD + tid, d);
#pragma unroll
            for (int k = 0; k < 3; ++k) at[k * plane] = t[k];
        }
    }
}

// ── hand-over to the one-position step ─────────────────────────────────────
// The last prompt position's rows of x become the step's x and planes
// (xs[3][DEC_MAX_BATCH][d]); the position counter names that position.
__global__ __launch_bounds__(256) void prefill_last_kernel(const float* __restrict__ px, int cp, int p,
                                                           float* __restrict__ x, uint16_t* __restrict__ xs, int d,
                                                           int* __restrict__ tctr, int t) {
    const int b = blockIdx.x;
    for (int k = threadIdx.x; k < d; k += blockDim.x) {
        const float v = px[((int64_t)b * cp + p) * d + k];
        x[(int64_t)b * d + k] = v;
        uint16_t tm[3];
        split_terms(v, tm);
#pragma unroll
        for (int q = 0; q < 3; ++q) xs[(int64_t)(q * DEC_MAX_BATCH + b) * d + k] = tm[q];
    }
    if (b == 0 && threadIdx.x == 0) *tctr = t;
}

constexpr int LOGIT_FT = 4;  // feature tiles per wave of the LM head

template <int EPI, int FT, int RT, int PD>
int launch_gemm(const PrefillGemm& p, int slice_steps, hipStream_t s) {
    const int64_t fgroups = ceil_div(ceil_div(p.n, TILE_N), FT), rgroups = ceil_div(ceil_div(p.rows, 16), RT);
    // Waves of one workgroup share their rows' fragments through the CU's
    // cache; fewer per workgroup where that leaves CUs without one.
    int nw = 4;
    while (nw > 1 && ceil_div(fgroups, nw) * rgroups < 256) nw /= 2;
    const int64_t grid = ceil_div(fgroups, nw) * rgroups;
    hipLaunchKernelGGL((prefill_gemm_kernel<EPI, FT, RT, PD>), dim3((unsigned)grid), dim3(nw * WAVE), 0, s, p,
                       slice_steps, (int)rgroups);
    return launch_check("prefill_gemm_kernel");
}

template <int EPI>
int dispatch_gemm(const PrefillGemm& p, int slice_steps, hipStream_t s) {
    // 64 x 32 outputs per wave from two waves per SIMD on, else 32 x 16.
    const int64_t wide = ceil_div(ceil_div(p.n, TILE_N), 4) * ceil_div(ceil_div(p.rows, 16), 2);
    if (EPI == PREFILL_LOGITS || wide >= 1024) {
        if (p.rows > 16) return launch_gemm<EPI, 4, 2, 2>(p, slice_steps, s);
        return launch_gemm<EPI, 4, 1, 4>(p, slice_steps, s);
    }
    return launch_gemm<EPI, 2, 1, 6>(p, slice_steps, s);
}

template <int HD, int Q>
int launch_attn(const float* q, const float* kc, const float* vc, uint16_t* os, int64_t plane, int batch, int heads,
                int tmax, float scale, int t0, int cp, hipStream_t s) {
    const int sld = (t0 + cp + 3) & ~3;
    const size_t lds = ((size_t)Q * sld + (size_t)Q * ATT_BLOCK * 4) * sizeof(float);
    hipLaunchKernelGGL((prefill_attn_kernel<HD, Q>), dim3(batch * heads, (unsigned)ceil_div(cp, Q)), dim3(ATT_BLOCK),
                       lds, s, q, kc, vc, os, plane, heads, tmax, scale, t0, cp, sld);
    return launch_check("prefill_attn_kernel");
}

template <int HD>
int dispatch_attn(const float* q, const float* kc, const float* vc, uint16_t* os, int64_t plane, int batch, int heads,
                  int tmax, float scale, int t0, int cp, hipStream_t s) {
    // Four queries per workgroup while their scores leave room for two
    // workgroups per CU, else one (its scores fit as the step's do).
    constexpr int Q = 4;
    if (((size_t)Q * (t0 + cp + 3) + (size_t)Q * ATT_BLOCK * 4) * sizeof(float) <= 60 * 1024)
        return launch_attn<HD, Q>(q, kc, vc, os, plane, batch, heads, tmax, scale, t0, cp, s);
    return launch_attn<HD, 1>(q, kc, vc, os, plane, batch, heads, tmax, scale, t0, cp, s);
}

}  // namespace

int prefill_part_groups(int n) { return (int)ceil_div(ceil_div(n, TILE_N), LOGIT_FT); }

int prefill_embed(const uint16_t* emb, const int* tokens, float* x, uint16_t* xs, int64_t plane, int d, int vocab,
                  int batch, int cp, int t0, hipStream_t s) {
    hipLaunchKernelGGL(prefill_embed_kernel, dim3(batch * cp), dim3(256), 0, s, emb, tokens, x, xs, plane, d, vocab,
                       batch, cp, t0);
    return launch_check("prefill_embed_kernel");
}

int prefill_rms(const float* x, float2* rms, int rows, int d, float eps, hipStream_t s) {
    hipLaunchKernelGGL(prefill_rms_kernel, dim3((unsigned)ceil_div(rows, RMS_ROWS)), dim3(RMS_ROWS * WAVE), 0, s, x,
                       rms, rows, d, eps);
    return launch_check("prefill_rms_kernel");
}

int prefill_gemm(int epi, const PrefillGemm& p, hipStream_t s) {
    if (p.rows <= 0 || p.cp <= 0 || p.n <= 0 || p.k <= 0 || p.k % KSTEP || (epi != PREFILL_LOGITS && p.n % TILE_N))
        return fail(MLXHIP_ERR_INVALID_ARGUMENT, "prefill gemm: unsupported shape n=%d k=%d rows=%d", p.n, p.k, p.rows);
    int slices = 0, width = 0;
    dec_gemv_slices(p.n, p.k, epi == PREFILL_LOGITS, &slices, &width);
    const int steps = width / KSTEP;
    switch (epi) {
        case PREFILL_QKV: return dispatch_gemm<PREFILL_QKV>(p, steps, s);
        case PREFILL_RESID: return dispatch_gemm<PREFILL_RESID>(p, steps, s);
        case PREFILL_SILU: return dispatch_gemm<PREFILL_SILU>(p, steps, s);
        default: return dispatch_gemm<PREFILL_LOGITS>(p, steps, s);
    }
}

int prefill_argmax(const uint64_t* part, int groups, int rows, int* argmax_out, int batch, int cp, int t0, int t_end,
                   hipStream_t s) {
    hipLaunchKernelGGL(prefill_argmax_kernel, dim3((unsigned)ceil_div(rows, 16)), dim3(256), 0, s, part, groups, rows,
                       argmax_out, batch, cp, t0, t_end);
    return launch_check("prefill_argmax_kernel");
}

int prefill_attention(const float* q, const float* kc, const float* vc, uint16_t* os, int64_t plane, int batch,
                      int heads, int hd, int tmax, float scale, int t0, int cp, hipStream_t s) {
    switch (hd) {
        case 8: return dispatch_attn<8>(q, kc, vc, os, plane, batch, heads, tmax, scale, t0, cp, s);
        case 16: return dispatch_attn<16>(q, kc, vc, os, plane, batch, heads, tmax, scale, t0, cp, s);
        case 32: return dispatch_attn<32>(q, kc, vc, os, plane, batch, heads, tmax, scale, t0, cp, s);
        case 64: return dispatch_attn<64>(q, kc, vc, os, plane, batch, heads, tmax, scale, t0, cp, s);
        case 128: return dispatch_attn<128>(q, kc, vc, os, plane, batch, heads, tmax, scale, t0, cp, s);
        case 256: return dispatch_attn<256>(q, kc, vc, os, plane, batch, heads, tmax, scale, t0, cp, s);
        default: return fail(MLXHIP_ERR_INVALID_ARGUMENT, "prefill attention: head_dim %d not in {8, 16, ..., 256}", hd);
    }
}

int prefill_last(const float* px, int cp, int p, float* x, uint16_t* xs, int d, int batch, int* tctr, int t,
                 hipStream_t s) {
    hipLaunchKernelGGL(prefill_last_kernel, dim3(batch), dim3(256), 0, s, px, cp, p, x, xs, d, tctr, t);
    return launch_check("prefill_last_kernel");
}

}  // namespace mlxhip
