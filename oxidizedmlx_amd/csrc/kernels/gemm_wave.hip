// gemm_wave.hip — f32 and 16-bit GEMM with K split over the waves of a
// workgroup, for products with too few tiles to fill the chip any other way
// (few rows, or a few hundred rows and columns), in one launch with no
// workspace.
//
// C_b[M,N] = op(A_b) * op(B_b), f32 sums; C in f32, or bf16 / f16 (round to
// nearest even) for 16-bit operands; replaces matmul
// (crates/mlx-core/src/cpu_kernels.rs:197-230) at these sizes.
//
// A workgroup of W waves owns a tile of C of MT x NT MFMA tiles (16 x 16 or
// 32 x 32: v_mfma_f32_16x16x4_f32 and 32x32x2, or 16x16x32 and 32x32x16 for
// 16 bits). K comes in runs of 16: a wave takes G runs at a time, one per lane
// group (G = 4 or 2, the k-slots of the MFMA), waves taking the groups of runs
// in turn, so each lane holds 16 consecutive k of its row of A and of its
// column of B, and lane group g's MFMA step i takes the i-th k (16 bits: the
// i-th 8 k) of its run. A K-contiguous operand is read with 16-byte loads, an
// MN-contiguous one with an element per load, coalesced across the lanes. No
// operand is used by two waves, so nothing goes through LDS and there is no
// barrier until the waves' partial tiles are added up there, in wave order
// (deterministic). The next group of runs is loaded while one is multiplied.
//
// f32 buffer loads need 4-byte alignment only, and 16-bit runs are shifted
// into place (load_run), so every alignment and leading dimension runs as it
// is (no packed copies); rows past the matrix take an offset past the
// descriptor's range (zeros), and the one group of runs that crosses the end
// of K is masked element by element.
//
// Bound, at the larger tiles, by the L1's rate for K-contiguous operands (64
// lanes of a load in 16 to 32 rows: 1024^3 bf16 14.0 us NT, 11.6 us NN), at
// the smaller ones by a load's latency, the reduction and the launch.
#include <algorithm>

#include "../common.hpp"
#include "../kernels.hpp"

namespace mlxhip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int RUN = 16;                      // k per lane group and step
constexpr uint32_t OOB_OFF = 0xFFFFFF00u;    // beyond every descriptor range (slices are < 2 GiB)
constexpr int BUF_FLAGS = 0x00020000;        // gfx9 buffer descriptor word 3 (32-bit data format)
constexpr int64_t SLICE_MAX_BYTES = int64_t(1) << 31;

constexpr int F32 = MLXHIP_DTYPE_F32, BF16 = MLXHIP_DTYPE_BF16, F16 = MLXHIP_DTYPE_F16;
template <int DT>
constexpr int ES = DT == F32 ? 4 : 2;  // bytes of an operand's element

struct WaveArgs {
    const char* a;
    const char* b;
    void* c;
    const float* bias;        // added to every row of C (null: none)
    int64_t sa, sb, sc, ldc;  // sa, sb in bytes
    int m, n, k, ct;          // ct: C's dtype
    uint32_t lda, ldb;        // leading dimensions in bytes
    uint32_t nrec_a, nrec_b;  // one operand slice's bytes
    int tiles_n, tiles_m;
};

// A lane's run of one operand and the MFMA steps that read it. f32: a value
// per step; 16 bits: 8 consecutive k per step, two to a dword.
template <int DT>
struct Run {
    static constexpr int STEPS = 2;
    uint32_t w[RUN / 2];
};
template <>
struct Run<F32> {
    static constexpr int STEPS = RUN;
    float w[RUN];
};

template <class V, int DT>
__device__ inline V eight(const Run<DT>& r, int e) {
    return __builtin_bit_cast(V, u32x4{r.w[4 * e], r.w[4 * e + 1], r.w[4 * e + 2], r.w[4 * e + 3]});
}

template <int S>
struct Mfma;
template <>
struct Mfma<16> {
    typedef f32x4 Acc;
    static constexpr int G = 4, E = 4;
    template <int DT>
    static __device__ inline Acc step(const Run<DT>& a, const Run<DT>& b, int e, Acc c) {
        if constexpr (DT == F32) return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w[e], b.w[e], c, 0, 0, 0);
        else if constexpr (DT == BF16)
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(eight<bf16x8>(a, e), eight<bf16x8>(b, e), c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f32_16x16x32_f16(eight<f16x8>(a, e), eight<f16x8>(b, e), c, 0, 0, 0);
    }
    // Accumulator element v of lane l is C[4 * (l / 16) + v][l % 16].
    static __device__ inline int row(int v, int g) { return 4 * g + v; }
};
template <>
struct Mfma<32> {
    typedef f32x16 Acc;
    static constexpr int G = 2, E = 16;
    template <int DT>
    static __device__ inline Acc step(const Run<DT>& a, const Run<DT>& b, int e, Acc c) {
        if constexpr (DT == F32) return __builtin_amdgcn_mfma_f32_32x32x2f32(a.w[e], b.w[e], c, 0, 0, 0);
        else if constexpr (DT == BF16)
            return __builtin_amdgcn_mfma_f32_32x32x16_bf16(eight<bf16x8>(a, e), eight<bf16x8>(b, e), c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f32_32x32x16_f16(eight<f16x8>(a, e), eight<f16x8>(b, e), c, 0, 0, 0);
    }
    // Accumulator element v of lane l is C[8 * (v / 4) + 4 * (l / 32) + v % 4][l % 32].
    static __device__ inline int row(int v, int g) { return 8 * (v >> 2) + 4 * g + (v & 3); }
};

// The lane's 16 k, k0 .. k0 + 15, of its row (or column) at byte offset
// `off` of k0 (OOB_OFF: outside the matrix). TAIL: the run may cross K.
template <bool KC, bool TAIL>
__device__ inline void load_run(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t ld, int k0, int K, Run<F32>& v) {
    if constexpr (KC) {
#pragma unroll
        for (int j = 0; j < RUN; j += 4) {
            const f32x4 t = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 4 * j, 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) v.w[j + e] = !TAIL || k0 + j + e < K ? t[e] : 0.0f;
        }
    } else {
#pragma unroll
        for (int e = 0; e < RUN; ++e) {
            if constexpr (TAIL)
                v.w[e] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(
                               rs, off != OOB_OFF && k0 + e < K ? off + (uint32_t)e * ld : OOB_OFF, 0, 0));
            else
                v.w[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, (uint32_t)e * ld, 0));
        }
    }
}

// 16-bit operands: any 2-byte alignment. A K-contiguous run is read from the
// dword at or below its first element and shifted down by an element where
// that one is a dword's upper half; then a ninth dword holds its last one.
template <bool KC, bool TAIL, int DT>
__device__ inline void load_run(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t ld, int k0, int K, Run<DT>& v) {
    if constexpr (KC) {
        const bool odd = off != OOB_OFF && (off & 2);
        const uint32_t at = off & ~3u, sh = odd ? 16u : 0u;
        uint32_t t[RUN / 2 + 1];
#pragma unroll
        for (int j = 0; j < RUN / 2; j += 4) {
            const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(rs, at + 4 * j, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) t[j + e] = q[e];
        }
        t[RUN / 2] = __builtin_amdgcn_raw_buffer_load_b32(rs, odd ? at + 2 * RUN : OOB_OFF, 0, 0);
#pragma unroll
        for (int j = 0; j < RUN / 2; ++j) {
            v.w[j] = __builtin_amdgcn_alignbit(t[j + 1], t[j], sh);
            if constexpr (TAIL)
                v.w[j] &= (k0 + 2 * j < K ? 0x0000FFFFu : 0u) | (k0 + 2 * j + 1 < K ? 0xFFFF0000u : 0u);
        }
    } else {
#pragma unroll
        for (int j = 0; j < RUN / 2; ++j) {
            uint32_t h[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                if constexpr (TAIL)
                    h[e] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(
                        rs, off != OOB_OFF && k0 + 2 * j + e < K ? off + (uint32_t)(2 * j + e) * ld : OOB_OFF, 0, 0);
                else h[e] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, off, (uint32_t)(2 * j + e) * ld, 0);
            }
            v.w[j] = h[0] | h[1] << 16;
        }
    }
}

template <class T>
__device__ inline void store_row(void* c, int64_t at, float v) {
    static_cast<T*>(c)[at] = (T)v;  // 16 bits: round to nearest even
}

template <int DT, int TA, int TB, int S, int MT, int NT, int W>
__global__ __launch_bounds__(W * 64) void gemm_wave_kernel(WaveArgs g) {
    using M = Mfma<S>;
    constexpr int G = M::G, STEP = G * RUN;  // k per wave and step
    constexpr int ROWS = S * MT, COLS = S * NT, PITCH = COLS + 1;
    // Independent accumulator chains: MFMAs in flight, and shorter sums.
    constexpr int CH = S == 16 ? 4 : 4 / (MT * NT);
    __shared__ float part[W][ROWS * PITCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Tile order: each XCD a contiguous range of tiles, in groups of 4 tile rows.
    const int per_batch = g.tiles_m * g.tiles_n;
    const int total = (int)gridDim.x;
    int lin = (int)blockIdx.x;
    if ((total & 7) == 0) lin = (lin & 7) * (total >> 3) + (lin >> 3);
    const int bt = lin / per_batch, id = lin - bt * per_batch;
    constexpr int GROUP_M = 4;
    const int in_group = GROUP_M * g.tiles_n, first_m = (id / in_group) * GROUP_M;
    const int gsz = min(g.tiles_m - first_m, GROUP_M);
    const int m0 = (first_m + (id % in_group) % gsz) * ROWS, n0 = ((id % in_group) / gsz) * COLS;
    const int r = lane % S, lg = lane / S;

    // 16 bits: from the dword at or below the slice's first element (its
    // byte phase goes into the offsets) to the end of its last dword.
    const uintptr_t pa = reinterpret_cast<uintptr_t>(g.a + (int64_t)bt * g.sa);
    const uintptr_t pb = reinterpret_cast<uintptr_t>(g.b + (int64_t)bt * g.sb);
    const uint32_t fa = DT == F32 ? 0u : (uint32_t)(pa & 2), fb = DT == F32 ? 0u : (uint32_t)(pb & 2);
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc((void*)(pa - fa), (short)0, (int)((g.nrec_a + fa + 3) & ~3u), BUF_FLAGS);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc((void*)(pb - fb), (short)0, (int)((g.nrec_b + fb + 3) & ~3u), BUF_FLAGS);
    constexpr bool AK = TA == 0, BK = TB == 1;  // K-contiguous
    constexpr uint32_t EB = ES<DT>;
    const uint32_t ka = AK ? EB : g.lda, kb = BK ? EB : g.ldb;  // bytes per unit of k
    uint32_t oa[MT], ob[NT];
    bool oka[MT], okb[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int row = m0 + S * i + r;
        oka[i] = row < g.m;
        oa[i] = fa + (oka[i] ? (uint32_t)row * (AK ? g.lda : EB) : 0u);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int col = n0 + S * j + r;
        okb[j] = col < g.n;
        ob[j] = fb + (okb[j] ? (uint32_t)col * (BK ? g.ldb : EB) : 0u);
    }
    Run<DT> a[2][MT], b[2][NT];
    const int K = g.k;
    auto load = [&](int u, int s) {
        const int ks = s * STEP, k0 = ks + lg * RUN;
        // Runs past the end of K start outside the matrix.
        const bool in = k0 < K;
        if (ks + STEP <= K) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
                load_run<AK, false>(ra, oka[i] ? oa[i] + (uint32_t)k0 * ka : OOB_OFF, g.lda, k0, K, a[u][i]);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                load_run<BK, false>(rb, okb[j] ? ob[j] + (uint32_t)k0 * kb : OOB_OFF, g.ldb, k0, K, b[u][j]);
        } else {
#pragma unroll
            for (int i = 0; i < MT; ++i)
                load_run<AK, true>(ra, oka[i] && in ? oa[i] + (uint32_t)k0 * ka : OOB_OFF, g.lda, k0, K, a[u][i]);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                load_run<BK, true>(rb, okb[j] && in ? ob[j] + (uint32_t)k0 * kb : OOB_OFF, g.ldb, k0, K, b[u][j]);
        }
    };
    typename M::Acc acc[MT][NT][CH];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int q = 0; q < CH; ++q)
#pragma unroll
                for (int v = 0; v < M::E; ++v) acc[i][j][q][v] = 0.0f;
    auto multiply = [&](int u) {
#pragma unroll
        for (int e = 0; e < Run<DT>::STEPS; ++e)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    auto& c = acc[i][j][(u * Run<DT>::STEPS + e) % CH];
                    c = M::template step<DT>(a[u][i], b[u][j], e, c);
                }
    };
    const int steps = (K + STEP - 1) / STEP;
    if (wave < steps) load(0, wave);
    for (int s = wave; s < steps; s += 2 * W) {
        if (s + W < steps) load(1, s + W);
        __builtin_amdgcn_sched_barrier(0);  // the loads first, not next to their use
        multiply(0);
        if (s + W < steps) {
            if (s + 2 * W < steps) load(0, s + 2 * W);
            __builtin_amdgcn_sched_barrier(0);
            multiply(1);
        }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int v = 0; v < M::E; ++v) {
                float x = acc[i][j][0][v];
#pragma unroll
                for (int q = 1; q < CH; ++q) x += acc[i][j][q][v];
                part[wave][(S * i + M::row(v, lg)) * PITCH + S * j + r] = x;
            }
    __syncthreads();
    const int used = min(W, steps);  // waves without a run hold zeros
    for (int e = tid; e < ROWS * COLS; e += W * 64) {
        const int i = e / COLS, j = e % COLS;
        const int row = m0 + i, col = n0 + j;
        if (row < g.m && col < g.n) {
            float s = part[0][i * PITCH + j];
            for (int w = 1; w < used; ++w) s += part[w][i * PITCH + j];
            if (g.bias) s += g.bias[col];
            const int64_t at = (int64_t)bt * g.sc + (int64_t)row * g.ldc + col;
            if (DT == F32 || g.ct == F32) store_row<float>(g.c, at, s);
            else if (g.ct == BF16) store_row<__bf16>(g.c, at, s);
            else store_row<_Float16>(g.c, at, s);
        }
    }
}

enum Tile { T64, T32X64, T32, T16X32, T16, NO_TILE };

// f32: the tile with the least rounds of workgroups (one per CU) times the
// cycles a workgroup's k costs its CU, matrix cycles (rows x cols / 128) and
// operand loads together.
Tile pick(int64_t m, int64_t n, int64_t batch) {
    static constexpr struct {
        Tile tile;
        int rows, cols, cost2;  // cost in half cycles
    } options[] = {{T64, 64, 64, 88}, {T32X64, 32, 64, 50}, {T32, 32, 32, 28}, {T16X32, 16, 32, 17}, {T16, 16, 16, 10}};
    Tile best = T64;
    int64_t least = INT64_MAX;
    for (const auto& o : options) {
        const int64_t cost = ceil_div(ceil_div(m, o.rows) * ceil_div(n, o.cols) * batch, 256) * o.cost2;
        if (cost < least) {
            least = cost;
            best = o.tile;
        }
    }
    return best;
}

// 16 bits, where the operand loads are nearly all of a workgroup's time: the
// tile with the least rounds times nanoseconds per k, or NO_TILE where the
// kernels with operands staged through LDS are faster. Measured, us, bf16,
// NT/NN/TN, those kernels -> here:
//   one round of 16-wide tiles: 8 x 3072 x 768 9.7 -> 5.4, 8 x 768 x 3072
//   15.7/19/21 -> 7.2/8.0/10.2, 128 x 768 x 3072 16.7/20/22 -> 11/10/11;
//   32 x 32: 512^3 10.3 -> 6.1; 32 x 64: 512 x 1000 x 777 11 -> 8.1/7.9/9.1,
//   but 512 x 768 x 3072 16.7 against 21/19/20; 64 x 64, where the others
//   split K over workgroups: 1024^3 17.5 -> 14/11.6/13.1, but 1024 x 1024 x
//   256 6.3 against 8.6 and, unaligned, 900 x 1000 x 1023 12.0 against 15.1.
// A second round pays for few rows or columns only (8 x 32000 x 768 15 -> 12,
// 2048 x 768 x 768 17.4 against 22; 16 x 4096 x 1500 in 4 slices NT 13.4 ->
// 10.8, NN 13.6 against 14.6). Eight rows of a wide B stored [K][N] at
// long K are read in 32-byte pieces (8 x 4096 x 4096 NT 11.3 -> 8.9, NN 11.7
// against 16.5).
Tile pick16(int64_t m, int64_t n, int64_t k, int64_t batch, bool nt, bool aligned) {
    static constexpr struct {
        Tile tile;
        int rows, cols, rounds;
        double ns;
    } options[] = {{T64, 64, 64, 1, 8.5}, {T32X64, 32, 64, 1, 5.0}, {T32, 32, 32, 1, 3.0},
                   {T16X32, 16, 32, 4, 2.0}, {T16, 16, 16, 4, 1.2}};
    if (!nt && k > 1536 && ceil_div(m, 128) * ceil_div(n, 128) * batch >= 16) return NO_TILE;
    const bool few = std::min(m, n) <= 32;
    Tile best = NO_TILE;
    double least = 9000.0;  // ns
    for (const auto& o : options) {
        const int64_t rounds = ceil_div(ceil_div(m, o.rows) * ceil_div(n, o.cols) * batch, 256);
        if (rounds > (few && (nt || k <= 1024) ? o.rounds : 1) || (o.tile == T64 && !(aligned && k >= 512))) continue;
        const double cost = (double)rounds * o.ns * (double)k;
        if (cost < least) {
            least = cost;
            best = o.tile;
        }
    }
    return best;
}

int64_t slice_bytes(int64_t rows, int64_t cols, int64_t ld, int64_t es) { return ((rows - 1) * ld + cols) * es; }

template <int DT, int S, int MT, int NT, int W>
int launch_wave(int ta, int tb, WaveArgs& g, int64_t batch, hipStream_t s) {
    g.tiles_m = (int)ceil_div(g.m, S * MT);
    g.tiles_n = (int)ceil_div(g.n, S * NT);
    const dim3 grid((unsigned)((int64_t)g.tiles_m * g.tiles_n * batch)), block(W * 64);
    if (!ta && !tb) hipLaunchKernelGGL((gemm_wave_kernel<DT, 0, 0, S, MT, NT, W>), grid, block, 0, s, g);
    else if (!ta) hipLaunchKernelGGL((gemm_wave_kernel<DT, 0, 1, S, MT, NT, W>), grid, block, 0, s, g);
    else if (!tb) hipLaunchKernelGGL((gemm_wave_kernel<DT, 1, 0, S, MT, NT, W>), grid, block, 0, s, g);
    else hipLaunchKernelGGL((gemm_wave_kernel<DT, 1, 1, S, MT, NT, W>), grid, block, 0, s, g);
    return launch_check("gemm_wave_kernel");
}

template <int DT>
int launch_tile(int ta, int tb, bool aligned, WaveArgs& g, int64_t batch, hipStream_t s) {
    switch (DT == F32 ? pick(g.m, g.n, batch) : pick16(g.m, g.n, g.k, batch, !ta && tb, aligned)) {
        case T64: return launch_wave<DT, 32, 2, 2, 8>(ta, tb, g, batch, s);
        case T32X64: return launch_wave<DT, 32, 1, 2, 8>(ta, tb, g, batch, s);
        case T32: return launch_wave<DT, 32, 1, 1, 8>(ta, tb, g, batch, s);
        case T16X32: return launch_wave<DT, 16, 1, 2, 8>(ta, tb, g, batch, s);
        default: return launch_wave<DT, 16, 1, 1, 8>(ta, tb, g, batch, s);
    }
}

}  // namespace

bool gemm_wave_fits(int ab_dtype, int64_t m, int64_t n, int64_t k, int64_t batch, int64_t lda, int64_t ldb,
                    int ta, int tb, bool aligned) {
    if (m < 1 || n < 1 || k < 1 || m > INT32_MAX / 2 || n > INT32_MAX / 2 || k > INT32_MAX / 2) return false;
    // f32: where it is the faster one (measured against the kernels below it in
    // the dispatch, us, before -> here; N64 = tiles of 64 x 64): few tiles, or
    // a K long enough for the waves to share. 8 x 3072 x 768 12.2 -> 5.6, 128 x
    // 3072 x 768 22.6 -> 13.8, 512 x 768 x 3072 41 -> 40, 1024^3 (256) 35 -> 30,
    // 2048 x 768 x 768 (384) 50 -> 38; but 2048 x 2048 x 256 (1024) 27 against
    // 39, 256^3 x 32 (512) 17 against 21, 64^3 x 512 (512) 7 against 11. At most
    // 32 rows or columns: 8 x 32000 x 768 (500) 41 -> 19. Unaligned operands
    // need no packed copies here: 100 x 300 x 77 x 32 (320) 14 -> 9.
    const int64_t n64 = ceil_div(m, 64) * ceil_div(n, 64) * batch;
    const double fill = (double)(m * n) / ((double)(ceil_div(m, 128) * 128) * (double)(ceil_div(n, 128) * 128));
    const bool faster = n64 <= 96 || (k >= 128 && n64 <= 256) ||
                        (n64 <= 1024 && (!aligned || (k >= 128 && std::min(m, n) <= 32))) ||
                        (k >= 500 && n64 <= 576 && fill >= 0.75);
    if (ab_dtype == F32 ? !faster : pick16(m, n, k, batch, !ta && tb, aligned) == NO_TILE) return false;
    const int64_t es = ab_dtype == F32 ? 4 : 2;
    const int64_t a_bytes = ta ? slice_bytes(k, m, lda, es) : slice_bytes(m, k, lda, es);
    const int64_t b_bytes = tb ? slice_bytes(n, k, ldb, es) : slice_bytes(k, n, ldb, es);
    return a_bytes < SLICE_MAX_BYTES && b_bytes < SLICE_MAX_BYTES && lda < SLICE_MAX_BYTES / es &&
           ldb < SLICE_MAX_BYTES / es;
}

int gemm_wave(int ab_dtype, int c_dtype, int ta, int tb, int64_t m, int64_t n, int64_t k, int64_t batch, const void* a,
              int64_t lda, int64_t sa, const void* b, int64_t ldb, int64_t sb, void* c, int64_t ldc, int64_t sc,
              const float* bias, bool aligned, hipStream_t s) {
    const int64_t es = ab_dtype == F32 ? 4 : 2;
    WaveArgs g{};
    g.a = static_cast<const char*>(a), g.b = static_cast<const char*>(b), g.c = c, g.bias = bias;
    g.sa = sa * es, g.sb = sb * es, g.sc = sc, g.ldc = ldc;
    g.m = (int)m, g.n = (int)n, g.k = (int)k, g.ct = c_dtype;
    g.lda = (uint32_t)(lda * es), g.ldb = (uint32_t)(ldb * es);
    g.nrec_a = (uint32_t)(ta ? slice_bytes(k, m, lda, es) : slice_bytes(m, k, lda, es));
    g.nrec_b = (uint32_t)(tb ? slice_bytes(n, k, ldb, es) : slice_bytes(k, n, ldb, es));
    if (ab_dtype == F32) return launch_tile<F32>(ta, tb, aligned, g, batch, s);
    return ab_dtype == BF16 ? launch_tile<BF16>(ta, tb, aligned, g, batch, s) : launch_tile<F16>(ta, tb, aligned, g, batch, s);
}

}  // namespace mlxhip
