// gemm_wave.hip — f32 GEMM with K split over the waves of a workgroup, for
// products with too few tiles to fill the chip any other way (few rows, or a
// few hundred rows and columns), in one launch with no workspace.
//
// C_b[M,N] = op(A_b) * op(B_b), f32 operands and output; replaces matmul
// (crates/mlx-core/src/cpu_kernels.rs:197-230) at these sizes.
//
// A workgroup of W waves owns a tile of C of MT x NT MFMA tiles (16 x 16 on
// v_mfma_f32_16x16x4_f32 or 32 x 32 on v_mfma_f32_32x32x2_f32). K comes in
// runs of 16: a wave takes G runs at a time, one per lane group (G = 4 or 2,
// the k-slots of the MFMA), waves taking the groups of runs in turn. Lane
// group g's MFMA step i takes k = run(g) + i, so each lane holds 16
// consecutive k of its row of A and of its column of B: a K-contiguous
// operand is read with four 16-byte loads, an MN-contiguous one with 16
// 4-byte loads that are coalesced across the lanes. No operand is used by
// two waves, so nothing goes through LDS and there is no barrier until the
// waves' partial tiles are added up there, in wave order (deterministic). The
// next group of runs is loaded while one is multiplied.
//
// Buffer loads need 4-byte alignment only, so every alignment and leading
// dimension runs as it is (no packed copies); rows past the matrix take an
// offset past the descriptor's range (zeros), and the one group of runs that
// crosses the end of K is masked element by element.
#include <algorithm>

#include "../common.hpp"
#include "../kernels.hpp"

namespace mlxhip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int RUN = 16;                      // k per lane group and step
constexpr uint32_t OOB_OFF = 0xFFFFFF00u;    // beyond every descriptor range (slices are < 2 GiB)
constexpr int BUF_FLAGS = 0x00020000;        // gfx9 buffer descriptor word 3 (32-bit data format)
constexpr int64_t SLICE_MAX_BYTES = int64_t(1) << 31;

struct WaveArgs {
    const float* a;
    const float* b;
    float* c;
    const float* bias;        // added to every row of C (null: none)
    int64_t sa, sb, sc, ldc;
    int m, n, k;
    uint32_t lda4, ldb4;      // leading dimensions in bytes
    uint32_t nrec_a, nrec_b;  // descriptor ranges: one operand slice's bytes
    int tiles_n, tiles_m;
};

template <int S>
struct Mfma;
template <>
struct Mfma<16> {
    typedef f32x4 Acc;
    static constexpr int G = 4, E = 4;
    static __device__ inline Acc step(float a, float b, Acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    // Accumulator element v of lane l is C[4 * (l / 16) + v][l % 16].
    static __device__ inline int row(int v, int g) { return 4 * g + v; }
};
template <>
struct Mfma<32> {
    typedef f32x16 Acc;
    static constexpr int G = 2, E = 16;
    static __device__ inline Acc step(float a, float b, Acc c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
    // Accumulator element v of lane l is C[8 * (v / 4) + 4 * (l / 32) + v % 4][l % 32].
    static __device__ inline int row(int v, int g) { return 8 * (v >> 2) + 4 * g + (v & 3); }
};

// The lane's 16 k, k0 .. k0 + 15, of its row (or column) at byte offset
// `off` of k0 (OOB_OFF: outside the matrix). TAIL: the run may cross K.
template <bool KC, bool TAIL>
__device__ inline void load_run(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t ld4, int k0, int K, float (&v)[RUN]) {
    if constexpr (KC) {
#pragma unroll
        for (int j = 0; j < RUN; j += 4) {
            const f32x4 t = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 4 * j, 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) v[j + e] = !TAIL || k0 + j + e < K ? t[e] : 0.0f;
        }
    } else {
#pragma unroll
        for (int e = 0; e < RUN; ++e) {
            if constexpr (TAIL)
                v[e] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(
                               rs, off != OOB_OFF && k0 + e < K ? off + (uint32_t)e * ld4 : OOB_OFF, 0, 0));
            else
                v[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, (uint32_t)e * ld4, 0));
        }
    }
}

template <int TA, int TB, int S, int MT, int NT, int W>
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

    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc((void*)(g.a + (int64_t)bt * g.sa), (short)0, (int)g.nrec_a, BUF_FLAGS);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc((void*)(g.b + (int64_t)bt * g.sb), (short)0, (int)g.nrec_b, BUF_FLAGS);
    constexpr bool AK = TA == 0, BK = TB == 1;  // K-contiguous
    const uint32_t ka4 = AK ? 4u : g.lda4, kb4 = BK ? 4u : g.ldb4;  // bytes per unit of k
    uint32_t oa[MT], ob[NT];
    bool oka[MT], okb[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int row = m0 + S * i + r;
        oka[i] = row < g.m;
        oa[i] = oka[i] ? (uint32_t)row * (AK ? g.lda4 : 4u) : 0u;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int col = n0 + S * j + r;
        okb[j] = col < g.n;
        ob[j] = okb[j] ? (uint32_t)col * (BK ? g.ldb4 : 4u) : 0u;
    }
    float a[2][MT][RUN], b[2][NT][RUN];
    const int K = g.k;
    auto load = [&](int u, int s) {
        const int ks = s * STEP, k0 = ks + lg * RUN;
        // Runs past the end of K start outside the matrix.
        const bool in = k0 < K;
        if (ks + STEP <= K) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
                load_run<AK, false>(ra, oka[i] ? oa[i] + (uint32_t)k0 * ka4 : OOB_OFF, g.lda4, k0, K, a[u][i]);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                load_run<BK, false>(rb, okb[j] ? ob[j] + (uint32_t)k0 * kb4 : OOB_OFF, g.ldb4, k0, K, b[u][j]);
        } else {
#pragma unroll
            for (int i = 0; i < MT; ++i)
                load_run<AK, true>(ra, oka[i] && in ? oa[i] + (uint32_t)k0 * ka4 : OOB_OFF, g.lda4, k0, K, a[u][i]);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                load_run<BK, true>(rb, okb[j] && in ? ob[j] + (uint32_t)k0 * kb4 : OOB_OFF, g.ldb4, k0, K, b[u][j]);
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
        for (int e = 0; e < RUN; ++e)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j][e % CH] = M::step(a[u][i][e], b[u][j][e], acc[i][j][e % CH]);
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
    float* cb = g.c + (int64_t)bt * g.sc;
    const int used = min(W, steps);  // waves without a run hold zeros
    for (int e = tid; e < ROWS * COLS; e += W * 64) {
        const int i = e / COLS, j = e % COLS;
        const int row = m0 + i, col = n0 + j;
        if (row < g.m && col < g.n) {
            float s = part[0][i * PITCH + j];
            for (int w = 1; w < used; ++w) s += part[w][i * PITCH + j];
            if (g.bias) s += g.bias[col];
            cb[(int64_t)row * g.ldc + col] = s;
        }
    }
}

// The tile: the one with the least rounds of workgroups (one per CU) times
// the cycles a workgroup's k costs its CU, matrix cycles (rows x cols / 128)
// and operand loads together.
enum Tile { T64, T32X64, T32, T16X32, T16 };
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

int64_t slice_bytes(int64_t rows, int64_t cols, int64_t ld) { return ((rows - 1) * ld + cols) * 4; }

template <int S, int MT, int NT, int W>
int launch_wave(int ta, int tb, WaveArgs& g, int64_t batch, hipStream_t s) {
    g.tiles_m = (int)ceil_div(g.m, S * MT);
    g.tiles_n = (int)ceil_div(g.n, S * NT);
    const dim3 grid((unsigned)((int64_t)g.tiles_m * g.tiles_n * batch)), block(W * 64);
    if (!ta && !tb) hipLaunchKernelGGL((gemm_wave_kernel<0, 0, S, MT, NT, W>), grid, block, 0, s, g);
    else if (!ta) hipLaunchKernelGGL((gemm_wave_kernel<0, 1, S, MT, NT, W>), grid, block, 0, s, g);
    else if (!tb) hipLaunchKernelGGL((gemm_wave_kernel<1, 0, S, MT, NT, W>), grid, block, 0, s, g);
    else hipLaunchKernelGGL((gemm_wave_kernel<1, 1, S, MT, NT, W>), grid, block, 0, s, g);
    return launch_check("gemm_wave_kernel");
}

}  // namespace

bool gemm_wave_f32_fits(int64_t m, int64_t n, int64_t k, int64_t batch, int64_t lda, int64_t ldb, int ta, int tb,
                        bool aligned) {
    if (m < 1 || n < 1 || k < 1 || m > INT32_MAX / 2 || n > INT32_MAX / 2 || k > INT32_MAX / 2) return false;
    // Where it is the faster one (measured against the kernels below it in
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
    if (!faster) return false;
    const int64_t a_bytes = ta ? slice_bytes(k, m, lda) : slice_bytes(m, k, lda);
    const int64_t b_bytes = tb ? slice_bytes(n, k, ldb) : slice_bytes(k, n, ldb);
    return a_bytes < SLICE_MAX_BYTES && b_bytes < SLICE_MAX_BYTES && lda < SLICE_MAX_BYTES / 4 &&
           ldb < SLICE_MAX_BYTES / 4;
}

int gemm_wave_f32(int ta, int tb, int64_t m, int64_t n, int64_t k, int64_t batch, const float* a, int64_t lda,
                  int64_t sa, const float* b, int64_t ldb, int64_t sb, float* c, int64_t ldc, int64_t sc,
                  const float* bias, hipStream_t s) {
    WaveArgs g{};
    g.a = a, g.b = b, g.c = c, g.bias = bias;
    g.sa = sa, g.sb = sb, g.sc = sc, g.ldc = ldc;
    g.m = (int)m, g.n = (int)n, g.k = (int)k;
    g.lda4 = (uint32_t)(lda * 4), g.ldb4 = (uint32_t)(ldb * 4);
    g.nrec_a = (uint32_t)(ta ? slice_bytes(k, m, lda) : slice_bytes(m, k, lda));
    g.nrec_b = (uint32_t)(tb ? slice_bytes(n, k, ldb) : slice_bytes(k, n, ldb));
    switch (pick(m, n, batch)) {
        case T64: return launch_wave<32, 2, 2, 8>(ta, tb, g, batch, s);
        case T32X64: return launch_wave<32, 1, 2, 8>(ta, tb, g, batch, s);
        case T32: return launch_wave<32, 1, 1, 8>(ta, tb, g, batch, s);
        case T16X32: return launch_wave<16, 1, 2, 8>(ta, tb, g, batch, s);
        default: return launch_wave<16, 1, 1, 8>(ta, tb, g, batch, s);
    }
}

}  // namespace mlxhip
