// The projections of a pass over a few rows (the batched decode step, a short prompt) on the
// matrix cores: Y[n][rows] = X[n][cols] W^T with W [rows][cols] and X [n][cols] bf16 row-major,
// f32 accumulation, Y bf16 or f32 (the reference's Gpu::gemm, gpu.rs:1098-1149). At one row the
// decode GEMV (gemv.hip) is the right kernel; past 64 rows the work is a compute-bound GEMM,
// the tiled kernels further down.
#include "device.h"

namespace {

constexpr uint32_t RSRC_WORD3 = 0x00020000;
constexpr uint32_t OFF_NONE = 0xFFFFFFF0u;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint64_t bytes) {
    // A byte count past 4 GiB - 16 is clamped there: offsets are 32-bit.
    const uint32_t n = bytes > OFF_NONE ? OFF_NONE : (uint32_t)bytes;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)n, RSRC_WORD3);
}

// CPOL: the cache policy (0 the default; CPOL_NT non-temporal, for a stream read once).
constexpr int CPOL_NT = 2;
template <int CPOL = 0>
__device__ __forceinline__ uint4 bload(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, CPOL);
    return make_uint4((uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]);
}

}  // namespace

// ---- a few rows: Y[n][rows] = X[n][cols] W^T for n <= 64, bandwidth-bound ----
// The batched decode step's projections and a short prompt's. Every W row is read once, so the
// kernel streams W at the HBM rate and the few-row matrix-core products cost nothing beside it:
//  - Block b takes the RG row groups of 16 W rows 16 RG b .. 16 RG b + 16 RG - 1 over all of K;
//    its V wavefronts (V = blockDim / 64, chosen by the host with RG so the launch holds enough
//    loads in flight) take its steps of 32 columns in turn (wavefront w: steps w, w + V, ..), so
//    at any time a block reads one contiguous run of each of its panels.
//  - W is read with a non-temporal hint (each byte read once), X with the default policy (every
//    block reads it, from the L2). Measured on MI355X on the batched Qwen3-8B and -32B shapes
//    (W and X in panels): 3-19 % faster than each wavefront reading its own quarter of K with the
//    default policy.
//  - A step is TT x RG 16 x 16 x 32 products (TT tiles of 16 tokens, RG row groups) whose A
//    operand is X (row = token, zero past n) and B operand W (column = W row): lane l loads
//    16 bytes, columns k0 + 8 (l / 16) .. + 7, of W row 16 (RG b + g) + l % 16 and of X row
//    16 tt + l % 16; the 4 lane groups cover 64 contiguous bytes of each row. One X piece
//    serves the RG row groups, so X (read from the L2 by every block) costs TT / RG of W's loads.
//  - U steps are in flight per wavefront: the slot a product has consumed is refilled at once
//    with the wavefront's step U ahead, so U - 1 steps stay in flight while one multiplies. A piece past K
//    (or a token past n, a W row past rows) is a raw buffer load at an offset past the buffer,
//    which returns zeros without touching memory.
//  - The wavefronts' partial tiles are summed in LDS in wavefront order (deterministic).
// flags: FEW_F32 Y f32 (else bf16); FEW_X_PANEL X in panels (below); FEW_Y_PANEL Y in panels
// (bf16); FEW_W_PANEL W in panels (rows a multiple of 16; with SwiGLU the [gate; up] matrix of
// 2 rows rows in panels, so gate and up panels do not mix). GLU: SwiGLU over the packed [gate; up] W of 2 rows rows: the block also takes the up
// rows rows + 16 (RG b + g) .., and writes act[t][r] = bf16(g / (1 + e^-g) u) of the
// bf16-rounded g and u, in f64 (x0ne_swiglu_bf16 of the bf16 projection).
//
// Panels: a [n][cols] bf16 matrix stored as ceil(n / 16) panels of [cols / 8][16][8]: element
// (t, k) at ((t / 16 * cols / 8 + k / 8) 16 + t % 16) 8 + k % 8. One step's X operand is then one
// contiguous KiB; row-major, its 16 rows lie cols apart and meet in the same L2 channels, which
// costs the W stream up to a fifth of its rate at 16 rows (measured on MI355X). W is laid out the
// same way for the same reason: row-major, each step reads 64 bytes of 16 rows cols apart, and
// the W stream of the Qwen3 decode shapes runs at 3.1-5.1 TB/s; in panels each step reads one
// contiguous KiB and a block's steps run through its panel in order, 3.7-5.9 TB/s (MI355X).
namespace {

constexpr uint32_t FEW_F32 = 1, FEW_X_PANEL = 2, FEW_Y_PANEL = 4, FEW_W_PANEL = 8;

template <int TT, int RG, int U, bool GLU, int MAXV>
__device__ __forceinline__ void few_rows(const bf16_t* __restrict__ w, const bf16_t* __restrict__ x,
                                         void* __restrict__ y, uint32_t rows, uint32_t cols, uint32_t n,
                                         uint32_t flags, f32x4* part) {
    constexpr int KINDS = GLU ? 2 : 1;
    const uint32_t b = blockIdx.x, V = blockDim.x >> 6;
    const bool out_f32 = flags & FEW_F32, x_panel = flags & FEW_X_PANEL, y_panel = flags & FEW_Y_PANEL;
    const bool w_panel = flags & FEW_W_PANEL;
    // Grid-uniform exits for a launch that does not fit.
    if (b * 16 * RG >= rows || n == 0 || n > 16 * TT || cols % 8 != 0 || V > MAXV || flags > 15 ||
        (out_f32 && (GLU || y_panel)) || (y_panel && rows % 8 != 0) || (w_panel && rows % 16 != 0))
        return;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15, q4 = lane >> 4;
    // Panels hold whole tiles of 16 rows.
    const auto xr = rsrc(x, (uint64_t)(x_panel ? (n + 15) / 16 * 16 : n) * cols * 2);
    const auto wr = rsrc(w, (uint64_t)KINDS * rows * cols * 2);
    const uint32_t steps = (cols + 31) / 32;
    f32x4 acc[KINDS][RG][TT];
#pragma unroll
    for (int kd = 0; kd < KINDS; ++kd)
#pragma unroll
        for (int g = 0; g < RG; ++g)
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) acc[kd][g][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 xa[U][TT], wb[U][KINDS][RG];
    auto request = [&](int u, uint32_t s) {
        const uint32_t k = 32 * s + 8 * q4;
        const bool in = s < steps && k < cols;  // a K tail: pieces past the row read zeros
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            const uint32_t t = 16 * tt + r;
            const uint32_t off = x_panel ? (uint32_t)panel_index(t, k, cols) * 2 : (t * cols + k) * 2;
            xa[u][tt] = bload<>(xr, in && t < n ? off : OFF_NONE);
        }
#pragma unroll
        for (int kd = 0; kd < KINDS; ++kd)
#pragma unroll
            for (int g = 0; g < RG; ++g) {
                const uint32_t row = 16 * (RG * b + g) + r;
                const uint32_t wrow = kd * rows + row;
                wb[u][kd][g] = bload<CPOL_NT>(wr, !(in && row < rows) ? OFF_NONE
                                         : w_panel ? (uint32_t)panel_index(wrow, k, cols) * 2
                                                   : (wrow * cols + k) * 2);
            }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) request(u, wave + V * u);
    for (uint32_t s0 = wave; s0 < steps; s0 += U * V) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int kd = 0; kd < KINDS; ++kd)
#pragma unroll
                for (int g = 0; g < RG; ++g)
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt) acc[kd][g][tt] = mfma(xa[u][tt], wb[u][kd][g], acc[kd][g][tt]);
            request(u, s0 + V * (U + u));
        }
    }
    // part[(((kd V + wave) RG + g) TT + tt) 64 + lane]
    auto at = [&](uint32_t kd, uint32_t v, uint32_t g, uint32_t tt) { return (((kd * V + v) * RG + g) * TT + tt) * 64 + lane; };
#pragma unroll
    for (int kd = 0; kd < KINDS; ++kd)
#pragma unroll
        for (int g = 0; g < RG; ++g)
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) part[at(kd, wave, g, tt)] = acc[kd][g][tt];
    lds_barrier();
    // Wavefront w sums row groups w, w + V, ..: the V partials of each in wavefront order.
    for (uint32_t g = wave; g < (uint32_t)RG; g += V) {
        const uint32_t wrow = 16 * (RG * b + g) + r;
        if (wrow >= rows) continue;
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            f32x4 sg = part[at(0, 0, g, tt)], su = GLU ? part[at(1, 0, g, tt)] : f32x4{0.f, 0.f, 0.f, 0.f};
            for (uint32_t v = 1; v < V; ++v) {
                sg += part[at(0, v, g, tt)];
                if (GLU) su += part[at(1, v, g, tt)];
            }
            // sg[i]: token 16 tt + 4 (lane / 16) + i, W row wrow.
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t t = 16 * tt + 4 * q4 + i;
                if (t >= n) continue;
                const size_t o = y_panel ? panel_index(t, wrow, rows) : (size_t)t * rows + wrow;
                if (GLU) {
                    const double gv = (double)bf2f(f2bf(sg[i])), uv = (double)bf2f(f2bf(su[i]));
                    static_cast<bf16_t*>(y)[o] = f2bf((float)(gv / (1.0 + exp(-gv)) * uv));
                } else if (out_f32) {
                    static_cast<float*>(y)[o] = sg[i];
                } else {
                    static_cast<bf16_t*>(y)[o] = f2bf(sg[i]);
                }
            }
        }
    }
}

}  // namespace

// x0ne_gemm_few_t{TT}_r{RG}[_swiglu]_bf16: grid (ceil(rows / (16 RG))), block 64 V threads
// (V <= MAXV); n in 1 .. 16 TT; cols a multiple of 8 (of 8 and rows of 8 for a Y panel); X, W
// below 4 GiB - 16 bytes; flags as above (FEW_F32 = 1 not with SwiGLU or a Y panel).
#define X0NE_FEW(NAME, TT, RG, U, GLU, MAXV)                                                                     \
    extern "C" __global__ void __launch_bounds__(64 * MAXV)                                                       \
        NAME(const bf16_t* __restrict__ w, const bf16_t* __restrict__ x, void* __restrict__ y, uint32_t rows,     \
             uint32_t cols, uint32_t n, uint32_t flags) {                                                         \
        __shared__ f32x4 part[(GLU ? 2 : 1) * MAXV * RG * TT * 64];                                               \
        few_rows<TT, RG, U, GLU, MAXV>(w, x, y, rows, cols, n, flags, part);                                      \
    }
#ifndef X0NE_FEW_NO_TABLE
X0NE_FEW(x0ne_gemm_few_t1_r1_bf16, 1, 1, 12, false, 8)
X0NE_FEW(x0ne_gemm_few_t1_r2_bf16, 1, 2, 4, false, 8)
X0NE_FEW(x0ne_gemm_few_t1_r4_bf16, 1, 4, 8, false, 8)
X0NE_FEW(x0ne_gemm_few_t1_r8_bf16, 1, 8, 4, false, 8)
X0NE_FEW(x0ne_gemm_few_t1_r1_swiglu_bf16, 1, 1, 4, true, 8)
X0NE_FEW(x0ne_gemm_few_t1_r2_swiglu_bf16, 1, 2, 4, true, 8)
X0NE_FEW(x0ne_gemm_few_t2_r1_bf16, 2, 1, 8, false, 8)
X0NE_FEW(x0ne_gemm_few_t2_r2_bf16, 2, 2, 4, false, 8)
X0NE_FEW(x0ne_gemm_few_t2_r1_swiglu_bf16, 2, 1, 4, true, 8)
X0NE_FEW(x0ne_gemm_few_t4_r1_bf16, 4, 1, 4, false, 8)
X0NE_FEW(x0ne_gemm_few_t4_r1_swiglu_bf16, 4, 1, 4, true, 8)
#endif

// ---- a few rows balanced over the CUs: one block per CU, an equal run of the steps ----
// Where the 16-row groups are between one and two per CU (the Qwen3-32B O and down projections:
// 320 groups on 256 CUs), whole groups per block leave CUs idle (RG 2: 160 blocks) or doubled
// (RG 1). Here the steps of all groups, group-major (G groups x S steps of 32 columns), are cut
// into runs of T steps, one run per block and one block per CU, and the block's V wavefronts
// take its run's steps in turn (wavefront w: steps Lb + w, Lb + w + V, ..), so every block
// streams the same bytes as one contiguous run through the panels (a run crosses a group's end
// where one panel ends and the next begins).
//  - A wavefront sums its steps in order, one accumulator at a time: where its next step is in
//    the next group, the sums go to LDS (slot g - g0), so its loads never wait on a store.
//  - The block sums each group's wavefront partials in wavefront order. A group inside its run is
//    written at once. A group cut between runs (at most two blocks meet in a group here) is
//    finished by the last of its blocks to count: each stores its sums in slot (g, block - first
//    block of g) through agent-scope stores (coherent across the XCDs' L2s), waits for their
//    acknowledgment and counts in cnt[g]; the one that completes the count adds the slots in
//    slot order, writes Y and sets the count back to 0 for the next launch.
// Every sum's order is fixed by (rows, cols, T, V): the same bits whatever n, the timing or
// which block finishes a group. Measured on MI355X (32B down, 16 rows, 262 MB): 48.1 against
// 53.0 us for RG 2 (160 blocks); shapes whose groups are not cut this way (the 8B projections,
// SwiGLU, 640 or 1600 groups) measured no faster than whole groups per block.
namespace {

__device__ __forceinline__ void bal_put(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float bal_get(const float* p) {
    return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int U, int MAXG, int MAXV>
__device__ __forceinline__ void few_bal(const bf16_t* __restrict__ w, const bf16_t* __restrict__ x,
                                        void* __restrict__ y, uint32_t rows, uint32_t cols, uint32_t n,
                                        uint32_t flags, uint32_t T, float* __restrict__ ws,
                                        uint32_t* __restrict__ cnt, f32x4* stash) {
    const bool out_f32 = flags & FEW_F32, y_panel = flags & FEW_Y_PANEL;
    const uint32_t S = (cols + 31) / 32, G = rows / 16, V = blockDim.x >> 6;
    const uint64_t total = (uint64_t)G * S;
    // Grid-uniform exits for a launch that does not fit: a run touches at most MAXG groups and
    // gives every wavefront a step; X and W in panels.
    if (n == 0 || n > 16 || cols % 8 != 0 || rows % 16 != 0 || T < V || (uint64_t)T > (uint64_t)(MAXG - 2) * S + 1 ||
        total >= (1ull << 31) || V > MAXV || S < V || flags > 15 || !(flags & FEW_W_PANEL) || !(flags & FEW_X_PANEL) ||
        (out_f32 && y_panel) || (y_panel && rows % 8 != 0) || ws == nullptr || cnt == nullptr)
        return;
    const uint32_t b = blockIdx.x;
    if ((uint64_t)b * T >= total) return;  // block-uniform
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15, q4 = lane >> 4;
    const uint32_t Lb = b * T, Le = (uint32_t)min<uint64_t>((uint64_t)Lb + T, total), g0 = Lb / S;
    const uint32_t cmax = (S + T - 1) / T + 1;  // blocks that can meet in one group
    const auto xr = rsrc(x, (uint64_t)16 * cols * 2);
    const auto wr = rsrc(w, (uint64_t)rows * cols * 2);
    f32x4* mine = stash + (size_t)wave * MAXG * 64 + lane;
#pragma unroll
    for (int j = 0; j < MAXG; ++j) mine[j * 64] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 xa[U], wb[U];
    // Requests run through the wavefront's steps: (rg, rs) is request rq's group and step.
    const uint32_t L0 = Lb + wave;
    uint32_t rq = L0, rg = L0 / S, rs = L0 - rg * S;
    auto request = [&](int u) {
        const uint32_t k = 32 * rs + 8 * q4;
        const bool in = rq < Le && k < cols;  // a K tail: pieces past the row read zeros
        xa[u] = bload<>(xr, in && r < n ? (uint32_t)panel_index(r, k, cols) * 2 : OFF_NONE);
        wb[u] = bload<CPOL_NT>(wr, in ? (uint32_t)panel_index(16 * rg + r, k, cols) * 2 : OFF_NONE);
        rq += V;
        rs += V;
        if (rs >= S) {
            rs -= S;
            ++rg;
        }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) request(u);
    uint32_t cq = L0, cg = L0 / S, cs = L0 - cg * S;  // the consumed step, its group and place
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    for (uint32_t q0 = L0; q0 < Le; q0 += U * V) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (cq < Le) {  // wavefront-uniform
                acc = mfma(xa[u], wb[u], acc);
                cq += V;
                cs += V;
                if (cs >= S) {  // this wavefront's part of group cg ends: its sums to LDS
                    mine[(cg - g0) * 64] = acc;
                    acc = f32x4{0.f, 0.f, 0.f, 0.f};
                    cs -= S;
                    ++cg;
                }
            }
            request(u);
        }
    }
    if (cs != 0) mine[(cg - g0) * 64] = acc;  // the run ends inside group cg
    lds_barrier();
    // sg[i]: token 4 (lane / 16) + i, W row 16 g + lane % 16.
    auto emit = [&](uint32_t g, const f32x4& sg) {
        const uint32_t wrow = 16 * g + r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t t = 4 * q4 + i;
            if (t >= n) continue;
            const size_t o = y_panel ? panel_index(t, wrow, rows) : (size_t)t * rows + wrow;
            if (out_f32)
                static_cast<float*>(y)[o] = sg[i];
            else
                static_cast<bf16_t*>(y)[o] = f2bf(sg[i]);
        }
    };
    auto slot = [&](uint32_t g, uint32_t c) { return ws + ((size_t)g * cmax + c) * 256 + lane * 4; };
    const uint32_t ng = (Le - 1) / S - g0 + 1;
    // Wavefront w finishes the block's groups w, w + V, ..
    for (uint32_t j = wave; j < ng; j += V) {
        const uint32_t g = g0 + j;
        f32x4 sg = stash[j * 64 + lane];
        for (uint32_t v = 1; v < V; ++v) sg += stash[(v * MAXG + j) * 64 + lane];
        const uint32_t fb = (uint32_t)((uint64_t)g * S / T), lb = (uint32_t)(((uint64_t)g * S + S - 1) / T);
        if (fb == lb) {
            emit(g, sg);
            continue;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) bal_put(slot(g, b - fb) + e, sg[e]);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the slot acknowledged, then the count
        uint32_t old = 0;
        if (lane == 0) old = __hip_atomic_fetch_add(cnt + g, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_readfirstlane(old) != lb - fb) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) sg[e] = bal_get(slot(g, 0) + e);
        for (uint32_t c = 1; c <= lb - fb; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) sg[e] += bal_get(slot(g, c) + e);
        emit(g, sg);
        if (lane == 0) __hip_atomic_store(cnt + g, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

}  // namespace

// x0ne_gemm_few_bal_bf16: grid ceil(G S / T) for G = rows / 16 groups and S = ceil(cols / 32)
// steps, block 64 V threads (V <= 8, V <= T <= 4 S + 1); n in 1 .. 16; rows a multiple of 16,
// cols of 8; X and W in panels (flags FEW_X_PANEL | FEW_W_PANEL, FEW_F32 or FEW_Y_PANEL as
// above; no SwiGLU); ws: G (ceil(S / T) + 1) 256 floats, cnt: G words, zero before the first
// launch and left zero by every launch. Launches sharing ws and cnt must not overlap.
extern "C" __global__ void __launch_bounds__(512)
    x0ne_gemm_few_bal_bf16(const bf16_t* __restrict__ w, const bf16_t* __restrict__ x, void* __restrict__ y,
                           uint32_t rows, uint32_t cols, uint32_t n, uint32_t flags, uint32_t T, float* __restrict__ ws,
                           uint32_t* __restrict__ cnt) {
    __shared__ f32x4 stash[8 * 6 * 64];
    few_bal<8, 6, 8>(w, x, y, rows, cols, n, flags, T, ws, cnt, stash);
}

// ---- exact sums: Y[n][rows] = X[n][cols] W^T, every product summed in f64 ----
// The exact mode's prefill passes (the f64 sums of the exact GEMV, gemv.hip, over many rows):
// W [rows][cols] and X [n][cols] bf16 row-major, the products exact on the f64 matrix cores
// (v_mfma_f64_16x16x4_f64, W the A operand: 16 features x 4 k; X the B operand: 4 k x 16
// tokens), f64 accumulators, and Y = bf16(f32(sum)) or f32(sum): the exact GEMV's rounding.
//  - A wavefront owns 16 TF features x 16 TT tokens over all of K and works alone (no LDS, no
//    barrier): at 64 cycles per product on MI355X the matrix cores, not the loads, bound it, so
//    its operands come straight from memory (the L2), one step of 32 columns ahead.
//  - In a step lane l loads 16 bytes, columns k0 + 8 (l / 16) .. + 7, of W row 16 f + l % 16
//    and of X row 16 t + l % 16; product e (0..7) of the step feeds element e of both, so lane
//    group l / 16 supplies column k0 + 8 (l / 16) + e and each product sums 4 columns.
//  - Each output is summed in a fixed order (steps, then products within a step, then the
//    product's own 4 columns): the same bits from call to call, within f64 rounding of the
//    oracle's sequential sum.
//  - A wavefront's steps run one after the other (8 x 16 products of 64 cycles per step at
//    64 x 64 outputs), so a launch is as long as the fullest SIMD's wavefronts: 333 x 24576 x 4096
//    in 64 x 64 tiles is 2.25 wavefronts per SIMD and takes the time of 3. The host picks the
//    tile (16 x 16, 32 x 32, 48 x 48 or 64 x 32) and the slices of K (exact_gemm); with ks > 1
//    the steps are cut into ks equal runs, wavefront (tile, slice) writes its f64 partial sums
//    to ws[slice][token][feature], and x0ne_gemm_f64_reduce adds the slices in slice order.
// Wavefronts are numbered tokens fastest, then slices, so neighbouring wavefronts share W rows.
namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

template <int TF, int TT>
__device__ __forceinline__ void gemm_f64(const bf16_t* __restrict__ w, const bf16_t* __restrict__ x,
                                         void* __restrict__ y, uint32_t rows, uint32_t cols, uint32_t n,
                                         uint32_t out_f32, uint32_t ks, double* __restrict__ ws) {
    const uint32_t lane = threadIdx.x & 63, V = blockDim.x >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tiles_t = (n + 16 * TT - 1) / (16 * TT), tiles_f = (rows + 16 * TF - 1) / (16 * TF);
    const uint32_t id = blockIdx.x * V + wave;
    if (cols % 8 != 0 || out_f32 > 1 || ks == 0 || (ks > 1 && ws == nullptr) ||
        (uint64_t)id >= (uint64_t)tiles_f * tiles_t * ks)
        return;  // wavefront-uniform; no barrier
    const uint32_t tile = id / (tiles_t * ks) * tiles_t + id % tiles_t, slice = id / tiles_t % ks;
    const uint32_t ft = tile / tiles_t, tt = tile % tiles_t, r = lane & 15, q = lane >> 4;
    const auto wr = rsrc(w, (uint64_t)rows * cols * 2);
    const auto xr = rsrc(x, (uint64_t)n * cols * 2);
    f64x4 acc[TF][TT];
#pragma unroll
    for (int f = 0; f < TF; ++f)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[f][t] = f64x4{0.0, 0.0, 0.0, 0.0};
    uint4 a[2][TF], b[2][TT];
    const uint32_t all = (cols + 31) / 32, s_lo = all * slice / ks, steps = all * (slice + 1) / ks;
    auto load = [&](int buf, uint32_t s) {
        const uint32_t k = 32 * s + 8 * q;
        const bool in = s < steps && k < cols;  // a K tail: pieces past the row read zeros
#pragma unroll
        for (int f = 0; f < TF; ++f) {
            const uint32_t row = 16 * (TF * ft + f) + r;
            a[buf][f] = bload<>(wr, in && row < rows ? (row * cols + k) * 2 : OFF_NONE);
        }
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const uint32_t tok = 16 * (TT * tt + t) + r;
            b[buf][t] = bload<>(xr, in && tok < n ? (tok * cols + k) * 2 : OFF_NONE);
        }
    };
    auto elem = [](const uint4& v, int e) -> double {
        const uint32_t u = e < 2 ? v.x : e < 4 ? v.y : e < 6 ? v.z : v.w;
        return (double)((e & 1) ? bf_hi(u) : bf_lo(u));
    };
    auto step = [&](int buf) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            double av[TF], bv[TT];
#pragma unroll
            for (int f = 0; f < TF; ++f) av[f] = elem(a[buf][f], e);
#pragma unroll
            for (int t = 0; t < TT; ++t) bv[t] = elem(b[buf][t], e);
#pragma unroll
            for (int f = 0; f < TF; ++f)
#pragma unroll
                for (int t = 0; t < TT; ++t) acc[f][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[f], bv[t], acc[f][t], 0, 0, 0);
        }
    };
    // Steps in pairs, so each register set is named statically, and no way out between the two: with
    // one the compiler keeps a second copy of the accumulators and moves them over every pair.
    load(0, s_lo);
    uint32_t s = s_lo;
    for (; s + 1 < steps; s += 2) {
        load(1, s + 1);
        step(0);
        load(0, s + 2);
        step(1);
    }
    if (s < steps) step(0);
    // acc[f][t][i]: feature 16 (TF ft + f) + l / 16 + 4 i, token 16 (TT tt + t) + l % 16 (the
    // f64 product's result rows interleave over the lane groups).
#pragma unroll
    for (int f = 0; f < TF; ++f)
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const uint32_t tok = 16 * (TT * tt + t) + r;
            if (tok >= n) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t feat = 16 * (TF * ft + f) + q + 4 * i;
                if (feat >= rows) continue;
                if (ks > 1) {
                    ws[((size_t)slice * n + tok) * rows + feat] = acc[f][t][i];
                    continue;
                }
                const float v = (float)acc[f][t][i];
                if (out_f32)
                    static_cast<float*>(y)[(size_t)tok * rows + feat] = v;
                else
                    static_cast<bf16_t*>(y)[(size_t)tok * rows + feat] = f2bf(v);
            }
        }
}

}  // namespace

// x0ne_gemm_f64_t{TT}[f{TF}]_bf16 (TF 4 unless named): grid ceil(ceil(rows / (16 TF))
// ceil(n / (16 TT)) ks / V), block 64 V threads (any V); cols a multiple of 8; W and X below
// 4 GiB - 16 bytes; out_f32 0 (bf16 Y) or 1 (f32 Y); ks 1 (Y written) or more (the partial sums
// into ws: [ks][n][rows] f64, then x0ne_gemm_f64_reduce).
#define X0NE_GEMM_F64(NAME, TF, TT)                                                                               \
    extern "C" __global__ void __launch_bounds__(256)                                                              \
        NAME(const bf16_t* __restrict__ w, const bf16_t* __restrict__ x, void* __restrict__ y, uint32_t rows,      \
             uint32_t cols, uint32_t n, uint32_t out_f32, uint32_t ks, double* __restrict__ ws) {                 \
        gemm_f64<TF, TT>(w, x, y, rows, cols, n, out_f32, ks, ws);                                                 \
    }
// t1 and t4 (64 x 16, 64 x 64) are for callers of the kernel table, who name them. exact_gemm does
// without: of 962 shapes swept t4 was faster than the pick on 5, by at most 4 % (4096 x 12288 by 256).
X0NE_GEMM_F64(x0ne_gemm_f64_t1_bf16, 4, 1)
X0NE_GEMM_F64(x0ne_gemm_f64_t2_bf16, 4, 2)
X0NE_GEMM_F64(x0ne_gemm_f64_t4_bf16, 4, 4)
X0NE_GEMM_F64(x0ne_gemm_f64_t1f1_bf16, 1, 1)
X0NE_GEMM_F64(x0ne_gemm_f64_t2f2_bf16, 2, 2)
X0NE_GEMM_F64(x0ne_gemm_f64_t3f3_bf16, 3, 3)

// ---- exact sums for a few rows: 4-token quads ----
// The same product for n <= 32 rows of X on v_mfma_f64_4x4x4f64, which computes 4 blocks b of
// D[4][4] += A[4][4] B[4][4] with lane l = 16 k + 4 b + x holding A_b[x][k], B_b[k][x] and
// D_b[l / 16][x] (about 18 cycles per product against 64 for the 16x16x4 product, the same f64
// rate): A is W as in gemm_f64 (lane l loads row 16 f + l % 16, columns k0 + 8 (l / 16) ..), B
// the quad's 4 tokens (lane l loads token 4 t + l % 4, the same columns), so a wavefront covers
// 16 TF features x 4 TQ tokens without padding 20 rows to 32. D of lane l: feature
// 16 f + 4 ((l % 16) / 4) + l / 16, token 4 t + l % 4.
namespace {

template <int TF, int TQ>
__device__ __forceinline__ void gemm_f64_quads(const bf16_t* __restrict__ w, const bf16_t* __restrict__ x,
                                               void* __restrict__ y, uint32_t rows, uint32_t cols, uint32_t n,
                                               uint32_t out_f32, uint32_t ks, double* __restrict__ ws) {
    const uint32_t lane = threadIdx.x & 63, V = blockDim.x >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tiles_f = (rows + 16 * TF - 1) / (16 * TF);
    const uint32_t id = blockIdx.x * V + wave;
    if (cols % 8 != 0 || out_f32 > 1 || ks == 0 || (ks > 1 && ws == nullptr) || n > 4u * TQ ||
        (uint64_t)id >= (uint64_t)tiles_f * ks)
        return;  // wavefront-uniform; no barrier
    const uint32_t ft = id / ks, slice = id % ks;
    const uint32_t r = lane & 15, q = lane >> 4, xq = lane & 3;
    const auto wr = rsrc(w, (uint64_t)rows * cols * 2);
    const auto xr = rsrc(x, (uint64_t)n * cols * 2);
    double acc[TF][TQ];
#pragma unroll
    for (int f = 0; f < TF; ++f)
#pragma unroll
        for (int t = 0; t < TQ; ++t) acc[f][t] = 0.0;
    uint4 a[2][TF], b[2][TQ];
    const uint32_t all = (cols + 31) / 32, s_lo = all * slice / ks, steps = all * (slice + 1) / ks;
    auto load = [&](int buf, uint32_t s) {
        const uint32_t k = 32 * s + 8 * q;
        const bool in = s < steps && k < cols;
#pragma unroll
        for (int f = 0; f < TF; ++f) {
            const uint32_t row = 16 * (TF * ft + f) + r;
            a[buf][f] = bload<>(wr, in && row < rows ? (row * cols + k) * 2 : OFF_NONE);
        }
#pragma unroll
        for (int t = 0; t < TQ; ++t) {
            const uint32_t tok = 4 * t + xq;
            b[buf][t] = bload<>(xr, in && tok < n ? (tok * cols + k) * 2 : OFF_NONE);
        }
    };
    auto elem = [](const uint4& v, int e) -> double {
        const uint32_t u = e < 2 ? v.x : e < 4 ? v.y : e < 6 ? v.z : v.w;
        return (double)((e & 1) ? bf_hi(u) : bf_lo(u));
    };
    auto step = [&](int buf) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            double av[TF], bv[TQ];
#pragma unroll
            for (int f = 0; f < TF; ++f) av[f] = elem(a[buf][f], e);
#pragma unroll
            for (int t = 0; t < TQ; ++t) bv[t] = elem(b[buf][t], e);
#pragma unroll
            for (int f = 0; f < TF; ++f)
#pragma unroll
                for (int t = 0; t < TQ; ++t) acc[f][t] = __builtin_amdgcn_mfma_f64_4x4x4f64(av[f], bv[t], acc[f][t], 0, 0, 0);
        }
    };
    load(0, s_lo);
    uint32_t s = s_lo;
    for (; s + 1 < steps; s += 2) {
        load(1, s + 1);
        step(0);
        load(0, s + 2);
        step(1);
    }
    if (s < steps) step(0);
#pragma unroll
    for (int f = 0; f < TF; ++f)
#pragma unroll
        for (int t = 0; t < TQ; ++t) {
            const uint32_t tok = 4 * t + xq, feat = 16 * (TF * ft + f) + 4 * (r / 4) + q;
            if (tok >= n || feat >= rows) continue;
            if (ks > 1) {
                ws[((size_t)slice * n + tok) * rows + feat] = acc[f][t];
                continue;
            }
            const float v = (float)acc[f][t];
            if (out_f32)
                static_cast<float*>(y)[(size_t)tok * rows + feat] = v;
            else
                static_cast<bf16_t*>(y)[(size_t)tok * rows + feat] = f2bf(v);
        }
}

}  // namespace

// x0ne_gemm_f64_q{TQ}_bf16: x0ne_gemm_f64_t*_bf16's arguments for 1 <= n <= 4 TQ rows; grid
// ceil(ceil(rows / 64) ks / V), block 64 V threads (any V).
#define X0NE_GEMM_F64_Q(TQ)                                                                                       \
    extern "C" __global__ void __launch_bounds__(256) x0ne_gemm_f64_q##TQ##_bf16(                                 \
        const bf16_t* __restrict__ w, const bf16_t* __restrict__ x, void* __restrict__ y, uint32_t rows,          \
        uint32_t cols, uint32_t n, uint32_t out_f32, uint32_t ks, double* __restrict__ ws) {                      \
        gemm_f64_quads<4, TQ>(w, x, y, rows, cols, n, out_f32, ks, ws);                                            \
    }
X0NE_GEMM_F64_Q(1)
X0NE_GEMM_F64_Q(2)
X0NE_GEMM_F64_Q(3)
X0NE_GEMM_F64_Q(4)
X0NE_GEMM_F64_Q(5)
X0NE_GEMM_F64_Q(6)
X0NE_GEMM_F64_Q(7)
X0NE_GEMM_F64_Q(8)

// x0ne_gemm_f64_reduce: y[t][f] = the f32 (out_f32 1) or bf16 of the f32 of sum over slices 0 ..
// ks - 1, in that order, of ws[slice][t][f] (f64); grid ceil(n rows / 256), block 256.
extern "C" __global__ void __launch_bounds__(256)
    x0ne_gemm_f64_reduce(const double* __restrict__ ws, void* __restrict__ y, uint32_t rows, uint32_t n, uint32_t ks,
                         uint32_t out_f32) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x, total = (uint64_t)rows * n;
    if (i >= total || ks == 0 || out_f32 > 1) return;
    double sum = ws[i];
    for (uint32_t s = 1; s < ks; ++s) sum += ws[(uint64_t)s * total + i];
    if (out_f32)
        static_cast<float*>(y)[i] = (float)sum;
    else
        static_cast<bf16_t*>(y)[i] = f2bf((float)sum);
}

// x0ne_panel_bf16: a row-major [rows][cols] bf16 matrix copied into 16-row panels (element (r, k)
// at panel_index(r, k, cols)), one 16-byte chunk per thread in destination order, so the writes
// are contiguous; grid ceil(rows cols / 8 / 256), block 256. rows a multiple of 16 and cols of 8,
// else nothing is written. The source and destination must not overlap.
extern "C" __global__ void __launch_bounds__(256)
    x0ne_panel_bf16(const bf16_t* __restrict__ src, bf16_t* __restrict__ dst, uint32_t rows, uint32_t cols) {
    if (rows % 16 != 0 || cols % 8 != 0) return;  // grid-uniform
    const uint64_t c8 = cols / 8, j = (uint64_t)blockIdx.x * 256 + threadIdx.x;  // destination chunk
    if (j >= (uint64_t)rows * c8) return;
    const uint64_t r = j / (16 * c8) * 16 + j % 16, k8 = j / 16 % c8;
    reinterpret_cast<uint4*>(dst)[j] = reinterpret_cast<const uint4*>(src)[r * c8 + k8];
}

// ---- many rows: Y[n][rows] = X[n][cols] W^T, compute-bound, on the matrix cores ----
// The prefill passes' projections (2048 rows of X at Qwen3 widths: 0.07-0.41 TFLOP a launch).
// A block of NWF x NWT wavefronts computes a tile of BF = NWF WF output features (W rows) by
// BT = NWT WT tokens (X rows); wavefront (wf, wt) holds WF x WT of it in f32 accumulators as
// (WF / 16) x (WT / 16) products v_mfma_f32_16x16x32_bf16 with W as the A operand (16 features x
// 32 k) and X as the B operand (16 tokens x 32 k), so each lane ends with 4 consecutive
// features of one token and stores them as one 8-byte (bf16) or 16-byte (f32) write.
//  - K passes in stages of 64 columns (two 32-column steps) through a ring of STAGES buffers in
//    LDS, filled by direct buffer-to-LDS loads (buffer_load_dwordx4 ... lds: no registers, no
//    VALU) issued STAGES stages ahead. One barrier per stage.
//  - The operands of each 32-column step are read from LDS into a second register set while the
//    products of the step before run, and the next stage's loads are issued among them, one read
//    or load between every few products, so the matrix cores wait for neither: 2048 x 24576 x 4096
//    317 us (1.30 PFLOP/s; a library product of that shape 322), x 6144 x 4096 95 (87), x 4096 x
//    12288 173 (175), x 4096 x 4096 64 (61).
//  - LDS holds 16 rows x 64 columns of an operand as 2 KiB, the two fragments (16 rows x 32 k)
//    that the products read; either layout is read without bank conflicts (256 bytes per clock,
//    measured on gfx950). Operands in 16-row panels (device.h: [rows / 16][cols / 8][16][8]): a
//    fragment is 1 KiB contiguous in memory and in LDS, in lane order. Row-major operands: one
//    load instruction fetches 8 rows x 128 bytes, whole cache lines, 8 neighbouring lanes on
//    each; row r's 16-byte chunk c lies at slot 8 (r % 8) + (c ^ r % 8) of its KiB, so that the
//    16 rows that a product reads at one chunk fall in different banks. Against 16 rows x 64
//    bytes per load (half a line each, no two neighbouring lanes on one): 2048 x 24576 x 4096
//    447 -> 344 us, x 6144 x 4096 141 -> 100, panels 357 -> 334-343 and 105 -> 97-103
//    (rotating weights).
//  - A load past the matrix (a token past n, a feature past rows, k past cols) is a buffer load
//    at an offset past the buffer: zeros, no memory touched.
//  - A launch of few tiles cuts K into `slices` equal runs of stages (x0ne_gemm_tile_plan): block
//    (slice, tile) writes its f32 sums to parts[slice][token][feature] and
//    x0ne_gemm_tiles_reduce adds the slices in slice order. 200 x 4096 x 12288: 64 tiles, 158 us;
//    32 tiles of 256 x 128 in 8 slices, 40 us with the reduction (floor 16 us, W at 6.5 TB/s).
//  - Blocks in launch order go round the 8 XCDs (each with its own L2): they are renumbered so
//    each XCD takes a contiguous run of (slice, tile), tiles fastest, and a slice's tiles are
//    ordered TILE_GROUP feature tiles wide, tokens slowest, so the blocks an XCD holds at once
//    share their W and X pieces in its L2 (with 8 slices, each XCD reads its own eighth of K).
// Each output is summed over k by one wavefront per slice in a fixed order: bit-reproducible, and
// with one slice the same bits whatever the tile, the operands' layout or the number of tokens.
namespace {

constexpr int TILE_GROUP = 4;  // feature tiles side by side in one run of tiles
constexpr uint32_t TILE_F32 = 1, TILE_W_PANEL = 2, TILE_X_PANEL = 4;

constexpr int TILE_K = 2;  // 32-column steps per stage

template <int WF, int WT, int NWF, int NWT, int STAGES>
struct TileCfg {
    static constexpr int NW = NWF * NWT;
    static constexpr int BF = NWF * WF, BT = NWT * WT;  // block tile: features x tokens
    static constexpr int WFR = BF / 16, XFR = BT / 16;   // 16-row groups per stage
    static constexpr int FR = WFR + XFR;
    static constexpr int LOADS = TILE_K * FR / NW;       // load instructions per wavefront per stage
    static constexpr int GROUP = TILE_K * 1024;          // LDS bytes of a group's stage
    static constexpr int BYTES = FR * GROUP;             // one stage in LDS
    static constexpr int RA = WF / 16, RB = WT / 16;     // fragments a wavefront reads per step
    static_assert(FR % NW == 0 && WF % 16 == 0 && WT % 16 == 0, "tile shape");
    static_assert(STAGES >= 2 && STAGES * BYTES <= 160 * 1024, "LDS");
};

typedef int i32x4 __attribute__((ext_vector_type(4)));

// A raw buffer descriptor (the 48-bit base, stride 0, `bytes` records, word 3 of
// make_buffer_rsrc) as four scalar words, for the load below.
__device__ __forceinline__ i32x4 rsrc_words(const void* base, uint64_t bytes) {
    const uint64_t a = (uint64_t)base;
    const uint32_t n = bytes > OFF_NONE ? OFF_NONE : (uint32_t)bytes;
    return i32x4{(int)(uint32_t)a, (int)((uint32_t)(a >> 32) & 0xFFFFu), (int)n, (int)RSRC_WORD3};
}

// One direct buffer-to-LDS load (buffer_load_dwordx4 ... lds): lane l's 16 bytes at byte offset
// off + soff of the buffer (zeros past it) land at LDS byte lds + 16 l. Written as an instruction of
// its own so the compiler adds no wait of its own for it: the loop below counts these loads and
// waits for them itself. M0 holds the LDS address; nothing else in these kernels uses M0.
__device__ __forceinline__ void load_lds16(const i32x4& r, uint32_t lds, uint32_t off, uint32_t soff) {
    // The descriptor, the LDS address and soff are wavefront-uniform; read from lane 0 so they are
    // scalar registers whatever the compiler concluded.
    const i32x4 u = {__builtin_amdgcn_readfirstlane(r[0]), __builtin_amdgcn_readfirstlane(r[1]),
                     __builtin_amdgcn_readfirstlane(r[2]), __builtin_amdgcn_readfirstlane(r[3])};
    asm volatile("s_mov_b32 m0, %1\n\tbuffer_load_dwordx4 %0, %2, %3 offen lds" ::"v"(off),
                 "s"(__builtin_amdgcn_readfirstlane(lds)), "s"(u), "s"(__builtin_amdgcn_readfirstlane(soff))
                 : "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const uint8_t* p) {
    return __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)(p));
}

// s_waitcnt lgkmcnt(0) (vmcnt and expcnt at their maxima) through the compiler's builtin, so its
// own wait bookkeeping knows the LDS reads are done.
constexpr int WAIT_LGKM0 = 0xC07F;

template <int WF, int WT, int NWF, int NWT, int STAGES>
__device__ __forceinline__ void gemm_tiles(const bf16_t* __restrict__ w, const bf16_t* __restrict__ x,
                                           void* __restrict__ y, uint32_t rows, uint32_t cols, uint32_t n,
                                           uint32_t flags, uint32_t slices, float* __restrict__ parts, uint8_t* lds) {
    using C = TileCfg<WF, WT, NWF, NWT, STAGES>;
    const uint32_t tiles_f = (rows + C::BF - 1) / C::BF, tiles_t = (n + C::BT - 1) / C::BT;
    const uint32_t tiles = tiles_f * tiles_t, total = tiles * slices;
    // Launch id -> (slice, tile): ids alternate over the 8 XCDs, so block b runs on XCD b % 8; the
    // XCD's blocks b % 8, b % 8 + 8, .. take a contiguous run of total / 8 (and one of the rest).
    const uint32_t b = blockIdx.x, xcd = b & 7;
    const uint32_t id = xcd * (total >> 3) + min(xcd, total & 7) + (b >> 3);
    const uint32_t slice = id / tiles, seq = id - slice * tiles;
    const uint32_t group = seq / (TILE_GROUP * tiles_t), in_group = seq % (TILE_GROUP * tiles_t);
    const uint32_t width = min((uint32_t)TILE_GROUP, tiles_f - group * TILE_GROUP);
    const uint32_t f0 = (group * TILE_GROUP + in_group % width) * C::BF, t0 = in_group / width * C::BT;

    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wf = wave % NWF, wt = wave / NWF;
    const bool w_panel = flags & TILE_W_PANEL, x_panel = flags & TILE_X_PANEL;
    // Panels hold whole groups of 16 rows.
    const i32x4 wr = rsrc_words(w, (uint64_t)(w_panel ? (rows + 15) / 16 * 16 : rows) * cols * 2);
    const i32x4 xr = rsrc_words(x, (uint64_t)(x_panel ? (n + 15) / 16 * 16 : n) * cols * 2);
    const uint32_t all = (cols + 32 * TILE_K - 1) / (32 * TILE_K), c8 = cols / 8;
    // This slice's stages: first, first + 1, .. (counted from 0 below).
    const uint32_t first = (uint32_t)((uint64_t)all * slice / slices);
    const uint32_t stages = (uint32_t)((uint64_t)all * (slice + 1) / slices) - first;

    // This wavefront's loads of a stage: load h (0, 1) of 16-row group g = wave + NW (q / 2) (W's
    // groups first). In panels lane l fetches row l % 16, columns 32 h + 8 (l / 16) .. + 7 of the
    // stage; row-major, row 8 h + l / 8, columns 8 ((l % 8) ^ (l / 8)) .. + 7. A lane's offset in
    // its operand is voff[q] (past the buffer for a row that does not exist) and, the same for
    // every lane, w_step or x_step per stage; a stage that reaches past cols checks its columns.
    uint32_t voff[C::LOADS], chunk0[C::LOADS];
#pragma unroll
    for (int q = 0; q < C::LOADS; ++q) {
        const int h = q % TILE_K, g = (int)wave + C::NW * (q / TILE_K);
        const bool is_w = g < C::WFR;
        const uint32_t g16 = ((is_w ? f0 : t0) >> 4) + (uint32_t)(is_w ? g : g - C::WFR);
        const bool panel = is_w ? w_panel : x_panel;
        const uint32_t row = 16 * g16 + (panel ? 0 : 8 * h + (lane >> 3));
        chunk0[q] = panel ? 4 * h + (lane >> 4) : (lane & 7) ^ (lane >> 3);
        voff[q] = row >= (is_w ? rows : n) ? OFF_NONE
                  : panel                  ? g16 * c8 * 256 + 1024 * h + 16 * lane
                                           : row * cols * 2 + 16 * chunk0[q];
    }
    const uint32_t w_step = TILE_K * (w_panel ? 1024 : 64), x_step = TILE_K * (x_panel ? 1024 : 64);
    const uint32_t lds0 = lds_addr(lds) + wave * C::GROUP;
    auto load = [&](uint32_t s, int q) {
        const int h = q % TILE_K, g = C::NW * (q / TILE_K);
        const bool is_w = (int)wave + g < C::WFR;
        uint32_t off = voff[q];
        if (4 * TILE_K * (first + s + 1) > c8 && 4 * TILE_K * (first + s) + chunk0[q] >= c8) off = OFF_NONE;
        load_lds16(is_w ? wr : xr, lds0 + (s % STAGES) * C::BYTES + g * C::GROUP + h * 1024, off,
                   (first + s) * (is_w ? w_step : x_step));
    };

    f32x4 acc[C::RA][C::RB];
#pragma unroll
    for (int i = 0; i < C::RA; ++i)
#pragma unroll
        for (int j = 0; j < C::RB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 a0[C::RA], b0[C::RB], a1[C::RA], b1[C::RB];
    // Where lane l finds row l % 16, columns 32 kk + 8 (l / 16) .. + 7 of a group's stage.
    uint32_t w_at[TILE_K], x_at[TILE_K];
#pragma unroll
    for (int kk = 0; kk < TILE_K; ++kk) {
        const uint32_t r = lane & 15, c = 4 * kk + (lane >> 4);
        const uint32_t in_panel = kk * 1024 + lane * 16, in_rows = (r >> 3) * 1024 + ((r & 7) * 8 + (c ^ (r & 7))) * 16;
        w_at[kk] = (w_panel ? in_panel : in_rows) + wf * C::RA * C::GROUP;
        x_at[kk] = (x_panel ? in_panel : in_rows) + (C::WFR + wt * C::RB) * C::GROUP;
    }
    auto read = [&](uint32_t s, int kk, uint4 (&a)[C::RA], uint4 (&bx)[C::RB]) {
        const uint8_t* src = lds + (s % STAGES) * C::BYTES;
#pragma unroll
        for (int i = 0; i < C::RA; ++i) a[i] = *reinterpret_cast<const uint4*>(src + w_at[kk] + i * C::GROUP);
#pragma unroll
        for (int j = 0; j < C::RB; ++j) bx[j] = *reinterpret_cast<const uint4*>(src + x_at[kk] + j * C::GROUP);
    };
    // One step: the products of (a, bx); among them, evenly, the reads of the next step's operands
    // (step kk of stage s) into (na, nb) and, with LOAD, the loads of stage ls. The order is as
    // written: the loads in one run in front of the products left the matrix cores idle for it
    // (2048 x 24576 x 4096 346 -> 317 us; in the first half of the step 333).
    auto step = [&](const uint4 (&a)[C::RA], const uint4 (&bx)[C::RB], uint32_t s, int kk, uint4 (&na)[C::RA],
                    uint4 (&nb)[C::RB], bool loads, uint32_t ls) {
        const uint8_t* src = lds + (s % STAGES) * C::BYTES;
        constexpr int R = C::RA + C::RB, M = C::RA * C::RB;
        int m = 0;
#pragma unroll
        for (int g = 0; g < R; ++g) {
            if (loads)
#pragma unroll
                for (int q = g * C::LOADS / R; q < (g + 1) * C::LOADS / R; ++q) load(ls, q);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (; m < (g + 1) * M / R; ++m)
                acc[m / C::RB][m % C::RB] = mfma(a[m / C::RB], bx[m % C::RB], acc[m / C::RB][m % C::RB]);
            __builtin_amdgcn_sched_barrier(0);
            if (g < C::RA)
                na[g] = *reinterpret_cast<const uint4*>(src + w_at[kk] + g * C::GROUP);
            else
                nb[g - C::RA] = *reinterpret_cast<const uint4*>(src + x_at[kk] + (g - C::RA) * C::GROUP);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Prologue: stages 0 .. STAGES - 1 in flight, stage 0 complete (this wavefront's loads: at
    // most the later stages' in flight; then the barrier: every wavefront's), its first step's
    // operands read.
#pragma unroll
    for (int p = 0; p < STAGES; ++p)
        if ((uint32_t)p < stages) {
#pragma unroll
            for (int q = 0; q < C::LOADS; ++q) load(p, q);
        }
    if (stages >= (uint32_t)STAGES) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::LOADS * (STAGES - 1)) : "memory");
    } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    asm volatile("s_barrier" ::: "memory");
    read(0, 0, a0, b0);
    // The two steps of stage s alternate between the register sets; each step's products run while
    // the next step's operands are read. Before its last step: stage s + 1 complete in this
    // wavefront (at most min(stages - s - 2, STAGES - 2) later stages' loads in flight) and its own
    // reads of stage s done; the barrier: the same in every wavefront, so stage s's slot is no
    // longer read and takes stage s + STAGES. The last step's reads fetch stage s's again (harmless,
    // they keep the reads unconditional).
    auto turn = [&](uint32_t s) {
        if (s + 1 < stages) {
            if (stages - s - 2 >= (uint32_t)(STAGES - 2)) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::LOADS * (STAGES - 2)) : "memory");
            } else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
        }
        __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);
        asm volatile("s_barrier" ::: "memory");
    };
    static_assert(TILE_K == 2, "two steps per stage");
    uint32_t s = 0;
    for (; s + STAGES < stages; ++s) {
        step(a0, b0, s, 1, a1, b1, false, 0);
        turn(s);
        step(a1, b1, s + 1, 0, a0, b0, true, s + STAGES);
    }
    for (; s < stages; ++s) {
        step(a0, b0, s, 1, a1, b1, false, 0);
        turn(s);
        step(a1, b1, s + 1 < stages ? s + 1 : s, 0, a0, b0, false, 0);
    }

    // acc[i][j][r]: feature f0 + WF wf + 16 i + 4 (lane / 16) + r, token t0 + WT wt + 16 j + lane % 16.
    const bool out_f32 = flags & TILE_F32;
#pragma unroll
    for (int j = 0; j < C::RB; ++j) {
        const uint32_t t = t0 + WT * wt + 16 * j + (lane & 15);
        if (t >= n) continue;
#pragma unroll
        for (int i = 0; i < C::RA; ++i) {
            const uint32_t f = f0 + WF * wf + 16 * i + 4 * (lane >> 4);
            if (f >= rows) continue;
            const f32x4 v = acc[i][j];
            const size_t o = (size_t)t * rows + f;
            if (slices > 1) {
                *reinterpret_cast<f32x4*>(parts + (size_t)slice * n * rows + o) = v;
            } else if (out_f32) {
                *reinterpret_cast<f32x4*>(static_cast<float*>(y) + o) = v;
            } else {
                const uint32_t lo = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
                const uint32_t hi = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
                *reinterpret_cast<uint2*>(static_cast<bf16_t*>(y) + o) = make_uint2(lo, hi);
            }
        }
    }
}

}  // namespace

// Tiled GEMM kernels: grid ceil(rows / BF) ceil(n / BT) slices, block 64 NWF NWT; rows a multiple
// of 4, cols of 8 (and rows of 16 with W in panels), W and X below 4 GiB - 16 bytes, Y 8-byte
// (bf16) or 16-byte (f32) aligned; flags TILE_F32 | TILE_W_PANEL | TILE_X_PANEL; slices at most
// the stages of K, parts [slices][n][rows] f32 when more than one.
#define X0NE_TILES(NAME, WF, WT, NWF, NWT, STAGES)                                                              \
    extern "C" __global__ void __launch_bounds__(64 * NWF * NWT)                                                      \
        NAME(const bf16_t* __restrict__ w, const bf16_t* __restrict__ x, void* __restrict__ y, uint32_t rows,         \
             uint32_t cols, uint32_t n, uint32_t flags, uint32_t slices, float* __restrict__ parts) {                 \
        __shared__ __attribute__((aligned(1024))) uint8_t lds[STAGES * TileCfg<WF, WT, NWF, NWT, STAGES>::BYTES];     \
        if (rows % 4 != 0 || cols % 8 != 0 || n == 0 || slices == 0 || ((flags & TILE_W_PANEL) && rows % 16 != 0))    \
            return;                                                                                                   \
        gemm_tiles<WF, WT, NWF, NWT, STAGES>(w, x, y, rows, cols, n, flags, slices, parts, lds);                      \
    }
// Block tiles from sweeps on MI355X: 256 x 256 of 8 wavefronts (64 features x 128 tokens each; two per
// SIMD; four stages of 32 columns in their place: 5-7 % slower row-major, level in panels), 256 x 128
// of 8 and 128 x 128 of 4 (64 x 64 each), 64 x 64 of 4 (32 x 32 each, two blocks per CU) and 16 x 16 of
// one (ten blocks). 128 x 32 of two wavefronts was best for none of the Qwen3 projections but 10240 x
// 5120 by 17 to 32 (26 us, 64 x 64 28), and far off the best on 16384 columns. The small tiles
// stream W at 4-6 TB/s where the few-row kernels above, which read 64 bytes of 16 rows per load,
// reach 1-4 on row-major W: 16 x 51200 x 5120 147 -> 106 us, 64 x 24576 x 4096 129 -> 47.
X0NE_TILES(x0ne_gemm_tiles_256x256_bf16, 64, 128, 4, 2, 2)
X0NE_TILES(x0ne_gemm_tiles_256x128_bf16, 64, 64, 4, 2, 3)
X0NE_TILES(x0ne_gemm_tiles_128x128_bf16, 64, 64, 2, 2, 4)
X0NE_TILES(x0ne_gemm_tiles_64x64_bf16, 32, 32, 2, 2, 4)
X0NE_TILES(x0ne_gemm_tiles_16x16_bf16, 16, 16, 1, 1, 4)

// x0ne_gemm_tiles_reduce: y[t][f] = the f32 (flags TILE_F32) or bf16 of the sum over slices, in
// slice order, of parts[slice][t][f]; one thread per 4 features, grid ceil(n rows / 4 / 256),
// block 256; rows a multiple of 4. Bound by the parts' reads (from the L2 and the Infinity Cache).
extern "C" __global__ void __launch_bounds__(256)
    x0ne_gemm_tiles_reduce(const float* __restrict__ parts, void* __restrict__ y, uint32_t rows, uint32_t n,
                           uint32_t flags, uint32_t slices) {
    const uint64_t quads = (uint64_t)n * rows / 4, i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (rows % 4 != 0 || i >= quads) return;
    const f32x4* p = reinterpret_cast<const f32x4*>(parts) + i;
    f32x4 v = p[0];
    for (uint32_t s = 1; s < slices; ++s) v += p[s * quads];
    if (flags & TILE_F32) {
        static_cast<f32x4*>(y)[i] = v;
    } else {
        const uint32_t lo = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
        const uint32_t hi = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
        static_cast<uint2*>(y)[i] = make_uint2(lo, hi);
    }
}

// ---- typed launchers of the tiled GEMM (called by the runtime) ----

#include <algorithm>
#include <cmath>

#include "launch.h"

namespace {

struct TileKind {
    const void* fn;
    uint32_t bf, bt;  // block tile: features x tokens
    uint32_t threads;
    // The plan's estimate, us on MI355X: a round of blocks' start and end (a CU holds `resident` blocks at
    // once), one stage of a block alone on its CU, and one stage of each block where several share a
    // CU (0: they take turns).
    uint32_t resident;
    double fixed, stage, shared;
};

TileKind tile_kind(int tile) {
    switch (tile) {
        case X0NE_TILE_256x256: return {(const void*)&x0ne_gemm_tiles_256x256_bf16, 256, 256, 512, 1, 8.1, 1.52, 0};
        case X0NE_TILE_256x128: return {(const void*)&x0ne_gemm_tiles_256x128_bf16, 256, 128, 512, 1, 4.0, 0.96, 0};
        case X0NE_TILE_128x128: return {(const void*)&x0ne_gemm_tiles_128x128_bf16, 128, 128, 256, 1, 2.5, 0.83, 0};
        case X0NE_TILE_64x64: return {(const void*)&x0ne_gemm_tiles_64x64_bf16, 64, 64, 256, 2, 1.4, 0.26, 0.25};
        case X0NE_TILE_16x16: return {(const void*)&x0ne_gemm_tiles_16x16_bf16, 16, 16, 64, 10, 0.75, 0.155, 0.038};
        default: return {nullptr, 0, 0, 0, 1, 0, 0, 0};
    }
}

uint64_t tile_count(const TileKind& k, uint32_t rows, uint32_t n) {
    return (uint64_t)((rows + k.bf - 1) / k.bf) * ((n + k.bt - 1) / k.bt);
}

}  // namespace

// The tile and the K slices for a shape: the pair that an estimate of the time puts first. The
// estimate is a block's time per round and per stage over the blocks of the fullest CU, not less than
// W's stream (9.5 TB/s and 2 us) or the tiles' reads from the L2 (19.5 TB/s); 1.065 times it where
// all slices start on the same memory channels (rows and slices of whole 4 KiB: 4096 x 8192 by 2 in
// 3 slices 18.0 us, in 4 20.4; 4096 x 12288 by 17 in 3 28.3, in 4 23.8); and for several slices
// the reduction (1 us and the parts at 2.3 TB/s). The constants are fitted to sweeps on MI355X of the
// 12 Qwen3-0.6B, -8B and -32B projections by 2 to 2048 rows, row-major and in panels, and of a grid
// of 4 to 65536 x 8 to 16384 by 2 to 1000, weights rotating: over the projections the picked pair takes
// 1.0 % longer than the best one on average and 18 % at worst, over the grid 2.0 and 30 % (a round's
// blocks without their start and end, no 128 x 128, and 128 x 32: 1.9 and 20 %, 4.0 and 93 %: 65536 x
// 128 by 512 57 us in 64 x 64 tiles, 31 in 256 x 256).
X0neTilePlan x0ne_gemm_tile_plan(uint32_t rows, uint32_t cols, uint32_t n, uint32_t cus, uint64_t parts_bytes) {
    const uint32_t stages = (cols + 63) / 64;
    X0neTilePlan best = {X0NE_TILE_256x256, 1};
    double best_us = 1e30;
    auto four = [](double a) { return a * a * a * a; };
    for (int tile : {X0NE_TILE_16x16, X0NE_TILE_64x64, X0NE_TILE_128x128, X0NE_TILE_256x128, X0NE_TILE_256x256}) {
        const TileKind k = tile_kind(tile);
        const uint64_t tiles = tile_count(k, rows, n), part = (uint64_t)n * rows * 4;
        const double stream = 2.0 + 2.0 * rows * cols / 9.5e6, reads = (double)tiles * stages * (k.bf + k.bt) * 128 / 19.5e6;
        for (uint32_t slices : {1u, 2u, 3u, 4u, 6u, 8u, 12u, 16u}) {
            if (tiles * slices * k.threads > UINT32_MAX) break;  // more than HIP launches
            // A slice holds at least 4 stages, and all slices' blocks come to a few per CU at most.
            if (slices > 1 && (slices > stages / 4 || slices * part > parts_bytes || tiles * slices > 24ull * cus)) break;
            const double per_cu = std::ceil((double)(tiles * slices) / cus), rounds = std::ceil(per_cu / k.resident);
            const double steps = std::ceil((double)stages / slices);
            double us = rounds * k.fixed + steps * (k.shared > 0 ? std::max(per_cu * k.shared, k.stage) : per_cu * k.stage);
            us = std::sqrt(std::sqrt(four(us) + four(stream) + four(reads)));
            if (slices > 1) {
                if (cols % 2048 == 0 && stages % slices == 0 && stages / slices % 32 == 0) us *= 1.065;
                us += 1.0 + (double)slices * part / 2.3e6;
            }
            if (us < best_us) best_us = us, best = {tile, slices};
        }
    }
    return best;
}

hipError_t x0ne_launch_gemm_tiles(X0neTilePlan plan, const void* w, const void* x, void* y, uint32_t rows, uint32_t cols,
                                  uint32_t n, uint32_t flags, float* parts, hipStream_t s) {
    const TileKind k = tile_kind(plan.tile);
    uint32_t slices = plan.slices;
    if (!k.fn || rows % 4 != 0 || cols % 8 != 0 || n == 0 || flags > 7 || ((flags & TILE_W_PANEL) && rows % 16 != 0) ||
        slices == 0 || (slices > 1 && (!parts || slices > (cols + 63) / 64)))
        return hipErrorInvalidValue;
    const uint64_t blocks = tile_count(k, rows, n) * slices;
    if (blocks > 0x7FFFFFFFull) return hipErrorInvalidValue;
    void* args[] = {(void*)&w, (void*)&x, (void*)&y, (void*)&rows, (void*)&cols, (void*)&n, (void*)&flags, (void*)&slices, (void*)&parts};
    const hipError_t e = x0ne_launch(k.fn, dim3((uint32_t)blocks), dim3(k.threads), args, 0, s);
    if (e != hipSuccess || slices == 1) return e;
    void* rargs[] = {(void*)&parts, (void*)&y, (void*)&rows, (void*)&n, (void*)&flags, (void*)&slices};
    return x0ne_launch((const void*)&x0ne_gemm_tiles_reduce, dim3((uint32_t)(((uint64_t)n * rows / 4 + 255) / 256)),
                       dim3(256), rargs, 0, s);
}
