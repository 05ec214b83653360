// GQA decode attention over the paged KV arena, for gfx950 (64-lane wavefronts).
//
// Semantics follow x0ne-core/kernels/cuda/attention.cu: the query at position pos[0] attends
// keys 0..pos[0] (ctx = min(pos + 1, max_ctx)); q head h reads kv head h / (q_heads / kv_heads);
// scores q.k / sqrt(128); softmax with the maximum subtracted; f32 accumulation. Split-K
// (attention.cu:161-251): the keys are cut in tiles at absolute positions, a block of slice y
// takes its share of them and writes a partial state (m, l, o[128]) per q head at
// state[(h * P + y) * 132]; the merge (attention.cu:253-280) combines slices 0..active-1 in that
// fixed order. The result depends on the inputs, ctx and P only.
//
// The layout and the work split are this build's own, shaped for CDNA:
//  - K planes are paged [pages][kv_heads][16][128] bf16 (key rows), V planes
//    [pages][kv_heads][128][16] (dim-major: the operand layout of the matrix-core P V),
//    page_table[pos / 16] the physical page. A tile is 64 keys (4 pages); a block is 4
//    wavefronts. Slice y of P takes a contiguous run of tiles (a multiple of 4), its wavefront w
//    the tiles w, w + 4, ... of the run, so a block reads 256 consecutive keys at a time.
//  - The fp32 kernels run on the matrix cores (attend_wave_mfma): S^T = K Q^T and O = P V as
//    16x16x32 bf16 products with fp32 accumulation, the G q heads of a kv head padded to 16, the
//    tiles of a wavefront pipelined (the next tile's K and V requested while the current one is
//    computed) through branch-free buffer loads.
//  - The f64 (exact) mode and the per-head kernels run on the vector units (attend_wave): lane
//    (r = lane / 16, b = lane % 16) holds dims 8b..8b+7 of key rows 4i + r; its partial dot
//    products are summed over the 16 lanes of a row by a transposing butterfly (each step halves
//    the vector), scores and weights pass once through LDS, and lane d accumulates dims d and
//    d + 64 over the tile's keys.
//  - The 4 wavefronts' states are merged in LDS; a block that covers the whole context (ctx of at
//    most 256, or P = 1) writes the output directly, without a state, a counter or a second pass.
//  - The fused variant starts with the QK-norm + RoPE of its G q heads (into LDS) and, in the
//    block that owns position pos, the K/V write of that position's row (rope.cu:7-47), so a
//    decode step's attention is one launch.
#include "device.h"
#include "kernels.h"

namespace {

constexpr int WAVES = 4;
constexpr int BLOCK = 64 * WAVES;
constexpr uint32_t BLOCK_TILES = WAVES;  // tiles of 64 keys per block-tile
constexpr uint32_t MERGE_MAX = 256;      // most slices a merge takes (P is capped at this)

// The split of ctx keys over P slices: tiles of 64 keys, each slice a contiguous run of `per`
// tiles (a multiple of the 4 a block takes at a time), `active` slices holding at least one.
// Slice y takes tiles [y per, min((y + 1) per, ntiles)); wavefront w of its block the tiles
// y per + w, + 4, ..., so the block reads 256 consecutive keys at a time.
struct Split {
    uint32_t ntiles, per, active;
};
__device__ __forceinline__ Split split_of(uint32_t ctx, uint32_t P) {
    Split s;
    s.ntiles = (ctx + X0NE_SPLIT_TILE - 1) / X0NE_SPLIT_TILE;
    const uint32_t groups = (s.ntiles + BLOCK_TILES - 1) / BLOCK_TILES;  // 4-tile groups
    s.per = BLOCK_TILES * ((groups + P - 1) / P);
    s.active = (s.ntiles + s.per - 1) / s.per;
    return s;
}

// Every LDS write this wavefront issued is done, and no memory access moves across this point.
__device__ __forceinline__ void wave_lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// The accumulation type T is float (the decode path) or double (the exact mode, whose sums
// follow the f64 oracle).
__device__ __forceinline__ float acc_exp(float x) { return expf(x); }
__device__ __forceinline__ double acc_exp(double x) { return exp(x); }
__device__ __forceinline__ float acc_fma(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double acc_fma(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float acc_max(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double acc_max(double a, double b) { return fmax(a, b); }
__device__ __forceinline__ float acc_wave_sum(float v) { return wave_sum(v); }
__device__ __forceinline__ double acc_wave_sum(double v) { return wave_sum_d(v); }
template <class T>
__device__ __forceinline__ T acc_wave_max(T v) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) v = acc_max(v, (T)__shfl_xor(v, o, 64));
    return v;
}

// One step of the transposing butterfly: lanes b and b ^ 2^K exchange halves of an N-vector;
// the lane whose bit K is 0 keeps the lower half, its partner the upper.
template <int N, int K, class T>
__device__ __forceinline__ void butterfly_step(T* a, uint32_t b) {
    constexpr int H = N >> 1;
    const bool bit = (b >> K) & 1u;
#pragma unroll
    for (int j = 0; j < H; ++j) {
        const T send = bit ? a[j] : a[j + H];
        const T keep = bit ? a[j + H] : a[j];
        a[j] = keep + __shfl_xor(send, 1 << K, 64);
    }
}

// Sum over the 16 lanes of a row, transposing: lane b (of a row) ends with values
// (N/16) * rev4(b) + e, e < N/16, of the original vector, in a[0..N/16).
template <int N, class T>
__device__ __forceinline__ void butterfly16(T* a, uint32_t b) {
    butterfly_step<N, 0>(a, b);
    butterfly_step<N / 2, 1>(a, b);
    butterfly_step<N / 4, 2>(a, b);
    butterfly_step<N / 8, 3>(a, b);
}

__device__ __forceinline__ uint32_t rev4(uint32_t b) {
    return ((b & 1u) << 3) | ((b & 2u) << 1) | ((b & 4u) >> 1) | ((b & 8u) >> 3);
}

// One wavefront: the G q heads in qs (G x 128 f32, LDS) over kv head kh, tiles t0, t0 + tstep,
// ... below ntiles. Leaves per head the running max m, the sum l (whole, every lane) and
// o = sum exp(s - m) v for dims lane and lane + 64. lds: this wavefront's 2 * G * 64 values. A
// wavefront without a tile leaves m = -inf.
template <int G, class T>
__device__ __forceinline__ void attend_wave(const float* qs, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
                                            const uint32_t* __restrict__ pages, uint32_t kh, uint32_t kv_heads,
                                            uint32_t ctx, uint32_t t0, uint32_t tstep, uint32_t t_end, T scale,
                                            T* lds, T m[G], T l[G], T o[G][2]) {
    constexpr int HGMAX = sizeof(T) == 4 ? 4 : 2;  // heads per score pass (registers)
    constexpr int HG = G < HGMAX ? G : HGMAX;
    constexpr int PASSES = G / HG;
    T* s_lds = lds;           // [G][64] scores of the tile's keys
    T* p_lds = lds + G * 64;  // [G][64] their softmax weights
    const uint32_t lane = threadIdx.x & 63, r = lane >> 4, b = lane & 15;
    const uint32_t ntiles = (ctx + X0NE_SPLIT_TILE - 1) / X0NE_SPLIT_TILE;

    T lsum[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        m[g] = -INFINITY;
        lsum[g] = 0;
        o[g][0] = 0;
        o[g][1] = 0;
    }

    const uint32_t tend = min(t_end, ntiles);
    for (uint32_t t = t0; t < tend; t += tstep) {
        const uint32_t base = t * X0NE_SPLIT_TILE;
        // Rows 4i + r of the tile: page base/16 + i/4, slot 4 (i % 4) + r. A page is looked up
        // only when its first key is below ctx (the table holds ceil(ctx / 16) pages at least).
        uint32_t pg[4];
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) {
            const uint32_t first = base + X0NE_PAGE * ii;
            pg[ii] = first < ctx ? pages[first / X0NE_PAGE] : 0u;
        }
        uint32_t off[16];
        bool valid[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            valid[i] = base + 4 * i + r < ctx;
            off[i] = ((pg[i >> 2] * kv_heads + kh) * X0NE_PAGE + 4 * (i & 3) + r) * X0NE_HEAD_DIM + 8 * b;
        }
        // K and V together (the f64 mode loads V after the scores, for registers). K: rows 4i + r,
        // dims 8b..8b+7. V (dim-major pages): vv[4 pp + 2 dh + kk] holds keys 16 pp + 8 kk ..
        // + 7 of the tile at dim lane + 64 dh. Rows past ctx are zero (their weight is 0, and a
        // zero keeps a value that is not a number out of the sum).
        uint4 kv[16], vv[16];
        auto load_v = [&] {
#pragma unroll
            for (int pp = 0; pp < 4; ++pp) {
                const bool live = base + X0NE_PAGE * pp < ctx;
                const bf16_t* vp = vc + (size_t)(pg[pp] * kv_heads + kh) * X0NE_HEAD_DIM * X0NE_PAGE;
#pragma unroll
                for (int dh = 0; dh < 2; ++dh)
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk)
                        vv[4 * pp + 2 * dh + kk] =
                            live ? *reinterpret_cast<const uint4*>(vp + (lane + 64 * dh) * X0NE_PAGE + 8 * kk)
                                 : make_uint4(0, 0, 0, 0);
            }
        };
#pragma unroll
        for (int i = 0; i < 16; ++i)
            kv[i] = valid[i] ? *reinterpret_cast<const uint4*>(kc + off[i]) : make_uint4(0, 0, 0, 0);
        if constexpr (sizeof(T) == 4) load_v();

#pragma unroll
        for (int pass = 0; pass < PASSES; ++pass) {
            T qf[HG][8];
#pragma unroll
            for (int g = 0; g < HG; ++g) {
                const float4 q0 = *reinterpret_cast<const float4*>(qs + (pass * HG + g) * X0NE_HEAD_DIM + 8 * b);
                const float4 q1 = *reinterpret_cast<const float4*>(qs + (pass * HG + g) * X0NE_HEAD_DIM + 8 * b + 4);
                qf[g][0] = q0.x; qf[g][1] = q0.y; qf[g][2] = q0.z; qf[g][3] = q0.w;
                qf[g][4] = q1.x; qf[g][5] = q1.y; qf[g][6] = q1.z; qf[g][7] = q1.w;
            }
            T part[16 * HG];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const T k0 = bf_lo(kv[i].x), k1 = bf_hi(kv[i].x), k2 = bf_lo(kv[i].y), k3 = bf_hi(kv[i].y);
                const T k4 = bf_lo(kv[i].z), k5 = bf_hi(kv[i].z), k6 = bf_lo(kv[i].w), k7 = bf_hi(kv[i].w);
#pragma unroll
                for (int g = 0; g < HG; ++g) {
                    T d = qf[g][0] * k0;
                    d = acc_fma(qf[g][1], k1, d);
                    d = acc_fma(qf[g][2], k2, d);
                    d = acc_fma(qf[g][3], k3, d);
                    d = acc_fma(qf[g][4], k4, d);
                    d = acc_fma(qf[g][5], k5, d);
                    d = acc_fma(qf[g][6], k6, d);
                    d = acc_fma(qf[g][7], k7, d);
                    part[i * HG + g] = d;
                }
            }
            butterfly16<16 * HG>(part, b);
            // Lane holds values HG * rev4(b) + e: row slot i = v / HG, head g = v % HG.
#pragma unroll
            for (int e = 0; e < HG; ++e) {
                const uint32_t v = HG * rev4(b) + e;
                const uint32_t i = v / HG, g = v % HG;
                const uint32_t row = 4 * i + r;
                const T s = (base + row < ctx) ? part[e] * scale : (T)-INFINITY;
                s_lds[(pass * HG + g) * 64 + row] = s;
            }
        }
        wave_lds_sync();
        if constexpr (sizeof(T) == 8) load_v();

        // Online softmax, lane = key of the tile.
        T alpha[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const T s = s_lds[g * 64 + lane];
            const T mn = acc_max(m[g], acc_wave_max(s));  // key `base` is below ctx: mn is finite
            alpha[g] = acc_exp(m[g] - mn);
            const T p = acc_exp(s - mn);
            lsum[g] = lsum[g] * alpha[g] + p;
            m[g] = mn;
            p_lds[g * 64 + lane] = p;
        }
        wave_lds_sync();

#pragma unroll
        for (int g = 0; g < G; ++g) {
            o[g][0] *= alpha[g];
            o[g][1] *= alpha[g];
        }
        // Keys past ctx inside a live page hold anything: their values are taken as 0.
#pragma unroll
        for (int pp = 0; pp < 4; ++pp)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                const uint4 w0 = vv[4 * pp + kk], w1 = vv[4 * pp + 2 + kk];
                const uint32_t u0[4] = {w0.x, w0.y, w0.z, w0.w}, u1[4] = {w1.x, w1.y, w1.z, w1.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t key = X0NE_PAGE * pp + 8 * kk + e;
                    const bool ok = base + key < ctx;
                    const T v0 = ok ? (T)((e & 1) ? bf_hi(u0[e >> 1]) : bf_lo(u0[e >> 1])) : (T)0;
                    const T v1 = ok ? (T)((e & 1) ? bf_hi(u1[e >> 1]) : bf_lo(u1[e >> 1])) : (T)0;
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        const T p = p_lds[g * 64 + key];
                        o[g][0] = acc_fma(p, v0, o[g][0]);
                        o[g][1] = acc_fma(p, v1, o[g][1]);
                    }
                }
            }
        wave_lds_sync();  // the next tile rewrites s_lds and p_lds
    }
    // Whole sums: l over the 64 keys' lanes (o is whole in each lane already).
#pragma unroll
    for (int g = 0; g < G; ++g) l[g] = acc_wave_sum(lsum[g]);
}

// ---- the matrix-core path (fp32 accumulation) ----
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16x16x32(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two values to bf16 (f2bf's rounding), in one word: one v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    const bf16x2 v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
}

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;

// Raw buffer resources (gfx9 word 3): a load whose bytes are not all below `bytes` gives zeros
// and touches no memory, so a key past the context or a prefetch past the last tile needs no
// branch, and the compiler's waits before a use cover only the loads that use needs.
constexpr int RSRC_WORD3 = 0x00020000;
constexpr uint32_t OFF_NONE = 0xFFFFFFF0u;  // an offset past any plane: the load gives zeros

__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, RSRC_WORD3);
}

// The default cache policy: a non-temporal hint on the K/V tiles measured no faster at short
// contexts and 12 % slower at 32k keys on MI355X.
__device__ __forceinline__ uint4 bload16(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t uniform_off = 0) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)uniform_off, 0);
    return make_uint4((uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]);
}
// One word through the vector memory path: a page-table entry fetched ahead this way is waited
// for by the in-order vector count, not by the LDS count every LDS read in between waits on.
__device__ __forceinline__ uint32_t bload4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
}

// One wavefront on the matrix cores (v_mfma_f32_16x16x32_bf16; lane l: row or column l % 16,
// k = 8 (l / 16) .. + 7 of a 32-wide step; result rows 4 (l / 16) .. + 3, column l % 16). The
// G q heads are the 16 columns of S^T = K Q^T (heads past G are zero) and the 16 rows of
// O = P V. For a tile of 64 keys: four 16-key blocks X0, Y0, X1, Y1 of S^T (block (kp, h)
// row m is key 32 kp + 8 (m / 4) + 4 h + m % 4, so lane l ends with keys 32 kp + 8 (l / 16) +
// 0..7 of its head: the k = 8 (l / 16) .. + 7 slice of P's 32-key step kp, in registers), four
// 32-dim steps each; then P V over two 32-key steps and 8 blocks of 16 dims, V read from the
// dim-major pages (8 consecutive keys of one dim = 16 bytes). P enters as bf16 hi + lo (two
// products), so its rounding is about 2^-16 relative, below the fp32 accumulation's own.
//
// The tiles of a wavefront are pipelined: tile t + 1's K is requested right after tile t's
// S^T, its V right after tile t's P V, and the page-table entries a tile ahead of that, so a
// load is in flight while the matrix cores work. The planes are addressed by 32-bit byte
// offsets (a plane below 4 GiB - 16 bytes); only OFF_NONE falls outside their resources.
// prologue(qb) runs once the first tile's loads are issued and fills qb[s], the B operand of Q^T
// for step s (every wavefront of the block calls it: it may hold a barrier). fx names the key
// whose K and V rows come from LDS rather than from the loads. ctx bounds the keys the
// wavefront reads (ctx rows exist in the cache); ctx_col, at most ctx, those its lane's column
// attends (a causal prefill row's own position + 1; the decode query's is ctx). The first tile
// a wavefront takes holds a key below every column's ctx_col. Leaves m (running max) and l (sum)
// of head l % 16 in lane l, and o[nb][i] = O[head 4 (l / 16) + i][dim 16 nb + l % 16].
//
// The K and V rows of position pos as the block that writes them holds them in LDS: the
// wavefront whose tile holds pos takes them from there, since its loads may be served before the
// block's own write of that row lands (tile = ~0u: no such key).
struct NewRow {
    uint32_t tile, key;  // pos / 64 and pos % 64
    const bf16_t* k;     // LDS, 128 bf16: the rotated K row (16-byte aligned)
    const bf16_t* v;     // LDS, 128 bf16: the V row
};
// first_pages, when given, holds tile t0's four page-table entries, read before ctx was known.
template <class Prologue>
__device__ __forceinline__ void attend_wave_mfma(Prologue&& prologue, const NewRow& fx, const bf16_t* __restrict__ kc,
                                                 const bf16_t* __restrict__ vc, const uint32_t* __restrict__ pages, uint32_t kh, uint32_t kv_heads,
                                                 uint32_t ctx, uint32_t ctx_col, uint32_t t0, uint32_t tstep,
                                                 uint32_t t_end, float scale, float& m_out, float& l_out, f32x4 o[8],
                                                 const uint32_t* first_pages = nullptr) {
    const uint32_t lane = threadIdx.x & 63, n = lane & 15, q4 = lane >> 4;
    const uint32_t ntiles = min(t_end, (ctx + X0NE_SPLIT_TILE - 1) / X0NE_SPLIT_TILE);  // this wavefront's end
    const auto kr = plane_rsrc(kc, OFF_NONE), vr = plane_rsrc(vc, OFF_NONE);
    // Scores in units of log2 (scale log2 e folded in), so each weight is one exp2.
    const float scale2 = scale * LOG2E;
    float m_run = -INFINITY, lsum = 0.f;
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) o[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t head_b = kh * X0NE_PAGE * X0NE_HEAD_DIM * 2;             // kv head's block in a page, bytes
    const uint32_t page_b = kv_heads * X0NE_PAGE * X0NE_HEAD_DIM * 2;       // one page of one plane, bytes

    // Page-table entries of a tile (0 for pages past the context; their loads read nothing).
    auto tile_pages = [&](uint32_t t, uint32_t pg[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t first = t * X0NE_SPLIT_TILE + X0NE_PAGE * i;
            pg[i] = (t < ntiles && first < ctx) ? pages[first / X0NE_PAGE] : 0u;
        }
    };
    auto load_k = [&](uint32_t t, const uint32_t pg[4], uint4 (&ka)[2][2][4]) {
        const uint32_t base = t * X0NE_SPLIT_TILE;
#pragma unroll
        for (int kp = 0; kp < 2; ++kp)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t key = 32 * kp + 8 * (n >> 2) + 4 * h + (n & 3);
                const bool ok = t < ntiles && base + key < ctx;
                const uint32_t row = pg[key / X0NE_PAGE] * page_b + head_b + (key % X0NE_PAGE) * X0NE_HEAD_DIM * 2 + 16 * q4;
#pragma unroll
                for (int st = 0; st < 4; ++st) ka[kp][h][st] = bload16(kr, ok ? row + 64 * st : OFF_NONE);
            }
    };
    auto load_v = [&](uint32_t t, const uint32_t pg[4], uint4 (&vb)[2][8]) {
        const uint32_t base = t * X0NE_SPLIT_TILE;
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
            const uint32_t pp = 2 * kp + (q4 >> 1);
            const bool live = t < ntiles && base + X0NE_PAGE * pp < ctx;
            const uint32_t col = pg[pp] * page_b + head_b + 16 * (q4 & 1);
#pragma unroll
            for (int nb = 0; nb < 8; ++nb)
                vb[kp][nb] = bload16(vr, live ? col + (16 * nb + n) * X0NE_PAGE * 2 : OFF_NONE);
        }
    };

    uint32_t pg[4], pg_next[4];
    uint4 ka[2][2][4], vb[2][8];
    // Loads only for tiles that exist (wavefront-uniform branches): a load past the last tile
    // would still cost its address cycles in the CU's memory pipeline.
    if (first_pages) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            pg[i] = (t0 < ntiles && t0 * X0NE_SPLIT_TILE + X0NE_PAGE * i < ctx) ? first_pages[i] : 0u;
    } else {
        tile_pages(t0, pg);
    }
    if (t0 < ntiles) {
        load_k(t0, pg, ka);
        load_v(t0, pg, vb);
    }
    tile_pages(t0 + tstep, pg_next);
    uint4 qb[4];
    prologue(qb);  // while the first tile is in flight

    for (uint32_t t = t0; t < ntiles; t += tstep) {
        const uint32_t base = t * X0NE_SPLIT_TILE;
        if (t == fx.tile) {  // wavefront-uniform: key fx.key of this tile is the new row
            const uint32_t r = fx.key & 31, ksel = fx.key >> 5, hsel = (r >> 2) & 1u;
            if (n == 4 * (r >> 3) + (r & 3)) {
#pragma unroll
                for (int kp = 0; kp < 2; ++kp)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        if (kp == (int)ksel && h == (int)hsel) {
#pragma unroll
                            for (int st = 0; st < 4; ++st)
                                ka[kp][h][st] = *reinterpret_cast<const uint4*>(fx.k + 32 * st + 8 * q4);
                        }
            }
        }
        // S^T = K Q^T, then tile t + 1's K.
        f32x4 sacc[2][2];
#pragma unroll
        for (int kp = 0; kp < 2; ++kp)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int st = 0; st < 4; ++st) acc = mfma16x16x32(ka[kp][h][st], qb[st], acc);
                sacc[kp][h] = acc;
            }
        if (t + tstep < ntiles) load_k(t + tstep, pg_next, ka);
        // Scale, mask, and the online softmax of head n over the lane's 16 keys and the 3 other
        // lanes of the head (l ^ 16, l ^ 32).
        float sc[2][2][4];
        float mx = -INFINITY;
#pragma unroll
        for (int kp = 0; kp < 2; ++kp)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t key = 32 * kp + 8 * q4 + 4 * h + i;
                    sc[kp][h][i] = base + key < ctx_col ? sacc[kp][h][i] * scale2 : -INFINITY;
                    mx = fmaxf(mx, sc[kp][h][i]);
                }
        mx = rows_max(mx);
        const float mn = fmaxf(m_run, mx);  // key `base` is below ctx: mn is finite
        const float alpha = __builtin_amdgcn_exp2f(m_run - mn);
        m_run = mn;
        float psum = 0.f;
#pragma unroll
        for (int kp = 0; kp < 2; ++kp)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    sc[kp][h][i] = __builtin_amdgcn_exp2f(sc[kp][h][i] - mn);
                    psum += sc[kp][h][i];
                }
        lsum = lsum * alpha + psum;
        // O rows are heads 4 q4 + i: their factors come from lanes 4 q4 + i.
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float ai = __shfl(alpha, 4 * q4 + i, 64);
#pragma unroll
            for (int nb = 0; nb < 8; ++nb) o[nb][i] *= ai;
        }
        // Keys past ctx in a live page hold anything: their V values are taken as 0 (their weight
        // is 0, and 0 times a value that is not a number would not be).
        if (base + X0NE_SPLIT_TILE > ctx) {
#pragma unroll
            for (int kp = 0; kp < 2; ++kp) {
                const uint32_t k0 = base + 32 * kp + 8 * q4;
                const uint32_t valid = k0 >= ctx ? 0u : min(ctx - k0, 8u);  // keys kept, from the first
#pragma unroll
                for (int nb = 0; nb < 8; ++nb) {
                    uint32_t w[4] = {vb[kp][nb].x, vb[kp][nb].y, vb[kp][nb].z, vb[kp][nb].w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t keep = (2 * e + 1 < valid ? 0xFFFF0000u : 0u) | (2 * e < valid ? 0xFFFFu : 0u);
                        w[e] &= keep;
                    }
                    vb[kp][nb] = make_uint4(w[0], w[1], w[2], w[3]);
                }
            }
        }
        if (t == fx.tile && q4 == ((fx.key >> 3) & 3u)) {  // the new row's V: key fx.key % 8 of the lane's 8
            const uint32_t vsel = fx.key >> 5, e = fx.key & 7u;
            const uint32_t shift = 16 * (e & 1u), keep = shift ? 0x0000FFFFu : 0xFFFF0000u;
#pragma unroll
            for (int kp = 0; kp < 2; ++kp)
                if (kp == (int)vsel) {
#pragma unroll
                    for (int nb = 0; nb < 8; ++nb) {
                        uint32_t w[4] = {vb[kp][nb].x, vb[kp][nb].y, vb[kp][nb].z, vb[kp][nb].w};
                        const uint32_t val = (uint32_t)fx.v[16 * nb + n] << shift;
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (j == (int)(e >> 1)) w[j] = (w[j] & keep) | val;
                        vb[kp][nb] = make_uint4(w[0], w[1], w[2], w[3]);
                    }
                }
        }
        // O += P V, P as bf16 hi + lo; then tile t + 1's V and the pages of tile t + 2.
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
            float pv[8], lo[8];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pv[i] = sc[kp][0][i];
                pv[4 + i] = sc[kp][1][i];
            }
            uint32_t hw[4], lw[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                hw[j] = pack_bf16(pv[2 * j], pv[2 * j + 1]);
                lo[2 * j] = pv[2 * j] - bf_lo(hw[j]);  // exact
                lo[2 * j + 1] = pv[2 * j + 1] - bf_hi(hw[j]);
                lw[j] = pack_bf16(lo[2 * j], lo[2 * j + 1]);
            }
            const uint4 ahi = make_uint4(hw[0], hw[1], hw[2], hw[3]);
            const uint4 alo = make_uint4(lw[0], lw[1], lw[2], lw[3]);
#pragma unroll
            for (int nb = 0; nb < 8; ++nb) {
                o[nb] = mfma16x16x32(ahi, vb[kp][nb], o[nb]);
                o[nb] = mfma16x16x32(alo, vb[kp][nb], o[nb]);
            }
        }
        if (t + tstep < ntiles) load_v(t + tstep, pg_next, vb);
#pragma unroll
        for (int i = 0; i < 4; ++i) pg[i] = pg_next[i];
        tile_pages(t + 2 * tstep, pg_next);
    }
    const float l = rows_sum(lsum);
    m_out = m_run * LN2;  // back to natural units for the merges
    l_out = l;
}

// The shared memory of one block: q of its heads, each wavefront's exchange area, each
// wavefront's state for the block merge, each wavefront's slice weights for a global merge.
// VEC = false: the matrix-core kernels' (no vector-path q or exchange area).
template <int G, class T = float, bool VEC = true>
struct AttnShared {
    float qs[VEC ? G : 1][X0NE_HEAD_DIM];            // the vector-unit paths' q
    alignas(16) bf16_t qh[G][X0NE_HEAD_DIM];         // the matrix-core path's q (bf16)
    alignas(16) bf16_t knew[X0NE_HEAD_DIM], vnew[X0NE_HEAD_DIM];  // the fused variant's new K/V row
    T xch[VEC ? WAVES : 1][VEC ? 2 * G * 64 : 1];
    T wm[WAVES][G], wl[WAVES][G];
    T wo[WAVES][G][X0NE_HEAD_DIM];
    T wf[WAVES][G], mh[G], lh[G];  // the block merge's factors, maximum and sum per head
    float f[sizeof(T) == 4 ? WAVES : 1][MERGE_MAX];  // the exact mode has no global merge
    uint32_t last;
};


// The split states of the last-block merge are written and read only through agent-scope atomic
// stores and loads: coherent across the device (they bypass the per-XCD L2's write-back caching),
// so the count that elects the merging block needs no L2 writeback before it, only the stores'
// acknowledgments (a release fence would write the whole L2 back: ~4 µs per block measured).
__device__ __forceinline__ void state_put(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float state_get(const float* p) {
    return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Merge of one q head's slices 0..active-1 (FlashInfer's: M = max m_y, f_y = exp(m_y - M),
// l = sum l_y f_y, o = sum o_y f_y; one rounding, of o / l), the sums in a fixed order so the
// result depends on the states only. One wavefront; lane y holds slice y's (m, l) (and y + 64,
// ...), lane d owns dims d and d + 64 of o. Every load of a chunk of MERGE_CHUNK slices (their
// (m, l) and o values) is issued before any is used, so a merge of up to MERGE_CHUNK slices costs
// one round trip to memory. f: this wavefront's LDS for `active` floats. Every active slice saw a
// key, so each m is finite. The caller has made other workgroups' states visible (their release,
// its acquire): the loads are coherent.
constexpr uint32_t MERGE_CHUNK = 32;
template <class Store>
__device__ __forceinline__ void merge_head(const float* __restrict__ s, Store&& store, uint32_t active, float* f) {
    const uint32_t lane = threadIdx.x & 63;
    constexpr int MLK = MERGE_MAX / 64;
    float mv[MLK], lv[MLK];
#pragma unroll
    for (int k = 0; k < MLK; ++k) {
        const uint32_t y = lane + 64 * k;
        if (64 * k < active) {  // wave-uniform
            mv[k] = y < active ? state_get(s + (size_t)y * X0NE_SPLIT_STATE) : -INFINITY;
            lv[k] = y < active ? state_get(s + (size_t)y * X0NE_SPLIT_STATE + 1) : 0.f;
        }
    }
    float a[MERGE_CHUNK], b[MERGE_CHUNK];
    auto request = [&](uint32_t y0) {
#pragma unroll
        for (uint32_t k = 0; k < MERGE_CHUNK; ++k)
            if (y0 + k < active) {  // wave-uniform
                const float* st = s + (size_t)(y0 + k) * X0NE_SPLIT_STATE + 4;
                a[k] = state_get(st + lane);
                b[k] = state_get(st + lane + 64);
            }
    };
    request(0);
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < MLK; ++k)
        if (64 * k < active) mx = fmaxf(mx, mv[k]);
    mx = wave_max(mx);
    float lp = 0.f;
#pragma unroll
    for (int k = 0; k < MLK; ++k) {
        const uint32_t y = lane + 64 * k;
        if (64 * k < active && y < active) {
            const float fy = expf(mv[k] - mx);
            f[y] = fy;
            lp += lv[k] * fy;
        }
    }
    const float l = wave_sum(lp);
    wave_lds_sync();
    float o0 = 0.f, o1 = 0.f;
    for (uint32_t y0 = 0; y0 < active; y0 += MERGE_CHUNK) {
#pragma unroll
        for (uint32_t k = 0; k < MERGE_CHUNK; ++k)
            if (y0 + k < active) {
                o0 = fmaf(a[k], f[y0 + k], o0);
                o1 = fmaf(b[k], f[y0 + k], o1);
            }
        if (y0 + MERGE_CHUNK < active) request(y0 + MERGE_CHUNK);
    }
    store(lane, f2bf(o0 / l));
    store(lane + 64, f2bf(o1 / l));
    wave_lds_sync();
}

// The 4 wavefronts' states of a block merged (in wave order, a wavefront without a key skipped),
// per head g and dim d: threads 0..G-1 first take each head's maximum, factors and sum into LDS;
// then thread t takes the (g, d) pairs t, t + 256, ... and calls f(g, d, m, l, o). Every thread
// of the block calls it (it holds a barrier), after the wavefronts' states are in LDS.
template <int G, class T, bool V, class F>
__device__ __forceinline__ void block_merge(AttnShared<G, T, V>& sh, F f) {
    const uint32_t t = threadIdx.x;
    if (t < (uint32_t)G) {
        T mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) mx = acc_max(mx, sh.wm[w][t]);
        T l = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const bool seen = sh.wm[w][t] != (T)-INFINITY;  // the wavefront saw a key
            const T fw = seen ? acc_exp(sh.wm[w][t] - mx) : (T)0;
            sh.wf[w][t] = fw;
            if (seen) l += sh.wl[w][t] * fw;
        }
        sh.mh[t] = mx;
        sh.lh[t] = l;
    }
    lds_barrier();
    for (uint32_t k = t; k < (uint32_t)G * X0NE_HEAD_DIM; k += BLOCK) {
        const uint32_t g = k / X0NE_HEAD_DIM, d = k % X0NE_HEAD_DIM;
        T o = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w)
            if (sh.wm[w][g] != (T)-INFINITY) o += sh.wo[w][g][d] * sh.wf[w][g];
        f(g, d, sh.mh[g], sh.lh[g], o);
    }
}

// One head row's pair (lane i: elements i and i + 64) and its norm weights, as loaded.
struct RopeIn {
    float a, b, wa, wb;
};
__device__ __forceinline__ RopeIn rope_in(const bf16_t* __restrict__ src, const bf16_t* __restrict__ nw) {
    constexpr uint32_t HALF = X0NE_HEAD_DIM / 2;
    const uint32_t i = threadIdx.x & 63;
    return {bf2f(src[i]), bf2f(src[i + HALF]), bf2f(nw[i]), bf2f(nw[i + HALF])};
}

// QK-norm + RoPE of one head row (oracle/src/lib.rs:95-110; rope.cu:7-47): lane i owns the pair
// (i, i + 64); RMSNorm and the rotation in f64 by the angle whose cosine and sine are c and s.
// Returns the two rotated values, unrounded.
__device__ __forceinline__ void rope_rotate_cs(const RopeIn& r, double c, double s, float eps, float* ra,
                                               float* rb) {
    const double ss = wave_sum_d((double)r.a * (double)r.a + (double)r.b * (double)r.b);
    const double scale = 1.0 / sqrt(ss / (double)X0NE_HEAD_DIM + (double)eps);
    const double na = (double)r.a * scale * (double)r.wa;
    const double nb = (double)r.b * scale * (double)r.wb;
    *ra = (float)(na * c - nb * s);
    *rb = (float)(nb * c + na * s);
}

// rope_rotate_cs in two steps: the RMS norm, which does not depend on the position, then the
// rotation; the same operations in the same order, so the same bits.
struct RopeNormed {
    double na, nb;
};
__device__ __forceinline__ RopeNormed rope_norm(const RopeIn& r, float eps) {
    const double ss = wave_sum_d((double)r.a * (double)r.a + (double)r.b * (double)r.b);
    const double scale = 1.0 / sqrt(ss / (double)X0NE_HEAD_DIM + (double)eps);
    return {(double)r.a * scale * (double)r.wa, (double)r.b * scale * (double)r.wb};
}
__device__ __forceinline__ void rope_turn(const RopeNormed& n, double c, double s, float* ra, float* rb) {
    *ra = (float)(n.na * c - n.nb * s);
    *rb = (float)(n.nb * c + n.na * s);
}

// The angle of lane i is the f32 product pos * inv_freq[i] (invf), its sine and cosine in f64.
__device__ __forceinline__ void rope_rotate(const RopeIn& r, float invf, uint32_t pos, float eps, float* ra,
                                            float* rb) {
    const double angle = (double)((float)pos * invf);
    rope_rotate_cs(r, cos(angle), sin(angle), eps, ra, rb);
}

__device__ __forceinline__ void rope_pair(const bf16_t* __restrict__ src, const bf16_t* __restrict__ nw,
                                          const float* __restrict__ inv_freq, uint32_t pos, float eps, float* ra,
                                          float* rb) {
    rope_rotate(rope_in(src, nw), inv_freq[threadIdx.x & 63], pos, eps, ra, rb);
}

struct AttnArgs {
    const bf16_t* q;         // non-fused: [q_heads][128]
    const bf16_t* qkv;       // fused: the packed [q; k; v] row
    const bf16_t* q_norm;    // fused
    const bf16_t* k_norm;    // fused
    const float* inv_freq;   // fused
    const double* rope_cs;   // fused: cos and sin per position below max_ctx and lane (x0ne_rope_table_f64)
    bf16_t* k_cache;         // written by the fused variant at pos
    bf16_t* v_cache;
    const uint32_t* pages;
    float* state;
    uint32_t* counter;       // null: the merge kernel follows
    bf16_t* out;
    const uint32_t* pos;
    uint32_t q_heads, kv_heads, max_ctx, splits;
    float scale, eps;
    uint32_t out_panel;      // 0: out row-major [q_heads][128]; t + 1: row t of out in panels
};

// Where dim d of q head h goes: out row-major, or row t = out_panel - 1 of a [..][q_heads 128]
// matrix in panels (the batched step's X layout, device.h).
__device__ __forceinline__ size_t out_index(const AttnArgs& a, uint32_t h, uint32_t d) {
    const uint32_t k = h * X0NE_HEAD_DIM + d;
    return a.out_panel ? panel_index(a.out_panel - 1, k, a.q_heads * X0NE_HEAD_DIM) : (size_t)k;
}

// A wavefront's state into the block's LDS for the block merge.
template <int G, class T, bool V>
__device__ __forceinline__ void stash_wave(AttnShared<G, T, V>& sh, const T m[G], const T l[G], const T o[G][2]) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            sh.wm[wave][g] = m[g];
            sh.wl[wave][g] = l[g];
        }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
        sh.wo[wave][g][lane] = o[g][0];
        sh.wo[wave][g][lane + 64] = o[g][1];
    }
}

// ---- the exact mode (f64 scores, softmax and sums) ----
//
// The exact mode follows the f64 oracle's arithmetic (oracle/src/lib.rs:149-176): scores are
// exact bf16 x bf16 products summed in f64 and scaled by the f64 1/sqrt(128), the softmax and
// the weighted V sums are f64, and the result is rounded f64 -> f32 -> bf16. Only the order of
// the f64 additions differs from the oracle's, which moves a result by about 1e-16 relative:
// far below the bf16 rounding step the outputs are compared at.
//
// The work unit is one 16-key page of one kv head (4 KiB of K rows and 4 KiB of dim-major V).
// Slices are the split-K slices of the fp32 kernels (split_of: runs of 64-key tiles, P of them);
// inside a slice the 4 wavefronts take its pages in turn (wavefront w: pages w, w + 4, ...), so a
// short context spreads over every wavefront of the block. The products and their sums run on
// the f64 matrix cores: v_mfma_f64_4x4x4f64 computes 4 blocks b of D[4][4] += A[4][4] B[4][4],
// lane l = 16 k + 4 b + x holding A_b[x][k], B_b[k][x] and D_b[l / 16][x] (measured on gfx950).
//  - scores S^T: block b's rows are keys 4 b .. 4 b + 3 of the page, its columns 4 q heads, its
//    k 4 dims: lane l supplies K[key 4 b + x][dim 32 k + t] at product t (64 contiguous bytes of
//    its key) and q[head x][dim 32 k + t] (32 f64 values held in registers from the prologue);
//    32 products over the 128 dims, in 4 interleaved chains of 8 (t % 4) added at the end, leave
//    lane l with the score of key 4 b + l / 16 for head x;
//  - the online softmax per head over the lanes of its column (xor 4, 8, 16, 32);
//  - O += P V: rows are the 4 heads, k 4 keys, block b's columns dims 16 i + 4 b .. + 3 for
//    product i (0..7): lane l supplies P[head x][key 4 k + s] at step s (through LDS) and
//    V[key 4 k + s][dim 16 i + 4 b + x] (8 contiguous bytes of each of its 8 dims), and ends
//    with O[head l / 16][dim 16 i + 4 b + x] in 8 accumulators.
// A group of 8 q heads runs both sets of 4 columns; of 1 or 2 the columns repeat the heads.
// The next page's K and V are in flight while a page is summed, its page-table entry one page
// further ahead (a vector load, so the LDS waits in between do not wait for it); slice 0 requests
// its first entry together with pos and the RoPE factors before the first page, so the
// dependent chain of a short context is pos/page -> K,V -> sums.

struct ExactShared {
    // q heads, bf16-rounded, as f64; the page weights (per wavefront, head, key) and rescale
    // factors; the new K/V row; the block merge's states; the last block's slice factors.
    // qd[head][d / 32][d % 32]: each quarter row padded to 34, so the 16 quarters a read of the
    // q operand meets (4 heads x 4 quarters) fall in distinct LDS banks.
    double qd[8][4][34];
    double pw[WAVES][8][X0NE_PAGE];
    double alpha[WAVES][8];
    alignas(16) bf16_t knew[X0NE_HEAD_DIM], vnew[X0NE_HEAD_DIM];
    double wm[WAVES][8], wl[WAVES][8];
    double wo[WAVES][8][X0NE_HEAD_DIM];
    double wf[WAVES][8], mh[8];
    double f[WAVES][MERGE_MAX];
    uint32_t last;
};

constexpr uint32_t EXACT_CHUNK = 40;  // slices whose f64 o values the exact merge loads at once

// The exact kernel's slices: runs of whole 64-key tiles (a wavefront's page each per tile). The
// finest split that fills P slices costs a second round trip in the merge past EXACT_CHUNK
// slices; longer runs that keep one round trip are taken unless they add more than two pages per
// wavefront per extra round trip saved (a page costs about 1.5 us, a round trip about 3 us). Two
// tiles stay in one slice: a second page per wavefront costs less than the cross-slice merge. On
// MI355X at 8 kv heads, P 64, against runs of at least 4 tiles: 164 keys 12.8 -> 11.5 us, 300
// keys 17.4 -> 11.4, 1024 keys 18.1 -> 12.8, 2048 keys 18.8 -> 15.6; 8k to 32k unchanged.
__device__ __forceinline__ Split split_exact(uint32_t ctx, uint32_t P) {
    Split s;
    s.ntiles = (ctx + X0NE_SPLIT_TILE - 1) / X0NE_SPLIT_TILE;
    if (s.ntiles <= 2) {
        s.per = s.ntiles;
        s.active = 1;
        return s;
    }
    const uint32_t fine = (s.ntiles + P - 1) / P;
    const uint32_t cap = min(P, EXACT_CHUNK);
    const uint32_t one = (s.ntiles + cap - 1) / cap;
    const uint32_t rounds = ((s.ntiles + fine - 1) / fine + EXACT_CHUNK - 1) / EXACT_CHUNK;
    s.per = one - fine <= 2 * (rounds - 1) ? one : fine;
    s.active = (s.ntiles + s.per - 1) / s.per;
    return s;
}

__device__ __forceinline__ void dstate_put(double* p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double dstate_get(const double* p) {
    return __hip_atomic_load(const_cast<double*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint2 bload8(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
    return make_uint2((uint32_t)v[0], (uint32_t)v[1]);
}

// bf16 element e (0..7) of 8 packed in a uint4, as f64.
__device__ __forceinline__ double bf_of(const uint4& v, int e) {
    const uint32_t u = e < 2 ? v.x : e < 4 ? v.y : e < 6 ? v.z : v.w;
    return (double)((e & 1) ? bf_hi(u) : bf_lo(u));
}

template <int G>
__device__ __forceinline__ void exact_block(const AttnArgs& a, ExactShared& sh) {
    constexpr int HS = G > 4 ? G / 4 : 1;  // sets of 4 head columns
    const uint32_t kh = blockIdx.x, y = blockIdx.y, P = a.splits;
    if (P == 0 || P > MERGE_MAX || kh >= a.kv_heads || a.q_heads != (uint32_t)G * a.kv_heads) return;  // uniform
    const uint32_t t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t kq = lane >> 4, bq = (lane >> 2) & 3, x = lane & 3;
    const uint32_t h0 = kh * G, q_dim = a.q_heads * X0NE_HEAD_DIM, kv_dim = a.kv_heads * X0NE_HEAD_DIM;
    const uint32_t seq_pages = (a.max_ctx + X0NE_PAGE - 1) / X0NE_PAGE;

    // Before pos: the q rows this wavefront ropes (heads wave, wave + 4, ...), in the last
    // wavefront kv head kh's K and V rows, their RMS norms (which do not depend on pos), and in
    // slice 0 the first page's table entry (slice 0's wavefront w starts at page w whatever the
    // context; clamped inside the table).
    constexpr int QPW = (G + WAVES - 1) / WAVES;
    RopeIn qin[QPW], kin{};
    bf16_t vrow[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < QPW; ++j) {
        const uint32_t g = wave + WAVES * j;
        qin[j] = g < (uint32_t)G ? rope_in(a.qkv + (h0 + g) * X0NE_HEAD_DIM, a.q_norm) : RopeIn{};
    }
    const float invf = a.inv_freq[lane];
    if (wave == WAVES - 1) {
        kin = rope_in(a.qkv + q_dim + kh * X0NE_HEAD_DIM, a.k_norm);
        const bf16_t* vs = a.qkv + q_dim + kv_dim + kh * X0NE_HEAD_DIM;
        vrow[0] = vs[lane];
        vrow[1] = vs[lane + 64];
    }
    const uint32_t first_entry = y == 0 ? a.pages[min(wave, seq_pages - 1)] : 0u;
    RopeNormed qnm[QPW], knm{};
#pragma unroll
    for (int j = 0; j < QPW; ++j)
        if (wave + WAVES * j < (uint32_t)G) qnm[j] = rope_norm(qin[j], a.eps);
    if (wave == WAVES - 1) knm = rope_norm(kin, a.eps);

    const uint32_t pos = a.pos[0];
    const uint32_t ctx = min(pos + 1u, a.max_ctx);
    const Split sp = split_exact(ctx, P);
    if (y >= sp.active) return;  // block-uniform: a slice past the context
    // The RoPE factors at pos (the table's below max_ctx, else computed alike) before any page.
    double rc, rs;
    if (pos < a.max_ctx) {
        const double2 cs = *reinterpret_cast<const double2*>(a.rope_cs + 2 * ((size_t)pos * (X0NE_HEAD_DIM / 2) + lane));
        rc = cs.x;
        rs = cs.y;
    } else {
        const double angle = (double)((float)pos * invf);
        rc = cos(angle);
        rs = sin(angle);
    }
    const uint32_t npages = (ctx + X0NE_PAGE - 1) / X0NE_PAGE;
    const uint32_t run_begin = y * sp.per * (X0NE_SPLIT_TILE / X0NE_PAGE);
    const uint32_t run_end = min((y + 1) * sp.per * (X0NE_SPLIT_TILE / X0NE_PAGE), npages);
    const uint32_t new_page = pos < a.max_ctx ? pos / X0NE_PAGE : ~0u;
    const bool owner = new_page >= run_begin && new_page < run_end;

    // Page-table entry and plane byte offsets of page p of this kv head: K key 4 bq + x's dims
    // 32 kq .. + 31 (four 16-byte pieces); V keys 4 kq .. + 3 of dims 16 i + 4 bq + x (8 bytes
    // each, i = 0..7).
    const auto kr = plane_rsrc(a.k_cache, OFF_NONE), vr = plane_rsrc(a.v_cache, OFF_NONE);
    const auto pr_ = plane_rsrc(a.pages, run_end * 4);  // entries past the run read 0
    const uint32_t page_b = a.kv_heads * X0NE_PAGE * X0NE_HEAD_DIM * 2, head_b = kh * X0NE_PAGE * X0NE_HEAD_DIM * 2;
    // (kept in a vector register: only the load offsets use it, so nothing waits for it early)
    auto entry = [&](uint32_t p) -> uint32_t { return bload4(pr_, p < run_end ? 4 * p : OFF_NONE); };
    auto load_page = [&](uint32_t p, uint32_t pg, uint4 (&kk)[4], uint2 (&vv)[8]) {
        const bool live = p < run_end;
        const uint32_t kb = pg * page_b + head_b + (4 * bq + x) * X0NE_HEAD_DIM * 2 + 64 * kq;
        const uint32_t vb = pg * page_b + head_b + ((4 * bq + x) * X0NE_PAGE + 4 * kq) * 2;
#pragma unroll
        for (int j = 0; j < 4; ++j) kk[j] = bload16(kr, live ? kb + 16 * j : OFF_NONE);
#pragma unroll
        for (int i = 0; i < 8; ++i) vv[i] = bload8(vr, live ? vb + 16 * i * X0NE_PAGE * 2 : OFF_NONE);
    };
    uint32_t p = run_begin + wave;
    uint4 kc[4], kn[4];
    uint2 vc[8], vn[8];
    uint32_t pg = y == 0 ? (p < run_end ? first_entry : 0u) : entry(p);
    load_page(p, pg, kc, vc);
    uint32_t pg_next = entry(p + WAVES);

    // RoPE while the first page is in flight; the owner's last wavefront writes position pos's K
    // row and V column and keeps them in LDS.
#pragma unroll
    for (int j = 0; j < QPW; ++j) {
        const uint32_t g = wave + WAVES * j;
        if (g < (uint32_t)G) {
            float ra, rb;
            rope_turn(qnm[j], rc, rs, &ra, &rb);
            sh.qd[g][lane / 32][lane % 32] = (double)bf_round(ra);
            sh.qd[g][lane / 32 + 2][lane % 32] = (double)bf_round(rb);
        }
    }
    if (owner && wave == WAVES - 1) {
        float ra, rb;
        rope_turn(knm, rc, rs, &ra, &rb);
        const bf16_t k0 = f2bf(ra), k1 = f2bf(rb);
        const uint32_t at = kv_row(a.pages, pos, kh, a.kv_heads);
        a.k_cache[at + lane] = k0;
        a.k_cache[at + lane + 64] = k1;
        const uint32_t vat = v_slot(a.pages, pos, kh, a.kv_heads);
        a.v_cache[vat + lane * X0NE_PAGE] = vrow[0];
        a.v_cache[vat + (lane + 64) * X0NE_PAGE] = vrow[1];
        sh.knew[lane] = k0;
        sh.knew[lane + 64] = k1;
        sh.vnew[lane] = vrow[0];
        sh.vnew[lane + 64] = vrow[1];
    }
    lds_barrier();  // q and the new row in LDS; the page loads stay in flight
    // This lane's q operand: head column x of each set (a group of 1 or 2 repeats its heads),
    // dims 32 kq .. + 31.
    double qv[HS][32];
#pragma unroll
    for (int hs = 0; hs < HS; ++hs) {
        const uint32_t h = G >= 4 ? 4 * hs + x : x % (uint32_t)G;
#pragma unroll
        for (int d = 0; d < 32; d += 2) {
            const double2 v = *reinterpret_cast<const double2*>(&sh.qd[h][kq][d]);
            qv[hs][d] = v.x;
            qv[hs][d + 1] = v.y;
        }
    }

    const double scale = 1.0 / sqrt((double)X0NE_HEAD_DIM);
    double m[HS], lsum[HS];
    double o[HS][8];
#pragma unroll
    for (int hs = 0; hs < HS; ++hs) {
        m[hs] = -INFINITY;
        lsum[hs] = 0.0;
#pragma unroll
        for (int i = 0; i < 8; ++i) o[hs][i] = 0.0;
    }

    for (; p < run_end; p += WAVES) {
        const uint32_t pg_after = entry(p + 2 * WAVES);  // requested before the page it follows
        if (p + WAVES < run_end) load_page(p + WAVES, pg_next, kn, vn);
        const uint32_t base = p * X0NE_PAGE;
        if (p == new_page) {  // wavefront-uniform: the new row from LDS, not from its write
            const uint32_t e = pos % X0NE_PAGE;
            if (4 * bq + x == e) {
#pragma unroll
                for (int j = 0; j < 4; ++j) kc[j] = *reinterpret_cast<const uint4*>(sh.knew + 32 * kq + 8 * j);
            }
            if (e / 4 == kq) {
                const uint32_t sel = e % 4, shift = 16 * (sel & 1u), keep = shift ? 0x0000FFFFu : 0xFFFF0000u;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint32_t val = (uint32_t)sh.vnew[16 * i + 4 * bq + x] << shift;
                    if (sel < 2)
                        vc[i].x = (vc[i].x & keep) | val;
                    else
                        vc[i].y = (vc[i].y & keep) | val;
                }
            }
        }
        // Scores: key 4 bq + l / 16 of the page for head column x of each set.
        double sc[HS];
        {
            double acc[HS][4];
#pragma unroll
            for (int hs = 0; hs < HS; ++hs)
#pragma unroll
                for (int c4 = 0; c4 < 4; ++c4) acc[hs][c4] = 0.0;
#pragma unroll
            for (int d = 0; d < 32; ++d) {
                const double kd = bf_of(kc[d / 8], d % 8);
#pragma unroll
                for (int hs = 0; hs < HS; ++hs)
                    acc[hs][d % 4] = __builtin_amdgcn_mfma_f64_4x4x4f64(kd, qv[hs][d], acc[hs][d % 4], 0, 0, 0);
            }
#pragma unroll
            for (int hs = 0; hs < HS; ++hs) sc[hs] = (acc[hs][0] + acc[hs][1]) + (acc[hs][2] + acc[hs][3]);
        }
        // Online softmax per head column over the page's 16 keys (the lanes of column x).
        const bool in = base + 4 * bq + kq < ctx;
        double pr[HS];
#pragma unroll
        for (int hs = 0; hs < HS; ++hs) {
            const double s = in ? sc[hs] * scale : -INFINITY;
            double mx = s;
#pragma unroll
            for (int o2 = 4; o2 < 64; o2 <<= 1) mx = fmax(mx, __shfl_xor(mx, o2, 64));
            const double mn = fmax(m[hs], mx);  // key `base` is below ctx: mn is finite
            const double al = exp(m[hs] - mn);
            pr[hs] = exp(s - mn);
            lsum[hs] = lsum[hs] * al + pr[hs];
            m[hs] = mn;
            sh.pw[wave][4 * hs + x][4 * bq + kq] = pr[hs];
            if (lane < 4) sh.alpha[wave][4 * hs + x] = al;
        }
        wave_lds_sync();
        // V of keys past ctx taken as 0 (their weight is 0, and 0 times a value that is not a
        // number would not be); then O rescaled and O += P V.
        if (base + X0NE_PAGE > ctx) {
            const uint32_t k0 = base + 4 * kq;
            const uint32_t valid = k0 >= ctx ? 0u : min(ctx - k0, 4u);
            const uint32_t mlo = (valid > 1 ? 0xFFFF0000u : 0u) | (valid > 0 ? 0xFFFFu : 0u);
            const uint32_t mhi = (valid > 3 ? 0xFFFF0000u : 0u) | (valid > 2 ? 0xFFFFu : 0u);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                vc[i].x &= mlo;
                vc[i].y &= mhi;
            }
        }
#pragma unroll
        for (int hs = 0; hs < HS; ++hs) {
            const double al = sh.alpha[wave][4 * hs + kq];
#pragma unroll
            for (int i = 0; i < 8; ++i) o[hs][i] *= al;
        }
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
            double pv[HS];
#pragma unroll
            for (int hs = 0; hs < HS; ++hs) pv[hs] = sh.pw[wave][4 * hs + x][4 * kq + s4];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t w = s4 < 2 ? vc[i].x : vc[i].y;
                const double vd = (double)((s4 & 1) ? bf_hi(w) : bf_lo(w));
#pragma unroll
                for (int hs = 0; hs < HS; ++hs) o[hs][i] = __builtin_amdgcn_mfma_f64_4x4x4f64(pv[hs], vd, o[hs][i], 0, 0, 0);
            }
        }
        wave_lds_sync();  // the next page rewrites pw and alpha
#pragma unroll
        for (int j = 0; j < 4; ++j) kc[j] = kn[j];
#pragma unroll
        for (int i = 0; i < 8; ++i) vc[i] = vn[i];
        pg_next = pg_after;
    }
    // This wavefront's state: each head's m and l (the lane sums over the column's 16 lanes),
    // its o (lane l: head 4 hs + l / 16, dims 16 i + 4 bq + x).
#pragma unroll
    for (int hs = 0; hs < HS; ++hs) {
        double l = lsum[hs];
#pragma unroll
        for (int o2 = 4; o2 < 64; o2 <<= 1) l += __shfl_xor(l, o2, 64);
        const uint32_t g = 4 * hs + x;
        if (lane < 4 && g < (uint32_t)G) {
            sh.wm[wave][g] = m[hs];
            sh.wl[wave][g] = l;
        }
        const uint32_t go = 4 * hs + kq;
        if (go < (uint32_t)G) {
#pragma unroll
            for (int i = 0; i < 8; ++i) sh.wo[wave][go][16 * i + 4 * bq + x] = o[hs][i];
        }
    }
    lds_barrier();
    // The block's 4 wavefronts merged per head, in wave order: thread 4 g + w forms wavefront
    // w's factor for head g (the block's exps side by side), then every thread adds its outputs'
    // terms. Wavefront 0 always has a page, so each maximum is finite, and a wavefront without
    // one (m -inf, l and o 0) adds +0.
    if (t < 4 * (uint32_t)G) {
        const uint32_t g = t / 4, w = t % 4;
        double mx = -INFINITY;
#pragma unroll
        for (int v = 0; v < WAVES; ++v) mx = fmax(mx, sh.wm[v][g]);
        sh.wf[w][g] = exp(sh.wm[w][g] - mx);
        if (w == 0) sh.mh[g] = mx;
    }
    lds_barrier();
    const bool whole = sp.active == 1;
    double* st_base = reinterpret_cast<double*>(a.state);
#pragma unroll
    for (uint32_t i = t; i < (uint32_t)G * X0NE_HEAD_DIM; i += BLOCK) {
        const uint32_t g = i / X0NE_HEAD_DIM, d = i % X0NE_HEAD_DIM;
        const double mx = sh.mh[g];
        double l = 0.0, ov = 0.0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const double fw = sh.wf[w][g];
            l += sh.wl[w][g] * fw;
            ov += sh.wo[w][g][d] * fw;
        }
        if (whole) {
            a.out[(size_t)(h0 + g) * X0NE_HEAD_DIM + d] = f2bf((float)(ov / l));
        } else {
            double* st = st_base + ((size_t)(h0 + g) * P + y) * X0NE_SPLIT_STATE;
            dstate_put(st + 4 + d, ov);
            if (d == 0) {
                dstate_put(st, mx);
                dstate_put(st + 1, l);
            }
        }
    }
    if (whole) return;
    // Without counters (a null pointer) the states are left for the caller and no block merges:
    // grid-uniform, so no block counts at address 0.
    if (a.counter == nullptr) return;
    // The slices' states acknowledged, then the count; the block that completes it merges each
    // head's slices 0 .. active - 1 in that order (M = max m, f = exp(m - M), l = sum l f,
    // o = sum o f; one rounding of o / l), and sets the count back to 0 for the next step.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t == 0)
        sh.last = __hip_atomic_fetch_add(a.counter + kh, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                  sp.active - 1;
    __syncthreads();
    if (!sh.last) return;  // block-uniform
    const uint32_t active = sp.active;
    for (uint32_t g = wave; g < (uint32_t)G; g += WAVES) {
        const double* s = st_base + (size_t)(h0 + g) * P * X0NE_SPLIT_STATE;
        double* f = sh.f[wave];
        // The slices' m and l (lane l: slices l, l + 64, ...) and the first EXACT_CHUNK slices'
        // o values are requested together, before any is used: one round trip to memory for up
        // to EXACT_CHUNK slices. Later chunks of o follow one round trip each, summed in slice
        // order.
        double av[EXACT_CHUNK], bv[EXACT_CHUNK];
        auto request = [&](uint32_t y0) {
#pragma unroll
            for (uint32_t k = 0; k < EXACT_CHUNK; ++k)
                if (y0 + k < active) {  // wave-uniform
                    const double* so = s + (size_t)(y0 + k) * X0NE_SPLIT_STATE + 4;
                    av[k] = dstate_get(so + lane);
                    bv[k] = dstate_get(so + lane + 64);
                }
        };
        constexpr int ML = MERGE_MAX / 64;
        double mv[ML], lv[ML];
#pragma unroll
        for (int j = 0; j < ML; ++j) {
            const uint32_t yy = lane + 64 * j;
            mv[j] = -INFINITY;
            lv[j] = 0.0;
            if (64 * j < active && yy < active) {
                mv[j] = dstate_get(s + (size_t)yy * X0NE_SPLIT_STATE);
                lv[j] = dstate_get(s + (size_t)yy * X0NE_SPLIT_STATE + 1);
            }
        }
        request(0);
        // Maximum and sum over the lanes that hold slices: butterflies over the smallest power
        // of two of lanes covering them (lane 0's group), then lane 0's sum for every lane.
        uint32_t span = 1;
        while (span < active && span < 64) span <<= 1;
        double mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < ML; ++j) mx = fmax(mx, mv[j]);
        for (uint32_t o2 = 1; o2 < span; o2 <<= 1) mx = fmax(mx, __shfl_xor(mx, (int)o2, 64));
        double lp = 0.0;
#pragma unroll
        for (int j = 0; j < ML; ++j) {
            const uint32_t yy = lane + 64 * j;
            if (64 * j < active && yy < active) {
                const double fy = exp(mv[j] - mx);
                f[yy] = fy;
                lp += lv[j] * fy;
            }
        }
        for (uint32_t o2 = 1; o2 < span; o2 <<= 1) lp += __shfl_xor(lp, (int)o2, 64);
        const double l = __shfl(lp, 0, 64);
        wave_lds_sync();
        double o0 = 0.0, o1 = 0.0;
        for (uint32_t y0 = 0; y0 < active; y0 += EXACT_CHUNK) {
#pragma unroll
            for (uint32_t k = 0; k < EXACT_CHUNK; ++k)
                if (y0 + k < active) {
                    o0 = fma(av[k], f[y0 + k], o0);
                    o1 = fma(bv[k], f[y0 + k], o1);
                }
            if (y0 + EXACT_CHUNK < active) request(y0 + EXACT_CHUNK);
        }
        a.out[(size_t)(h0 + g) * X0NE_HEAD_DIM + lane] = f2bf((float)(o0 / l));
        a.out[(size_t)(h0 + g) * X0NE_HEAD_DIM + lane + 64] = f2bf((float)(o1 / l));
        wave_lds_sync();
    }
    __syncthreads();
    if (t == 0) __hip_atomic_store(a.counter + kh, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // next step
}

// Block (kv head kh, slice y) of the grouped kernel on the matrix cores: q heads kh G .. kh G +
// G - 1. The loads that do not depend on pos (the q rows, or the packed qkv rows and norm
// weights of the fused variant) are issued first, the first tile's page-table entries and K/V as
// soon as pos is known, and the QK-norm + RoPE runs while those are in flight. In the fused
// variant the block owning pos's tile writes that position's K and V rows to their page and
// keeps them in LDS for its wavefront that attends them, so no wavefront waits for that write.
template <int G, bool FUSED>
__device__ __forceinline__ void attn_group_block(const AttnArgs& a, AttnShared<G, float, false>& sh) {
    const uint32_t kh = blockIdx.x, y = blockIdx.y, P = a.splits;
    // Block-uniform exits for a launch that does not fit the geometry, before any load.
    if (P > MERGE_MAX || kh >= a.kv_heads || a.q_heads != (uint32_t)G * a.kv_heads) return;
    const uint32_t t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t h0 = kh * G, q_dim = a.q_heads * X0NE_HEAD_DIM, kv_dim = a.kv_heads * X0NE_HEAD_DIM;

    // Requested before pos: the fused variant's q rows wave, wave + 4, ... of the group (and in
    // the last wavefront kv head kh's K and V rows), or the plain variant's q values.
    constexpr int QPW = (G + WAVES - 1) / WAVES;             // q heads a wavefront ropes
    constexpr int QV = (G * X0NE_HEAD_DIM + BLOCK - 1) / BLOCK;  // plain: q values per thread
    RopeIn qin[QPW], kin{};
    bf16_t vrow[2] = {0, 0}, qv[QV];
    float invf = 0.f;
    if (FUSED) {
#pragma unroll
        for (int j = 0; j < QPW; ++j) {
            const uint32_t g = wave + WAVES * j;
            qin[j] = g < (uint32_t)G ? rope_in(a.qkv + (h0 + g) * X0NE_HEAD_DIM, a.q_norm) : RopeIn{};
        }
        invf = a.inv_freq[lane];
        if (wave == WAVES - 1) {
            kin = rope_in(a.qkv + q_dim + kh * X0NE_HEAD_DIM, a.k_norm);
            const bf16_t* vs = a.qkv + q_dim + kv_dim + kh * X0NE_HEAD_DIM;
            vrow[0] = vs[lane];
            vrow[1] = vs[lane + 64];
        }
    } else {
#pragma unroll
        for (int j = 0; j < QV; ++j) {
            const uint32_t k = t + BLOCK * j;
            qv[j] = k < (uint32_t)G * X0NE_HEAD_DIM ? a.q[(size_t)h0 * X0NE_HEAD_DIM + k] : (bf16_t)0;
        }
    }

    // Slice 0's wavefront w starts at tile w whatever the context: its page-table entries are
    // requested with pos rather than after it (clamped below max_ctx, unused past ctx).
    uint32_t first_pages[4] = {0u, 0u, 0u, 0u};
    if (y == 0) {
        const uint32_t last_page = (a.max_ctx + X0NE_PAGE - 1) / X0NE_PAGE - 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) first_pages[i] = a.pages[min(4 * wave + i, last_page)];
    }

    const uint32_t pos = a.pos[0];
    const uint32_t ctx = min(pos + 1u, a.max_ctx);
    const Split sp = split_of(ctx, P);
    if (y >= sp.active) return;  // block-uniform: a slice past the context
    const uint32_t active = sp.active;
    const uint32_t t_begin = y * sp.per + wave, t_end = (y + 1) * sp.per;
    const bool owner = FUSED && pos < a.max_ctx && y == (pos / X0NE_SPLIT_TILE) / sp.per;
    // This lane's cosine and sine at pos: the table's below max_ctx, else computed alike.
    double rc = 0.0, rs = 0.0;
    if (FUSED) {
        if (pos < a.max_ctx) {
            const double2 v = *reinterpret_cast<const double2*>(a.rope_cs + 2 * ((size_t)pos * (X0NE_HEAD_DIM / 2) + lane));
            rc = v.x;
            rs = v.y;
        } else {
            const double angle = (double)((float)pos * invf);
            rc = cos(angle);
            rs = sin(angle);
        }
    }
    const NewRow fx = {owner ? pos / X0NE_SPLIT_TILE : ~0u, pos % X0NE_SPLIT_TILE, sh.knew, sh.vnew};

    // q into LDS as bf16 (the rotated values rounded, as the engine stores q), then the B operand
    // of Q^T: head lane % 16, dims 32 st + 8 (lane / 16) .., heads past G zero.
    auto prologue = [&](uint4 qb[4]) {
        if (FUSED) {
#pragma unroll
            for (int j = 0; j < QPW; ++j) {
                const uint32_t g = wave + WAVES * j;
                if (g < (uint32_t)G) {
                    float ra, rb;
                    rope_rotate_cs(qin[j], rc, rs, a.eps, &ra, &rb);
                    sh.qh[g][lane] = f2bf(ra);
                    sh.qh[g][lane + 64] = f2bf(rb);
                }
            }
            if (owner && wave == WAVES - 1) {  // the K/V write of position pos, and its LDS copy
                float ra, rb;
                rope_rotate_cs(kin, rc, rs, a.eps, &ra, &rb);
                const bf16_t k0 = f2bf(ra), k1 = f2bf(rb);
                const uint32_t at = kv_row(a.pages, pos, kh, a.kv_heads);
                a.k_cache[at + lane] = k0;
                a.k_cache[at + lane + 64] = k1;
                const uint32_t vat = v_slot(a.pages, pos, kh, a.kv_heads);
                a.v_cache[vat + lane * X0NE_PAGE] = vrow[0];
                a.v_cache[vat + (lane + 64) * X0NE_PAGE] = vrow[1];
                sh.knew[lane] = k0;
                sh.knew[lane + 64] = k1;
                sh.vnew[lane] = vrow[0];
                sh.vnew[lane + 64] = vrow[1];
            }
        } else {
#pragma unroll
            for (int j = 0; j < QV; ++j) {
                const uint32_t k = t + BLOCK * j;
                if (k < (uint32_t)G * X0NE_HEAD_DIM) sh.qh[k / X0NE_HEAD_DIM][k % X0NE_HEAD_DIM] = qv[j];
            }
        }
        lds_barrier();  // q and the new row in LDS; the loads in flight stay in flight
        const uint32_t n = lane & 15, q4 = lane >> 4;
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            const uint4 v = *reinterpret_cast<const uint4*>(&sh.qh[n < (uint32_t)G ? n : 0][32 * st + 8 * q4]);
            qb[st] = n < (uint32_t)G ? v : make_uint4(0, 0, 0, 0);
        }
    };
    float mw, lw;
    f32x4 ow[8];
    attend_wave_mfma(prologue, fx, a.k_cache, a.v_cache, a.pages, kh, a.kv_heads, ctx, ctx, t_begin, BLOCK_TILES, t_end,
                     a.scale, mw, lw, ow, y == 0 ? first_pages : nullptr);
    {
        const uint32_t n = lane & 15, q4 = lane >> 4;
        if (q4 == 0 && n < (uint32_t)G) {
            sh.wm[wave][n] = mw;
            sh.wl[wave][n] = lw;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t h = 4 * q4 + i;
            if (h < (uint32_t)G) {
#pragma unroll
                for (int nb = 0; nb < 8; ++nb) sh.wo[wave][h][16 * nb + n] = ow[nb][i];
            }
        }
    }
    lds_barrier();

    if (active == 1) {  // one block holds the whole context: the output directly
        block_merge<G, float>(sh, [&](uint32_t g, uint32_t d, float, float lv, float ov) {
            a.out[out_index(a, h0 + g, d)] = f2bf(ov / lv);
        });
        return;
    }
    block_merge<G, float>(sh, [&](uint32_t g, uint32_t d, float mv, float lv, float ov) {
        float* st = a.state + ((size_t)(h0 + g) * P + y) * X0NE_SPLIT_STATE;
        state_put(st + 4 + d, ov);
        if (d == 0) {
            state_put(st, mv);
            state_put(st + 1, lv);
        }
    });
    if (a.counter == nullptr) return;  // grid-uniform: the merge kernel follows
    // Every thread's state stores acknowledged (coherent), then the count: the block that brings
    // it to `active` sees every slice's state.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t == 0)
        sh.last = __hip_atomic_fetch_add(a.counter + kh, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == active - 1;
    __syncthreads();
    if (!sh.last) return;  // block-uniform
    for (uint32_t g = wave; g < (uint32_t)G; g += WAVES)
        merge_head(a.state + (size_t)(h0 + g) * P * X0NE_SPLIT_STATE,
                   [&](uint32_t d, bf16_t v) { a.out[out_index(a, h0 + g, d)] = v; }, active, sh.f[wave]);
    __syncthreads();
    if (t == 0) __hip_atomic_store(a.counter + kh, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // next step
}

// ---- causal prefill on the matrix cores ----
//
// Block (kv head kh, row block) serves the G q heads of kv head kh for RB = 128 / G rows of q
// ([rows][q_heads][128] bf16, at positions pos0 + row): its 128 columns (column c: row
// r0 + c / G, head kh G + c % G) go 32 to a wavefront, as two groups of 16 (the 16 columns of a
// product). The keys pass in tiles of 64 (4 pages) staged in LDS once per block and read by all
// 4 wavefronts (K by products, V dim-major, chunks swizzled against bank conflicts);
// each K or V piece a wavefront reads serves both groups.
// Per tile and column group: S^T = K Q^T (16 products; the S^T blocks X0, Y0, X1, Y1 of the
// decode wavefront, which leave each lane the 8 keys of its P row for a 32-key step), a
// per-column causal mask (keys up to the column's own position; skipped for a tile inside every
// limit of the wavefront), the online softmax in units of log2 (the rescale of O skipped when no
// maximum of the group moved), and O += P V with P rounded to bf16 (16 products). The next
// tile's loads are in flight while a tile is multiplied (two LDS buffers). Each column's output
// goes straight to out ([rows][q_heads][128], or in 16-row panels). The heavier half of the row blocks is dispatched
// first, heaviest first, then the lighter half, lightest first. Keys at or past the block's context are read as zeros (V) or masked (K); no page past
// the context is read. Two blocks share a CU (2 x 64 KiB of LDS, at most 256 registers per
// lane), so one block's products overlap the other's softmax and loads.
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) v = min(v, (uint32_t)__shfl_xor((int)v, o, 64));
    return v;
}
constexpr int PF_CG = 2;              // column groups of 16 per wavefront
constexpr int PF_NW = X0NE_PREFILL_THREADS / 64;  // wavefronts per block
static_assert(PF_NW * 16 * PF_CG == X0NE_PREFILL_COLS, "columns per prefill block");
// LDS tiles without padding, in KiB of 8 rows x 128 bytes whose 16-byte chunks are placed by an XOR
// of the row, so that the 16 rows x 4 chunks that a product's operand reads meet in no bank (gfx950:
// 256 bytes per clock, measured over single access patterns) and neither do 8 neighbouring lanes'
// stores. The layout before, by rows of the tile, spent 38 % of the LDS cycles in conflicts.
// K: the keys of a product's 16 rows together: block (kp, h) holds keys 32 kp + 8 a + 4 h + j as rows
// n = 4 a + j, dims 0..63 in front of 64..127. V: row = dim, 64 keys of 2 bytes.
// Element index of 16-byte chunk c (dims 8 c ..) of key r, and of chunk c (keys 8 c ..) of dim d.
__device__ __forceinline__ uint32_t pf_chunk(uint32_t row, uint32_t c) {
    return ((row >> 3) * 64 + (row & 7) * 8 + (c ^ (row & 7))) * 8;
}
__device__ __forceinline__ uint32_t pf_k_at(uint32_t kp, uint32_t h, uint32_t n, uint32_t c) {
    return ((kp * 2 + h) * 2 + (c >> 3)) * 1024 + pf_chunk(n, c & 7);
}
__device__ __forceinline__ uint32_t pf_k_key(uint32_t r, uint32_t c) {
    return pf_k_at(r >> 5, (r >> 2) & 1, 4 * ((r >> 3) & 3) + (r & 3), c);
}

struct PrefillShared {
    alignas(1024) bf16_t k[2][X0NE_SPLIT_TILE * X0NE_HEAD_DIM];
    alignas(1024) bf16_t v[2][X0NE_HEAD_DIM * X0NE_SPLIT_TILE];
};

template <int G, int CG, bool OUT_PANEL = false, int NW = 4>
__device__ __forceinline__ void prefill_block(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache,
                                              const bf16_t* __restrict__ v_cache, const uint32_t* __restrict__ pages,
                                              bf16_t* __restrict__ out, uint32_t p0, uint32_t rows, uint32_t q_heads,
                                              uint32_t kv_heads, uint32_t max_ctx, float scale, PrefillShared& sh) {
    constexpr uint32_t COLS = NW * 16 * CG;  // columns per block: CG groups of 16 per wavefront
    constexpr uint32_t RB = COLS / G;
    constexpr uint32_t NT = 64 * NW, J = 1024 / NT;  // threads; K (and V) chunks of a tile per thread
    static_assert(1024 % NT == 0, "a tile's 1024 chunks over the block's threads");
    // Dispatch order: the first half of the row blocks heaviest first, then the second half
    // lightest first, so the two blocks that share a CU (block i and block i + half the grid)
    // hold a heavy and a light row block (four 2048-row passes: 245.5 against 251.4 µs mean).
    const uint32_t ny = gridDim.y, half = (ny + 1) / 2, y = blockIdx.y;
    const uint32_t kh = blockIdx.x, rb = y < half ? ny - 1 - y : y - half;
    const uint32_t r0 = rb * RB;
    if (kh >= kv_heads || q_heads != (uint32_t)G * kv_heads || r0 >= rows || max_ctx == 0 || blockDim.x != NT)
        return;  // block-uniform
    const uint32_t t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t n = lane & 15, q4 = lane >> 4;
    const uint32_t ctx = min(p0 + min(r0 + RB, rows), max_ctx);  // keys the block reads
    const uint32_t ntiles = (ctx + X0NE_SPLIT_TILE - 1) / X0NE_SPLIT_TILE;
    const uint32_t npages = (ctx + X0NE_PAGE - 1) / X0NE_PAGE;
    const float scale2 = scale * LOG2E;

    // The lane's CG columns (one per group): their q pieces (the B operand of Q^T for each
    // 32-dim step) and causal limits; a column past the rows attends key 0 only and is not written.
    uint4 qb[CG][4];
    uint32_t ctx_col[CG];
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
        const uint32_t c = 16 * CG * wave + 16 * cg + n, r = r0 + c / G, h = kh * G + c % G;
        const bool live = r < rows;
        ctx_col[cg] = live ? min(p0 + r + 1, max_ctx) : 1u;
        const bf16_t* qr = q + ((size_t)(live ? r : 0) * q_heads + h) * X0NE_HEAD_DIM + 8 * q4;
#pragma unroll
        for (int st = 0; st < 4; ++st)
            qb[cg][st] = live ? *reinterpret_cast<const uint4*>(qr + 32 * st) : make_uint4(0, 0, 0, 0);
    }

    // A tile's K and V pieces for this thread: K chunk i = t + NT j is page i / 256, key
    // (i / 16) % 16, 16-byte piece i % 16; V chunk i is page i / 256, dim v_dim(i), keys
    // 8 (i % 2) .. + 7 of the page. A wavefront's V loads cover 32 dims of a page (1 KiB
    // contiguous), and 8 neighbouring lanes hold dims 2 apart, so their LDS chunks differ.
    // Their loads are issued by fetch() and waited for only by stash(), after a tile's products. The
    // thread's chunk j of a tile is in the tile's page j: its page-table entry is the same for the
    // whole block, so it is a scalar, requested one tile before the K and V (an entry past the
    // context is the last one again: those keys are masked), and a load's address is a lane's constant
    // plus a scalar.
    static_assert(NT == 256 && J == X0NE_SPLIT_TILE / X0NE_PAGE, "chunk j of a thread is in page j of the tile");
    auto v_dim = [](uint32_t i) { return 32 * ((i >> 6) & 3) + 8 * ((i >> 4) & 3) + 2 * ((i >> 1) & 3) + ((i >> 3) & 1); };
    auto v_half = [](uint32_t i) { return i & 1; };
    uint4 kr[J], vr[J];
    const auto kres = plane_rsrc(k_cache, OFF_NONE), vres = plane_rsrc(v_cache, OFF_NONE);
    const uint32_t k_lane = (((t >> 4) & 15) * X0NE_HEAD_DIM + 8 * (t & 15)) * 2;
    const uint32_t v_lane = (v_dim(t) * X0NE_PAGE + 8 * v_half(t)) * 2;
    uint32_t pe[J];  // entries of the next tile to fetch
    auto entries = [&](uint32_t tile) {
#pragma unroll
        for (int j = 0; j < (int)J; ++j) pe[j] = pages[min(4 * tile + j, npages - 1)];
    };
    auto fetch = [&](uint32_t tile) {
#pragma unroll
        for (int j = 0; j < (int)J; ++j) {
            const uint32_t at = __builtin_amdgcn_readfirstlane((pe[j] * kv_heads + kh) * (X0NE_PAGE * X0NE_HEAD_DIM * 2));
            kr[j] = bload16(kres, k_lane, at);
            vr[j] = bload16(vres, v_lane, at);
        }
    };
    auto stash = [&](uint32_t tile, int buf) {
        // Keys at or past ctx hold anything: V zeros there (their weight is 0, and 0 times a value
        // that is not a number would not be). Only a tile that reaches ctx has such keys.
        const bool edge = X0NE_SPLIT_TILE * (tile + 1) > ctx;  // block-uniform
        if (edge) {
#pragma unroll
            for (int j = 0; j < (int)J; ++j) {
                const uint32_t i = t + NT * j, pi = i >> 8;
                const uint32_t key0 = X0NE_SPLIT_TILE * tile + X0NE_PAGE * pi + 8 * v_half(i);
                const uint32_t valid = key0 >= ctx ? 0u : min(ctx - key0, 8u);
                uint32_t w[4] = {vr[j].x, vr[j].y, vr[j].z, vr[j].w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    w[e] &= (2 * e + 1 < (int)valid ? 0xFFFF0000u : 0u) | (2 * e < (int)valid ? 0xFFFFu : 0u);
                vr[j] = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
#pragma unroll
        for (int j = 0; j < (int)J; ++j) {
            const uint32_t i = t + NT * j, pi = i >> 8, r = 16 * pi + ((i >> 4) & 15), d = v_dim(i);
            *reinterpret_cast<uint4*>(&sh.k[buf][pf_k_key(r, i & 15)]) = kr[j];
            *reinterpret_cast<uint4*>(&sh.v[buf][pf_chunk(d, 2 * pi + v_half(i))]) = vr[j];
        }
    };

    float m_run[CG], lsum[CG];
    f32x4 o[CG][8];
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
        m_run[cg] = -INFINITY;
        lsum[cg] = 0.f;
    }
#pragma unroll
    for (int cg = 0; cg < CG; ++cg)
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) o[cg][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

    // A tile wholly below every limit of the wavefront's columns needs no mask.
    uint32_t lim = ctx_col[0];
#pragma unroll
    for (int cg = 1; cg < CG; ++cg) lim = min(lim, ctx_col[cg]);
    const uint32_t wave_lim = __builtin_amdgcn_readfirstlane(wave_min_u32(lim));

    entries(0);
    fetch(0);
    entries(1);
    stash(0, 0);
    __syncthreads();
    for (uint32_t tile = 0; tile < ntiles; ++tile) {
        const int buf = tile & 1;
        if (tile + 1 < ntiles) {  // block-uniform; in flight during the products
            fetch(tile + 1);
            entries(tile + 2);
        }
        const bf16_t* K = sh.k[buf];
        const bf16_t* V = sh.v[buf];
        const uint32_t base = X0NE_SPLIT_TILE * tile;
        // S^T blocks (kp, h) for every column group: one K piece serves all of them.
        f32x4 s[CG][2][2];
#pragma unroll
        for (int kp = 0; kp < 2; ++kp)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                // A row n: key 32 kp + 8 (n >> 2) + 4 h + (n & 3)
                f32x4 acc[CG];
#pragma unroll
                for (int cg = 0; cg < CG; ++cg) acc[cg] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int st = 0; st < 4; ++st) {
                    const uint4 kk = *reinterpret_cast<const uint4*>(K + pf_k_at(kp, h, n, 4 * st + q4));
#pragma unroll
                    for (int cg = 0; cg < CG; ++cg) acc[cg] = mfma16x16x32(kk, qb[cg][st], acc[cg]);
                }
#pragma unroll
                for (int cg = 0; cg < CG; ++cg) s[cg][kp][h] = acc[cg];
            }
        // s[cg][kp][h][i] is the score of key base + 32 kp + 8 q4 + 4 h + i for the lane's column
        // of group cg. Causal mask: keys at or past the column's limit score -inf.
        if (base + X0NE_SPLIT_TILE > wave_lim) {  // wavefront-uniform
#pragma unroll
            for (int cg = 0; cg < CG; ++cg) {
                const int left = (int)ctx_col[cg] - (int)(base + 8 * q4);  // keys of the lane below the limit
#pragma unroll
                for (int kp = 0; kp < 2; ++kp)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (32 * kp + 4 * h + i >= left) s[cg][kp][h][i] = -INFINITY;
            }
        }
        // Online softmax per column group in units of log2 (the scale folded into the exponent);
        // P rounded to bf16 for the P V product (relative error 2^-9 per weight, so at most
        // max|V| / 512 in an output, against the reference's max|V| / 128; the row sums l are
        // of the unrounded weights).
        uint4 phi[CG][2];
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) {
            float mx = -INFINITY;
#pragma unroll
            for (int kp = 0; kp < 2; ++kp)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[cg][kp][h][i]);
            mx = rows_max(mx);
            // Key 0 is in every column's first tile, so m_run is finite from there on.
            const float mn = fmaxf(m_run[cg], mx * scale2);
            const float alpha = __builtin_amdgcn_exp2f(m_run[cg] - mn);
            m_run[cg] = mn;
            float sc[2][2][4];
            float psum = 0.f;
#pragma unroll
            for (int kp = 0; kp < 2; ++kp)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        sc[kp][h][i] = __builtin_amdgcn_exp2f(fmaf(s[cg][kp][h][i], scale2, -mn));
                        psum += sc[kp][h][i];
                    }
            lsum[cg] = lsum[cg] * alpha + psum;
            if (__any(alpha != 1.f)) {  // multiplying by 1 changes nothing: skipped when no max moved
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float ai = __shfl(alpha, 4 * q4 + i, 64);
#pragma unroll
                    for (int nb = 0; nb < 8; ++nb) o[cg][nb][i] *= ai;
                }
            }
#pragma unroll
            for (int kp = 0; kp < 2; ++kp) {
                float pv[8];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    pv[i] = sc[kp][0][i];
                    pv[4 + i] = sc[kp][1][i];
                }
                uint32_t hw[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) hw[j] = pack_bf16(pv[2 * j], pv[2 * j + 1]);
                phi[cg][kp] = make_uint4(hw[0], hw[1], hw[2], hw[3]);
            }
        }
        // O += P V: the V piece (keys 32 kp + 8 q4 .., dim 16 nb + n) serves every group.
#pragma unroll
        for (int kp = 0; kp < 2; ++kp)
#pragma unroll
            for (int nb = 0; nb < 8; ++nb) {
                const uint32_t d = 16 * nb + n;
                const uint4 vb = *reinterpret_cast<const uint4*>(V + pf_chunk(d, 4 * kp + q4));
#pragma unroll
                for (int cg = 0; cg < CG; ++cg) o[cg][nb] = mfma16x16x32(phi[cg][kp], vb, o[cg][nb]);
            }
        if (tile + 1 < ntiles) stash(tile + 1, buf ^ 1);  // the other buffer was last read before the barrier
        __syncthreads();
    }
    // o[cg][nb][i] = O[column 16 cg + 4 q4 + i of the wavefront][dim 16 nb + n]; lane c < 16 of
    // the group holds column c's sum once the 4 lanes of a column are added.
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
        const float l = rows_sum(lsum[cg]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t cl = 4 * q4 + i, c = 16 * CG * wave + 16 * cg + cl;
            const float lc = __shfl(l, (int)cl, 64);
            const uint32_t rc = r0 + c / G;
            if (rc < rows) {
                const uint32_t k0 = (kh * G + c % G) * X0NE_HEAD_DIM;
                bf16_t* op = out + (size_t)rc * q_heads * X0NE_HEAD_DIM + k0;
#pragma unroll
                for (int nb = 0; nb < 8; ++nb) {
                    const bf16_t v = f2bf(o[cg][nb][i] / lc);
                    if (OUT_PANEL)
                        out[panel_index(rc, k0 + 16 * nb + n, q_heads * X0NE_HEAD_DIM)] = v;
                    else
                        op[16 * nb + n] = v;
                }
            }
        }
    }
}

}  // namespace

// x0ne_attention_prefill_g{G}_bf16: the causal prefill of x0ne_attention_prefill_bf16 (same
// arguments and semantics) on the matrix cores for G q heads per kv head; grid (kv_heads,
// ceil(rows / (128 / G))), block 256, two wavefronts per SIMD.
#define X0NE_PREFILL_GROUP(G)                                                                                      \
    extern "C" __global__ void __launch_bounds__(X0NE_PREFILL_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) \
        x0ne_attention_prefill_g##G##_bf16(                                                                       \
        const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,    \
        const uint32_t* __restrict__ pages, bf16_t* __restrict__ out, const uint32_t* __restrict__ pos0,          \
        uint32_t rows, uint32_t q_heads, uint32_t kv_heads, uint32_t max_ctx, float scale) {                       \
        __shared__ PrefillShared sh;                                                                               \
        prefill_block<G, PF_CG, false, PF_NW>(q, k_cache, v_cache, pages, out, pos0[0], rows, q_heads, kv_heads,     \
                                              max_ctx, scale, sh);                                                 \
    }                                                                                                              \
    /* The same with out in 16-row panels (device.h) of q_heads 128 columns: the prefill pass's O      */          \
    /* projection reads it so.                                                                          */          \
    extern "C" __global__ void __launch_bounds__(X0NE_PREFILL_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) \
        x0ne_attention_prefill_panel_g##G##_bf16(                                                                 \
        const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,    \
        const uint32_t* __restrict__ pages, bf16_t* __restrict__ out, const uint32_t* __restrict__ pos0,          \
        uint32_t rows, uint32_t q_heads, uint32_t kv_heads, uint32_t max_ctx, float scale) {                       \
        __shared__ PrefillShared sh;                                                                               \
        prefill_block<G, PF_CG, true, PF_NW>(q, k_cache, v_cache, pages, out, pos0[0], rows, q_heads, kv_heads,      \
                                             max_ctx, scale, sh);                                                  \
    }                                                                                                              \
    /* The panel kernel over several sequences of `rows` rows, one per blockIdx.z: sequence s has the   */          \
    /* rows from s stride on of q and out (stride a multiple of 16: whole panels), pos0[s] and the      */          \
    /* seq_pages page-table entries from s seq_pages on. 512 rows of one sequence are 128 blocks for    */          \
    /* 512 places on the chip; four sequences fill them in one launch.                                  */          \
    extern "C" __global__ void __launch_bounds__(X0NE_PREFILL_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) \
        x0ne_attention_prefill_seqs_g##G##_bf16(                                                                  \
        const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,    \
        const uint32_t* __restrict__ pages, bf16_t* __restrict__ out, const uint32_t* __restrict__ pos0,          \
        uint32_t rows, uint32_t q_heads, uint32_t kv_heads, uint32_t max_ctx, float scale, uint32_t stride,         \
        uint32_t seq_pages) {                                                                                      \
        __shared__ PrefillShared sh;                                                                               \
        const size_t at = (size_t)blockIdx.z * stride * q_heads * X0NE_HEAD_DIM;                                   \
        if (stride % 16 != 0) return;                                                                              \
        prefill_block<G, PF_CG, true, PF_NW>(q + at, k_cache, v_cache, pages + (size_t)blockIdx.z * seq_pages,     \
                                             out + at, pos0[blockIdx.z], rows, q_heads, kv_heads, max_ctx, scale,  \
                                             sh);                                                                  \
    }
X0NE_PREFILL_GROUP(1)
X0NE_PREFILL_GROUP(2)
X0NE_PREFILL_GROUP(4)
X0NE_PREFILL_GROUP(8)

// ---- causal prefill in the exact mode (f64 scores, softmax and sums) ----
//
// The exact mode's prefill passes: the arithmetic of the exact decode kernel (exact bf16 x bf16
// products summed in f64, the f64 scale 1/sqrt(128), an f64 online softmax with the maximum
// subtracted, f64 weighted V sums, the result rounded f64 -> f32 -> bf16) for every row of the
// pass, on the f64 matrix cores: v_mfma_f64_16x16x4f64, lane l supplying A[l % 16][l / 16] and
// B[l / 16][l % 16] and holding D[l / 16 + 4 i][l % 16], i = 0..3. Block (kv head kh, row
// block) serves 64 columns (column c: row r0 + c / G, head kh G + c % G), 16 to each of its 4
// wavefronts; the keys pass in tiles of 64 staged in LDS once per block (K swizzled by key, V
// dim-major swizzled by dim), the next tile's loads in flight while one is summed:
//  - scores S^T per 16-key block kb: A = K, product row r holding key 16 kb + 4 (r % 4) + r / 4,
//    so that lane l's results are the 4 consecutive keys 16 kb + 4 (l / 16) + i; k = dims
//    32 (l / 16) + j at product j; B = the wavefront's 16 q columns, lane l holding column
//    l % 16's dims 32 (l / 16) .. + 31 as f64 in registers for the whole pass;
//  - the online softmax per column: lane l holds 16 of its column's 64 keys, the other 48 sit in
//    lanes l ^ 16, l ^ 32, l ^ 48;
//  - O^T += V^T P^T: A = V^T (row = dim 16 db + l % 16, k = the key of step (kb, i),
//    16 kb + 4 (l / 16) + i: 4 consecutive keys of one dim, one 8-byte LDS read), B = P^T, whose
//    value at lane l is the lane's own weight of that key (no exchange); D = O^T, lane l holding
//    dims 16 db + l / 16 + 4 i of column l % 16 in 8 accumulators.
// Keys at or past a column's own position + 1 score -inf; V of keys at or past the block's
// context is zeroed in LDS (its weight is 0, and 0 times a value that is not a number would
// not be). Each output depends on its column's own inputs and the fixed order above.
namespace {

typedef double px_f64x4 __attribute__((ext_vector_type(4)));
constexpr uint32_t PX_COLS = X0NE_PREFILL_EXACT_COLS;       // columns per block
constexpr uint32_t PX_BLOCK = X0NE_PREFILL_EXACT_THREADS;

struct PrefillExactShared {
    alignas(16) bf16_t k[X0NE_SPLIT_TILE * X0NE_HEAD_DIM];  // [key][16 chunks of 8 dims], chunk c at c ^ (key % 16)
    alignas(16) bf16_t v[X0NE_HEAD_DIM * X0NE_SPLIT_TILE];  // [dim][8 chunks of 8 keys], chunk c at c ^ (dim % 8)
};

template <int G>
__device__ __forceinline__ void prefill_exact_block(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache,
                                                    const bf16_t* __restrict__ v_cache,
                                                    const uint32_t* __restrict__ pages, bf16_t* __restrict__ out,
                                                    uint32_t p0, uint32_t rows, uint32_t q_heads, uint32_t kv_heads,
                                                    uint32_t max_ctx, PrefillExactShared& sh) {
    constexpr uint32_t RB = PX_COLS / G;
    const uint32_t kh = blockIdx.x, r0 = blockIdx.y * RB;
    if (kh >= kv_heads || q_heads != (uint32_t)G * kv_heads || r0 >= rows || max_ctx == 0 || blockDim.x != PX_BLOCK)
        return;  // block-uniform
    const uint32_t t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t n16 = lane & 15, q4 = lane >> 4;
    const uint32_t ctx = min(p0 + min(r0 + RB, rows), max_ctx);  // keys the block reads
    const uint32_t ntiles = (ctx + X0NE_SPLIT_TILE - 1) / X0NE_SPLIT_TILE;
    const uint32_t npages = (ctx + X0NE_PAGE - 1) / X0NE_PAGE;
    // This lane's column 16 wave + l % 16: its row and key limit (keys below p0 + row + 1; a
    // column past the rows attends key 0 only and is not written), and its q dims 32 q4 .. + 31.
    const uint32_t col = 16 * wave + n16, r = r0 + col / G;
    const bool live = r < rows;
    const uint32_t lim = live ? min(p0 + r + 1, max_ctx) : 1u;
    double qv[32];
    {
        const uint4* qp = reinterpret_cast<const uint4*>(
            q + ((size_t)(live ? r : r0) * q_heads + kh * G + col % G) * X0NE_HEAD_DIM + 32 * q4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint4 u = live ? qp[j] : make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 8; ++e) qv[8 * j + e] = bf_of(u, e);
        }
    }
    // A tile's K chunk i (i = t + 256 j): key i / 16, dims 8 (i % 16) ..; V chunk i: dim i / 8,
    // keys 8 (i % 8) .. of the tile.
    constexpr int J = X0NE_SPLIT_TILE * X0NE_HEAD_DIM / 8 / PX_BLOCK;
    const auto kres = plane_rsrc(k_cache, OFF_NONE), vres = plane_rsrc(v_cache, OFF_NONE);
    uint4 kr[J], vr[J];
    auto fetch = [&](uint32_t tile) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const uint32_t i = t + PX_BLOCK * j;
            const uint32_t key = X0NE_SPLIT_TILE * tile + i / 16, kp = key / X0NE_PAGE;
            const uint32_t pb = (kp < npages ? pages[kp] : 0u) * kv_heads + kh;
            kr[j] = bload16(kres, kp < npages ? ((pb * X0NE_PAGE + key % X0NE_PAGE) * X0NE_HEAD_DIM + 8 * (i % 16)) * 2
                                              : OFF_NONE);
            const uint32_t d = i / 8, vkey = X0NE_SPLIT_TILE * tile + 8 * (i % 8), vp = vkey / X0NE_PAGE;
            const uint32_t vb = (vp < npages ? pages[vp] : 0u) * kv_heads + kh;
            vr[j] = bload16(vres, vp < npages ? ((vb * X0NE_HEAD_DIM + d) * X0NE_PAGE + vkey % X0NE_PAGE) * 2 : OFF_NONE);
        }
    };
    auto stash = [&](uint32_t tile) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const uint32_t i = t + PX_BLOCK * j, key = i / 16, kc = i % 16;
            *reinterpret_cast<uint4*>(&sh.k[key * X0NE_HEAD_DIM + 8 * (kc ^ (key % 16))]) = kr[j];
            const uint32_t d = i / 8, vc = i % 8, key0 = X0NE_SPLIT_TILE * tile + 8 * vc;
            const uint32_t valid = key0 >= ctx ? 0u : min(ctx - key0, 8u);
            uint32_t w4[4] = {vr[j].x, vr[j].y, vr[j].z, vr[j].w};
#pragma unroll
            for (int e = 0; e < 4; ++e)
                w4[e] &= (2 * e + 1 < (int)valid ? 0xFFFF0000u : 0u) | (2 * e < (int)valid ? 0xFFFFu : 0u);
            *reinterpret_cast<uint4*>(&sh.v[d * X0NE_SPLIT_TILE + 8 * (vc ^ (d % 8))]) = make_uint4(w4[0], w4[1], w4[2], w4[3]);
        }
    };
    const double scale = 1.0 / sqrt((double)X0NE_HEAD_DIM);
    double m = -INFINITY, lsum = 0.0;
    px_f64x4 o[8];
#pragma unroll
    for (int db = 0; db < 8; ++db) o[db] = px_f64x4{0.0, 0.0, 0.0, 0.0};
    fetch(0);
    for (uint32_t tile = 0; tile < ntiles; ++tile) {
        __syncthreads();  // the tile before is summed
        stash(tile);
        if (tile + 1 < ntiles) fetch(tile + 1);  // block-uniform; in flight while this tile is summed
        __syncthreads();
        // Scores of keys 16 kb + 4 q4 + i against the lane's column.
        double sc[16];
        {
            const uint32_t kt = 4 * (n16 % 4) + n16 / 4;  // the key of product row l % 16 in a block of 16
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                const uint32_t key = 16 * kb + kt;
                uint4 kv[4];
#pragma unroll
                for (int c4 = 0; c4 < 4; ++c4)
                    kv[c4] = *reinterpret_cast<const uint4*>(&sh.k[key * X0NE_HEAD_DIM + 8 * ((4 * q4 + c4) ^ (key % 16))]);
                px_f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int j = 0; j < 32; ++j)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(bf_of(kv[j / 8], j % 8), qv[j], acc, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[4 * kb + i] = acc[i];
            }
        }
        // The online softmax of the lane's column over the tile's 64 keys.
        double mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const uint32_t key = X0NE_SPLIT_TILE * tile + 16 * (e / 4) + 4 * q4 + e % 4;
            sc[e] = key < lim ? sc[e] * scale : -INFINITY;
            mx = fmax(mx, sc[e]);
        }
        mx = fmax(mx, __shfl_xor(mx, 16, 64));
        mx = fmax(mx, __shfl_xor(mx, 32, 64));
        const double mn = fmax(m, mx);  // key 0 is in every column's first tile: mn is finite
        const double al = exp(m - mn);
        double ps = 0.0;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            sc[e] = exp(sc[e] - mn);
            ps += sc[e];
        }
        lsum = lsum * al + ps;
        m = mn;
#pragma unroll
        for (int db = 0; db < 8; ++db) o[db] *= al;
        // O^T += V^T P^T over the tile's keys, 4 per product.
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
            for (int db = 0; db < 8; ++db) {
                const uint32_t d = 16 * db + n16;
                const uint2 vv = *reinterpret_cast<const uint2*>(
                    &sh.v[d * X0NE_SPLIT_TILE + 8 * ((2 * kb + q4 / 2) ^ (d % 8)) + 4 * (q4 % 2)]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t w = i < 2 ? vv.x : vv.y;
                    const double vd = (double)((i & 1) ? bf_hi(w) : bf_lo(w));
                    o[db] = __builtin_amdgcn_mfma_f64_16x16x4f64(vd, sc[4 * kb + i], o[db], 0, 0, 0);
                }
            }
    }
    // The column's weight sum over its 4 lanes (the same association in each).
    lsum += __shfl_xor(lsum, 16, 64);
    lsum += __shfl_xor(lsum, 32, 64);
    if (!live) return;
    bf16_t* op = out + ((size_t)r * q_heads + kh * G + col % G) * X0NE_HEAD_DIM;
#pragma unroll
    for (int db = 0; db < 8; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) op[16 * db + q4 + 4 * i] = f2bf((float)(o[db][i] / lsum));
}

}  // namespace

// x0ne_attention_prefill_exact_g{G}_bf16: the causal prefill of x0ne_attention_prefill_bf16
// (same arguments; `scale` unused: the f64 1/sqrt(128)) in the exact mode's arithmetic, for G q
// heads per kv head; grid (kv_heads, ceil(rows / (64 / G))), block 256.
#define X0NE_PREFILL_EXACT(G)                                                                                      \
    extern "C" __global__ void __launch_bounds__(PX_BLOCK) x0ne_attention_prefill_exact_g##G##_bf16(              \
        const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,    \
        const uint32_t* __restrict__ pages, bf16_t* __restrict__ out, const uint32_t* __restrict__ pos0,          \
        uint32_t rows, uint32_t q_heads, uint32_t kv_heads, uint32_t max_ctx, float scale) {                       \
        __shared__ PrefillExactShared sh;                                                                          \
        prefill_exact_block<G>(q, k_cache, v_cache, pages, out, pos0[0], rows, q_heads, kv_heads, max_ctx, sh);     \
    }
X0NE_PREFILL_EXACT(1)
X0NE_PREFILL_EXACT(2)
X0NE_PREFILL_EXACT(4)
X0NE_PREFILL_EXACT(8)

namespace {

// One q head per block (group sizes without a grouped kernel, the per-head witness, prefill):
// q head row q_row over kv head kh, ctx keys, slice y of P; the output directly when the block
// holds the whole context (and out_h is given), else a state at state_h[y * 132].
__device__ __forceinline__ void attn_head_block(const bf16_t* __restrict__ q_row, const bf16_t* __restrict__ kc,
                                                const bf16_t* __restrict__ vc, const uint32_t* __restrict__ pages,
                                                uint32_t kh, uint32_t kv_heads, uint32_t ctx, uint32_t y, uint32_t P,
                                                float scale, float* state_h, bf16_t* out_h, AttnShared<1>& sh) {
    const uint32_t t = threadIdx.x, wave = t >> 6;
    if (t < X0NE_HEAD_DIM) sh.qs[0][t] = bf2f(q_row[t]);
    __syncthreads();
    float m[1], l[1], o[1][2];
    const Split sp = split_of(ctx, P);
    attend_wave<1, float>(&sh.qs[0][0], kc, vc, pages, kh, kv_heads, ctx, y * sp.per + wave, BLOCK_TILES, (y + 1) * sp.per,
                          scale, sh.xch[wave], m, l, o);
    stash_wave<1, float>(sh, m, l, o);
    __syncthreads();
    if (sp.active == 1 && out_h != nullptr) {
        block_merge<1, float>(sh, [&](uint32_t, uint32_t d, float, float lv, float ov) { out_h[d] = f2bf(ov / lv); });
        return;
    }
    block_merge<1, float>(sh, [&](uint32_t, uint32_t d, float mv, float lv, float ov) {
        float* st = state_h + (size_t)y * X0NE_SPLIT_STATE;
        st[4 + d] = ov;
        if (d == 0) {
            st[0] = mv;
            st[1] = lv;
        }
    });
}

}  // namespace

// Split-K, one block (4 wavefronts) per (kv head, slice) serving the G q heads of the group:
// grid (kv_heads, P), block 256. With counter != 0 the last block of a kv head to finish merges
// its G heads into out (same code and order as x0ne_attention_merge_bf16, so the same bits) and
// sets counter[kh] back to 0; with counter == 0 and more than one active slice, out is unused and
// the merge kernel follows. With one active slice (ctx <= 256 or P = 1) the block writes out.
//
// The fused variant x0ne_attention_rope_decode_g*_bf16 takes the packed qkv row instead of q:
// it applies QK-norm + RoPE to its q heads and writes the K/V row of position pos into its page
// (the work of x0ne_qk_norm_rope_kv_write_bf16 for one decode row), then attends.
//
// x0ne_attention_rope_decode_batch_g*_bf16 is the fused variant for B independent sequences,
// grid (kv_heads, P, B): sequence b = blockIdx.z has its packed qkv row at qkv + b (q_heads + 2
// kv_heads) 128, its page table at pages + b seq_pages (its own pages of the shared K/V planes),
// its position at pos[b], its split state and counters after b (q_heads P) states and b kv_heads
// counters, and its output is row b of out, a [B][q_heads 128] matrix in panels (device.h): the
// X operand of the batched O projection.
//
// x0ne_attention_rope_decode_exact_g*_bf16 is the fused variant of the exact mode: the same
// arguments, f64 scores, softmax and sums with the f64 scale 1/sqrt(128) (`scale` is unused),
// grid (kv_heads, P); its split state is f64 (m, l, -, -, o[128] at state + (h P + y) 132
// doubles: twice x0ne_split_state_bytes), merged in f64 by the last block of each kv head.
#define X0NE_SPLIT_GROUP(G)                                                                                        \
    extern "C" __global__ void __launch_bounds__(256) x0ne_attention_decode_split_g##G##_bf16(                    \
        const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,    \
        const uint32_t* __restrict__ pages, float* __restrict__ state, uint32_t* __restrict__ counter,           \
        bf16_t* __restrict__ out, const uint32_t* __restrict__ pos, uint32_t q_heads, uint32_t kv_heads,         \
        uint32_t max_ctx, uint32_t splits, float scale) {                                                         \
        __shared__ AttnShared<G, float, false> sh;                                                                 \
        AttnArgs a = {};                                                                                           \
        a.q = q;                                                                                                   \
        a.k_cache = const_cast<bf16_t*>(k_cache);                                                                  \
        a.v_cache = const_cast<bf16_t*>(v_cache);                                                                  \
        a.pages = pages;                                                                                           \
        a.state = state;                                                                                           \
        a.counter = counter;                                                                                       \
        a.out = out;                                                                                               \
        a.pos = pos;                                                                                               \
        a.q_heads = q_heads;                                                                                       \
        a.kv_heads = kv_heads;                                                                                     \
        a.max_ctx = max_ctx;                                                                                       \
        a.splits = splits;                                                                                         \
        a.scale = scale;                                                                                           \
        attn_group_block<G, false>(a, sh);                                                                         \
    }                                                                                                              \
    extern "C" __global__ void __launch_bounds__(256) x0ne_attention_rope_decode_g##G##_bf16(                     \
        const bf16_t* __restrict__ qkv, const bf16_t* __restrict__ q_norm, const bf16_t* __restrict__ k_norm,    \
        const float* __restrict__ inv_freq, const double* __restrict__ rope_cs, bf16_t* __restrict__ k_cache,    \
        bf16_t* __restrict__ v_cache, const uint32_t* __restrict__ pages, float* __restrict__ state,             \
        uint32_t* __restrict__ counter, bf16_t* __restrict__ out, const uint32_t* __restrict__ pos,              \
        uint32_t q_heads, uint32_t kv_heads, uint32_t max_ctx, uint32_t splits, float scale, float eps) {         \
        __shared__ AttnShared<G, float, false> sh;                                                                 \
        AttnArgs a = {};                                                                                           \
        a.qkv = qkv;                                                                                               \
        a.q_norm = q_norm;                                                                                         \
        a.k_norm = k_norm;                                                                                         \
        a.inv_freq = inv_freq;                                                                                     \
        a.rope_cs = rope_cs;                                                                                       \
        a.k_cache = k_cache;                                                                                       \
        a.v_cache = v_cache;                                                                                       \
        a.pages = pages;                                                                                           \
        a.state = state;                                                                                           \
        a.counter = counter;                                                                                       \
        a.out = out;                                                                                               \
        a.pos = pos;                                                                                               \
        a.q_heads = q_heads;                                                                                       \
        a.kv_heads = kv_heads;                                                                                     \
        a.max_ctx = max_ctx;                                                                                       \
        a.splits = splits;                                                                                         \
        a.scale = scale;                                                                                           \
        a.eps = eps;                                                                                               \
        attn_group_block<G, true>(a, sh);                                                                          \
    }                                                                                                              \
    extern "C" __global__ void __launch_bounds__(256) x0ne_attention_rope_decode_batch_g##G##_bf16(               \
        const bf16_t* __restrict__ qkv, const bf16_t* __restrict__ q_norm, const bf16_t* __restrict__ k_norm,    \
        const float* __restrict__ inv_freq, const double* __restrict__ rope_cs, bf16_t* __restrict__ k_cache,    \
        bf16_t* __restrict__ v_cache, const uint32_t* __restrict__ pages, float* __restrict__ state,             \
        uint32_t* __restrict__ counter, bf16_t* __restrict__ out, const uint32_t* __restrict__ pos,              \
        uint32_t q_heads, uint32_t kv_heads, uint32_t max_ctx, uint32_t splits, float scale, float eps,          \
        uint32_t seq_pages) {                                                                                      \
        __shared__ AttnShared<G, float, false> sh;                                                                 \
        const size_t b = blockIdx.z;                                                                               \
        AttnArgs a = {};                                                                                           \
        a.qkv = qkv + b * (q_heads + 2 * kv_heads) * X0NE_HEAD_DIM;                                                \
        a.q_norm = q_norm;                                                                                         \
        a.k_norm = k_norm;                                                                                         \
        a.inv_freq = inv_freq;                                                                                     \
        a.rope_cs = rope_cs;                                                                                       \
        a.k_cache = k_cache;                                                                                       \
        a.v_cache = v_cache;                                                                                       \
        a.pages = pages + b * seq_pages;                                                                           \
        a.state = state + b * q_heads * splits * X0NE_SPLIT_STATE;                                                 \
        a.counter = counter + b * kv_heads;                                                                        \
        a.out = out;                                                                                               \
        a.out_panel = (uint32_t)b + 1;                                                                             \
        a.pos = pos + b;                                                                                           \
        a.q_heads = q_heads;                                                                                       \
        a.kv_heads = kv_heads;                                                                                     \
        a.max_ctx = max_ctx;                                                                                       \
        a.splits = splits;                                                                                         \
        a.scale = scale;                                                                                           \
        a.eps = eps;                                                                                               \
        attn_group_block<G, true>(a, sh);                                                                          \
    }                                                                                                              \
    extern "C" __global__ void __launch_bounds__(256) x0ne_attention_rope_decode_exact_g##G##_bf16(               \
        const bf16_t* __restrict__ qkv, const bf16_t* __restrict__ q_norm, const bf16_t* __restrict__ k_norm,    \
        const float* __restrict__ inv_freq, const double* __restrict__ rope_cs, bf16_t* __restrict__ k_cache,    \
        bf16_t* __restrict__ v_cache, const uint32_t* __restrict__ pages, float* __restrict__ state,             \
        uint32_t* __restrict__ counter, bf16_t* __restrict__ out, const uint32_t* __restrict__ pos,              \
        uint32_t q_heads, uint32_t kv_heads, uint32_t max_ctx, uint32_t splits, float scale, float eps) {         \
        __shared__ ExactShared sh;                                                                                 \
        AttnArgs a = {};                                                                                           \
        a.qkv = qkv;                                                                                               \
        a.q_norm = q_norm;                                                                                         \
        a.k_norm = k_norm;                                                                                         \
        a.inv_freq = inv_freq;                                                                                     \
        a.rope_cs = rope_cs;                                                                                       \
        a.k_cache = k_cache;                                                                                       \
        a.v_cache = v_cache;                                                                                       \
        a.pages = pages;                                                                                           \
        a.state = state;                                                                                           \
        a.counter = counter;                                                                                       \
        a.out = out;                                                                                               \
        a.pos = pos;                                                                                               \
        a.q_heads = q_heads;                                                                                       \
        a.kv_heads = kv_heads;                                                                                     \
        a.max_ctx = max_ctx;                                                                                       \
        a.splits = splits;                                                                                         \
        a.eps = eps;                                                                                               \
        exact_block<G>(a, sh);                                                                                     \
    }
X0NE_SPLIT_GROUP(1)
X0NE_SPLIT_GROUP(2)
X0NE_SPLIT_GROUP(4)
X0NE_SPLIT_GROUP(8)

// Split-K, one block per (q head, slice), for group sizes without a grouped kernel:
// grid (q_heads, P), block 256. The merge kernel follows unless one slice holds the context, in
// which case the block writes out itself.
extern "C" __global__ void __launch_bounds__(256)
    x0ne_attention_decode_split_bf16(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache,
                                     const bf16_t* __restrict__ v_cache, const uint32_t* __restrict__ pages,
                                     float* __restrict__ state, bf16_t* __restrict__ out,
                                     const uint32_t* __restrict__ pos, uint32_t q_heads, uint32_t kv_heads,
                                     uint32_t max_ctx, uint32_t splits, float scale) {
    __shared__ AttnShared<1> sh;
    const uint32_t h = blockIdx.x, y = blockIdx.y;
    if (h >= q_heads || y >= splits || kv_heads == 0 || q_heads % kv_heads != 0) return;
    const uint32_t kh = h / (q_heads / kv_heads);
    const uint32_t ctx = min(pos[0] + 1u, max_ctx);
    if (y >= split_of(ctx, splits).active) return;
    attn_head_block(q + (size_t)h * X0NE_HEAD_DIM, k_cache, v_cache, pages, kh, kv_heads, ctx, y, splits, scale,
                    state + (size_t)h * splits * X0NE_SPLIT_STATE, out + (size_t)h * X0NE_HEAD_DIM, sh);
}

// Merge of the split-K states: grid (q_heads), block 64, active = min(P, ceil(ctx / 256)). With
// one active slice the split kernel wrote out already and this does nothing.
extern "C" __global__ void __launch_bounds__(64)
    x0ne_attention_merge_bf16(const float* __restrict__ state, bf16_t* __restrict__ out,
                              const uint32_t* __restrict__ pos, uint32_t max_ctx, uint32_t splits) {
    __shared__ float f[MERGE_MAX];
    const uint32_t h = blockIdx.x;
    const uint32_t ctx = min(pos[0] + 1u, max_ctx);
    const uint32_t active = split_of(ctx, splits).active;
    if (active <= 1 || splits > MERGE_MAX) return;
    bf16_t* out_h = out + (size_t)h * X0NE_HEAD_DIM;
    merge_head(state + (size_t)h * splits * X0NE_SPLIT_STATE, [&](uint32_t d, bf16_t v) { out_h[d] = v; }, active, f);
}

// Per-head decode over the whole context in one block (the reference's E2 witness,
// attention.cu:9-81): grid (q_heads), block 256; one slice, normalised in the block.
extern "C" __global__ void __launch_bounds__(256)
    x0ne_attention_decode_bf16(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache,
                               const bf16_t* __restrict__ v_cache, const uint32_t* __restrict__ pages,
                               bf16_t* __restrict__ out, const uint32_t* __restrict__ pos, uint32_t q_heads,
                               uint32_t kv_heads, uint32_t max_ctx, float scale) {
    __shared__ AttnShared<1> sh;
    const uint32_t h = blockIdx.x;
    if (h >= q_heads || kv_heads == 0 || q_heads % kv_heads != 0) return;
    const uint32_t kh = h / (q_heads / kv_heads);
    const uint32_t ctx = min(pos[0] + 1u, max_ctx);
    attn_head_block(q + (size_t)h * X0NE_HEAD_DIM, k_cache, v_cache, pages, kh, kv_heads, ctx, 0, 1, scale, nullptr,
                    out + (size_t)h * X0NE_HEAD_DIM, sh);
}

// Causal prefill: rows at positions pos0[0] + r over the cache (already holding their keys).
// grid (q_heads, rows), block 256: one block per (q head, row), the decode arithmetic over keys
// 0..min(pos0 + r, max_ctx - 1). q and out are [rows][q_heads][128].
extern "C" __global__ void __launch_bounds__(256)
    x0ne_attention_prefill_bf16(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache,
                                const bf16_t* __restrict__ v_cache, const uint32_t* __restrict__ pages,
                                bf16_t* __restrict__ out, const uint32_t* __restrict__ pos0, uint32_t rows,
                                uint32_t q_heads, uint32_t kv_heads, uint32_t max_ctx, float scale) {
    __shared__ AttnShared<1> sh;
    const uint32_t h = blockIdx.x, row = blockIdx.y;
    if (row >= rows || h >= q_heads || kv_heads == 0 || q_heads % kv_heads != 0) return;
    const uint32_t kh = h / (q_heads / kv_heads);
    const uint32_t ctx = min(pos0[0] + row + 1u, max_ctx);
    const size_t at = ((size_t)row * q_heads + h) * X0NE_HEAD_DIM;
    attn_head_block(q + at, k_cache, v_cache, pages, kh, kv_heads, ctx, 0, 1, scale, nullptr, out + at, sh);
}
