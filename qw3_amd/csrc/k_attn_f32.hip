// k_attn_f32.hip -- causal GQA attention over f32 caches (head_dim 64 or 128) on the
// f32 matrix cores, for one new token or many.
//
// Semantics: kernels_b.zig:29-133. Query rows of one kv head are numbered
// R = t * group + (head in the group), so 16 consecutive rows share every K/V row they
// attend whatever the group size (1 token x 16 heads, 2 x 8, 8 x 2). A wavefront takes
// 16 rows and streams 16-position tiles:
//   S^T[16 pos x 16 rows] = K . Q^T       D / 4 v_mfma_f32_16x16x4_f32
//   O^T[D x 16 rows]     += V^T . P^T     D / 4 of them
// Everything is f32: products, sums, weights.
//
// K and V go from memory straight into operands, 16 bytes a lane, with no LDS. The
// k slots of a product may be any elements as long as both operands agree, and so may
// the rows of O^T: lane (c, g) = (lane % 16, lane / 16) loads K dims 16 j + 4 g + [0, 4)
// of position c and feeds them to four products; V dims 64 u + 4 c + [0, 4) of position
// 4 g + i, each of the four a row of its own O^T block. S^T leaves lane (c, g) with the
// scores of positions 4 g + i for query row c, which is the P^T operand of the PV
// product over k slots 4 g + i.
//
// What bounds it: decode, the bytes (16 KB per tile and 2048 matrix-core cycles is
// 32 B a cycle and CU, 2.5 times the HBM rate); prefill, the f32 matrix cores. So decode
// spreads the positions of a row tile over the 4 wavefronts of a workgroup (WS 4,
// combined through LDS) and over workgroups; prefill gives each wavefront its own row
// tile (WS 1: the four read the same K/V rows at about the same time, one L2 read each).
// One workgroup per (token, head) reading whole K rows per thread (the generic kernel,
// which other head sizes keep) took 757 us at 3000 positions of 32 q / 4 kv heads x 128
// and 480 us for a 500-token prompt; the attention blocks around them went from 782 to
// 21 us and from 575 to 117 us (norm, rope and append in one launch included).
#include "ds5_common.hpp"

namespace {

constexpr int kRows = ds5idx::kAfRows, kPos = ds5idx::kAfPos;  // query rows and positions of a tile
constexpr int kWaves = ds5idx::kAfWaves;
constexpr int kThreads = kWaves * 64;

struct AttnF32Params {
    const float* q;
    const float* k_cache;
    const float* v_cache;
    float* out;
    float* part_o;   // [n_tokens * n_q_heads, n_splits, D]
    float* part_ml;  // [n_tokens * n_q_heads, n_splits, 2]
    uint32_t pos, n_tokens, n_q_heads, group, max_ctx;
    uint32_t chunk, n_splits;  // positions per split
    float scale;
};

// exp(d) of a score less its reference. The scores stay as they are (not in units of log2,
// where a finite score above 2.4e38 would overflow): only the difference is scaled.
DS5_DEVICE_INLINE float weight_of(float d) { return fast_exp2(d * kLog2e); }

DS5_DEVICE_INLINE f32x4 mfma_f32_16x16x4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <int D>
struct Tile {
    f32x4 k[D / 16];
    f32x4 v[4][D / 64];
};

// Rows at or past `end` re-read row end - 1: their scores are masked.
template <int D>
DS5_DEVICE_INLINE void load_tile(Tile<D>& t, const float* kb, const float* vb, uint32_t p0, uint32_t end, int c, int g) {
    const float* kr = kb + (uint64_t)ds5idx::af_load_pos(p0 + c, end) * D + 4 * g;
#pragma unroll
    for (int j = 0; j < D / 16; j++) t.k[j] = *(const f32x4*)(kr + 16 * j);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float* vr = vb + (uint64_t)ds5idx::af_load_pos(p0 + 4 * g + i, end) * D + 4 * c;
#pragma unroll
        for (int u = 0; u < D / 64; u++) t.v[i][u] = *(const f32x4*)(vr + 64 * u);
    }
}

template <int D, int WS>
__global__ __launch_bounds__(kThreads) void attn_f32_kernel(const AttnF32Params p) {
    constexpr int NU = D / 64, OROW = D + 4;
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t n_rows = p.n_tokens * p.group, kvh = blockIdx.y;
    // the last row tiles (the longest contexts) first
    const uint32_t bx = gridDim.x - 1 - blockIdx.x;
    const uint32_t R0 = ds5idx::af_row0(bx, wave, WS == 1);
    if (R0 >= n_rows) return;  // WS 1: wave-uniform, no barrier follows; WS 4: never
    const uint32_t R = min(R0 + c, n_rows - 1), t = R / p.group;
    const uint64_t row = (uint64_t)t * p.n_q_heads + kvh * p.group + R % p.group;
    const uint32_t lim = p.pos + t;  // last position of this lane's row
    const uint32_t first_lim = p.pos + R0 / p.group, last_lim = p.pos + (min(R0 + kRows, n_rows) - 1) / p.group;
    const uint32_t start = blockIdx.z * p.chunk;
    if (start > last_lim) return;  // uniform over what shares a barrier: no row reaches this split
    const uint32_t end = min(start + p.chunk, last_lim + 1);
    const float* kb = p.k_cache + (uint64_t)kvh * p.max_ctx * D;
    const float* vb = p.v_cache + (uint64_t)kvh * p.max_ctx * D;

    f32x4 q[D / 16];
#pragma unroll
    for (int j = 0; j < D / 16; j++) q[j] = *(const f32x4*)(p.q + row * D + 16 * j + 4 * g);

    f32x4 O[NU][4];
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
        for (int e = 0; e < 4; e++) O[u][e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;  // l: this lane's positions only

    auto compute = [&](const Tile<D>& tl, uint32_t p0) {
        f32x4 s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = s0;
#pragma unroll
        for (int j = 0; j < D / 16; j += 2)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                s0 = mfma_f32_16x16x4(tl.k[j][i], q[j][i], s0);
                s1 = mfma_f32_16x16x4(tl.k[j + 1][i], q[j + 1][i], s1);
            }
        // positions past a row's own (or the split's) are masked: uniform test first
        const bool edge = p0 + kPos - 1 > first_lim || p0 + kPos > end;
        float s[4];
#pragma unroll
        for (int i = 0; i < 4; i++) s[i] = (s0[i] + s1[i]) * p.scale;
        if (edge) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t at = p0 + 4 * g + i;
                if (at > lim || at >= end) s[i] = -INFINITY;
            }
        }
        float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
        mx = swap32_op(swap16_op(mx, OpMax{}), OpMax{});
        const float m_new = fmaxf(m, mx);
        // a row without a score yet keeps weights of 0 (-inf - -inf would be NaN)
        const float ref = m_new == -INFINITY ? 0.0f : m_new;
        const float alpha = weight_of(m - ref);
        float w[4];
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = weight_of(s[i] - ref);
        l = l * alpha + ((w[0] + w[1]) + (w[2] + w[3]));
        m = m_new;
        if (__ballot(alpha != 1.0f)) {
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int e = 0; e < 4; e++) O[u][e] *= alpha;
        }
        if (edge) {
            // 0 x inf: a V row that some query row does not attend must not reach it, so
            // a non-finite V in an edge tile takes the products one by one
            bool bad = false;
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int u = 0; u < NU; u++)
#pragma unroll
                    for (int e = 0; e < 4; e++) bad |= !(fabsf(tl.v[i][u][e]) <= 3.4028235e38f);
            if (__builtin_expect(__ballot(bad) != 0, 0)) {
                for (int gg = 0; gg < 4; gg++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float wi = __shfl(w[i], 16 * gg + c, 64);
                        const uint32_t at = p0 + 4 * gg + i;
                        const bool seen = at <= lim && at < end;
#pragma unroll
                        for (int u = 0; u < NU; u++)
#pragma unroll
                            for (int e = 0; e < 4; e++)
#pragma unroll
                                for (int k = 0; k < 4; k++) {
                                    const float v = __shfl(tl.v[i][u][e], 16 * gg + 4 * g + k, 64);
                                    if (seen) O[u][e][k] = __builtin_fmaf(wi, v, O[u][e][k]);
                                }
                    }
                return;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int e = 0; e < 4; e++) O[u][e] = mfma_f32_16x16x4(tl.v[i][u][e], w[i], O[u][e]);
    };

    // one tile ahead, in two register sets
    constexpr uint32_t STEP = WS * kPos;
    uint32_t p0 = start + (WS == 1 ? 0 : wave * kPos);
    if (p0 < end) {  // wave-uniform
        Tile<D> ta, tb;
        load_tile<D>(ta, kb, vb, p0, end, c, g);
        for (;;) {
            if (p0 + STEP >= end) {
                compute(ta, p0);
                break;
            }
            load_tile<D>(tb, kb, vb, p0 + STEP, end, c, g);
            compute(ta, p0);
            p0 += STEP;
            if (p0 + STEP >= end) {
                compute(tb, p0);
                break;
            }
            load_tile<D>(ta, kb, vb, p0 + STEP, end, c, g);
            compute(tb, p0);
            p0 += STEP;
        }
    }
    l = swap32_op(swap16_op(l, OpAdd{}), OpAdd{});

    // O[u][e][k] of lane (c, g): row c, dim 64 u + 16 g + 4 k + e
    if constexpr (WS == 1) {
        if (R0 + c < n_rows) {
            const int to = ds5idx::af_store(lim, start, p.chunk);
            const bool single = to == ds5idx::kAfOut;
            float* dst = single ? p.out + row * D : p.part_o + (row * p.n_splits + blockIdx.z) * D;
            if (to != ds5idx::kAfNone) {
                const float den = single ? l : 1.0f;
#pragma unroll
                for (int u = 0; u < NU; u++)
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        *(f32x4*)(dst + 64 * u + 16 * g + 4 * k) =
                            f32x4{O[u][0][k], O[u][1][k], O[u][2][k], O[u][3][k]} / den;
                if (!single && g == 0) *(float2*)(p.part_ml + (row * p.n_splits + blockIdx.z) * 2) = float2{m, l};
            }
        }
    } else {
        __shared__ __attribute__((aligned(16))) float s_o[kWaves][kRows * OROW];
        __shared__ float s_m[kWaves][kRows], s_l[kWaves][kRows];
        if (g == 0) {
            s_m[wave][c] = m;
            s_l[wave][c] = l;
        }
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int k = 0; k < 4; k++)
                *(f32x4*)&s_o[wave][c * OROW + 64 * u + 16 * g + 4 * k] =
                    f32x4{O[u][0][k], O[u][1][k], O[u][2][k], O[u][3][k]};
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < kRows * (D / 4); i += kThreads) {
            const uint32_t r = i / (D / 4), d0 = 4 * (i % (D / 4)), Rr = R0 + r;
            if (Rr >= n_rows) break;
            const uint32_t tr = Rr / p.group;
            const uint64_t orow = (uint64_t)tr * p.n_q_heads + kvh * p.group + Rr % p.group;
            const int to = ds5idx::af_store(p.pos + tr, start, p.chunk);
            if (to == ds5idx::kAfNone) continue;
            float M = s_m[0][r];
#pragma unroll
            for (int w = 1; w < kWaves; w++) M = fmaxf(M, s_m[w][r]);
            const float ref = M == -INFINITY ? 0.0f : M;
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            float lt = 0.0f;
#pragma unroll
            for (int w = 0; w < kWaves; w++) {
                const float f = weight_of(s_m[w][r] - ref);
                // a wavefront without a score for the row has weight 0 and O 0
                acc += *(const f32x4*)&s_o[w][r * OROW + d0] * f;
                lt += s_l[w][r] * f;
            }
            if (to == ds5idx::kAfOut) {
                *(f32x4*)(p.out + orow * D + d0) = acc / lt;
            } else {
                *(f32x4*)(p.part_o + (orow * p.n_splits + blockIdx.z) * D + d0) = acc;
                if (d0 == 0) *(float2*)(p.part_ml + (orow * p.n_splits + blockIdx.z) * 2) = float2{M, lt};
            }
        }
    }
}

// The splits of one query row, in split order within each of the slots, then the slots
// in order: thread (slot, column) folds splits slot, slot + SLOTS, ... of one float4.
template <int D>
__global__ __launch_bounds__(256) void attn_f32_merge_kernel(const AttnF32Params p) {
    constexpr int COLS = D / 4, SLOTS = 256 / COLS, BATCH = 4;
    __shared__ f32x4 s_o[SLOTS][COLS];
    __shared__ float2 s_ml[SLOTS];
    const uint64_t row = blockIdx.x;
    const uint32_t t = (uint32_t)(row / p.n_q_heads);
    const uint32_t ns = ds5idx::af_row_splits(p.pos + t, p.chunk);
    if (ns <= 1) return;  // written by its split
    const int col = threadIdx.x % COLS, slot = threadIdx.x / COLS;
    const float2* ml_row = (const float2*)p.part_ml + row * p.n_splits;
    const float* o_row = p.part_o + row * p.n_splits * D + 4 * col;
    float m = -INFINITY, l = 0.0f;
    f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t s0 = slot; s0 < ns; s0 += SLOTS * BATCH) {
        float2 ml[BATCH];
        f32x4 os[BATCH];
#pragma unroll
        for (int k = 0; k < BATCH; k++) {
            const uint32_t s = min(s0 + SLOTS * k, ns - 1);
            ml[k] = ml_row[s];
            os[k] = *(const f32x4*)(o_row + (uint64_t)s * D);
        }
#pragma unroll
        for (int k = 0; k < BATCH; k++) {
            if (s0 + SLOTS * k >= ns) break;
            const float mn = fmaxf(m, ml[k].x), ref = mn == -INFINITY ? 0.0f : mn;
            const float a = weight_of(m - ref), w = weight_of(ml[k].x - ref);
            l = l * a + ml[k].y * w;
            o = o * a + os[k] * w;
            m = mn;
        }
    }
    s_o[slot][col] = o;
    if (col == 0) s_ml[slot] = float2{m, l};
    __syncthreads();
    if (slot == 0) {
        float M = s_ml[0].x;
#pragma unroll
        for (int k = 1; k < SLOTS; k++) M = fmaxf(M, s_ml[k].x);
        const float ref = M == -INFINITY ? 0.0f : M;
        float lt = 0.0f;
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < SLOTS; k++) {
            const float w = weight_of(s_ml[k].x - ref);
            lt += s_ml[k].y * w;
            acc += s_o[k][col] * w;
        }
        *(f32x4*)(p.out + row * D + 4 * col) = acc / lt;
    }
}

template <int D>
int launch_d(ds5_hip_ctx* ctx, const AttnF32Params& p, const AttnF32Plan& plan, uint32_t n_kv_heads) {
    const dim3 grid(plan.wave_rows ? (plan.row_tiles + kWaves - 1) / kWaves : plan.row_tiles, n_kv_heads, p.n_splits);
    if (plan.wave_rows)
        DS5_TIMED_LAUNCH(ctx, "attn_f32_kernel", (attn_f32_kernel<D, 1>), grid, dim3(kThreads), 0, ctx->stream, p);
    else
        DS5_TIMED_LAUNCH(ctx, "attn_f32_kernel", (attn_f32_kernel<D, kWaves>), grid, dim3(kThreads), 0, ctx->stream, p);
    if (int rc = ds5_after_launch(ctx, "attn_f32_kernel")) return rc;
    if (p.n_splits == 1) return DS5_OK;
    DS5_TIMED_LAUNCH(ctx, "attn_f32_merge_kernel", attn_f32_merge_kernel<D>, dim3(p.n_tokens * p.n_q_heads), dim3(256), 0,
                     ctx->stream, p);
    return ds5_after_launch(ctx, "attn_f32_merge_kernel");
}

}  // namespace

AttnF32Plan attn_f32_plan(uint32_t cu_count, uint32_t pos, uint32_t n_tokens, uint32_t n_q_heads, uint32_t n_kv_heads,
                          uint32_t head_dim) {
    const uint32_t group = n_q_heads / n_kv_heads, cu = cu_count ? cu_count : 256;
    const uint64_t L = (uint64_t)pos + n_tokens;
    AttnF32Plan pl{};
    pl.row_tiles = (uint32_t)(((uint64_t)n_tokens * group + kRows - 1) / kRows);
    // a wavefront per row tile once those fill the SIMDs; below, a workgroup per row tile
    const uint64_t units = (uint64_t)pl.row_tiles * n_kv_heads;
    pl.wave_rows = units >= 2ull * cu;
    const uint64_t step = pl.wave_rows ? kPos : kWaves * kPos;
    const uint64_t want = pl.wave_rows ? (4ull * 4 * cu + units - 1) / units : (2ull * cu + units - 1) / units;
    const uint64_t least = pl.wave_rows ? 128 : step;  // a split's partials cost about a 100-position tile row
    uint64_t chunk = (L + want - 1) / want;
    chunk = std::max<uint64_t>(least, (chunk + step - 1) / step * step);
    const uint64_t most = ds5_max_splits((uint64_t)n_tokens * n_q_heads, head_dim);
    if (most < 2) chunk = L;
    else chunk = std::max<uint64_t>(chunk, (L + most * step - 1) / (most * step) * step);
    pl.chunk = (uint32_t)std::min<uint64_t>(chunk, 0xfffffff0u);
    pl.n_splits = (uint32_t)((L + pl.chunk - 1) / pl.chunk);
    return pl;
}

int launch_attn_f32(ds5_hip_ctx* ctx, const GenericAttnLaunch& a) {
    if (a.n_tokens == 0) return DS5_OK;
    AttnF32Plan plan = attn_f32_plan(ctx->cu_count, a.pos, a.n_tokens, a.n_q_heads, a.n_kv_heads, a.head_dim);
    if (plan.n_splits > 1 && !ctx->split_buf) {  // one split needs no partials
        plan.n_splits = 1;
        plan.chunk = 0xffffffffu;
    }
    AttnF32Params p{};
    p.q = a.q;
    p.k_cache = (const float*)a.k_cache;
    p.v_cache = (const float*)a.v_cache;
    p.out = a.out;
    if (plan.n_splits > 1) {
        p.part_o = (float*)ctx->split_buf;
        p.part_ml = p.part_o + (size_t)a.n_tokens * a.n_q_heads * plan.n_splits * a.head_dim;
    }
    p.pos = a.pos;
    p.n_tokens = a.n_tokens;
    p.n_q_heads = a.n_q_heads;
    p.group = a.n_q_heads / a.n_kv_heads;
    p.max_ctx = a.max_ctx;
    p.chunk = plan.chunk;
    p.n_splits = plan.n_splits;
    p.scale = a.scale;
    return a.head_dim == 128 ? launch_d<128>(ctx, p, plan, a.n_kv_heads) : launch_d<64>(ctx, p, plan, a.n_kv_heads);
}
