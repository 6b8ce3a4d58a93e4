// k_matmul.hip -- the projection matmul of the step before the attention path:
// out[m, n] = x[m, k] . W^T, W a GGUF-layout weight of n rows of k elements in
// f32 or Q8_0 (34-byte blocks: an f16 scale, then 32 int8; value = f32(scale) * q).
//
// Semantics: kernels_a.zig:136-163 (matmul) and :39-62 (dotRow). The reference
// sums each output serially in k order; here each output is a fixed-order tree
// of per-block partial sums (scale * sum_i q_i x_i per block, then a wavefront
// reduction), so results agree to rounding, not bit for bit.
//
// Decode-shaped products (m = a few tokens) are weight-bandwidth bound: every
// weight byte is read once per pass of up to MT tokens. matmul_rows_kernel
// gives each wavefront one weight row: lane L owns the 32-element blocks
// b = L + 64 j of the row (a 2048-wide Q8_0 row, 64 blocks, is one load sweep),
// and the wavefront reduces the row's partial sums. The workgroup (8 rows)
// stages the pass's x once in LDS: read per wavefront from L2 instead, x costs
// as many bytes as the weights themselves. Q8_0 blocks are only 2-byte aligned:
// a lane reads the nine dwords covering its block from the dword boundary below
// it and realigns the bytes in registers.
#include <type_traits>

#include "ds5_common.hpp"

namespace {

constexpr int kMmThreads = 512;  // 8 wavefronts, one weight row each


// Up to kMatmulGroupMax weight matrices sharing x, in one launch: entry e owns
// the workgroups (row kernel) or column tiles (GEMM) [wg0[e], wg0[e + 1]).
struct WeightGroup {
    const uint8_t* w[kMatmulGroupMax];
    float* out[kMatmulGroupMax];
    const float* res[kMatmulGroupMax];  // residual added to out (nullptr: none)
    uint32_t n[kMatmulGroupMax];
    uint32_t wg0[kMatmulGroupMax];
    uint32_t count;
};

// Every field of a group in one scalar round trip: the entry selection below
// would otherwise load each entry's fields only after testing the previous
// entry (a chain of dependent argument loads before the first memory access).
#define DS5_GROUP_ARGS(g) \
    "s"((g).w[0]), "s"((g).w[1]), "s"((g).w[2]), "s"((g).w[3]), "s"((g).out[0]), "s"((g).out[1]), "s"((g).out[2]), \
        "s"((g).out[3]), "s"((g).res[0]), "s"((g).res[1]), "s"((g).res[2]), "s"((g).res[3]), "s"((g).n[0]), \
        "s"((g).n[1]), "s"((g).n[2]), "s"((g).n[3]), "s"((g).wg0[0]), "s"((g).wg0[1]), "s"((g).wg0[2]), \
        "s"((g).wg0[3]), "s"((g).count)
static_assert(kMatmulGroupMax == 4, "DS5_GROUP_ARGS lists four entries");

// MT tokens per pass, JB blocks per lane (k <= 2048 * JB).
// Launch: grid.x = sum of ceil(n[e] / 8), one pass of tokens m0..m0+MT-1. Rows
// past n (an entry's last workgroup) load row n - 1 and store nothing: every
// wavefront reaches the barrier.
// NORM: x is first normalised, x' = (x * inv) * nw with inv of the reference GPU
// kernel's tree order (tree_rms_inv; rows of more than 256 elements), as the
// workgroup stages it: ds5_hip_rms_norm then the product, bit for bit, with the
// norm worked out while the weights are in flight.
template <int MT, int JB, bool Q8, bool NORM>
__global__ __launch_bounds__(kMmThreads) void matmul_rows_kernel(const float* __restrict__ x, const WeightGroup g,
                                                                 uint32_t m, uint32_t k, uint32_t m0,
                                                                 const float* __restrict__ nw, float eps) {
    // this workgroup's entry (uniform; selected without indexing the argument arrays,
    // with selects rather than branches so that every field loads in one round trip)
    // (out may be the residual itself: each output is read, then written, by one lane)
    const uint8_t* __restrict__ w = g.w[0];
    float* out = g.out[0];
    const float* res = g.res[0];
    uint32_t n = g.n[0], wg = blockIdx.x;
#pragma unroll
    for (int e = 1; e < kMatmulGroupMax; e++) {
        const bool take = (uint32_t)e < g.count && blockIdx.x >= g.wg0[e];
        w = take ? g.w[e] : w;
        out = take ? g.out[e] : out;
        res = take ? g.res[e] : res;
        n = take ? g.n[e] : n;
        wg = take ? blockIdx.x - g.wg0[e] : wg;
    }

    // x in LDS: float4 chunk i of block b of token t at t * kXChunks + 8 b + (i ^ (b & 7)),
    // so the 16-byte reads of 8 consecutive lanes (one block each) hit distinct banks
    constexpr int kXChunks = JB * 512;                                  // float4 chunks of one token's x
    constexpr int kXPer = (kXChunks + kMmThreads - 1) / kMmThreads;     // chunks each thread stages
    __shared__ float4 xs[MT * kXChunks];

    const int lane = threadIdx.x & 63;
    const uint32_t row = min(wg * (kMmThreads / 64) + (threadIdx.x >> 6), n - 1);
    const uint32_t nb = k / 32, kc = k / 4;
    const uint64_t row_bytes = Q8 ? (uint64_t)nb * kQ8Bytes : (uint64_t)k * 4;
    const uint32_t mt = min((uint32_t)MT, m - m0);

    // 1. this thread's share of x (tokens past mt re-read token mt - 1; never stored)
    float4 xv[MT][kXPer];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int u = 0; u < kXPer; u++) {
            const uint32_t e = min(threadIdx.x + (uint32_t)kMmThreads * u, kc - 1);
            xv[t][u] = ((const float4*)x)[(uint64_t)(m0 + min((uint32_t)t, mt - 1)) * kc + e];
        }
    float4 wn[NORM ? kXPer : 1];
    if constexpr (NORM) {
#pragma unroll
        for (int u = 0; u < kXPer; u++) wn[u] = ((const float4*)nw)[min(threadIdx.x + (uint32_t)kMmThreads * u, kc - 1)];
    }

    // 2. the row's weights, all in flight before x is needed (loads complete in
    //    issue order, so staging x waits for x alone)
    constexpr int kWDw = Q8 ? 9 : 32;  // dwords per lane and block
    uint32_t d[JB][kWDw];
    uint32_t sh[JB];
#pragma unroll
    for (int j = 0; j < JB; j++) {
        const uint32_t b = min(lane + 64u * j, nb - 1);
        if constexpr (Q8) {
            // byte offset from w (w is 4-byte aligned, so offset & 3 is the block's)
            const uint64_t off = row * row_bytes + (uint64_t)b * kQ8Bytes;
            sh[j] = (uint32_t)off & 3u;
            const uint32_t* p = (const uint32_t*)(w + (off - sh[j]));
#pragma unroll
            for (int i = 0; i < 9; i++) d[j][i] = p[i];
        } else {
            const uint4* p = (const uint4*)(w + row * row_bytes + (uint64_t)b * 128);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint4 v = p[i];
                d[j][4 * i] = v.x;
                d[j][4 * i + 1] = v.y;
                d[j][4 * i + 2] = v.z;
                d[j][4 * i + 3] = v.w;
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // 3. stage x, then each lane takes the x of its blocks
    auto slot = [&](int t, uint32_t e) { return t * kXChunks + (e & ~7u) + ((e & 7u) ^ ((e >> 3) & 7u)); };
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int u = 0; u < kXPer; u++) {
            const uint32_t e = threadIdx.x + (uint32_t)kMmThreads * u;
            if (e < kc) xs[slot(t, e)] = xv[t][u];
        }
    __syncthreads();
    if constexpr (NORM) {
        // each token's partials from the staged row (element i: chunk i / 4, lane i % 4),
        // the tree, then the staged row rewritten as (x * inv) * nw
        __shared__ float s_part[kTreeParts];
        __shared__ float s_inv;
        const float* xf = (const float*)xs;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            float sq = 0.0f;
            if (threadIdx.x < kTreeParts)
                for (uint32_t i = threadIdx.x; i < k; i += kTreeParts) {
                    const float v = xf[4 * slot(t, i >> 2) + (i & 3)];
                    sq = __builtin_fmaf(v, v, sq);
                }
            const float inv = tree_rms_inv(sq, k, eps, s_part, &s_inv);
#pragma unroll
            for (int u = 0; u < kXPer; u++) {
                const uint32_t e = threadIdx.x + (uint32_t)kMmThreads * u;
                const float4 v = xv[t][u], ww = wn[u];
                if (e < kc)
                    xs[slot(t, e)] = float4{v.x * inv * ww.x, v.y * inv * ww.y, v.z * inv * ww.z, v.w * inv * ww.w};
            }
        }
        __syncthreads();
    }

    // 4. per-block partial sums (x of the lane's block read from LDS just before
    //    use), then the wavefront's fixed-order reduction
    float acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) acc[t] = 0.0f;
#pragma unroll
    for (int j = 0; j < JB; j++) {
        const uint32_t b = min(lane + 64u * j, nb - 1);
        float xr[MT][32];
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float4 v = xs[t * kXChunks + 8 * b + (i ^ (b & 7))];
                xr[t][4 * i] = v.x;
                xr[t][4 * i + 1] = v.y;
                xr[t][4 * i + 2] = v.z;
                xr[t][4 * i + 3] = v.w;
            }
        if (lane + 64u * j >= nb) continue;
        if constexpr (Q8) {
            const Q8Block blk = q8_unpack(d[j], sh[j]);
#pragma unroll
            for (int t = 0; t < MT; t++) acc[t] = __builtin_fmaf(blk.scale, q8_dot(blk.q, xr[t]), acc[t]);
        } else {
#pragma unroll
            for (int t = 0; t < MT; t++) {
                float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int i = 0; i < 32; i++)
                    s[i & 3] = __builtin_fmaf(__builtin_bit_cast(float, d[j][i]), xr[t][i], s[i & 3]);
                acc[t] += (s[0] + s[1]) + (s[2] + s[3]);
            }
        }
    }
    const bool live = wg * (kMmThreads / 64) + (threadIdx.x >> 6) < n;
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const float v = wave_allreduce(acc[t], OpAdd{});
        if (lane == 0 && live && (uint32_t)t < mt) {
            const uint64_t o = (uint64_t)(m0 + t) * n + row;
            out[o] = res ? res[o] + v : v;  // the reference's add(residual, proj)
        }
    }
}

// ---------------------------------------------------------------------------
// Prefill-shaped products (many tokens): Q8_0 GEMM on the f16 matrix cores.
//
// out[m, n] = sum_b scale[n, b] * sum_{e < 32} x[m, 32 b + e] * q[n, 32 b + e].
// The int8 q are exact in f16. Each x row is first scaled by a power of two,
// x' = x * 2^(14 - E) with 2^E <= max |x row| < 2^(E+1), so |x'| < 2^15 fits
// f16, and split into two f16 parts, x' = hi + lo (lo the f16 rounding of
// x' - hi): 22 significant bits, and no overflow or loss of range whatever
// the row's magnitude. Per 32-element block and 32 x 32 output tile, four
// v_mfma_f32_32x32x16_f16 (lo, lo, hi, hi: two products of 16 elements each) into a
// zeroed temporary, then acc += scale * tmp in f32 (the scale belongs to the weight
// row: one per lane in the result layout); the epilogue undoes the row's power of two
// exactly.
//
// matmul_x_split_kernel writes the two planes and the row exponents into the
// context workspace; matmul_q8_mfma_kernel then only copies x tiles.
//
// GEMM workgroup: 32 TM tokens x 128 weight rows, four wavefronts, each all the tokens of
// its own 32 weight rows (v_mfma_f32_32x32x16_f16: two products of 16 k per plane and
// block), so a weight row is converted to f16 once, in the registers that multiply it.
// What bounds it: the matrix cores (with random data the card's clock falls to about 1.7
// GHz under them), then the memory pipe of the CU, which takes 64 B a cycle: a block's 22
// KB (x planes and raw q) are 344 of its 512 matrix-core cycles. So every load is
// direct-to-LDS (inline asm with explicit vmcnt waits: the compiler's would cover the later
// blocks' loads too) and is issued between two products: issued together after the barrier
// the six took 390 cycles in which no product ran. x comes two blocks ahead into a ring of
// three stages, q three; one workgroup barrier per block. A 128-row tile takes 1160 cycles
// per block alone on a CU and 1740 beside a second one. Against the previous kernel (16 x 16
// tiles of 8 wavefronts, q converted through LDS by all of them, loads issued together):
// m 203, n 9216, k 4096: 112 -> 72 us; m 500, n 5120, k 2048: 60 -> 43 us; 2048 tokens:
// 138 -> 133 us, and 150 -> 128 us with the attention epilogue.
//
// LDS: x rows are 32 halves (four 16-byte chunks) with chunk c of row r stored at
// c ^ ((r >> 2) & 3): the 32-row operand reads run at 220 of the 256 B a cycle (measured;
// 16-row reads of the same layout reach half of it).
//
// MFMA operand layout (32x32x16): lane l supplies row / column l % 32 and eight k of half
// l / 32; which k does not matter as long as x and q agree: half h takes elements
// 16 h + 8 j + [0, 8) of the block in product j, so a lane's q are 16 consecutive bytes.
// Result element (8 (i / 4) + 4 (l / 32) + i % 4, l % 32) is in register i of lane l.
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kGemmCols = 128;  // columns of a tile of four wavefronts

constexpr int kSplitThreads = 256;
constexpr int kXExpBias = 14;  // scaled rows have max |x'| in [2^14, 2^15)

// Workspace bytes of the split x: hi and lo planes of m x k halves, m exponents.
inline size_t x_split_bytes(uint32_t m, uint32_t k) { return (size_t)m * k * 4 + (size_t)m * 4; }

// The rope angles of a prefill's tokens, made by the x split of the attention
// block's projection (one workgroup per token): cs[t] holds cos then sin of
// (pos_t * freq_scale) * inv_freq[i], i < half.
struct XSplitRope {
    const int32_t* positions;
    float* cs;
    uint32_t half;
    float freq_scale;
};

// Row `row` of the split planes from load(c) (float4 chunk c of the row's k values):
// max |v|, its exponent E, then hi / lo of v * 2^(14 - E). A row of zeros (or with a
// non-finite maximum) keeps E = 0. red: kSplitThreads / 64 floats of LDS.
template <class F>
__device__ __forceinline__ void split_row(F load, uint64_t row, uint32_t k, uint16_t* __restrict__ hi,
                                          uint16_t* __restrict__ lo, int* __restrict__ row_exp, float* red) {
    const uint32_t kc = k / 4;
    float mx = 0.0f;
    for (uint32_t c = threadIdx.x; c < kc; c += kSplitThreads) {
        const float4 v = load(c);
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
    mx = wave_allreduce(mx, OpMax{});
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    // floor(log2 mx): frexp gives mx = f * 2^x with f in [0.5, 1)
    const int e = (mx > 0.0f && mx <= 3.4028235e38f) ? __builtin_amdgcn_frexp_expf(mx) - 1 : 0;
    const int sh = kXExpBias - e;
    if (threadIdx.x == 0) row_exp[row] = e;
    uint2* h2 = (uint2*)(hi + row * k);
    uint2* l2 = (uint2*)(lo + row * k);
    for (uint32_t c = threadIdx.x; c < kc; c += kSplitThreads) {
        const float4 v = load(c);
        const float f[4] = {v.x, v.y, v.z, v.w};
        uint32_t hb[4], lb[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float s = __builtin_ldexpf(f[i], sh);
            const _Float16 h = (_Float16)s;
            hb[i] = __builtin_bit_cast(uint16_t, h);
            lb[i] = __builtin_bit_cast(uint16_t, (_Float16)(s - (float)h));
        }
        h2[c] = uint2{hb[0] | (hb[1] << 16), hb[2] | (hb[3] << 16)};
        l2[c] = uint2{lb[0] | (lb[1] << 16), lb[2] | (lb[3] << 16)};
    }
}

// One workgroup per x row: split_row of x. ROPE: also the
// row's token's rope cos / sin. nw (if not null): the row is first normalised,
// x' = (x * inv) * nw with inv in the reference GPU kernel's tree order
// (tree_rms_inv), exactly as ds5_hip_rms_norm writes rows of more than 256
// elements.
template <bool ROPE>
__global__ __launch_bounds__(kSplitThreads) void matmul_x_split_kernel(const float* __restrict__ x,
                                                                       uint16_t* __restrict__ hi,
                                                                       uint16_t* __restrict__ lo,
                                                                       int* __restrict__ row_exp, uint32_t k,
                                                                       XSplitRope rope, RopeTable table,
                                                                       const float* __restrict__ nw, float eps) {
    static_assert(kSplitThreads >= kTreeParts, "one tree partial per thread");
    __shared__ float red[kSplitThreads / 64];
    __shared__ float s_part[kTreeParts];
    __shared__ float s_inv;
    const uint64_t row = blockIdx.x;
    if constexpr (ROPE) {
        const float pos = (float)rope.positions[row];
        for (uint32_t i = threadIdx.x; i < rope.half; i += kSplitThreads) {
            const float ang = qk_rope_angle(pos, rope.freq_scale, table.inv[i]);
            rope.cs[row * 2 * rope.half + i] = cosf(ang);
            rope.cs[row * 2 * rope.half + rope.half + i] = sinf(ang);
        }
    }
    const float4* xr = (const float4*)(x + row * k);
    float inv = 1.0f;
    if (nw) {  // uniform
        float sq = 0.0f;
        for (uint32_t i = threadIdx.x; i < k; i += kTreeParts) {
            const float v = x[row * k + i];
            sq = __builtin_fmaf(v, v, sq);
        }
        inv = tree_rms_inv(sq, k, eps, s_part, &s_inv);
    }
    auto load = [&](uint32_t c) {
        const float4 v = xr[c];
        if (!nw) return v;
        const float4 w = ((const float4*)nw)[c];
        return float4{v.x * inv * w.x, v.y * inv * w.y, v.z * inv * w.z, v.w * inv * w.w};
    };
    split_row(load, row, k, hi, lo, row_exp, red);
}

// The planes of a MoE layer's expert products, for rows sorted by expert: row r of
// h = silu(g) * u (kernels_c.zig:70-72, silu(v) = v / (1 + exp(-v))) from the gate
// and up products g, u [rows, k] f32, split as matmul_x_split_kernel splits x.
__global__ __launch_bounds__(kSplitThreads) void moe_h_split_kernel(const float* __restrict__ g,
                                                                   const float* __restrict__ u,
                                                                   uint16_t* __restrict__ hi,
                                                                   uint16_t* __restrict__ lo,
                                                                   int* __restrict__ row_exp, uint32_t k) {
#pragma clang fp contract(off)
    __shared__ float red[kSplitThreads / 64];
    const uint64_t row = blockIdx.x;
    const float4* gr = (const float4*)(g + row * k);
    const float4* ur = (const float4*)(u + row * k);
    auto load = [&](uint32_t c) {
        const float4 a = gr[c], b = ur[c];
        return float4{a.x / (1.0f + expf(-a.x)) * b.x, a.y / (1.0f + expf(-a.y)) * b.y,
                      a.z / (1.0f + expf(-a.z)) * b.z, a.w / (1.0f + expf(-a.w)) * b.w};
    };
    split_row(load, row, k, hi, lo, row_exp, red);
}

// The same planes, one wavefront per row (rows of k <= 256 R elements): the row's h stays
// in registers between its maximum and its split, no barrier; the arithmetic of
// split_row operation for operation.
template <int R>
__global__ __launch_bounds__(256) void moe_h_split_rows_kernel(const float* __restrict__ g,
                                                               const float* __restrict__ u,
                                                               uint16_t* __restrict__ hi, uint16_t* __restrict__ lo,
                                                               int* __restrict__ row_exp, uint32_t k, uint32_t rows) {
#pragma clang fp contract(off)
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t row = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;  // wavefront-uniform; the kernel has no barrier
    const uint32_t kc = k / 4;
    const float4* gr = (const float4*)(g + row * k);
    const float4* ur = (const float4*)(u + row * k);
    float4 h[R];
    float mx = 0.0f;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t c = lane + 64 * r;
        h[r] = float4{0.0f, 0.0f, 0.0f, 0.0f};
        if (c < kc) {
            const float4 a = gr[c], b = ur[c];
            h[r] = float4{a.x / (1.0f + expf(-a.x)) * b.x, a.y / (1.0f + expf(-a.y)) * b.y,
                          a.z / (1.0f + expf(-a.z)) * b.z, a.w / (1.0f + expf(-a.w)) * b.w};
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(h[r].x), fabsf(h[r].y)), fmaxf(fabsf(h[r].z), fabsf(h[r].w))));
        }
    }
    mx = wave_allreduce(mx, OpMax{});
    const int e = (mx > 0.0f && mx <= 3.4028235e38f) ? __builtin_amdgcn_frexp_expf(mx) - 1 : 0;
    const int sh = kXExpBias - e;
    if (lane == 0) row_exp[row] = e;
    uint2* h2 = (uint2*)(hi + row * k);
    uint2* l2 = (uint2*)(lo + row * k);
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t c = lane + 64 * r;
        if (c < kc) {
            const float f[4] = {h[r].x, h[r].y, h[r].z, h[r].w};
            uint32_t hb[4], lb[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float s = __builtin_ldexpf(f[i], sh);
                const _Float16 hv = (_Float16)s;
                hb[i] = __builtin_bit_cast(uint16_t, hv);
                lb[i] = __builtin_bit_cast(uint16_t, (_Float16)(s - (float)hv));
            }
            h2[c] = uint2{hb[0] | (hb[1] << 16), hb[2] | (hb[3] << 16)};
            l2[c] = uint2{lb[0] | (lb[1] << 16), lb[2] | (lb[3] << 16)};
        }
    }
}

// Four int8 (one dword) as four f16: bytes biased to q + 128, placed under the
// f16 pattern 0x64 (1024 + q + 128, exact), then 1152 subtracted in f16.
__device__ __forceinline__ uint2 i8x4_to_f16x4(uint32_t u) {
    const uint32_t v = u ^ 0x80808080u;
    typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
    const h2_t bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    const h2_t a = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)) - bias;
    const h2_t b = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)) - bias;
    return uint2{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)};
}

// Workgroup barrier that orders LDS only: global loads stay in flight across it.
__device__ __forceinline__ void gemm_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ uint32_t gemm_lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}

// Wave-uniform 64-bit value made explicitly scalar (an asm "s" operand).
__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    return ((uint64_t)hi << 32) | (uint64_t)lo;
}

// Wait until at most N vector-memory operations of this wavefront are
// outstanding (the compiler does not count inline-asm loads).
template <int N>
__device__ __forceinline__ void wait_vm_only() {
    static_assert(N >= 0 && N < 16, "vmcnt field");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Direct-to-LDS load: 16 (DW = 4) or 4 (DW = 1) bytes per lane from base + off
// to LDS address lds + lane * 4 DW.
template <int DW>
__device__ __forceinline__ void lds_dma(uint32_t off, uint64_t base, uint32_t lds) {
    if constexpr (DW == 4)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds)
                     : "m0", "memory");
    else
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(base), "s"(lds)
                     : "m0", "memory");
}

// EPI = 1: the attention block's q / k / v projections (entries 0, 1, 2 of the
// group), tiles of 128 columns: a tile is 32 TM tokens of one head's 128 dims, and
// the epilogue turns it into what the prefill attention reads -- k: RMSNorm
// (serial sum) and rotation, f16 into the cache row pos + t of its kv head; v:
// f16 into the cache; q: RMSNorm, rotation, times q_scale, f16 into the q
// operand [t, n_q_heads, 128] -- with the arithmetic of the pre-pass (k) and of
// the attention kernel's own q operand (q) (the qk_* helpers), so the results
// equal the separate projection and step.
struct AttnPrepEpi {
    const float* q_norm;
    const float* k_norm;
    const float* cs;  // [m, 128]: cos of pairs 0..63, then sin
    f16* q16;
    f16* k_cache;
    f16* v_cache;
    uint32_t pos, n_q_heads, max_ctx;
    float eps, q_scale;
};

// GRP: the experts' products of a MoE layer over rows sorted by expert.
// Workgroup row tile y is tiles[y] = (first row, end row, expert): its rows are the
// sorted rows [first, end) (rows past the end read end - 1, a row of the same
// expert, and store nothing), its weights the expert's matrix, w + expert *
// w_stride; tiles past *count stop at once. Sorted row r reads plane row x_rows[r]
// (null: r) and its output goes to row out_rows[r] (null: r).
struct MoeGemmTiles {
    const uint4* tiles;
    const uint32_t* count;
    uint64_t w_stride;
    const uint32_t* x_rows;
    const uint32_t* out_rows;
};

// W wavefronts (32 columns each) make the tile. KS > 1: KS groups of W wavefronts share it,
// each with its own rings over its own range of blocks; the groups' sums add in group order
// at the end (W does not change the order).
template <int TM, int W, int KS, int EPI, bool GRP = false>
__global__ __launch_bounds__(64 * W * KS, W* KS <= 4 ? 2 : W * KS / 4) void matmul_q8_mfma_kernel(const uint16_t* __restrict__ xhi,
                                                                         const uint16_t* __restrict__ xlo,
                                                                         const int* __restrict__ row_exp,
                                                                         const WeightGroup g, uint32_t m, uint32_t k,
                                                                         const AttnPrepEpi ep, const MoeGemmTiles mt) {
    constexpr int BM = 32 * TM, BN = 32 * W, U = TM == 1 ? 1 : 2, kGroupThreads = 64 * W;
    static_assert(EPI == 0 || BN == kGemmCols, "the epilogue takes a head of 128 columns");
    asm volatile("" ::DS5_GROUP_ARGS(g), "s"(xhi), "s"(xlo), "s"(row_exp), "s"(m), "s"(k));
    // this workgroup's entry and column tile (uniform); out may be the residual itself
    // Workgroup L = y * gridDim.x + x runs on XCD L % 8. With gridDim.y a multiple of 8
    // (the launchers pad 8 or more row tiles to one), XCD q takes the row tiles q, q + 8,
    // ... with all their column tiles in a row, so a row tile's x rows come into one L2
    // (every (column, row tile) once; padding row tiles return at once).
    uint32_t bx = blockIdx.x, by = blockIdx.y;
    if (gridDim.y % 8 == 0) {
        const uint32_t L = blockIdx.y * gridDim.x + blockIdx.x, li = L / 8;
        bx = li % gridDim.x;
        by = L % 8 + 8 * (li / gridDim.x);
    }
    if (!GRP && by * BM >= m) return;  // workgroup-uniform, before any barrier
    const uint8_t* __restrict__ w = g.w[0];
    float* out = g.out[0];
    const float* res = g.res[0];
    uint32_t n = g.n[0], tile = bx;
    int entry = 0;
#pragma unroll
    for (int e = 1; e < kMatmulGroupMax; e++)
        if ((uint32_t)e < g.count && bx >= g.wg0[e]) {
            w = g.w[e];
            out = g.out[e];
            res = g.res[e];
            n = g.n[e];
            tile = bx - g.wg0[e];
            entry = e;
        }
    uint32_t m0 = by * BM;
    if constexpr (GRP) {
        if (by >= *mt.count) return;  // workgroup-uniform, before any barrier
        const uint4 te = mt.tiles[by];
        m0 = te.x;
        m = te.y;
        w += (uint64_t)te.z * mt.w_stride;
    }

    // LDS: rings of three x stages [hi, lo][row * 4 + swizzled chunk] and three raw q stages
    // of 2 KB per wavefront; EPI 1 reuses the bytes for a head's f32 tile
    constexpr int kX = 2 * BM * 64, kStages = 3, kQ = 2048, kQ0 = kStages * kX;
    constexpr int kGroup = kQ0 + kStages * W * kQ, kMain = KS * kGroup;
    static_assert((KS - 1) * TM * 16 * kGroupThreads * 4 <= kMain, "the groups' sums fit the rings");
    constexpr int kTileRow = 128 + 4;  // EPI 1 tile row stride in floats (16-byte rows, rows 4 banks apart)
    constexpr int kLdsBytes = EPI == 1 && BM * kTileRow * 4 > kMain ? BM * kTileRow * 4 : kMain;
    __shared__ __attribute__((aligned(16))) unsigned char smem[kLdsBytes];
    // the tile rows' power-of-two shifts and (GRP) output rows, for the epilogue: read there
    // from memory one by one they cost as much as the products (64 dependent loads a lane)
    __shared__ __attribute__((aligned(16))) int s_sh[BM];
    __shared__ __attribute__((aligned(16))) uint32_t s_orow[GRP ? BM : 4];

    const int lane = threadIdx.x & 63, r32 = lane & 31, h = lane >> 5;
    const uint32_t wave_id = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wave = wave_id % W, group = wave_id / W;
    const uint32_t n0 = tile * BN, col = 32 * wave + r32;
    const uint32_t nb = k / 32;
    const uint32_t row_bytes = nb * kQ8Bytes;  // below 2^31: the launchers' 32-bit offsets
    unsigned char* const ring = smem + group * kGroup;
    const uint32_t smem_lds = gemm_lds_addr(ring);
    // this group's blocks [first, first + iters) below nb: every group runs iters iterations
    // (the barriers), those past its blocks without loads or products
    // (past its end the last block is asked for again, so that every iteration has the same
    // loads outstanding; the loop ends on a full wait)
    uint32_t iters, first, blocks, bl;
    ds5idx::gemm_group_blocks(nb, group, KS, iters, first, blocks, bl);

    // x: load i of this wavefront fills bytes [1024 (wave + W i), +1024) of a stage, lane L
    // the 16 bytes at +16 L: plane, row r, slot L % 4 holding chunk (L % 4) ^ ((r >> 2) & 3).
    constexpr int NX = kX / 1024 / W;
    static_assert(NX >= 1 && NX * 1024 * W == kX && (BM * 64) % 1024 == 0, "whole 1 KB x loads inside one plane");
    uint32_t xoff[NX];  // byte offset in the plane: row min(m0 + r, m - 1), chunk c, block 0
#pragma unroll
    for (int i = 0; i < NX; i++) {
        const uint32_t o = 1024u * (wave + W * i) + 16u * lane;
        if (GRP && mt.x_rows) {  // uniform
            const uint32_t r = ds5idx::gemm_x_tile_row(o, BM);
            xoff[i] = ds5idx::gemm_x_off_row(r, (uint32_t)lane, mt.x_rows[min(m0 + r, m - 1)], k);
        } else {
            xoff[i] = ds5idx::gemm_x_off(o, (uint32_t)lane, BM, m0, m, k);
        }
    }
    auto issue_x = [&](uint32_t b, uint32_t stage, int i) {
        const uint32_t blk = wave + W * i;  // uniform
        const uint16_t* plane = blk * 1024 < BM * 64 ? xhi : xlo;
        lds_dma<4>(xoff[i], uniform_u64((uint64_t)(uintptr_t)plane + 64ull * b),
                   (uint32_t)__builtin_amdgcn_readfirstlane(smem_lds + stage * kX + 1024 * blk));
    };
    // raw q: row r of the wavefront's 32 takes 48 bytes, three 16-byte lanes with dwords
    // 0..3, 4..7 and 5..8 of the nine from the dword boundary at or below its block: 96
    // lanes of two loads (the others repeat the last, into the area's padding). 34 b is 0 mod
    // 4 for even b and 2 mod 4 for odd b: scalar base w + 34 b or w + 34 b - 2, lane offsets
    // per parity.
    uint32_t qe[2], qo[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t u = ds5idx::gemm_q_unit(i, (uint32_t)lane);
        ds5idx::gemm_q_off(ds5idx::gemm_q_dword(u), ds5idx::gemm_q_row(u, wave), n0, n, row_bytes, qe[i], qo[i]);
    }
    auto issue_q = [&](uint32_t b, uint32_t slot, int i) {
        const bool odd = b & 1;
        const uint64_t base = uniform_u64((uint64_t)(uintptr_t)w + (uint64_t)kQ8Bytes * b - (odd ? 2u : 0u));
        const uint32_t at = (uint32_t)__builtin_amdgcn_readfirstlane(smem_lds + kQ0 + (slot * W + wave) * kQ);
        lds_dma<4>(odd ? qo[i] : qe[i], base, at + 1024 * i);
    };
    constexpr int kVmPerBlock = NX + 2;

    // q operand: lane (r32, h) takes bytes 16 h .. 16 h + 15 of its column's block (dwords
    // 4 h .. 4 h + 4), converted to f16; the scale is in the h = 0 lanes' first dword.
    const bool s2 = (min(n0 + col, n - 1) * row_bytes) & 2u;  // even blocks start 2 mod 4
    struct QRaw {
        u32x4_t d;
        uint32_t d4;
    };
    auto q_raw = [&](uint32_t slot) {
        const unsigned char* row = ring + kQ0 + (slot * W + wave) * kQ + 48 * r32;
        return QRaw{*(const u32x4_t*)(row + 16 * h), *(const uint32_t*)(row + (h ? 44 : 16))};
    };
    // part p < 4: four elements; part 4: the scale, from the h = 0 half to both
    auto q_part = [&](f16x8_t& q0, f16x8_t& q1, float& scale, const QRaw& r, bool at2, int p) {
        if (p < 4) {
            const uint2 v = i8x4_to_f16x4(__builtin_amdgcn_perm(p < 3 ? r.d[p < 3 ? p + 1 : 3] : r.d4, r.d[p],
                                                                at2 ? 0x07060504u : 0x05040302u));
            u32x4_t w4 = __builtin_bit_cast(u32x4_t, p < 2 ? q0 : q1);
            w4[2 * (p & 1)] = v.x;
            w4[2 * (p & 1) + 1] = v.y;
            (p < 2 ? q0 : q1) = __builtin_bit_cast(f16x8_t, w4);
        } else {
            const uint32_t sb = at2 ? r.d[0] >> 16 : r.d[0] & 0xffffu;
            scale = f16_bits_to_f32(__builtin_amdgcn_permlane32_swap(sb, sb, false, false)[0]);
        }
    };

    if (threadIdx.x < BM) {
        const uint32_t row = min(m0 + threadIdx.x, m - 1);
        s_sh[threadIdx.x] = row_exp[GRP && mt.x_rows ? mt.x_rows[row] : row] - kXExpBias;
        if constexpr (GRP) s_orow[threadIdx.x] = mt.out_rows ? mt.out_rows[row] : row;
    }
    static_assert(BM <= kGroupThreads * KS, "a thread per tile row");

    f32x16 acc[TM];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][e] = 0.0f;

    // x operand of row subtile i, half j of the block: chunk 2 h + j of row 32 i + r32
    const uint32_t swz = (r32 >> 2) & 3;
    auto x_op = [&](const unsigned char* st, int plane, int i, int j) {
        return *(const f16x8_t*)(st + plane * BM * 64 + i * 2048 + r32 * 64 + ((2 * h + j) ^ swz) * 16);
    };
    // Iteration b: wait until only what the last iteration asked for is outstanding (block
    // b + 1's x, block b + 2's q), meet (block b's x is in LDS for everyone, and everyone is
    // done with block b - 1, whose stage block b + 2's x takes), ask for block b + 2's x and
    // block b + 3's q, multiply block b, convert block b + 1's q (the wavefront's own loads:
    // its own wait covers them) beside it.
    //
    // Within the block the products run in pairs of subtiles, two chains of four (lo, lo,
    // hi, hi) in turn. A slot is one product, the x operand read kAhead products early, and
    // four of the previous pair's scale multiply-adds (across blocks too): a wavefront keeps
    // the matrix core and the VALU busy by itself, the scheduling fences hold the order.
    constexpr int kAhead = 6;
    auto issue = [&](uint32_t b, uint32_t stage, uint32_t bq, uint32_t slot, int n) {
        if (n < NX) issue_x(b, stage, n);
        else if (n < NX + 2) issue_q(bq, slot, n - NX);
    };
#pragma unroll
    for (int n = 0; n < NX + 2; n++) issue(first, 0, first, 0, n);
    issue_q(min(first + 1, bl), 1, 0);
    issue_q(min(first + 1, bl), 1, 1);
#pragma unroll
    for (int n = 0; n < NX + 2; n++) issue(min(first + 1, bl), 1, min(first + 2, bl), 2, n);
    auto loop = [&](auto pairs) {
        constexpr int NP = decltype(pairs)::value, PS = 4 * U, NS = PS * NP;
        f32x16 t[2][2];  // [parity of the pair][subtile]
        float ps = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int e = 0; e < 16; e++) t[u / 2][u % 2][e] = 0.0f;
        f16x8_t q0 = {}, q1 = {};
        float sb = 0.0f;
        {
            wait_vm_only<kVmPerBlock>();
            const QRaw r = q_raw(0);
#pragma unroll
            for (int p = 0; p < 5; p++) q_part(q0, q1, sb, r, s2 != (bool)(first & 1), p);
        }
        uint32_t st = 0;
        auto block = [&](uint32_t i, auto par) {
            constexpr int P0 = decltype(par)::value;
            wait_vm_only<kVmPerBlock>();
            gemm_lds_sync();
            if (KS > 1 && i >= blocks) return;  // wavefront-uniform
            const uint32_t b = first + i;
            const unsigned char* at = ring + st * kX;
            const uint32_t st0 = st, st2 = st == 0 ? 2 : st - 1;  // b % 3, (b + 2) % 3
            st = st == 2 ? 0 : st + 1;
            f16x8_t xr[NS];
            auto read = [&](int n) {
                const int p = n / PS, s = n % PS / U, u = n % U;
                xr[n] = x_op(at, s < 2 ? 1 : 0, U * p + u, s & 1);
            };
#pragma unroll
            for (int n = 0; n < min(kAhead, NS); n++) read(n);
            const bool at2 = s2 != (bool)((b + 1) & 1);
            const QRaw nx = q_raw(st);
            f16x8_t n0q = q0, n1q = q1;
            float ns = sb;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < NS; n++) {
                const int p = n / PS, q = n % PS, s = q / U, u = q % U, cur = (P0 + p) & 1, pp = p == 0 ? NP - 1 : p - 1;
                if (n + kAhead < NS) read(n + kAhead);
                // one load per product or two: a load holds the wavefront's issue for as
                // long as the memory pipe needs for it (64 B a cycle and CU), which only
                // products in flight cover
                if constexpr (NS >= 2 * kVmPerBlock) {
                    if (n % 2 == 1) issue(min(b + 2, bl), st2, min(b + 3, bl), st0, n / 2);
                } else {
#pragma unroll
                    for (int v = n * kVmPerBlock / NS; v < (n + 1) * kVmPerBlock / NS; v++)
                        issue(min(b + 2, bl), st2, min(b + 3, bl), st0, v);
                }
                if (s == 0) {
                    f32x16 z;
#pragma unroll
                    for (int e = 0; e < 16; e++) z[e] = 0.0f;
                    t[cur][u] = mfma_32x32x16(xr[n], q0, z);
                } else {
                    t[cur][u] = mfma_32x32x16(xr[n], s & 1 ? q1 : q0, t[cur][u]);
                }
                const float sc = p == 0 ? ps : sb;
#pragma unroll
                for (int e = 4 * (q % 4); e < 4 * (q % 4) + 4; e++) {
                    float v = __builtin_fmaf(sc, t[cur ^ 1][q / 4][e], acc[U * pp + q / 4][e]);
                    asm volatile("" : "+v"(v));  // here, not sunk into a later block
                    acc[U * pp + q / 4][e] = v;
                }
                if (p == NP - 1 && q < 5) q_part(n0q, n1q, ns, nx, at2, q);
                if (PS < 5 && n == NS - 1) q_part(n0q, n1q, ns, nx, at2, 4);
                __builtin_amdgcn_sched_barrier(0);
            }
            ps = sb;
            q0 = n0q;
            q1 = n1q;
            sb = ns;
        };
        auto last = [&](auto par) {  // the last pair's sums
            constexpr int C = decltype(par)::value;
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int e = 0; e < 16; e++)
                    acc[U * (NP - 1) + u][e] = __builtin_fmaf(ps, t[C][u][e], acc[U * (NP - 1) + u][e]);
        };
        for (uint32_t i = 0; i < iters; i += 2) {
            block(i, std::integral_constant<int, 0>{});
            if (i + 1 < iters) block(i + 1, std::integral_constant<int, NP & 1>{});
        }
        if (NP & 1 && blocks % 2 == 0) last(std::integral_constant<int, NP & 1>{});  // uniform
        else last(std::integral_constant<int, (NP - 1) & 1>{});
        wait_vm_only<0>();  // the repeated loads, before their LDS is used or given up
    };
    // pairs of 32-row subtiles that hold rows (uniform); the others skip their products
    const uint32_t live = (uint32_t)__builtin_amdgcn_readfirstlane((int)((m - m0 + 63) / 64));
    static_assert(TM == 1 || TM == 2 || TM == 4, "tiles");
    if constexpr (TM > 2) {
        if (live >= TM / 2) loop(std::integral_constant<int, TM / 2>{});
        else loop(std::integral_constant<int, 1>{});
    } else {
        loop(std::integral_constant<int, 1>{});
    }

    if constexpr (KS > 1) {
        // the groups' sums to group 0, in group order
        float* part = reinterpret_cast<float*>(smem);
        __syncthreads();  // every group's last ring reads
        if (group > 0)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int e = 0; e < 16; e++)
                    part[(((group - 1) * TM + i) * 16 + e) * kGroupThreads + (threadIdx.x % kGroupThreads)] = acc[i][e];
        __syncthreads();
        if (group == 0)
#pragma unroll
            for (int q = 1; q < KS; q++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][e] += part[(((q - 1) * TM + i) * 16 + e) * kGroupThreads + threadIdx.x];
        if (EPI == 0 && group > 0) return;
    }

    if constexpr (EPI == 1) {
        // The tile's head goes through LDS; then thread t takes row t / 8 (+ kRowsPer, ...),
        // dims k8 + [0, 8) and 64 + k8 + [0, 8) (8 rope pairs), k8 = 8 (t % 8).
        constexpr int D = 128, HALF = 64, TROW = kTileRow, kRowsPer = kGroupThreads * KS / 8;
        const int r0 = threadIdx.x / 8, k8 = 8 * (threadIdx.x % 8);
        const float* nw = entry == 0 ? ep.q_norm : ep.k_norm;
        float w0[8], w1[8];
        if (entry != 2) {
            *(float4*)&w0[0] = *(const float4*)(nw + k8);
            *(float4*)&w0[4] = *(const float4*)(nw + k8 + 4);
            *(float4*)&w1[0] = *(const float4*)(nw + HALF + k8);
            *(float4*)&w1[4] = *(const float4*)(nw + HALF + k8 + 4);
        }
        float* tl = reinterpret_cast<float*>(smem);
        const uint32_t head = tile;  // column tile j of an entry is head j
        __syncthreads();  // every wavefront's last read of the bytes
        if (group == 0) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int lr = 32 * i + 8 * (e / 4) + 4 * h + e % 4;
                    tl[lr * TROW + col] = __builtin_ldexpf(acc[i][e], s_sh[lr]);
                }
        }
        __syncthreads();
#pragma unroll 1
        for (int r = r0; r < BM; r += kRowsPer) {
            const uint32_t tok = m0 + r;
            if (m0 + (r - r0) >= m) break;  // uniform: no rows left
            const bool ok = tok < m;
            const float* trow = tl + r * TROW;
            float x0[8], x1[8], c[8], sn[8];
            if (entry != 2) {
                const float* cs = ep.cs + (uint64_t)min(tok, m - 1) * D;
                *(float4*)&c[0] = *(const float4*)(cs + k8);
                *(float4*)&c[4] = *(const float4*)(cs + k8 + 4);
                *(float4*)&sn[0] = *(const float4*)(cs + HALF + k8);
                *(float4*)&sn[4] = *(const float4*)(cs + HALF + k8 + 4);
            }
            *(float4*)&x0[0] = *(const float4*)(trow + k8);
            *(float4*)&x0[4] = *(const float4*)(trow + k8 + 4);
            *(float4*)&x1[0] = *(const float4*)(trow + HALF + k8);
            *(float4*)&x1[4] = *(const float4*)(trow + HALF + k8 + 4);
            f16x8_t y0v, y1v;
            f16* dst;
            if (entry == 2) {  // v: f16 append
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    y0v[j] = (f16)x0[j];
                    y1v[j] = (f16)x1[j];
                }
                dst = ep.v_cache + ((uint64_t)head * ep.max_ctx + ep.pos + tok) * D;
            } else {
                if (entry == 0) {
                    // q: the thread's two quarters (pairs k8 .. k8 + 3 and k8 + 4 .. k8 + 7),
                    // then the head's 8 threads in the balanced tree's order (xor 1, 2, 4)
                    float ss = qk_quarter_sumsq(x0[0], x1[0], x0[1], x1[1], x0[2], x1[2], x0[3], x1[3]) +
                               qk_quarter_sumsq(x0[4], x1[4], x0[5], x1[5], x0[6], x1[6], x0[7], x1[7]);
#pragma unroll
                    for (int mm = 1; mm < 8; mm <<= 1) ss += __shfl_xor(ss, mm, 64);
                    const float r1 = rms_inv(ss, (float)D, ep.eps) * ep.q_scale;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        _Float16 o0, o1;
                        qk_q_pair(x0[j], x1[j], w0[j], w1[j], c[j], sn[j], r1, o0, o1);
                        y0v[j] = o0;
                        y1v[j] = o1;
                    }
                } else {  // k: the reference's serial sum of the row
                    const float inv = rms_inv(qk_serial_sumsq(trow, D), (float)D, ep.eps);
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        float y0, y1;
                        qk_rotate(qk_norm_mul(x0[j], inv, w0[j]), qk_norm_mul(x1[j], inv, w1[j]), c[j], sn[j], y0,
                                  y1);
                        y0v[j] = (f16)y0;
                        y1v[j] = (f16)y1;
                    }
                }
                dst = entry == 0 ? ep.q16 + ((uint64_t)tok * ep.n_q_heads + head) * D
                                 : ep.k_cache + ((uint64_t)head * ep.max_ctx + ep.pos + tok) * D;
            }
            if (ok) {
                *(f16x8_t*)(dst + k8) = y0v;
                *(f16x8_t*)(dst + HALF + k8) = y1v;
            }
        }
        return;
    }
    // rows 32 i + 8 v + 4 h + [0, 4) of the tile in acc[i][4 v ..]; every residual of a
    // subtile is asked for before the first store
    const uint32_t oc = n0 + col;
    if (oc >= n) return;
#pragma unroll
    for (int i = 0; i < TM; i++) {
        uint64_t o[16];
        float rv[16];
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const uint32_t lr = 32 * i + 8 * (e / 4) + 4 * h + e % 4;
            const uint32_t orow = GRP ? s_orow[lr] : min(m0 + lr, m - 1);
            o[e] = (uint64_t)orow * n + oc;
            rv[e] = 0.0f;
        }
        if (res) {  // uniform
#pragma unroll
            for (int e = 0; e < 16; e++) rv[e] = res[o[e]];
        }
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const uint32_t lr = 32 * i + 8 * (e / 4) + 4 * h + e % 4;
            const float v = __builtin_ldexpf(acc[i][e], s_sh[lr]);
            if (m0 + lr < m) out[o[e]] = res ? rv[e] + v : v;
        }
    }
}

// Any shape or alignment: one thread per output in the reference's serial order
// with every product and sum rounded on its own (bit-identical to dotRow).
__global__ __launch_bounds__(kMmThreads) void matmul_generic_kernel(const float* __restrict__ x, const uint8_t* __restrict__ w,
                                                                    uint32_t q8, float* out, const float* res, uint32_t m,
                                                                    uint32_t n, uint32_t k) {
#pragma clang fp contract(off)
    const uint64_t i = (uint64_t)blockIdx.x * kMmThreads + threadIdx.x;
    if (i >= (uint64_t)m * n) return;
    const uint64_t mi = i / n, ni = i % n;
    const float* xr = x + mi * k;
    float acc = 0.0f;
    if (q8) {
        const uint8_t* row = w + ni * ((uint64_t)k / 32 * kQ8Bytes);
        for (uint32_t b = 0; b < k / 32; b++) {
            const uint8_t* blk = row + (uint64_t)b * kQ8Bytes;
            const float scale = f16_bits_to_f32((uint32_t)blk[0] | ((uint32_t)blk[1] << 8));
            for (int e = 0; e < 32; e++) acc += (scale * (float)(int8_t)blk[2 + e]) * xr[32 * b + e];
        }
    } else {
        const float* row = (const float*)w + ni * k;
        for (uint32_t e = 0; e < k; e++) acc += row[e] * xr[e];
    }
    out[i] = res ? res[i] + acc : acc;
}

// out = x + y elementwise (kernels_a.zig:223-233): out may be x or y. Views that
// are not all 4-byte aligned go through byte copies.
__global__ __launch_bounds__(kMmThreads) void add_kernel(const uint8_t* x, const uint8_t* y, uint8_t* out, uint64_t n,
                                                         uint32_t aligned) {
    const uint64_t i = (uint64_t)blockIdx.x * kMmThreads + threadIdx.x;
    if (i >= n) return;
    if (aligned) {
        ((float*)out)[i] = ((const float*)x)[i] + ((const float*)y)[i];
    } else {
        float a, b;
        __builtin_memcpy(&a, x + 4 * i, 4);
        __builtin_memcpy(&b, y + 4 * i, 4);
        const float c = a + b;
        __builtin_memcpy(out + 4 * i, &c, 4);
    }
}

template <int MT, int JB, bool Q8, bool NORM>
int launch_rows(ds5_hip_ctx* ctx, const MatmulGroupLaunch& a, uint32_t m0) {
    constexpr uint32_t kRowsPerBlock = kMmThreads / 64;
    WeightGroup g{};
    uint32_t wgs = 0;
    for (uint32_t e = 0; e < a.count; e++) {
        g.w[g.count] = a.w[e];
        g.out[g.count] = a.out[e];
        g.res[g.count] = a.res[e];
        g.n[g.count] = a.n[e];
        g.wg0[g.count] = wgs;
        wgs += (a.n[e] + kRowsPerBlock - 1) / kRowsPerBlock;
        g.count += a.n[e] ? 1 : 0;  // entries without rows are dropped
    }
    if (wgs == 0) return DS5_OK;
    DS5_TIMED_LAUNCH(ctx, "matmul_rows_kernel", (matmul_rows_kernel<MT, JB, Q8, NORM>), dim3(wgs), dim3(kMmThreads), 0,
                     ctx->stream, a.x, g, a.m, a.k, m0, a.norm_w, a.norm_eps);
    return ds5_after_launch(ctx, "matmul_rows_kernel");
}


// Tokens per pass: up to 4 / JB (the x registers hold MT * JB * 32 floats per lane),
// and no more than the tokens there are (a 1-token decode runs MT = 1).
template <int JB, bool Q8, bool NORM>
int launch_passes(ds5_hip_ctx* ctx, const MatmulGroupLaunch& a) {
    constexpr uint32_t kMaxMt = 4 / JB;
    const uint32_t mt = a.m >= kMaxMt ? kMaxMt : (a.m >= 2 ? 2 : 1);
    for (uint32_t m0 = 0; m0 < a.m; m0 += mt) {
        int rc;
        if (mt == 4)
            rc = launch_rows<(kMaxMt >= 4 ? 4 : 1), JB, Q8, NORM>(ctx, a, m0);
        else if (mt == 2)
            rc = launch_rows<(kMaxMt >= 2 ? 2 : 1), JB, Q8, NORM>(ctx, a, m0);
        else
            rc = launch_rows<1, JB, Q8, NORM>(ctx, a, m0);
        if (rc) return rc;
    }
    return DS5_OK;
}

template <bool Q8, bool NORM>
int launch_rows_n(ds5_hip_ctx* ctx, const MatmulGroupLaunch& a) {
    const uint32_t nb = a.k / 32;
    if (nb <= 64) return launch_passes<1, Q8, NORM>(ctx, a);
    if (nb <= 128) return launch_passes<2, Q8, NORM>(ctx, a);
    return launch_passes<4, Q8, NORM>(ctx, a);
}

template <bool Q8>
int launch_rows_q(ds5_hip_ctx* ctx, const MatmulGroupLaunch& a) {
    return a.norm_w ? launch_rows_n<Q8, true>(ctx, a) : launch_rows_n<Q8, false>(ctx, a);
}

// Row tiles of a launch: 8 or more are padded to a multiple of 8 (the kernel's XCD order).
static uint32_t gemm_row_tiles(uint32_t m, uint32_t bm) {
    const uint32_t t = (m + bm - 1) / bm;
    return t >= 8 ? (t + 7) / 8 * 8 : t;
}

// 64-row tiles while those fill the CUs at most about once: a tile of twice the rows then
// only takes longer (m 100, n 2048, k 4096: 50 against 70 us; m 128, n 4096, k 2048: 26
// against 38; m 203, n 9216, k 4096, 288 tiles: 72 against 75). Above, 128 rows convert each
// weight half as often (m 500, n 5120, k 2048, 320 tiles: 42 against 46; 2048 tokens: 133
// against 162).
static bool gemm_half_tiles(const ds5_hip_ctx* ctx, uint32_t m, uint32_t cols) {
    const uint64_t cu = ctx->cu_count > 0 ? ctx->cu_count : 256;
    return ((uint64_t)m + 63) / 64 * cols <= cu + cu / 8;
}

// Split products: 32 columns a workgroup while tiles of 128 would fill half of the CUs (us,
// 32 / 128 columns, k 2048 and 4096: 64 such tiles, m 64, n 4096, 17 / 22 and 27 / 37; 128,
// m 128, n 4096, 25 / 25 and 42 / 42; 144, m 33, n 9216, 27 / 23 and 50 / 39): above, x is
// read four times as often and nothing is left idle.
static bool gemm_narrow_tiles(const ds5_hip_ctx* ctx, uint32_t m, uint32_t cols) {
    const uint64_t cu = ctx->cu_count > 0 ? ctx->cu_count : 256;
    return ((uint64_t)m + 31) / 32 * cols <= cu / 2;
}

// The split x: made once, shared by a group's products.
struct XPlanes {
    uint16_t *hi, *lo;
    int* row_exp;
};
XPlanes x_planes(void* ws, uint32_t m, uint32_t k) {
    uint16_t* hi = (uint16_t*)ws;
    return XPlanes{hi, hi + (size_t)m * k, (int*)(hi + 2 * (size_t)m * k)};
}

template <int TM, int W, int KS>
int launch_gemm(ds5_hip_ctx* ctx, const MatmulGroupLaunch& a, const XPlanes& xp) {
    WeightGroup g{};
    uint32_t tiles = 0;
    for (uint32_t e = 0; e < a.count; e++) {
        g.w[g.count] = a.w[e];
        g.out[g.count] = a.out[e];
        g.res[g.count] = a.res[e];
        g.n[g.count] = a.n[e];
        g.wg0[g.count] = tiles;
        tiles += (a.n[e] + 32 * W - 1) / (32 * W);
        g.count += a.n[e] ? 1 : 0;  // entries without rows are dropped
    }
    if (tiles == 0) return DS5_OK;
    DS5_TIMED_LAUNCH(ctx, "matmul_q8_mfma_kernel", (matmul_q8_mfma_kernel<TM, W, KS, 0>),
                     dim3(tiles, gemm_row_tiles(a.m, 32 * TM)), dim3(64 * W * KS), 0, ctx->stream, xp.hi, xp.lo, xp.row_exp,
                     g, a.m, a.k, AttnPrepEpi{}, MoeGemmTiles{});
    return ds5_after_launch(ctx, "matmul_q8_mfma_kernel");
}

}  // namespace

// The MoE experts' matrix-core path (rows sorted by expert): the tokens' x rows split,
// the grouped products (sorted rows gather their token's plane row), h = silu(g) * u
// split.
int launch_x_split_rows(ds5_hip_ctx* ctx, const float* x, uint32_t rows, uint32_t k, uint16_t* hi, uint16_t* lo,
                        int* row_exp) {
    if (rows == 0) return DS5_OK;
    DS5_TIMED_LAUNCH(ctx, "matmul_x_split_kernel", matmul_x_split_kernel<false>, dim3(rows), dim3(kSplitThreads), 0,
                     ctx->stream, x, hi, lo, row_exp, k, XSplitRope{}, RopeTable{}, nullptr, 0.0f);
    return ds5_after_launch(ctx, "matmul_x_split_kernel");
}

int launch_moe_h_split(ds5_hip_ctx* ctx, const float* g, const float* u, uint32_t rows, uint32_t k, uint16_t* hi,
                       uint16_t* lo, int* row_exp) {
    if (rows == 0) return DS5_OK;
    const dim3 g4((rows + 3) / 4);
    if (k <= 1024)
        DS5_TIMED_LAUNCH(ctx, "moe_h_split_kernel", moe_h_split_rows_kernel<4>, g4, dim3(256), 0, ctx->stream, g, u, hi,
                         lo, row_exp, k, rows);
    else if (k <= 2048)
        DS5_TIMED_LAUNCH(ctx, "moe_h_split_kernel", moe_h_split_rows_kernel<8>, g4, dim3(256), 0, ctx->stream, g, u, hi,
                         lo, row_exp, k, rows);
    else
        DS5_TIMED_LAUNCH(ctx, "moe_h_split_kernel", moe_h_split_kernel, dim3(rows), dim3(kSplitThreads), 0, ctx->stream,
                         g, u, hi, lo, row_exp, k);
    return ds5_after_launch(ctx, "moe_h_split_kernel");
}

template <int TM, int W, int KS>
static int launch_q8_gemm_grouped_t(ds5_hip_ctx* ctx, const uint16_t* hi, const uint16_t* lo, const int* row_exp,
                                    uint32_t k, const uint8_t* const* w, float* const* out, const uint32_t* n,
                                    uint32_t count, uint32_t max_tiles, const MoeGemmTiles& mt) {
    WeightGroup g{};
    uint32_t nt = 0;
    for (uint32_t e = 0; e < count; e++) {
        g.w[e] = w[e];
        g.out[e] = out[e];
        g.n[e] = n[e];
        g.wg0[e] = nt;
        nt += (n[e] + 32 * W - 1) / (32 * W);
    }
    g.count = count;
    if (nt == 0 || max_tiles == 0) return DS5_OK;
    DS5_TIMED_LAUNCH(ctx, "matmul_q8_mfma_kernel", (matmul_q8_mfma_kernel<TM, W, KS, 0, true>),
                     dim3(nt, gemm_row_tiles(max_tiles, 1)), dim3(64 * W * KS), 0, ctx->stream, hi, lo, row_exp, g, 0u, k,
                     AttnPrepEpi{}, mt);
    return ds5_after_launch(ctx, "matmul_q8_mfma_kernel");
}

int launch_q8_gemm_grouped(ds5_hip_ctx* ctx, const uint16_t* hi, const uint16_t* lo, const int* row_exp, uint32_t k,
                           const uint8_t* const* w, float* const* out, const uint32_t* n, uint32_t count,
                           const uint4* tiles, const uint32_t* n_tiles, uint32_t max_tiles, uint32_t tile_rows,
                           uint64_t w_stride, const uint32_t* x_rows, const uint32_t* out_rows) {
    const MoeGemmTiles mt{tiles, n_tiles, w_stride, x_rows, out_rows};
    if (tile_rows == 32)
        return launch_q8_gemm_grouped_t<1, 4, 1>(ctx, hi, lo, row_exp, k, w, out, n, count, max_tiles, mt);
    if (tile_rows == 64)
        return launch_q8_gemm_grouped_t<2, 4, 1>(ctx, hi, lo, row_exp, k, w, out, n, count, max_tiles, mt);
    if (tile_rows == 128)
        return launch_q8_gemm_grouped_t<4, 4, 1>(ctx, hi, lo, row_exp, k, w, out, n, count, max_tiles, mt);
    return ds5_fail(ctx, DS5_DEVICE_FAILURE, "moe: row tiles of %u rows", tile_rows);
}

// The rope table follows the x split at the next 16-byte boundary (the epilogue
// reads it in float4s).
static size_t qkv_prep_cs_offset(uint32_t m, uint32_t k) { return (x_split_bytes(m, k) + 15) & ~(size_t)15; }

size_t qkv_prep_workspace_bytes(uint32_t m, uint32_t k, uint32_t head_dim) {
    return qkv_prep_cs_offset(m, k) + (size_t)m * head_dim * sizeof(float);
}

int launch_qkv_prep(ds5_hip_ctx* ctx, const QkvPrepLaunch& a) {
    const XPlanes xp = x_planes(a.ws, a.m, a.k);
    float* cs = (float*)((char*)a.ws + qkv_prep_cs_offset(a.m, a.k));
    XSplitRope rope{a.positions, cs, a.head_dim / 2, a.freq_scale};
    DS5_TIMED_LAUNCH(ctx, "matmul_x_split_kernel", matmul_x_split_kernel<true>, dim3(a.m), dim3(kSplitThreads), 0,
                     ctx->stream, a.x, xp.hi, xp.lo, xp.row_exp, a.k, rope, *a.table, a.norm_w, a.norm_eps);
    if (int rc = ds5_after_launch(ctx, "matmul_x_split_kernel")) return rc;
    const uint32_t ns[3] = {a.n_q_heads * a.head_dim, a.n_kv_heads * a.head_dim, a.n_kv_heads * a.head_dim};
    const uint8_t* ws[3] = {a.wq, a.wk, a.wv};
    AttnPrepEpi ep{a.q_norm, a.k_norm, cs, a.q16, a.k_cache, a.v_cache, a.pos, a.n_q_heads, a.max_ctx, a.eps, a.q_scale};
    // one launch, or two where the weights' sizes put some on the split form and some not
    for (int split = 0; split < 2; split++) {
        WeightGroup g{};
        uint32_t tiles = 0;
        for (int e = 0; e < 3; e++) {  // all three keep their places: the epilogue goes by them
            g.w[e] = ws[e];
            g.n[e] = ns[e];
            g.wg0[e] = tiles;
            if (a.split[e] == (split != 0)) tiles += ns[e] / kGemmCols;
        }
        g.count = 3;
        if (tiles == 0) continue;
        auto launch = [&](auto tm, auto ks) {
            constexpr int TM = decltype(tm)::value, KS = decltype(ks)::value;
            DS5_TIMED_LAUNCH(ctx, "matmul_q8_mfma_kernel", (matmul_q8_mfma_kernel<TM, 4, KS, 1>),
                             dim3(tiles, gemm_row_tiles(a.m, 32 * TM)), dim3(256 * KS), 0, ctx->stream, xp.hi, xp.lo,
                             xp.row_exp, g, a.m, a.k, ep, MoeGemmTiles{});
        };
        using std::integral_constant;
        if (split) launch(integral_constant<int, 1>{}, integral_constant<int, 4>{});
        else if (gemm_half_tiles(ctx, a.m, tiles)) launch(integral_constant<int, 2>{}, integral_constant<int, 1>{});
        else launch(integral_constant<int, 4>{}, integral_constant<int, 1>{});
        if (int rc = ds5_after_launch(ctx, "matmul_q8_mfma_kernel")) return rc;
    }
    return DS5_OK;
}

// Tokens from which Q8_0 products run on the matrix cores (below, the row
// kernel's passes of up to 4 tokens re-read the weights less often than the
// GEMM wastes matrix-core work)
constexpr uint32_t kGemmMinM = 16;

// The row kernel needs x and out 16-byte aligned, k <= 8192, and f32 weights 16-byte
// aligned or Q8_0 weights 4-byte aligned. A Q8_0 block is read as the nine dwords
// from the dword boundary at or below it, which ends 2 bytes past the block when
// the block starts on a dword boundary; for the last block that stays inside the
// view only if the weights end on a dword boundary or the view has 2 more bytes.
// The GEMM reads x as float4 (x 16-byte aligned), stores single floats (out
// 4-byte aligned) and reads q as 16-byte loads of dwords 0..3, 4..7 and 5..8 of the same
// nine, with the same end condition. Its loads address an x plane and the
// weights with 32-bit byte offsets from a scalar base.
static bool gemm_offsets_fit(uint32_t m, uint32_t k, uint64_t w_end) {
    return (uint64_t)m * k * 2 < (1ull << 32) && w_end + 2 < (1ull << 32);
}

// Up to 128 tokens, four groups of wavefronts split a tile's blocks while the 32 x 128 tiles
// (one such workgroup fits a CU) are at most as many as the 256 CUs: unsplit, most CUs have
// no tile and the others wait for one block after the other. us, split and unsplit:
//   k 2048:  n 2048, m 32 (16 tiles) 14 and 29;  n 8192, m 128 (256) 29 and 32, m 129 (320)
//            43 and 32;  n 16384, m 64 (256) 29 and 33, m 65 (384) 45 and 34;  n 30011, m 32
//            (235) 30 and 34, m 33 (470) 49 and 34
//   k 4096:  n 9216, m 96 (216) 44 and 57, m 128 (288) 79 and 57;  n 16384, m 65 (384) 76 and 59
// Few blocks leave little to split: half as many tiles (k 96: n 300, m 64 (6) 8.4 and 9.5,
// n 4096, m 128 (128) 9.2 and 9.8, n 9216, m 64 (144) 9.9 and 10.0, n 12288, m 64 (192) 10.2
// and 10.2, n 30011, m 32 (235), k 256 12.1 and 11.3). Chosen from the product's own shape:
// in a group or in the attention block it adds in the same order.
static bool gemm_split(uint32_t m, uint32_t n, uint32_t k) {
    return m <= 128 && ((uint64_t)m + 31) / 32 * (((uint64_t)n + kGemmCols - 1) / kGemmCols) <= (k > 256 ? 256 : 128);
}

MatmulPath matmul_path(const MatmulLaunch& a, uint64_t w_len) {
    const uintptr_t x_addr = (uintptr_t)a.x, out_addr = (uintptr_t)a.out, w_addr = (uintptr_t)a.w;
    if (a.k % 32 != 0 || (x_addr & 15u)) return MatmulPath::Generic;
    if (!a.q8) return (a.k / 32 <= 256 && (out_addr & 15u) == 0 && (w_addr & 15u) == 0) ? MatmulPath::Rows
                                                                                         : MatmulPath::Generic;
    const uint64_t end = (uint64_t)a.n * (a.k / 32) * kQ8Bytes;
    if ((w_addr & 3u) || !((w_addr + end) % 4 == 0 || w_len >= end + 2)) return MatmulPath::Generic;
    const bool gemm = (out_addr & 3u) == 0 && gemm_offsets_fit(a.m, a.k, end);
    const MatmulPath gemm_path = gemm_split(a.m, a.n, a.k) ? MatmulPath::GemmSplit : MatmulPath::Gemm;
    if (a.m >= kGemmMinM && gemm) return gemm_path;
    if (a.k / 32 <= 256 && (out_addr & 15u) == 0) return MatmulPath::Rows;
    return gemm ? gemm_path : MatmulPath::Generic;
}

static int launch_generic(ds5_hip_ctx* ctx, const float* x, const uint8_t* w, bool q8, float* out, const float* res,
                          uint32_t m, uint32_t n, uint32_t k) {
    const uint64_t total = (uint64_t)m * n;
    const dim3 grid((unsigned)((total + kMmThreads - 1) / kMmThreads));
    DS5_TIMED_LAUNCH(ctx, "matmul_generic_kernel", matmul_generic_kernel, grid, dim3(kMmThreads), 0, ctx->stream, x, w,
                     (uint32_t)q8, out, res, m, n, k);
    return ds5_after_launch(ctx, "matmul_generic_kernel");
}

// The part of a group that takes `path`.
static MatmulGroupLaunch group_part(const MatmulGroupLaunch& a, const MatmulPath* paths, MatmulPath path) {
    MatmulGroupLaunch p = a;
    p.count = 0;
    for (uint32_t e = 0; e < a.count; e++)
        if (paths[e] == path) {
            p.w[p.count] = a.w[e];
            p.out[p.count] = a.out[e];
            p.res[p.count] = a.res[e];
            p.n[p.count++] = a.n[e];
        }
    return p;
}

// A group on the matrix cores: x split once, then a launch for the split products and one
// for the others.
static int launch_gemms(ds5_hip_ctx* ctx, const MatmulGroupLaunch& a, const MatmulPath* paths) {
    void* ws = nullptr;
    if (int rc = ds5_workspace(ctx, x_split_bytes(a.m, a.k), &ws)) return rc;
    const XPlanes xp = x_planes(ws, a.m, a.k);
    DS5_TIMED_LAUNCH(ctx, "matmul_x_split_kernel", matmul_x_split_kernel<false>, dim3(a.m), dim3(kSplitThreads), 0,
                     ctx->stream, a.x, xp.hi, xp.lo, xp.row_exp, a.k, XSplitRope{}, RopeTable{}, a.norm_w, a.norm_eps);
    if (int rc = ds5_after_launch(ctx, "matmul_x_split_kernel")) return rc;
    for (MatmulPath path : {MatmulPath::Gemm, MatmulPath::GemmSplit}) {
        const MatmulGroupLaunch p = group_part(a, paths, path);
        uint32_t cols = 0;
        for (uint32_t e = 0; e < p.count; e++) cols += (p.n[e] + kGemmCols - 1) / kGemmCols;
        if (cols == 0) continue;
        int rc;
        if (path == MatmulPath::Gemm)
            rc = gemm_half_tiles(ctx, a.m, cols) ? launch_gemm<2, 4, 1>(ctx, p, xp) : launch_gemm<4, 4, 1>(ctx, p, xp);
        else
            rc = gemm_narrow_tiles(ctx, a.m, cols) ? launch_gemm<1, 1, 4>(ctx, p, xp) : launch_gemm<1, 4, 4>(ctx, p, xp);
        if (rc) return rc;
    }
    return DS5_OK;
}

static int launch_same_path(ds5_hip_ctx* ctx, const MatmulGroupLaunch& a, MatmulPath path) {
    if (a.norm_w && (path == MatmulPath::Generic || a.k <= kRmsSerialMaxDim))
        return ds5_fail(ctx, DS5_DEVICE_FAILURE, "matmul: an in-kernel norm needs the row or GEMM path and k > %u",
                        kRmsSerialMaxDim);
    if (path == MatmulPath::Rows) return a.q8 ? launch_rows_q<true>(ctx, a) : launch_rows_q<false>(ctx, a);
    if (is_gemm(path)) {
        const MatmulPath paths[kMatmulGroupMax] = {path, path, path, path};
        return launch_gemms(ctx, a, paths);
    }
    for (uint32_t e = 0; e < a.count; e++)
        if (a.n[e])
            if (int rc = launch_generic(ctx, a.x, a.w[e], a.q8, a.out[e], a.res[e], a.m, a.n[e], a.k)) return rc;
    return DS5_OK;
}

int launch_matmul(ds5_hip_ctx* ctx, const MatmulLaunch& a, MatmulPath path) {
    MatmulGroupLaunch g{};
    g.x = a.x;
    g.q8 = a.q8;
    g.m = a.m;
    g.k = a.k;
    g.count = 1;
    g.w[0] = a.w;
    g.out[0] = a.out;
    g.res[0] = a.res;
    g.n[0] = a.n;
    return launch_matmul_group(ctx, g, &path);
}

int launch_add(ds5_hip_ctx* ctx, const void* x, const void* y, void* out, uint64_t n) {
    if (n == 0) return DS5_OK;
    const uint32_t aligned = (((uintptr_t)x | (uintptr_t)y | (uintptr_t)out) & 3u) == 0;
    const dim3 grid((unsigned)((n + kMmThreads - 1) / kMmThreads));
    DS5_TIMED_LAUNCH(ctx, "add_kernel", add_kernel, grid, dim3(kMmThreads), 0, ctx->stream, (const uint8_t*)x,
                     (const uint8_t*)y, (uint8_t*)out, n, aligned);
    return ds5_after_launch(ctx, "add_kernel");
}

// One launch for the whole group when every entry takes the same kernel (the matrix cores'
// two forms: one x split, a launch each); otherwise each entry on its own kernel, in order.
int launch_matmul_group(ds5_hip_ctx* ctx, const MatmulGroupLaunch& a, const MatmulPath* paths) {
    if (a.m == 0 || a.count == 0) return DS5_OK;
    bool same = true, gemm = true;
    for (uint32_t e = 0; e < a.count; e++) {
        same = same && paths[e] == paths[0];
        gemm = gemm && is_gemm(paths[e]);
    }
    if (same) return launch_same_path(ctx, a, paths[0]);
    if (a.norm_w && !(gemm && a.k > kRmsSerialMaxDim))
        return ds5_fail(ctx, DS5_DEVICE_FAILURE, "matmul: an in-kernel norm needs one kernel for the group and k > %u",
                        kRmsSerialMaxDim);
    if (gemm) return launch_gemms(ctx, a, paths);
    for (uint32_t e = 0; e < a.count; e++) {
        MatmulGroupLaunch one{};
        one.x = a.x;
        one.q8 = a.q8;
        one.m = a.m;
        one.k = a.k;
        one.count = 1;
        one.w[0] = a.w[e];
        one.out[0] = a.out[e];
        one.res[0] = a.res[e];
        one.n[0] = a.n[e];
        if (int rc = launch_same_path(ctx, one, paths[e])) return rc;
    }
    return DS5_OK;
}
