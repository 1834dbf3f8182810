// softmax(q k^T * scale) v for heads of 64 or 128 on the matrix cores, with the
// attention epilogue's head merge and per-head gate in the same pass
// (standalone/ltx_nn.py:22-26,227-235):
//
//   o[b, t, h, :]   = round_bf16(sum_j p_j v_j / sum_j p_j),  p_j = exp(scale q.k_j - m)
//   out[b, t, h, :] = round_bf16(o * 2*sigmoid(logit[b, t, h]))   (o itself without logits)
//
// q, k, v and out are token-major (batch, tokens, heads*D), as the projections
// make them.  Scores, running maximum, sums and output are fp32; p is rounded to
// bf16 for the second product.
//
// What bounds it: the card's power.  On 6144 x 6144 tokens, 32 heads of 128, it
// runs at 1.01-1.08 PFLOP/s (573-612 us from card to card) and the same launch on zeros,
// which switch nothing, at 1.63-1.66; torch's flash kernel 0.69 (865-916 us) on
// the same inputs.  So the split is taken for the least work beside the products:
// * Four waves of 32 queries share a 64-key tile in LDS (two workgroups a CU).
//   64 queries a wave (half the LDS reads, one wave a SIMD) 700-836 us; eight
//   waves sharing a tile 570-600 us here but 372-396 against 338-352 us on 4290
//   tokens, whose query tiles then fill the chip worse.
// * The scores are computed transposed (keys by queries): a lane then holds the
//   scores of one query, its maximum and sum need one exchange with lane ^ 32,
//   and its weights are already the second product's operand.
// * V is read from LDS by transposing reads, so neither operand is rearranged.
// * The second product of a tile and the scores of the next run as one stream,
//   LDS fragments four ahead: 592-602 us with the products apart.  The loads of the
//   next tile go between the products: 612 against 623 us (one card) with all of
//   them ahead of the stream, and without any loads (a timing copy) 11 % less.
// * The running maximum is exact in every tile.  Letting it lag up to 2^8 saves
//   2-4 %, but then a row's largest weight is no longer exactly 1 and its
//   rounding shows: relative error 2.26e-3 against 1.87e-3 (torch's 1.87e-3).
#include "ltxk_common.h"

#include <cfloat>
#include <type_traits>

namespace ltxk {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWaves = 4;
constexpr int kRows = 32 * kWaves;  // queries a workgroup, 32 a wave
constexpr int kKeys = 64;           // keys a tile
constexpr float kLarge = 4096.f;    // scaled scores whose products' rounding the weights may show

struct FlashParams {
    const uint16_t *q, *k, *v, *logits;
    uint16_t *out;
    float *part;            // split query tiles: each unit's weighted sums of v (128 x D)
    float2 *stats;          // and each of its rows' maximum and sum of weights (128)
    int64_t qbs, kbs, vbs;  // batch strides, elements
    uint32_t qts, kts, vts; // token strides, bytes
    int tq, tk, heads, q_tiles, tiles;
    int bh;                 // batch * heads
    int whole;              // query tiles of an XCD that one workgroup takes alone
    int rest, parts;        // the others, each cut into `parts` units over the keys
    float scale2;           // scale * log2(e)
};

// Query tile t of XCD x: all query tiles of a head go to one XCD, whose L2 then
// holds that head's keys and values (workgroups are dealt to the XCDs in turn).
__device__ __forceinline__ bool query_tile(const FlashParams &p, int xcd, int t, int &b, int &head, int &first)
{
    const int bh = t / p.q_tiles * 8 + xcd;
    b = bh / p.heads;
    head = bh % p.heads;
    first = t % p.q_tiles * kRows;
    return bh < p.bh;
}

// LDS position of 16-byte chunk c of a tile's row.  A row is D/8 chunks with no
// padding (the loads write LDS in lane order), so the chunks of a row are
// permuted instead.  K is read 16 bytes a lane down 16 rows of one chunk column,
// V as 4 rows x 64 bytes (a transposed read's four keys): with these
// permutations each such group covers 256 bytes of distinct banks.
template <int D>
__device__ __forceinline__ int k_pos(int row, int c)
{
    return D == 128 ? c ^ (row & 15) : c ^ ((row >> 1) & 7);
}
template <int D>
__device__ __forceinline__ int v_pos(int row, int c)
{
    return D == 128 ? c ^ (((row & 3) << 2) | ((row >> 2) & 3)) : c ^ ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
}

typedef __attribute__((address_space(3))) char lds_char;

// Part j of a wave's share of a 64-row tile: one load instruction moves 64 lanes
// x 16 bytes straight into LDS.  Rows past the last key repeat it (their scores
// are masked), so nothing outside the tensor is read.
template <int D>
constexpr int kLoads = kKeys * D * 2 / 1024 / kWaves;  // load instructions of a wave for a tile

template <int D, bool V>
__device__ __forceinline__ void load_part(rsrc_t r, char *lds, int j, int first_row, int last_row, uint32_t stride,
                                          int wave, int lane)
{
    const int at = wave * kLoads<D> + j;
    const int row = at * (1024 / (2 * D)) + lane / (D / 8);
    const int pos = lane % (D / 8);
    const int c = V ? v_pos<D>(row, pos) : k_pos<D>(row, pos);  // the permutations are involutions
    const uint32_t off = static_cast<uint32_t>(min(first_row + row, last_row)) * stride + c * 16;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_char *)(lds + at * 1024), 16, off, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 cat(bf16x4 a, bf16x4 b)
{
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

// The larger (sum) of a value over lanes l and l ^ 32, in both.
__device__ __forceinline__ float pair_max(float v)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float v)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The gate 2*sigmoid(logit), and a gated output: the output rounds to bf16 first,
// as the tensor that the gate multiplies does.
__device__ __forceinline__ float head_gate(uint16_t logit) { return 2.0f / (1.0f + expf(-bf16_to_f32(logit))); }
__device__ __forceinline__ float gated(float o, float gate) { return bf16_to_f32(f32_to_bf16(o)) * gate; }

// This wave's loads have landed and its LDS reads returned, then all waves'.
__device__ __forceinline__ void tile_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int D>
__global__ void __launch_bounds__(kWaves * 64, 2) flash_kernel(FlashParams p)
{
    constexpr int KS = D / 16;               // contraction steps of the scores
    constexpr int MT = D / 32;               // output tiles
    constexpr int NK = 2 * KS, NV = 4 * MT;  // K and V fragments of a tile
    constexpr int kAhead = 4;                // fragments read ahead of the products
    constexpr int kTileBytes = kKeys * D * 2;
    __shared__ __attribute__((aligned(1024))) char k0[kTileBytes];
    __shared__ __attribute__((aligned(1024))) char k1[kTileBytes];
    __shared__ __attribute__((aligned(1024))) char v0[kTileBytes];
    __shared__ __attribute__((aligned(1024))) char v1[kTileBytes];

    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    const bool split = j >= p.whole;
    const int unit = j - p.whole, part = split ? unit % p.parts : 0;
    int b, head, first;
    if (!query_tile(p, xcd, split ? p.whole + unit / p.parts : j, b, head, first)) return;
    const int t0 = split ? part * p.tiles / p.parts : 0;
    const int t1 = split ? (part + 1) * p.tiles / p.parts : p.tiles;
    const int n = t1 - t0;  // at least one tile: the host takes no more parts than tiles
    const int last = p.tk - 1;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l32 = lane & 31, half = lane >> 5;
    const rsrc_t kr = make_rsrc(p.k + b * p.kbs + head * D, static_cast<uint32_t>(last) * p.kts + 2 * D);
    const rsrc_t vr = make_rsrc(p.v + b * p.vbs + head * D, static_cast<uint32_t>(last) * p.vts + 2 * D);

    auto load_k = [&](int i, int part, char *dst) {
        load_part<D, false>(kr, dst, part, (t0 + i) * kKeys, last, p.kts, wave, lane);
    };
    auto load_v = [&](int i, int part, char *dst) {
        load_part<D, true>(vr, dst, part, (t0 + i) * kKeys, last, p.vts, wave, lane);
    };
#pragma unroll
    for (int c = 0; c < kLoads<D>; ++c) load_k(0, c, k0);

    // Queries: lane l holds query l % 32, elements 16 s + 8 (l/32) .. + 7.
    const int row = first + wave * 32 + l32;
    bf16x8 qf[KS];
    {
        const char *qp = reinterpret_cast<const char *>(p.q + b * p.qbs + head * D) +
                         static_cast<int64_t>(min(row, p.tq - 1)) * p.qts + half * 16;
#pragma unroll
        for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const bf16x8 *>(qp + s * 32);
    }

    // LDS byte offsets of this lane's fragments.  K: row l % 32 (+ 32 u), chunk
    // 2 s + half.  V (transposed reads of 4 keys x 16 columns by 16 lanes): rows
    // 16 s + 8 e + 4 half + (l%16)/4, columns 32 m + 16 (l/16 % 2) + 4 (l % 4).
    int k_off[KS], v_off[MT][2];
#pragma unroll
    for (int s = 0; s < KS; ++s) k_off[s] = l32 * 2 * D + k_pos<D>(l32, 2 * s + half) * 16;
    const int vi = lane & 15;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int r = 8 * e + 4 * half + (vi >> 2);
            const int c = 4 * m + 2 * ((lane >> 4) & 1) + ((vi & 3) >> 1);
            v_off[m][e] = r * 2 * D + v_pos<D>(r, c) * 16 + (vi & 1) * 8;
        }

    f32x16 o[MT] = {};
    f32x16 s[2];     // scores, transposed: register r of s[u] is key 32 u + 8 (r/4) + 4 half + r % 4 of query l % 32
    u32x4 w[4];      // weights, two a register, in the order of the scores
    float mx = 0.f;  // running maximum of the scaled scores (the same in lanes l and l ^ 32)
    float sum = 0.f; // this lane's share of the weights' sum

    // Fragment i of a K tile (contraction step i / 2 of keys 32 (i%2) ..) and of a
    // V tile (keys 16 (i / MT) .., columns 32 (i % MT) ..).
    auto k_frag = [&](const char *kt, int i) {
        return *reinterpret_cast<const bf16x8 *>(kt + k_off[i >> 1] + (i & 1) * 64 * D);
    };
    auto v_frag = [&](const char *vt, int i) {
        typedef __attribute__((address_space(3))) bf16x4 lds4;
        const int m = i % MT, st = i / MT;
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4 *)(vt + v_off[m][0] + st * 32 * D));
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4 *)(vt + v_off[m][1] + st * 32 * D));
        return cat(lo, hi);
    };
    // Matrix phase: a run of the stream of products that a tile takes, the weights
    // times V of the tile before (0 .. NV - 1), then its scores (NV .. NV + NK - 1),
    // with the LDS fragments read ahead of them and `loads(j)` between them.
    auto products = [&](auto from, auto to, const char *vp, const char *kc, auto loads)
                        __attribute__((always_inline)) {
        bf16x8 f[NV + NK];
        auto frag = [&](int j) { f[j] = j < NV ? v_frag(vp, j) : k_frag(kc, j - NV); };
#pragma unroll
        for (int j = from; j < from + kAhead; ++j) frag(j);
#pragma unroll
        for (int j = from; j < to; ++j) {
            if (j + kAhead < to) frag(j + kAhead);
            loads(j - from);
            if (j < NV) {
                o[j % MT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[j], __builtin_bit_cast(bf16x8, w[j / MT]),
                                                                    o[j % MT], 0, 0, 0);
            } else {
                const int i = j - NV;
                s[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[j], qf[i >> 1], i < 2 ? f32x16{} : s[i & 1], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Vector phase of tile i: its maximum, the rescale of what was summed so far
    // if a row's maximum grew, its weights.
    auto softmax = [&](int i) __attribute__((always_inline)) {
        if (i == n - 1) {  // keys past the last get weight zero
            const int valid = p.tk - (t0 + i) * kKeys;
            if (valid < kKeys)
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (32 * u + 8 * (r >> 2) + 4 * half + (r & 3) >= valid) s[u][r] = -INFINITY;
        }
        float t[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            t[c] = s[c >> 1][8 * (c & 1)];
#pragma unroll
            for (int r = 1; r < 8; ++r) t[c] = fmaxf(t[c], s[c >> 1][8 * (c & 1) + r]);
        }
        const float m = pair_max(fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]))) * p.scale2;
        if (i == 0) {
            mx = fmaxf(m, -FLT_MAX);  // finite, so that scores of -inf weigh zero
        } else if (__any(m > mx)) {
            const float nm = fmaxf(m, mx);
            const float a = __builtin_amdgcn_exp2f(mx - nm);
            mx = nm;
            sum *= a;
#pragma unroll
            for (int c = 0; c < MT; ++c)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[c][r] *= a;
        }
        // The maximum is a rounded product and the scores' products below are exact, so
        // the largest weight is 2^(a rounding of the maximum) instead of 1: past kLarge
        // that would come to show in bf16 (and past 2^31 overflow), so there the scores
        // round first (0.5 % of the time at 6144 tokens for the test).
        float scale2 = p.scale2;
        if (__any(fabsf(mx) > kLarge)) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 16; ++r) s[u][r] *= scale2;
            scale2 = 1.f;
        }
        float part[2] = {};
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j >> 3][2 * (j & 7)], scale2, -mx));
            const float y = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j >> 3][2 * (j & 7) + 1], scale2, -mx));
            part[0] += x;
            part[1] += y;
            w[j >> 2][j & 3] = pack_bf16x2(x, y);
        }
        sum += part[0] + part[1];
    };

    // Tile i: kc holds its keys, vp the values of tile i - 1.  Its values and the
    // next tile's keys (the last tile's once more after the last) load into the
    // other buffers between the products.
    using std::integral_constant;
    auto tile = [&](int i, auto from, const char *kc, const char *vp, char *kn, char *vn)
                    __attribute__((always_inline)) {
        constexpr int kEvery = from == 0 ? 3 : 2;
        const int next = min(i + 1, n - 1);
        products(from, integral_constant<int, NV + NK>{}, vp, kc, [&](int j) __attribute__((always_inline)) {
            if (j % kEvery) return;
            const int c = j / kEvery;
            if (c < kLoads<D>)
                load_v(i, c, vn);
            else if (c < 2 * kLoads<D>)
                load_k(next, c - kLoads<D>, kn);
        });
        softmax(i);
        __builtin_amdgcn_sched_barrier(0);
        tile_barrier();
    };
    constexpr integral_constant<int, 0> whole;
    tile_barrier();
    tile(0, integral_constant<int, NV>{}, k0, v1, k1, v0);
    for (int i = 1; i < n; i += 2) {
        tile(i, whole, k1, v0, k0, v1);
        if (i + 1 < n) tile(i + 1, whole, k0, v1, k1, v0);
    }
    products(whole, integral_constant<int, NV>{}, n & 1 ? v0 : v1, nullptr, [](int) {});

    // Lane l: query l % 32, columns 32 m + 8 j + 4 half + (0..3) in registers 4 j ..
    const float total = pair_sum(sum);
    if (split) {
        const int64_t u = (static_cast<int64_t>(xcd) * p.rest * p.parts + unit) * kRows + wave * 32 + l32;
        if (half == 0) p.stats[u] = make_float2(mx, total);
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                *reinterpret_cast<f32x4 *>(p.part + u * D + 32 * t + 8 * c + 4 * half) =
                    f32x4{o[t][4 * c], o[t][4 * c + 1], o[t][4 * c + 2], o[t][4 * c + 3]};
        return;
    }
    const float inv = 1.f / total;
    if (row >= p.tq) return;
    const int64_t tok = (static_cast<int64_t>(b) * p.tq + row) * p.heads + head;
    const float gate = p.logits ? head_gate(p.logits[tok]) : 1.f;
    uint16_t *op = p.out + tok * D + 4 * half;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float f[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) f[r] = gated(o[t][4 * c + r] * inv, gate);
            *reinterpret_cast<uint2 *>(op + 32 * t + 8 * c) =
                make_uint2(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]));
        }
}

// Merges the units of the split query tiles: 8 columns of one query a thread.
template <int D>
__global__ void __launch_bounds__(256) flash_merge_kernel(FlashParams p)
{
    constexpr int kChunks = D / 8;
    const int i = (blockIdx.x >> 3) * 256 + threadIdx.x, xcd = blockIdx.x & 7;
    const int c = i % kChunks, r = i / kChunks % kRows, t = i / kChunks / kRows;
    int b, head, first;
    if (!query_tile(p, xcd, p.whole + t, b, head, first) || first + r >= p.tq) return;
    const int64_t u = (static_cast<int64_t>(xcd) * p.rest + t) * p.parts * kRows + r;
    float m = -INFINITY;
    for (int k = 0; k < p.parts; ++k) m = fmaxf(m, p.stats[u + k * kRows].x);
    float acc[8] = {}, sum = 0.f;
    for (int k = 0; k < p.parts; ++k) {
        const float2 st = p.stats[u + k * kRows];
        const float w = __builtin_amdgcn_exp2f(st.x - m);
        const f32x4 *x = reinterpret_cast<const f32x4 *>(p.part + (u + k * kRows) * D + c * 8);
        const f32x4 lo = x[0], hi = x[1];
        sum += w * st.y;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc[e] = __builtin_fmaf(w, lo[e], acc[e]);
            acc[4 + e] = __builtin_fmaf(w, hi[e], acc[4 + e]);
        }
    }
    const int64_t tok = (static_cast<int64_t>(b) * p.tq + first + r) * p.heads + head;
    const float gate = p.logits ? head_gate(p.logits[tok]) : 1.f, inv = 1.f / sum;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = gated(acc[e] * inv, gate);
    *reinterpret_cast<u32x4 *>(p.out + tok * D + c * 8) = pack8v(acc);
}

// How a launch is cut.  The chip runs 64 workgroups an XCD at a time, so an
// XCD's query tiles past the last multiple of 64 would leave most of it idle for
// a whole tile's time: their keys are dealt to as many units as fit beside each
// other, each of at least four key tiles; the units' outputs are merged in fp32.
// 126 queries over 6144 keys, 32 heads of 64: 27 us for one batch item and 43 for
// four, against 308 and 323 for torch's flash kernel and about 60 for it over
// eight chunks of keys and ltxk_attn_combine; 4290 x 4290, heads of 128: 319 us.
struct FlashCut {
    int64_t q_tiles, tiles, whole, rest, parts;
};

FlashCut cut(int64_t bh, int64_t tokens_q, int64_t tokens_k)
{
    FlashCut c;
    c.q_tiles = (tokens_q + kRows - 1) / kRows;
    c.tiles = (tokens_k + kKeys - 1) / kKeys;
    const int64_t all = (bh + 7) / 8 * c.q_tiles;
    c.rest = all % 64;
    c.parts = 1;
    while (c.parts < 16 && c.rest * c.parts * 2 <= 64 && c.tiles >= c.parts * 2 * 4) c.parts *= 2;
    if (c.parts == 1) c.rest = 0;
    c.whole = all - c.rest;
    return c;
}

template <int D>
void launch(const FlashParams &p, hipStream_t s)
{
    flash_kernel<D><<<8u * (p.whole + p.rest * p.parts), kWaves * 64, 0, s>>>(p);
    if (p.rest) flash_merge_kernel<D><<<8u * (p.rest * (kRows * D / 8) / 256), 256, 0, s>>>(p);
}

}  // namespace
}  // namespace ltxk

using namespace ltxk;

extern "C" int64_t ltxk_attention_workspace_bytes(int64_t batch, int64_t tokens_q, int64_t tokens_k, int64_t heads,
                                                  int64_t head_dim)
{
    if (batch <= 0 || tokens_q <= 0 || tokens_k <= 0 || heads <= 0 || head_dim <= 0) return 0;
    const FlashCut c = cut(batch * heads, tokens_q, tokens_k);
    return 8 * c.rest * c.parts * kRows * (head_dim + 2) * 4;
}

extern "C" int ltxk_attention(void *out, const void *q, int64_t q_bstride, int64_t q_tstride, const void *k,
                              int64_t k_bstride, int64_t k_tstride, const void *v, int64_t v_bstride,
                              int64_t v_tstride, const void *logits, int64_t batch, int64_t tokens_q,
                              int64_t tokens_k, int64_t heads, int64_t head_dim, float scale, void *workspace,
                              int64_t workspace_bytes, void *stream)
{
    static const char *what = "attention";
    clear_error();
    if (batch < 0 || tokens_q < 0 || tokens_k < 0 || heads <= 0)
        return fail(LTXK_E_ARG, "%s: bad shape batch=%lld tokens_q=%lld tokens_k=%lld heads=%lld", what,
                    (long long)batch, (long long)tokens_q, (long long)tokens_k, (long long)heads);
    if (head_dim != 64 && head_dim != 128)
        return fail(LTXK_E_ARG, "%s: head_dim must be 64 or 128 (got %lld)", what, (long long)head_dim);
    if (batch == 0 || tokens_q == 0) return LTXK_OK;
    if (tokens_k == 0) return fail(LTXK_E_ARG, "%s: no keys", what);
    // the maximum is taken of the raw scores, and keys past the last are closed with -inf before the scaling
    const float scale2 = scale * 1.4426950408889634f;
    if (!(scale > 0.f && scale2 <= FLT_MAX))
        return fail(LTXK_E_ARG, "%s: scale must be positive and finite (got %g)", what, static_cast<double>(scale));
    if (!out || !q || !k || !v) return fail(LTXK_E_ARG, "%s: null out, q, k or v", what);
    if (!aligned16(out) || !aligned16(q) || !aligned16(k) || !aligned16(v) ||
        (reinterpret_cast<uintptr_t>(logits) & 1u))
        return fail(LTXK_E_ALIGN, "%s: out, q, k and v must be 16-byte aligned, logits 2-byte", what);
    for (int64_t st : {q_bstride, q_tstride, k_bstride, k_tstride, v_bstride, v_tstride})
        if (st < 0 || st % 8) return fail(LTXK_E_ALIGN, "%s: strides must be non-negative multiples of 8", what);
    const int64_t width = heads * head_dim;
    if (heads > (1 << 20) || batch > (1 << 20) || q_tstride < width || k_tstride < width || v_tstride < width)
        return fail(LTXK_E_ARG, "%s: token strides must cover heads*head_dim (%lld)", what, (long long)width);
    // the kernel addresses the rows of one batch item with 32-bit byte offsets
    const int64_t kMax = 0x7fffffff;
    if (q_tstride > kMax / 2 || tokens_q > kMax - 256 || (tokens_k + kKeys) > kMax / 2 / k_tstride ||
        (tokens_k + kKeys) > kMax / 2 / v_tstride)
        return fail(LTXK_E_ARG, "%s: a batch item's keys or values span 2^31 bytes or more", what);
    const FlashCut c = cut(batch * heads, tokens_q, tokens_k);
    // a launch holds fewer than 2^32 threads
    if (c.whole + c.rest * c.parts >= (int64_t{1} << 32) / (8 * kWaves * 64))
        return fail(LTXK_E_ARG, "%s: too many query tiles", what);
    if (c.rest && (!workspace || !aligned16(workspace) ||
                   workspace_bytes < ltxk_attention_workspace_bytes(batch, tokens_q, tokens_k, heads, head_dim)))
        return fail(LTXK_E_ARG, "%s: the workspace must hold ltxk_attention_workspace_bytes, 16-byte aligned", what);
    FlashParams p{};
    p.q = static_cast<const uint16_t *>(q);
    p.k = static_cast<const uint16_t *>(k);
    p.v = static_cast<const uint16_t *>(v);
    p.logits = static_cast<const uint16_t *>(logits);
    p.out = static_cast<uint16_t *>(out);
    p.part = static_cast<float *>(workspace);
    p.stats = reinterpret_cast<float2 *>(p.part + 8 * c.rest * c.parts * kRows * head_dim);
    p.qbs = q_bstride;
    p.kbs = k_bstride;
    p.vbs = v_bstride;
    p.qts = static_cast<uint32_t>(q_tstride * 2);
    p.kts = static_cast<uint32_t>(k_tstride * 2);
    p.vts = static_cast<uint32_t>(v_tstride * 2);
    p.tq = static_cast<int>(tokens_q);
    p.tk = static_cast<int>(tokens_k);
    p.heads = static_cast<int>(heads);
    p.bh = static_cast<int>(batch * heads);
    p.q_tiles = static_cast<int>(c.q_tiles);
    p.tiles = static_cast<int>(c.tiles);
    p.whole = static_cast<int>(c.whole);
    p.rest = static_cast<int>(c.rest);
    p.parts = static_cast<int>(c.parts);
    p.scale2 = scale2;
    if (head_dim == 128)
        launch<128>(p, static_cast<hipStream_t>(stream));
    else
        launch<64>(p, static_cast<hipStream_t>(stream));
    return check_launch(what);
}
