// y = round_bf16(x w^T + bias) for bf16 x (M, K) and w (N, K), for outputs that
// leave the chip's last wave of tiles nearly empty over a long K: the tiles past
// the last full wave are cut over K, and their parts' fp32 sums added in a second
// pass.
//
// What bounds it: the card's power and, with it, the loads beside the products.
// [1024, 188160] x [4096, 188160] takes 1214-1266 us, 1.25-1.30 PFLOP/s (the
// library's product, which leaves three of four compute units idle: 2100-2139 us,
// 0.74-0.75), [512, 16384] x [4096, 16384] 73 (86).  On zeros, 8192^3 runs at
// 1.72 PFLOP/s and 2.07 without its loads.  So:
// * 256 x 256 tiles (half the loads of 128 x 256, which ran 15 % slower), eight
//   waves of 128 x 64: four of 128 x 128 took 887 against 846 us on 8192^3.
// * Loads go straight to LDS, one between two products: in one run at the head of
//   a step 858 against 839 us.
// * x three steps deep and w two, all of the 160 KB: 839 against 846 with two of
//   each.  Steps of 32 elements in rings of three to five took 918-923 us (64-byte
//   row pieces).
// * Neighbouring tiles share an XCD and run its K in step: starting each workgroup
//   elsewhere in K took 1125 us.
#include "ltxk_common.h"

namespace ltxk {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) char lds_char;

constexpr int kTile = 256;  // rows of x and of w a workgroup
constexpr int kStep = 64;   // elements of K a step
constexpr int kWaves = 8;   // 2 along the rows of x, 4 along the rows of w
constexpr int kBand = 4;    // tiles of x that a band of the tile order holds (8: no difference)

struct GemmParams {
    const uint16_t *x, *w, *bias;
    uint16_t *y;
    float *part;  // (parts, rest) tiles of fp32 sums
    int m, n, k;
    int tiles_m, tiles_n;
    int whole, rest, parts;  // tiles that one workgroup takes alone; the others, cut into parts over K
};

// The rows of x and w that tile t takes: bands kBand tiles of x deep.
__device__ __forceinline__ void tile_rows(const GemmParams &p, int t, int &m0, int &n0)
{
    const int band = t / (kBand * p.tiles_n), at = t % (kBand * p.tiles_n);
    const int deep = min(kBand, p.tiles_m - band * kBand);
    m0 = (band * kBand + at % deep) * kTile;
    n0 = at / deep * kTile;
}

// LDS position of 16-byte chunk c (8 elements of K) of a tile's row: 16 rows of
// one chunk column, which a fragment read takes at a time, cover all banks.
__device__ __forceinline__ int chunk_pos(int row, int c) { return c ^ ((row >> 1) & 7); }

// 64 lanes x 16 bytes from memory straight to LDS at `lds`, through m0.  In assembly
// because the compiler, which cannot tell the buffers of a ring apart, would wait
// for every load in flight before each LDS read; it has no output register, and its
// wait is step_barrier's.  The wait states cover scalar operands that a vector
// instruction has just written, which the compiler does not see the load read.  It
// does not see m0 change either (a reserved register, whose clobber it ignores with
// a warning): nothing else in these kernels may use m0, such as an LDS load builtin,
// an indexed register or a message, and their assembly holds no other use.
__device__ __forceinline__ void load_lds(const u32x4 &rsrc, uint32_t lds, uint32_t off, uint32_t soff)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 ::"s"(lds), "v"(off), "s"(rsrc), "s"(soff)
                 : "memory");
}

// At most `N` of this wave's loads in flight (none without `more`) and its LDS
// reads returned, then all waves'.
template <int N>
__device__ __forceinline__ void step_barrier(bool more)
{
    asm volatile("" ::: "memory");
    if (more)
        __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | (N >> 4 << 14));  // vmcnt(N) lgkmcnt(0)
    else
        __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__global__ void __launch_bounds__(kWaves * 64, 2) gemm_kernel(GemmParams p)
{
    constexpr int MT = kTile / 64, NT = kTile / 128, F = MT + NT;  // 32-row tiles of a wave
    constexpr int L = kTile / 8 / kWaves;                          // loads of a wave for a step of x or w
    constexpr int kBytes = kTile * kStep * 2;
    // x: a ring of three steps, then w: of two
    __shared__ __attribute__((aligned(1024))) char smem[5 * kBytes];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l32 = lane & 31, half = lane >> 5;

    // A run of neighbouring tiles per XCD (workgroups are dealt to the XCDs in
    // turn), so that its L2 serves a tile of either side to several workgroups.
    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3, whole_per = p.whole >> 3;
    int tile, part = -1;
    if (j < whole_per) {
        tile = xcd * whole_per + j;
    } else {
        const int per = (p.rest * p.parts + 7) >> 3, unit = xcd * per + j - whole_per;
        if (unit >= p.rest * p.parts) return;
        part = unit / p.rest;
        tile = p.whole + unit % p.rest;
    }
    int m0, n0;
    tile_rows(p, tile, m0, n0);
    const int steps = p.k / kStep;
    const int first = part < 0 ? 0 : static_cast<int>(static_cast<int64_t>(part) * steps / p.parts);
    const int n = (part < 0 ? steps : static_cast<int>(static_cast<int64_t>(part + 1) * steps / p.parts)) - first;

    const uint64_t xa = reinterpret_cast<uint64_t>(p.x), wa = reinterpret_cast<uint64_t>(p.w);
    const u32x4 xr = {static_cast<uint32_t>(xa), static_cast<uint32_t>(xa >> 32) & 0xffff, 0xffffffffu, 0x00020000u};
    const u32x4 wr = {static_cast<uint32_t>(wa), static_cast<uint32_t>(wa >> 32) & 0xffff, 0xffffffffu, 0x00020000u};
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char *)smem));
    uint32_t xo[L], wo[L];
#pragma unroll
    for (int j = 0; j < L; ++j) {  // rows past the last repeat it; their results are not stored
        const int row = (wave * L + j) * 8 + (lane >> 3);
        const uint32_t c = chunk_pos(row, lane & 7) * 16, stride = static_cast<uint32_t>(p.k) * 2;
        xo[j] = static_cast<uint32_t>(min(m0 + row, p.m - 1)) * stride + c;
        wo[j] = static_cast<uint32_t>(min(n0 + row, p.n - 1)) * stride + c;
    }
    auto load_x = [&](int i, int j, int base) {
        load_lds(xr, __builtin_amdgcn_readfirstlane(lds0 + base + (wave * L + j) * 1024), xo[j],
                 __builtin_amdgcn_readfirstlane((first + i) * kStep * 2));
    };
    auto load_w = [&](int i, int j, int base) {
        load_lds(wr, __builtin_amdgcn_readfirstlane(lds0 + base + (wave * L + j) * 1024), wo[j],
                 __builtin_amdgcn_readfirstlane((first + i) * kStep * 2));
    };
    for (int i = 0; i < 2 && i < n; ++i) {
#pragma unroll
        for (int j = 0; j < L; ++j) load_x(i, j, i * kBytes);
#pragma unroll
        for (int j = 0; j < L; ++j) load_w(i, j, (3 + i) * kBytes);
    }
    if (n > 2)
#pragma unroll
        for (int j = 0; j < L; ++j) load_x(2, j, 2 * kBytes);

    int off[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) off[s] = l32 * 128 + chunk_pos(l32, 2 * s + half) * 16;
    const int wm = (wave >> 2) * (kTile / 2), wn = (wave & 3) * (kTile / 4);  // this wave's rows

    // acc[i][j]: lane l holds row 32 i + l % 32 of x; register r row 32 j + 8 (r/4) + 4 half + r % 4 of w
    f32x16 acc[MT][NT] = {};
    bf16x8 f[2][F];
    auto frag = [&](int xb, int wb, int s, int j) {
        const char *base = smem + off[s] + (j < MT ? xb + wm * 128 : wb + wn * 128);
        return *reinterpret_cast<const bf16x8 *>(base + (j < MT ? j : j - MT) * 4096);
    };
    step_barrier<L>(n > 2);
#pragma unroll
    for (int j = 0; j < F; ++j) f[0][j] = frag(0, 3 * kBytes, 0, j);
    int xb = 0, wb = 3 * kBytes;
    for (int i = 0; i < n; ++i) {
        const int xn = xb == 2 * kBytes ? 0 : xb + kBytes, wn_ = wb == 3 * kBytes ? 4 * kBytes : 3 * kBytes;
        const int xp = xb == 0 ? 2 * kBytes : xb - kBytes;  // x of step i - 1, that of i + 2 next
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            // before the last quarter: step i + 1 is there, and all waves have read
            // step i whole, so its w goes to step i + 2 here and its x to step i + 3
            // in the next step's first quarter, one load between two products
            if (s == 3) {
                step_barrier<L>(i + 2 < n);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int e = 0; e < MT * NT; ++e) {
                if (e < F) f[(s + 1) & 1][e] = s < 3 ? frag(xb, wb, s + 1, e) : frag(xn, wn_, 0, e);
                const int mi = e / NT, ni = e % NT;
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[s & 1][MT + ni], f[s & 1][mi], acc[mi][ni], 0, 0, 0);
                if (s == 3 && e < L && i + 2 < n) load_w(i + 2, e, wb);
                if (s == 0 && e < L && i > 0 && i + 2 < n) load_x(i + 2, e, xp);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        xb = xn;
        wb = wn_;
    }

    float *sums = part < 0 ? nullptr
                           : p.part + (static_cast<int64_t>(part) * p.rest + tile - p.whole) * (kTile * kTile);
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
        const int r = wm + mi * 32 + l32;
        if (m0 + r >= p.m) continue;
#pragma unroll
        for (int ni = 0; ni < NT; ++ni)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int c = wn + ni * 32 + 8 * q + 4 * half;
                if (n0 + c >= p.n) continue;
                f32x4 v = {acc[mi][ni][4 * q], acc[mi][ni][4 * q + 1], acc[mi][ni][4 * q + 2], acc[mi][ni][4 * q + 3]};
                if (sums) {
                    *reinterpret_cast<f32x4 *>(sums + r * kTile + c) = v;
                    continue;
                }
                if (p.bias)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] += bf16_to_f32(p.bias[n0 + c + e]);
                *reinterpret_cast<uint2 *>(p.y + static_cast<int64_t>(m0 + r) * p.n + n0 + c) =
                    make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
            }
    }
}

// Adds the parts of 8 outputs a thread, in their order, then the bias.
__global__ void __launch_bounds__(256) gemm_sum_kernel(GemmParams p)
{
    constexpr int kBlocks = kTile * kTile / 8 / 256;  // workgroups a tile
    const int t = blockIdx.x / kBlocks, i = (blockIdx.x % kBlocks * 256 + threadIdx.x) * 8;
    int m0, n0;
    tile_rows(p, p.whole + t, m0, n0);
    const int row = m0 + i / kTile, col = n0 + i % kTile;
    if (row >= p.m || col >= p.n) return;
    const float *s = p.part + static_cast<int64_t>(t) * (kTile * kTile) + i;
    f32x4 lo = {}, hi = {};
#pragma unroll 4
    for (int k = 0; k < p.parts; ++k, s += static_cast<int64_t>(p.rest) * (kTile * kTile)) {
        lo += *reinterpret_cast<const f32x4 *>(s);
        hi += *reinterpret_cast<const f32x4 *>(s + 4);
    }
    float f[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    if (p.bias) {
        float b[8];
        unpack8v(*reinterpret_cast<const u32x4 *>(p.bias + col), b);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] += b[e];
    }
    *reinterpret_cast<u32x4 *>(p.y + static_cast<int64_t>(row) * p.n + col) = pack8v(f);
}

// How an output is cut: the chip takes 256 tiles at a time, one a compute unit;
// the tiles past the last multiple of 256 are dealt to the units in parts of K, of
// at least 8 steps each.
struct GemmCut {
    int64_t tiles_m, tiles_n, whole, rest, parts;
};

GemmCut cut(int64_t m, int64_t n, int64_t k)
{
    GemmCut c;
    c.tiles_m = (m + kTile - 1) / kTile;
    c.tiles_n = (n + kTile - 1) / kTile;
    c.rest = c.tiles_m * c.tiles_n % 256;
    c.whole = c.tiles_m * c.tiles_n - c.rest;
    c.parts = 1;
    if (c.rest) {
        c.parts = 256 / c.rest;
        if (c.parts > k / kStep / 8) c.parts = k / kStep / 8;
        if (c.parts < 1) c.parts = 1;
    }
    return c;
}

// ------------------------------------------------- several layers, few rows --
// y_g = round_bf16(x w_g^T + bias_g) for up to four weights over the same few rows
// of x (an audio stream's q, k, v and gate projections) in one launch.  Layer by
// layer they take a launch and about 20 us of the host each: [126, 2048] x (3 x 2048
// + 32) 45 us on the device and 77 in eager calls, here 16 and 16.  What bounds it
// is each workgroup's own loads (65 of the 95 KB a us that loads alone reach), of
// which x is most: 128 rows of x and 32 of a weight a workgroup, so that 193 compute
// units work without a second pass.  Steps of 128 of K: 17 us with 64.
constexpr int kFewRows = 128, kFewCols = 32, kFewWaves = 4, kMaxLayers = 4;
constexpr int kFewStep = 2 * kStep;    // elements of K a step, as two tiles of kStep
constexpr int kFewX = 3, kFewW = 7;    // steps of x and of w in LDS

struct FewLayer {
    const uint16_t *w, *bias;
    uint16_t *y;
    int n, first;  // rows of w; its first column tile
};

struct FewParams {
    const uint16_t *x;
    FewLayer g[kMaxLayers];
    int m, k, tiles_m, tiles_n;
};

// Four waves load x and take 32 of its rows each; a fifth only loads w, whose
// rows come from memory: a wave's loads return in order, so beside x, which the L2
// holds, they could not run as far ahead.
__global__ void __launch_bounds__((kFewWaves + 1) * 64, 1) few_rows_kernel(FewParams p)
{
    constexpr int kXBytes = kFewRows * kFewStep * 2, kWBytes = kFewCols * kFewStep * 2, L = 8;  // loads of a wave a step
    __shared__ __attribute__((aligned(1024))) char smem[kFewX * kXBytes + kFewW * kWBytes];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l32 = lane & 31, half = lane >> 5;

    // a weight's tile goes to one XCD for all tiles of x
    const int t = (blockIdx.x >> 3) / p.tiles_m * 8 + (blockIdx.x & 7), m0 = (blockIdx.x >> 3) % p.tiles_m * kFewRows;
    if (t >= p.tiles_n) return;
    FewLayer g = p.g[0];
#pragma unroll
    for (int i = 1; i < kMaxLayers; ++i)
        if (t >= p.g[i].first) g = p.g[i];
    const int n0 = (t - g.first) * kFewCols, n = p.k / kFewStep;

    // rows past the last repeat it; their results are not stored
    const bool is_x = wave < kFewWaves;
    const uint64_t base = reinterpret_cast<uint64_t>(is_x ? p.x : g.w);
    const u32x4 rsrc = {static_cast<uint32_t>(base), static_cast<uint32_t>(base >> 32) & 0xffff, 0xffffffffu, 0x00020000u};
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char *)smem)) +
                          (is_x ? wave * 4096 : kFewX * kXBytes);
    uint32_t go[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = ((is_x ? wave : 0) * 4 + j) * 8 + (lane >> 3);
        const int at = is_x ? min(m0 + row, p.m - 1) : min(n0 + row, g.n - 1);
        go[j] = static_cast<uint32_t>(at) * (static_cast<uint32_t>(p.k) * 2) + chunk_pos(row, lane & 7) * 16;
    }
    auto load = [&](int i, int slot) {
#pragma unroll
        for (int j = 0; j < L; ++j)
            load_lds(rsrc,
                     __builtin_amdgcn_readfirstlane(lds0 + slot + (j >> 2) * ((is_x ? kFewRows : kFewCols) * kStep * 2) +
                                                    (j & 3) * 1024),
                     go[j & 3], __builtin_amdgcn_readfirstlane((2 * i + (j >> 2)) * kStep * 2));
    };
    // At barrier i step i is there and step i - 1 read by all: its slot takes the
    // load that is furthest ahead.
    if (!is_x) {
        for (int i = 0; i < kFewW - 1 && i < n; ++i) load(i, i * kWBytes);
        for (int i = 0; i < n; ++i) {
            step_barrier<(kFewW - 2) * L>(i + kFewW - 2 < n);
            if (i + kFewW - 1 < n) load(i + kFewW - 1, (i + kFewW - 1) % kFewW * kWBytes);
        }
        return;
    }
    for (int i = 0; i < kFewX - 1 && i < n; ++i) load(i, i * kXBytes);

    int off[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) off[s] = l32 * 128 + chunk_pos(l32, 2 * s + half) * 16;
    f32x16 acc2[2] = {};
    for (int i = 0; i < n; ++i) {
        step_barrier<(kFewX - 2) * L>(i + kFewX - 2 < n);
        const char *xs = smem + i % kFewX * kXBytes + wave * 4096, *ws = smem + kFewX * kXBytes + i % kFewW * kWBytes;
        bf16x8 xf[8], wf[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            xf[s] = *reinterpret_cast<const bf16x8 *>(xs + (s >> 2) * (kFewRows * kStep * 2) + off[s & 3]);
            wf[s] = *reinterpret_cast<const bf16x8 *>(ws + (s >> 2) * (kFewCols * kStep * 2) + off[s & 3]);
        }
        if (i + kFewX - 1 < n) load(i + kFewX - 1, (i + kFewX - 1) % kFewX * kXBytes);
#pragma unroll
        for (int s = 0; s < 8; ++s)
            acc2[s & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[s], xf[s], acc2[s & 1], 0, 0, 0);
    }
    const f32x16 acc = acc2[0] + acc2[1];

    const int row = m0 + wave * 32 + l32;
    if (row >= p.m) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int col = n0 + 8 * q + 4 * half;
        if (col >= g.n) continue;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[4 * q + e] + (g.bias ? bf16_to_f32(g.bias[col + e]) : 0.f);
        *reinterpret_cast<uint2 *>(g.y + static_cast<int64_t>(row) * g.n + col) =
            make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    }
}

}  // namespace
}  // namespace ltxk

using namespace ltxk;

extern "C" int64_t ltxk_linear_workspace_bytes(int64_t m, int64_t n, int64_t k)
{
    if (m <= 0 || n <= 0 || k <= 0) return 0;
    const GemmCut c = cut(m, n, k);
    return c.rest * c.parts * kTile * kTile * 4;
}

extern "C" int ltxk_linear(void *y, const void *x, const void *w, const void *bias, int64_t m, int64_t n, int64_t k,
                           void *workspace, int64_t workspace_bytes, void *stream)
{
    static const char *what = "linear";
    clear_error();
    if (m < 0 || n <= 0 || k <= 0) return fail(LTXK_E_ARG, "%s: bad shape m=%lld n=%lld k=%lld", what, (long long)m,
                                               (long long)n, (long long)k);
    if (n % 8 || k % kStep) return fail(LTXK_E_ARG, "%s: n must be a multiple of 8 and k of %d (got %lld, %lld)", what,
                                        kStep, (long long)n, (long long)k);
    if (m == 0) return LTXK_OK;
    if (!y || !x || !w) return fail(LTXK_E_ARG, "%s: null y, x or w", what);
    if (!aligned16(y) || !aligned16(x) || !aligned16(w) || !aligned16(bias))
        return fail(LTXK_E_ALIGN, "%s: y, x, w and bias must be 16-byte aligned", what);
    // operands are read through descriptors of 2^32 - 1 bytes, outputs counted by 32-bit tiles
    const int64_t kMax = int64_t{1} << 31;
    if (k >= kMax / 2 || m > (kMax - 1) / k || n > (kMax - 1) / k || m > kMax / n)
        return fail(LTXK_E_ARG, "%s: x or w holds 2^31 elements or more, or y more than 2^31", what);
    GemmParams p{};
    p.x = static_cast<const uint16_t *>(x);
    p.w = static_cast<const uint16_t *>(w);
    p.bias = static_cast<const uint16_t *>(bias);
    p.y = static_cast<uint16_t *>(y);
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = static_cast<int>(k);
    const GemmCut c = cut(m, n, k);
    if (c.rest && (!workspace || !aligned16(workspace) || workspace_bytes < ltxk_linear_workspace_bytes(m, n, k)))
        return fail(LTXK_E_ARG, "%s: the workspace must hold ltxk_linear_workspace_bytes, 16-byte aligned", what);
    p.part = static_cast<float *>(workspace);
    p.tiles_m = static_cast<int>(c.tiles_m);
    p.tiles_n = static_cast<int>(c.tiles_n);
    p.whole = static_cast<int>(c.whole);
    p.rest = static_cast<int>(c.rest);
    p.parts = static_cast<int>(c.parts);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const unsigned grid = 8u * static_cast<unsigned>(c.whole / 8 + (c.rest * c.parts + 7) / 8);
    gemm_kernel<<<grid, kWaves * 64, 0, s>>>(p);
    if (c.rest) gemm_sum_kernel<<<static_cast<unsigned>(c.rest) * (kTile * kTile / 8 / 256), 256, 0, s>>>(p);
    return check_launch(what);
}

extern "C" int ltxk_linear_layers(void *const *y, const void *x, const void *const *w, const void *const *bias,
                                  const int64_t *n, int64_t layers, int64_t m, int64_t k, void *stream)
{
    static const char *what = "linear_layers";
    clear_error();
    if (layers < 1 || layers > kMaxLayers)
        return fail(LTXK_E_ARG, "%s: 1 to %d layers (got %lld)", what, kMaxLayers, (long long)layers);
    if (m < 0 || k <= 0 || k % kFewStep)
        return fail(LTXK_E_ARG, "%s: bad shape m=%lld k=%lld (k a multiple of %d)", what, (long long)m, (long long)k,
                    kFewStep);
    if (!y || !w || !n) return fail(LTXK_E_ARG, "%s: null y, w or n", what);
    if (m == 0) return LTXK_OK;
    const int64_t kMax = int64_t{1} << 31;
    if (!x) return fail(LTXK_E_ARG, "%s: null x", what);
    if (!aligned16(x)) return fail(LTXK_E_ALIGN, "%s: x must be 16-byte aligned", what);
    if (k >= kMax / 2 || m > (kMax - 1) / k) return fail(LTXK_E_ARG, "%s: x holds 2^31 elements or more", what);
    FewParams p{};
    p.x = static_cast<const uint16_t *>(x);
    p.m = static_cast<int>(m);
    p.k = static_cast<int>(k);
    p.tiles_m = static_cast<int>((m + kFewRows - 1) / kFewRows);
    int64_t tiles = 0;
    for (int64_t i = 0; i < kMaxLayers; ++i) {
        FewLayer &g = p.g[i];
        if (i >= layers) {
            g.first = 0x7fffffff;  // no tile reaches it
            continue;
        }
        const void *b = bias ? bias[i] : nullptr;
        if (n[i] <= 0 || n[i] % 8)
            return fail(LTXK_E_ARG, "%s: layer %lld: n must be a positive multiple of 8 (got %lld)", what, (long long)i,
                        (long long)n[i]);
        if (n[i] > (kMax - 1) / k || m > kMax / n[i])
            return fail(LTXK_E_ARG, "%s: layer %lld: w holds 2^31 elements or more, or y more than 2^31", what,
                        (long long)i);
        if (!y[i] || !w[i]) return fail(LTXK_E_ARG, "%s: layer %lld: null y or w", what, (long long)i);
        if (!aligned16(y[i]) || !aligned16(w[i]) || !aligned16(b))
            return fail(LTXK_E_ALIGN, "%s: layer %lld: y, w and bias must be 16-byte aligned", what, (long long)i);
        g.w = static_cast<const uint16_t *>(w[i]);
        g.bias = static_cast<const uint16_t *>(b);
        g.y = static_cast<uint16_t *>(y[i]);
        g.n = static_cast<int>(n[i]);
        g.first = static_cast<int>(tiles);
        tiles += (n[i] + kFewCols - 1) / kFewCols;
    }
    p.tiles_n = static_cast<int>(tiles);
    const int64_t grid = 8 * ((tiles + 7) / 8) * p.tiles_m;
    if (grid >= kMax) return fail(LTXK_E_ARG, "%s: too many tiles", what);
    few_rows_kernel<<<static_cast<unsigned>(grid), (kFewWaves + 1) * 64, 0, static_cast<hipStream_t>(stream)>>>(p);
    return check_launch(what);
}
