// prefill.hip -- a prompt's tokens through the layers together.
//
// The reference feeds a prompt one token per step (examples/serve-demo.rs:
// 62-91), which reads every weight once per token.  Here all prompt tokens
// but the last go through each layer as one matrix product per projection
// (the last one is an ordinary decode step, which makes the logits); the KV
// cache, positions and step counts end up as the steps would leave them.
//
// Arithmetic: 32-bit values on the f16 matrix cores as pairs of halves
// (split.hpp, which says what a pair holds: 23 bits, down to a floor of 2^-39
// of the row's largest value).  A product is hi*hi + lo*hi + hi*lo, accumulated
// in f32 by the matrix cores; lo*lo, at most 2^-22 of it, is dropped.
// Activations carry one power of two per row, weights one per matrix row
// (pf_rowscale_kernel).  K and V are f16 in the cache, so the attention splits
// only the queries and the softmax weights (an f32 cache is attended in f32).
// Against 64 bits the sums are as far off as the steps' f32 sums, within half
// as much again (figures at pf_tile), and less than the steps' limbs from 2048
// columns on.  What that leaves a whole turn with: a cache entry now and then
// rounds to the neighbouring half, and the logits move by 1e-4 to 2e-4.
//
// No result depends on which other tokens share the launch: a row's sums run
// over the columns in an order fixed by the weights' shape and the prompt's
// length alone, whatever the number of clients.
#include "internal.hpp"

#include "prefill.hpp"
#include "split.hpp"

#include <math.h>

#include <algorithm>

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / EMU_WAVE;
constexpr int kTile = 32;  // matrix-core tile edge
constexpr int kStage = 64; // columns per pipeline stage (four 16-column slices)
constexpr int kPfMaxSplit = 8; // shares of the columns per product at most

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float16v mfma(half8 a, half8 b, float16v c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// ---- operand planes -------------------------------------------------------
// The left operand of a product: rows of K columns (padded with zeros to
// whole stages), cut into 32-row tiles and 16-column slices; slice s of tile
// t is 2 KB at 2048 * (t * K/16 + s): the hi halves, then the lo halves, each
// as the matrix cores take them (lane 32*kh + j: row j's columns 8kh..8kh+7).
__device__ __forceinline__ size_t plane_at(int row, int group, int slices) // 8-column group, its hi half
{
    return ((size_t)(row / kTile) * slices + (group >> 1)) * 2048 + (size_t)((group & 1) * kTile + row % kTile) * 16;
}

__device__ __forceinline__ void plane_store(uint8_t *planes, int row, int group, int slices, const float (&v)[8])
{
    half8 hi, lo;
    split8(v, hi, lo);
    uint8_t *p = planes + plane_at(row, group, slices);
    *reinterpret_cast<half8 *>(p) = hi;
    *reinterpret_cast<half8 *>(p + 1024) = lo;
}

__device__ __forceinline__ float block_max(float v, float *red)
{
    v = emu_wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float m = red[0];
    for (int i = 1; i < (int)(blockDim.x >> 6); ++i) m = fmaxf(m, red[i]);
    return m;
}

// One row into the planes by a workgroup of TH threads, thread i holding the
// row's 8-column groups i, i + TH, ... (G of them).  A row with an inf or NaN
// becomes zeros under a NaN scale: every product with it is NaN, as the limb
// kernels' spans are.
constexpr int kRowThreads = 512;
template <int G>
__device__ __forceinline__ void emit_row(const PfPlanes &P, int row, int cols, float *red, float (&v)[G][8])
{
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < G; ++j)
        if (8 * (int)(threadIdx.x + j * kRowThreads) < cols) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float a = fabsf(v[j][i]);
                amax = fmaxf(amax, a <= 3.402823466e38f ? a : INFINITY); // a NaN too
            }
        }
    amax = block_max(amax, red);
    const bool finite = amax <= 3.402823466e38f;
    float s, inv;
    pow2_scale(amax, s, inv);
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const int g = threadIdx.x + j * kRowThreads;
        if (g >= 2 * P.slices) continue;
        float w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = finite && 8 * g < cols ? v[j][i] * s : 0.0f; // rows are whole groups
        plane_store(P.q, row, g, P.slices, w);
    }
    if (threadIdx.x == 0) P.scale[row] = finite ? inv : __int_as_float(0x7fc00000);
}

__device__ __forceinline__ void ld8f(const float *p, float (&v)[8])
{
    const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// Eight columns of nks <= NS partial sums, added in order.  Straight-line
// code: slots past nks load the first slice again and are not added, so that
// every load is out before the first wait.
template <int NS> __device__ __forceinline__ void sum8(const float *p, int nks, size_t stride, float (&v)[8])
{
    float q[NS][8];
#pragma unroll
    for (int k = 0; k < NS; ++k) ld8f(p + (k < nks ? k : 0) * stride, q[k]);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        v[i] = q[0][i];
#pragma unroll
        for (int k = 1; k < NS; ++k) v[i] = k < nks ? v[i] + q[k][i] : v[i];
    }
}

// ---- weights --------------------------------------------------------------
// A lane of the product owns one weight row and one 8-column half (kh) of
// every 16-column slice.  load() reads what `PER` stages need of the row (a
// 256-column span; the router: one stage), in 16-byte pieces: the two lanes
// of a row read 32 neighbouring bytes, whose four 8-byte pieces belong to the
// two halves in turn, and swap the pieces that are the other's
// (v_permlane32_swap).  So each cache line of a row is asked for by a few
// back-to-back loads; with 8-byte loads per stage, lines left L1 between
// stages and were fetched again (gate|up of 4096 columns, 15 tokens: 60 us).
// part() gives the eight weights of slice j of stage q of the span, times the
// row's scale, as hi and lo halves.  slice() says which of the row's 16-column slices that is: the
// formats whose blocks interleave columns take the slices in the order their
// units hold them.

// 16 bytes at p + 16 kh; after swap32(), .xy and .zw are the row's 8-byte
// pieces kh and 2 + kh of the 32 at p.  load() only asks for them and
// settle(), a span later, swaps: swapping at once put a wait for memory into
// every span (15 tokens of Qwen3-8B: gate|up 42 -> 40 us, down 28 -> 24; at
// 511 tokens, 315 us of matrix cores, no difference).
__device__ __forceinline__ void swap32(uint4 &v)
{
    const auto x = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
    const auto y = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
    v = make_uint4(x[0], y[0], x[1], y[1]);
}
__device__ __forceinline__ uint2 half_of(const uint4 &v, int i) { return i ? make_uint2(v.z, v.w) : make_uint2(v.x, v.y); }
struct PfQ6K {
    static constexpr int PER = 4;
    struct Raw {
        uint4 ql[4], qh[2]; // 32-byte pieces; the halves are the units
        uint4 sc;
        uint32_t d;
    };
    static __device__ __forceinline__ int slice(int grp, int q, int j) { return 16 * grp + 8 * (q >> 1) + 2 * j + (q & 1); }
    static __device__ __forceinline__ void load(const uint8_t *row, int grp, int kh, int nb, Raw &r)
    {
        const uint8_t *b = row + (size_t)grp * 210;
#pragma unroll
        for (int i = 0; i < 4; ++i) r.ql[i] = ld16(b + 32 * i + 16 * kh);
#pragma unroll
        for (int i = 0; i < 2; ++i) r.qh[i] = ld16(b + 128 + 32 * i + 16 * kh);
        r.sc = ld16(b + 192);
        r.d = ld2(b + 208);
    }
    static __device__ __forceinline__ void settle(Raw &r)
    {
#pragma unroll
        for (int i = 0; i < 4; ++i) swap32(r.ql[i]);
#pragma unroll
        for (int i = 0; i < 2; ++i) swap32(r.qh[i]);
    }
    // q = 2 h + u: half h of the block, unit 2u + kh of the half
    static __device__ __forceinline__ void part(const Raw &r, int q, int kh, int j, float s, half8 &bh, half8 &bl)
    {
        const int h = q >> 1, u = q & 1;
        const uint32_t lo = 0x0f0f0f0fu, hi = 0x30303030u;
        const uint2 a = half_of(r.ql[2 * h + (j & 1)], u), c = half_of(r.qh[h], u);
        const int ns = 4 * (j >> 1);
        const uint32_t h0 = j < 2 ? c.x << (4 - 2 * j) : c.x >> (2 * j - 4);
        const uint32_t h1 = j < 2 ? c.y << (4 - 2 * j) : c.y >> (2 * j - 4);
        const uint32_t words[4] = {r.sc.x, r.sc.y, r.sc.z, r.sc.w};
        const int si = 8 * h + u + 2 * j; // scale of (half, 16 columns)
        const float m = h2f((uint16_t)r.d) * (float)(int8_t)(words[si >> 2] >> (8 * (si & 3))) * s;
        biased8<32>(((a.x >> ns) & lo) | (h0 & hi), ((a.y >> ns) & lo) | (h1 & hi), m, bh, bl);
    }
};
struct PfQ2K {
    static constexpr int PER = 4;
    struct Raw {
        uint4 qs[2]; // [half]; the halves are its 16-column runs
        uint4 sc;
        uint32_t dd;
    };
    static __device__ __forceinline__ int slice(int grp, int q, int j) { return PfQ6K::slice(grp, q, j); }
    static __device__ __forceinline__ void load(const uint8_t *row, int grp, int kh, int nb, Raw &r)
    {
        const uint8_t *b = row + (size_t)grp * 84;
#pragma unroll
        for (int i = 0; i < 2; ++i) r.qs[i] = ld16(b + 16 + 32 * i + 16 * kh);
        r.sc = ld16(b);
        r.dd = ld4(b + 80);
    }
    static __device__ __forceinline__ void settle(Raw &r)
    {
        swap32(r.qs[0]);
        swap32(r.qs[1]);
    }
    static __device__ __forceinline__ void part(const Raw &r, int q, int kh, int j, float s, half8 &bh, half8 &bl)
    {
        const int h = q >> 1, u = q & 1, si = 8 * h + 2 * j + u;
        const uint32_t words[4] = {r.sc.x, r.sc.y, r.sc.z, r.sc.w};
        const uint32_t packed = (words[si >> 2] >> (8 * (si & 3))) & 0xffu;
        const uint2 a = half_of(r.qs[h], u);
        codes8((a.x >> (2 * j)) & 0x03030303u, (a.y >> (2 * j)) & 0x03030303u,
               h2f((uint16_t)(r.dd & 0xffffu)) * (float)(packed & 15u) * s,
               -(h2f((uint16_t)(r.dd >> 16)) * (float)(packed >> 4)) * s, bh, bl);
    }
};
struct PfQ5K {
    static constexpr int PER = 4;
    struct Raw {
        uint4 qs[4], qh; // [64-column group]; the halves are its 16-column runs
        uint4 head;
    };
    static __device__ __forceinline__ int slice(int grp, int q, int j) { return 16 * grp + 4 * q + j; }
    static __device__ __forceinline__ void load(const uint8_t *row, int grp, int kh, int nb, Raw &r)
    {
        const uint8_t *b = row + (size_t)grp * 176;
#pragma unroll
        for (int i = 0; i < 4; ++i) r.qs[i] = ld16(b + 48 + 32 * i + 16 * kh);
        r.qh = ld16(b + 16 + 16 * kh);
        r.head = ld16(b);
    }
    static __device__ __forceinline__ void settle(Raw &r)
    {
#pragma unroll
        for (int i = 0; i < 4; ++i) swap32(r.qs[i]);
        swap32(r.qh);
    }
    static __device__ __forceinline__ void part(const Raw &r, int q, int kh, int j, float s, half8 &bh, half8 &bl)
    {
        const int half = j >> 1, index = 2 * q + half;
        const uint2 c = half_of(r.qs[q], j & 1), h = half_of(r.qh, j & 1);
        const uint32_t lo = 0x0f0f0f0fu;
        FmtQ5K::Raw f;
        f.s0 = r.head.y;
        f.s1 = r.head.z;
        f.s2 = r.head.w;
        uint32_t sc, m;
        FmtQ5K::scale_min(f, index, sc, m);
        codes8(((c.x >> (4 * half)) & lo) | (((h.x >> index) & 0x01010101u) << 4),
               ((c.y >> (4 * half)) & lo) | (((h.y >> index) & 0x01010101u) << 4),
               h2f((uint16_t)(r.head.x & 0xffffu)) * (float)sc * s, -(h2f((uint16_t)(r.head.x >> 16)) * (float)m) * s, bh,
               bl);
    }
};
struct PfQ8_0 {
    static constexpr int PER = 4;
    struct Raw {
        uint4 q[8]; // [block]; the halves are its 16-column runs
        uint32_t d[8];
    };
    static __device__ __forceinline__ int slice(int grp, int q, int j) { return 16 * grp + 4 * q + j; }
    static __device__ __forceinline__ void load(const uint8_t *row, int grp, int kh, int nb, Raw &r)
    {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int blk = 8 * grp + i < nb ? 8 * grp + i : nb - 1; // past the row: the planes hold zeros
            const uint8_t *b = row + (size_t)blk * 34;
            r.d[i] = ld2(b);
            r.q[i] = ld16(b + 2 + 16 * kh);
        }
    }
    static __device__ __forceinline__ void settle(Raw &r)
    {
#pragma unroll
        for (int i = 0; i < 8; ++i) swap32(r.q[i]);
    }
    static __device__ __forceinline__ void part(const Raw &r, int q, int kh, int j, float s, half8 &bh, half8 &bl)
    {
        const float d = h2f((uint16_t)r.d[2 * q + (j >> 1)]) * s;
        const uint2 c = half_of(r.q[2 * q + (j >> 1)], j & 1);
        biased8<128>(c.x ^ 0x80808080u, c.y ^ 0x80808080u, d, bh, bl);
    }
};
struct PfF32 { // the router's rows
    static constexpr int PER = 1;
    struct Raw {
        float4 v[4][2];
    };
    static __device__ __forceinline__ int slice(int grp, int q, int j) { return 4 * grp + j; }
    static __device__ __forceinline__ void load(const uint8_t *row, int grp, int kh, int nb, Raw &r) // nb: columns
    {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = kStage * grp + 16 * j + 8 * kh;
            const float4 *p = reinterpret_cast<const float4 *>(row) + (c < nb ? c : 0) / 4;
            r.v[j][0] = p[0];
            r.v[j][1] = p[1];
        }
    }
    static __device__ __forceinline__ void settle(Raw &) {}
    static __device__ __forceinline__ void part(const Raw &r, int q, int kh, int j, float s, half8 &bh, half8 &bl)
    {
        const float4 a = r.v[j][0], b = r.v[j][1];
        const float v[8] = {a.x * s, a.y * s, a.z * s, a.w * s, b.x * s, b.y * s, b.z * s, b.w * s};
        split8(v, bh, bl);
    }
};

// Per weight row, the power of two that keeps the row's scaled weights under
// 2^13 (a bound from the blocks' d and the formats' largest codes; f32 rows:
// the largest weight).  Eight lanes per row.
template <int ENC>
__global__ __launch_bounds__(kThreads) void pf_rowscale_kernel(const uint8_t *w, size_t row_bytes, int rows, int nb,
                                                               float *scale)
{
    const int row = blockIdx.x * (kThreads / 8) + threadIdx.x / 8, l = threadIdx.x & 7;
    const uint8_t *p = w + (size_t)(row < rows ? row : rows - 1) * row_bytes;
    float m = 0.0f;
    auto take = [&](float v) { m = fmaxf(m, v <= 3.402823466e38f ? v : INFINITY); };
    for (int b = l; b < nb; b += 8) {
        if constexpr (ENC == EMU_ENC_Q6_K) take(fabsf(h2f(ld2(p + (size_t)b * 210 + 208))) * 4096.0f);
        if constexpr (ENC == EMU_ENC_Q8_0) take(fabsf(h2f(ld2(p + (size_t)b * 34))) * 128.0f);
        if constexpr (ENC == EMU_ENC_Q5_K) {
            const uint32_t d = ld4(p + (size_t)b * 176);
            take(fabsf(h2f((uint16_t)d)) * 1953.0f + fabsf(h2f((uint16_t)(d >> 16))) * 63.0f);
        }
        if constexpr (ENC == EMU_ENC_Q2_K) {
            const uint32_t d = ld4(p + (size_t)b * 84 + 80);
            take(fabsf(h2f((uint16_t)d)) * 45.0f + fabsf(h2f((uint16_t)(d >> 16))) * 15.0f);
        }
        if constexpr (ENC == EMU_ENC_F32) take(fabsf(reinterpret_cast<const float *>(p)[b]));
    }
    m = fmaxf(m, emu_xor_lane<1>(m));
    m = fmaxf(m, emu_xor_lane<2>(m));
    m = fmaxf(m, emu_xor_lane<4>(m));
    float s, inv;
    pow2_scale(m, s, inv);
    if (l == 0 && row < rows) scale[row] = s;
}

// ---- the product ----------------------------------------------------------
// Tile: MT x 32 tokens by 128 weight rows, four wavefronts of 32 rows each.
// The tokens' planes come straight into LDS, one stage of the tallest tile or
// two of the others at a time, double buffered with one barrier each, and serve
// all four wavefronts; each lane decodes its own row's weights in registers, in
// the matrix cores' operand order, so weights never pass through LDS and are
// decoded once per MT x 32 tokens.
typedef const __attribute__((address_space(1))) void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

//
// pf_tile<D, MT, L> is one tile with its first L of MT token fragments live
// (the others hold no tokens): L is a constant in it, because a branch on the
// live count around each matrix instruction kept them from overlapping with
// the decode (gate|up of 4096 columns at 511 tokens: 335 us with them, 320 so).
template <class D, int MT, int L>
__device__ __forceinline__ void pf_tile(const PfGemm &g, uint8_t *lds, int a0, int count, int expert, int mat, int r0)
{
    constexpr int kFrags = MT * 4 * 2;              // 1 KB fragments per stage
    constexpr int PER = D::PER;                     // stages per weight load
    constexpr int SB = PER < 4 || MT == 4 ? 1 : 2;  // stages per LDS buffer
    constexpr int kBuf = SB * kFrags * 1024;
    const int tid = threadIdx.x, lane = tid & (EMU_WAVE - 1);
    const int w = __builtin_amdgcn_readfirstlane(tid / EMU_WAVE);
    const int ks = blockIdx.y;
    const int s0 = ks * g.split, s1 = min(g.stages, s0 + g.split);
    const int kh = lane >> 5, j32 = lane & 31;
    const int row = r0 + 32 * w + j32, rowc = row < g.rows ? row : g.rows - 1;
    const uint8_t *wp = (mat ? g.w1 : g.w0) + (size_t)expert * g.expert_stride + (size_t)rowc * g.row_bytes;
    const float sw = (mat ? g.ws1 : g.ws0)[(size_t)expert * g.ws_stride + rowc];
    const uint8_t *ap = g.a.q + (size_t)(a0 / kTile) * g.a.slices * 2048 + lane * 16;

    auto stage_a = [&](int grp, int q0, int buf) { // stages q0 .. q0 + SB - 1 of span grp
#pragma unroll
        for (int q = 0; q < SB; ++q) {
            if (SB > 1 && grp * PER + q0 + q >= s1) break; // uniform
#pragma unroll
            for (int f0 = 0; f0 < L * 8; f0 += kWaves) {
                const int f = f0 + w, mt = f >> 3, j = (f >> 1) & 3, p = f & 1; // wave-uniform
                __builtin_amdgcn_global_load_lds(
                    (gvoid *)(ap + ((size_t)mt * g.a.slices + D::slice(grp, q0 + q, j)) * 2048 + p * 1024),
                    (lvoid *)(lds + buf * kBuf + (q * kFrags + f) * 1024), 16, 0, 0);
            }
        }
    };
    // A stage's sums start from zero and are added to the total at its end.
    // Against 64 bits the values' projection is off by 1.36e-7 of its norm at
    // 576 columns and 1.5e-7 at 4096 so, by 1.94e-7 and 2.1e-7 with one addition
    // per 256-column span, and by more than twice that in one chain.  (The
    // small halves' products of a stage first, its hi * hi last: 1.1e-7 and
    // 1.3e-7, but the operands spill at four fragments: 512 tokens of Qwen3-8B
    // 28.1 -> 35.1 ms; the additions per stage cost 0.2.)
    float16v sum[L], acc[L];
#pragma unroll
    for (int m = 0; m < L; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) sum[m][i] = 0.0f;

    typename D::Raw cur, nxt;
    if (s0 < s1) {
        stage_a(s0 / PER, 0, 0);
        D::load(wp, s0 / PER, kh, g.nb, cur);
    }
    int buf = 0;
    for (int grp = s0 / PER; grp * PER < s1; ++grp) { // s0 is a multiple of PER
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int st = grp * PER + q;
            if (st >= s1) break; // uniform
            if (q % SB == 0) {
                __builtin_amdgcn_s_waitcnt(0x0f70); // vmcnt(0): this wavefront's fragments are in LDS
                __syncthreads();                    // everyone's are; the other buffer's readers are done
                if (st + SB < s1) stage_a(q + SB < PER ? grp : grp + 1, q + SB < PER ? q + SB : 0, buf ^ 1);
            }
            if (q == 0 && (grp + 1) * PER < s1) {
                D::load(wp, grp + 1, kh, g.nb, nxt);
                __builtin_amdgcn_sched_barrier(0); // asked for here, not where they are first used
            }
            if (q == 0) D::settle(cur);
            const uint8_t *ab = lds + buf * kBuf + (q % SB) * kFrags * 1024 + lane * 16;
#pragma unroll
            for (int m = 0; m < L; ++m)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                half8 bh, bl;
                D::part(cur, q, kh, j, sw, bh, bl);
                half8 ah[L], al[L];
#pragma unroll
                for (int m = 0; m < L; ++m) {
                    ah[m] = *reinterpret_cast<const half8 *>(ab + (m * 8 + j * 2) * 1024);
                    al[m] = *reinterpret_cast<const half8 *>(ab + (m * 8 + j * 2 + 1) * 1024);
                }
#pragma unroll
                for (int m = 0; m < L; ++m) acc[m] = mfma(ah[m], bh, acc[m]);
#pragma unroll
                for (int m = 0; m < L; ++m) acc[m] = mfma(al[m], bh, acc[m]);
#pragma unroll
                for (int m = 0; m < L; ++m) acc[m] = mfma(ah[m], bl, acc[m]);
            }
#pragma unroll
            for (int m = 0; m < L; ++m)
#pragma unroll
                for (int i = 0; i < 16; ++i) sum[m][i] += acc[m][i];
            if (q % SB == SB - 1) buf ^= 1;
        }
        cur = nxt;
    }
    if (row >= g.rows) return;
    const float inv = 1.0f / sw; // a power of two: exact
    float *out = g.out + (size_t)ks * g.ks_stride + (size_t)mat * g.mat_stride + row;
#pragma unroll
    for (int m = 0; m < L; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int t = m * kTile + 8 * (i >> 2) + 4 * kh + (i & 3);
            if (t < count) out[(size_t)(a0 + t) * g.rows] = sum[m][i] * inv * g.a.scale[a0 + t];
        }
}

template <class D, int MT> __global__ __launch_bounds__(kThreads, 2) void pf_gemm_kernel(PfGemm g)
{
    constexpr int SB = D::PER < 4 || MT == 4 ? 1 : 2;
    __shared__ __align__(16) uint8_t lds[2 * SB * MT * 8 * 1024];
    // Consecutive tiles go to one XCD (workgroups are dealt to the eight in
    // turn), so the token tiles that share weight rows share an L2.
    const int total = gridDim.x, xcd = blockIdx.x & 7, per = total >> 3, more = total & 7;
    const int id = xcd * per + (xcd < more ? xcd : more) + (blockIdx.x >> 3);
    const int tile = id % g.tok_tiles, rt = id / g.tok_tiles;
    const int row_tiles = (g.rows + 32 * kWaves - 1) / (32 * kWaves);
    const int mat = rt / row_tiles, r0 = (rt % row_tiles) * 32 * kWaves;
    int a0 = tile * MT * kTile, count = g.n - a0, expert = 0;
    if (g.tiles) {
        if (tile >= *g.n_tiles) return; // uniform
        const int4 t = g.tiles[tile];
        expert = t.x;
        a0 = t.y;
        count = t.z;
    }
    if (MT >= 2 && count > (MT / 2) * kTile)
        pf_tile<D, MT, MT>(g, lds, a0, count, expert, mat, r0);
    else if (MT == 4 && count > kTile)
        pf_tile<D, MT, MT == 4 ? 2 : 1>(g, lds, a0, count, expert, mat, r0);
    else
        pf_tile<D, MT, 1>(g, lds, a0, count, expert, mat, r0);
}

template <class D> void gemm_launch(const PfGemm &g, int mt, dim3 grid, hipStream_t s)
{
    if (mt == 1)
        hipLaunchKernelGGL((pf_gemm_kernel<D, 1>), grid, dim3(kThreads), 0, s, g);
    else if (mt == 2)
        hipLaunchKernelGGL((pf_gemm_kernel<D, 2>), grid, dim3(kThreads), 0, s, g);
    else
        hipLaunchKernelGGL((pf_gemm_kernel<D, 4>), grid, dim3(kThreads), 0, s, g);
}

// ---- row kernels: one workgroup per token ---------------------------------
template <class F>
__global__ __launch_bounds__(kThreads) void pf_embed_kernel(const uint8_t *embed, size_t row_bytes, int hidden,
                                                            const uint32_t *prompt, int stride, int t0, int tc,
                                                            float *h, float scale)
{
    const int r = blockIdx.x, c = r / tc, t = r % tc;
    const uint8_t *row = embed + (size_t)prompt[(size_t)c * stride + t0 + t] * row_bytes;
    for (int u = threadIdx.x; u < hidden / F::BE * F::UPB; u += kThreads) {
        const int blk = u / F::UPB, sub = u % F::UPB;
        typename F::Raw raw;
        F::load(row + (size_t)blk * F::BB, sub, raw);
        float *out = h + (size_t)r * hidden + blk * F::BE;
#pragma unroll
        for (int g = 0; g < F::G; ++g) {
            const Grp gp = F::group(raw, sub, g);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float v = grp_weight_exact<F::BIAS>(gp, i);
                out[F::col(sub, g) + i] = scale != 0.0f ? v * scale : v;
            }
        }
    }
}

// The residual stream between two products: partial sums (and a MoE layer's
// weighted experts) join it, then the next products' operands: with a gain
// the RMS-normalised row; in the Gemma form also the router's and the
// experts' inputs (both from the same row, see moe_gate_kernel).  NS: the
// partial sums' slices at most (0: none); rows are whole 8-column groups.
template <int G, int NS, bool MOE> __global__ __launch_bounds__(kRowThreads) void pf_rows_kernel(PfRows a)
{
    __shared__ float red[kRowThreads / EMU_WAVE];
    const int r = blockIdx.x, W = a.width;
    float v[G][8], ss = 0.0f;
    int n = 0, pos[8];
    float wt[8], ds[8];
    if constexpr (MOE) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int id = i < a.k ? a.ids[(size_t)r * a.k + i] : -1; // ascending: the valid ones lead
            const bool ok = id >= 0 && id < a.experts;
            n += ok ? 1 : 0;
            pos[i] = ok ? a.pos_of[(size_t)r * a.k + i] : 0;
            wt[i] = ok ? a.wts[(size_t)r * a.k + i] : 0.0f;
            ds[i] = ok && a.dscale ? a.dscale[id] : 1.0f;
        }
    }
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const int c = 8 * (threadIdx.x + j * kRowThreads);
        if (c >= W) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[j][i] = 0.0f;
            continue;
        }
        ld8f(a.x + (size_t)r * W + c, v[j]);
        if constexpr (NS > 0) {
            float q[8];
            sum8<NS>(a.part + (size_t)r * W + c, a.nks, a.ks_stride, q);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[j][i] = emu_resid_add(v[j][i], q[i], a.scale);
        }
        if constexpr (MOE) {
            float e[8][8];
#pragma unroll
            for (int k = 0; k < 8; ++k) ld8f(a.contrib + (size_t)pos[k < n ? k : 0] * W + c, e[k]);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float sum = 0.0f;
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (k < n) sum = __fadd_rn(sum, __fmul_rn(a.dscale ? __fmul_rn(e[k][i], ds[k]) : e[k][i], wt[k]));
                v[j][i] = emu_resid_add(v[j][i], sum, a.moe_scale);
            }
        }
        if (a.h) {
            float4 *h = reinterpret_cast<float4 *>(a.h + (size_t)r * W + c);
            h[0] = make_float4(v[j][0], v[j][1], v[j][2], v[j][3]);
            h[1] = make_float4(v[j][4], v[j][5], v[j][6], v[j][7]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) ss = __builtin_fmaf(v[j][i], v[j][i], ss);
    }
    if (!a.gain) { // plain operands of the row
        emit_row(a.p0, r, W, red, v);
        return;
    }
    const float tot = emu_block_sum(ss, red);
    // (row * f) * gain; Gemma's router input (row * rscale) * f
    auto emit = [&](const PfPlanes &P, const float *gain, float f, bool gain_first) {
        float w[G][8];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const int c = 8 * (threadIdx.x + j * kRowThreads);
            float g[8];
            ld8f(gain + (c < W ? c : 0), g);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                w[j][i] = gain_first ? __fmul_rn(__fmul_rn(v[j][i], g[i]), f) : __fmul_rn(__fmul_rn(v[j][i], f), g[i]);
        }
        emit_row(P, r, W, red, w);
    };
    if (a.p0.q) emit(a.p0, a.gain, 1.0f / sqrtf(tot / (float)W + a.eps), false);
    if (a.rscale) { // Gemma: router input (r * rscale) * (q / sqrt(W)), expert input (r * q) * gain2
        const float q = 1.0f / sqrtf(tot / (float)W + 1e-6f);
        emit(a.p1, a.rscale, q / sqrtf((float)W), true);
        emit(a.p2, a.gain2, q, false);
    }
}

// A gate|up pair's partial sums -> the activation -> the down product's
// operands.  rows_used (expert rows): the padded row count, and src < 0 marks
// padding.  Rows wider than 8192 in more than four shares (G 4, NS 8: prompts of
// few tokens) spill 110 registers; such a launch waits for its partial sums.
template <int G, int NS>
__global__ __launch_bounds__(kRowThreads) void pf_glu_kernel(const float *part, int nks, size_t ks_stride,
                                                             size_t mat_stride, int F, int act, PfPlanes P,
                                                             const int *rows_used, const int32_t *src)
{
    __shared__ float red[kRowThreads / EMU_WAVE];
    const int r = blockIdx.x;
    if (rows_used && (r >= *rows_used || src[r] < 0)) return; // uniform
    float v[G][8];
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const int c = 8 * (threadIdx.x + j * kRowThreads);
        const float *p = part + (size_t)r * F + (c < F ? c : 0);
        float u[8];
        sum8<NS>(p, nks, ks_stride, v[j]);
        sum8<NS>(p + mat_stride, nks, ks_stride, u);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[j][i] = emu_glu(v[j][i], u[i], act);
    }
    emit_row(P, r, F, red, v);
}

// ---- heads: QK-norm, RoPE, KV append --------------------------------------
// One wavefront per (token, head of q|k|v): queries go out as hi and lo
// halves under one power of two per (token, head), or in f32 where the cache
// holds f32 values, keys and values rounded to the cache's type (the arithmetic of attn_decode_kernel's preparation).
__device__ __forceinline__ void kv_store(void *cache, int kv_f16, size_t at, float v)
{
    if (kv_f16) static_cast<__half *>(cache)[at] = __float2half_rn(v);
    else static_cast<float *>(cache)[at] = v;
}

template <int HD, int NS>
__global__ __launch_bounds__(kThreads) void pf_heads_kernel(PfHeads a)
{
    constexpr int NP = HD / 2, PPL = (NP + EMU_WAVE - 1) / EMU_WAVE;
    const int lane = threadIdx.x & (EMU_WAVE - 1);
    const int item = blockIdx.y * kWaves + threadIdx.x / EMU_WAVE;
    const int r = blockIdx.x, client = r / a.tc, t = r % a.tc;
    const int nh = a.heads + 2 * a.kv_heads, width = nh * HD;
    if (item >= nh) return;
    const int pos = (int)a.positions[client] + t;
    const float *src = a.part + (size_t)r * width + (size_t)item * HD;
    const bool is_q = item < a.heads, is_v = item >= a.heads + a.kv_heads;
    const int kvh = is_q ? 0 : is_v ? item - a.heads - a.kv_heads : item - a.heads;
    const size_t cache = ((((size_t)client * a.layers + a.layer) * a.kv_heads + kvh) * a.context + pos) * HD;
    auto at = [&](int c) {
        float q[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) q[k] = src[(k < a.nks ? k : 0) * a.ks_stride + c];
        float v = q[0];
#pragma unroll
        for (int k = 1; k < NS; ++k) v = k < a.nks ? v + q[k] : v;
        return v;
    };
    if (is_v) {
        for (int c = lane; c < HD; c += EMU_WAVE) kv_store(a.v_cache, a.kv_f16, cache + c, at(c));
        return;
    }
    const float *gain = is_q ? a.q_norm : a.k_norm;
    const float2 *rope = a.rope + (size_t)pos * NP;
    float x[PPL], y[PPL];
    int ia[PPL], ib[PPL];
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
        const int i = lane + EMU_WAVE * j, ic = i < NP ? i : NP - 1;
        ia[j] = a.interleaved ? 2 * ic : ic;
        ib[j] = a.interleaved ? 2 * ic + 1 : ic + NP;
        x[j] = at(ia[j]);
        y[j] = at(ib[j]);
        if (i < NP) {
            ss = __builtin_fmaf(x[j], x[j], ss);
            ss = __builtin_fmaf(y[j], y[j], ss);
        }
    }
    if (gain) {
        const float s = 1.0f / sqrtf(wave_sum(ss) / (float)HD + a.eps);
#pragma unroll
        for (int j = 0; j < PPL; ++j) {
            x[j] = __fmul_rn(__fmul_rn(x[j], s), gain[ia[j]]);
            y[j] = __fmul_rn(__fmul_rn(y[j], s), gain[ib[j]]);
        }
    }
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
#pragma clang fp contract(off)
        const int i = lane + EMU_WAVE * j;
        const float2 cs = rope[i < NP ? i : NP - 1];
        const float l = x[j], h = y[j];
        if (a.rope_fma) {
            x[j] = __builtin_fmaf(l, cs.x, -(h * cs.y));
            y[j] = __builtin_fmaf(l, cs.y, h * cs.x);
        } else {
            x[j] = l * cs.x - h * cs.y;
            y[j] = h * cs.x + l * cs.y;
        }
        const float m = fmaxf(fabsf(x[j]), fabsf(y[j]));
        const bool nan = !(fabsf(x[j]) <= 3.402823466e38f) || !(fabsf(y[j]) <= 3.402823466e38f);
        amax = fmaxf(amax, nan ? INFINITY : m);
    }
    if (!is_q) {
#pragma unroll
        for (int j = 0; j < PPL; ++j)
            if (lane + EMU_WAVE * j < NP) {
                kv_store(a.k_cache, a.kv_f16, cache + ia[j], x[j]);
                kv_store(a.k_cache, a.kv_f16, cache + ib[j], y[j]);
            }
        return;
    }
    _Float16 *q = a.q + ((size_t)r * a.heads + item) * 2 * HD;
    if (!a.kv_f16) { // an f32 cache is attended in f32: the queries as they are, in the same bytes
        float *q32 = reinterpret_cast<float *>(q);
#pragma unroll
        for (int j = 0; j < PPL; ++j)
            if (lane + EMU_WAVE * j < NP) {
                q32[ia[j]] = x[j];
                q32[ib[j]] = y[j];
            }
        return;
    }
    amax = emu_wave_reduce(amax, [](float p, float q) { return fmaxf(p, q); });
    const bool finite = amax <= 3.402823466e38f;
    float s, inv;
    pow2_scale(amax, s, inv);
#pragma unroll
    for (int j = 0; j < PPL; ++j)
        if (lane + EMU_WAVE * j < NP) {
            const float v[2] = {finite ? x[j] * s : 0.0f, finite ? y[j] * s : 0.0f};
            const int c[2] = {ia[j], ib[j]};
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const _Float16 hi = (_Float16)v[e];
                q[c[e]] = hi;
                q[HD + c[e]] = (_Float16)(v[e] - (float)hi);
            }
        }
    if (lane == 0) a.q_scale[(size_t)r * a.heads + item] = finite ? inv : __int_as_float(0x7fc00000);
}

// ---- attention ------------------------------------------------------------
// Flash attention over the f16 cache, one workgroup per (32*WV query rows, kv
// head, client); a query row is a (token, head of the group) pair, so grouped
// heads share the K/V tiles.  Each wavefront owns 32 query rows and works on
// the transposes, S^T = K Q^T and O^T = V^T P^T: the scores leave the matrix
// cores with a lane's column its query row, so the softmax state is one value
// per lane, and the weights are already the next product's operand (its
// position order is the one the scores' registers have; V^T is read to match).
// 511 tokens, 32 heads on 8 of 128: 40 us per layer.
// Queries and weights are hi + lo halves; the weights carry a factor 2^15 so
// that small ones keep their bits.
constexpr int kAttnPos = 64; // positions per K/V tile
constexpr int kVStride = 68; // halves per V^T row in LDS: 8-byte reads of 32 rows touch every bank once

// One query row in f32 on one wavefront, as the decode step sums it.  For
// workgroups whose tiles hold an inf or NaN (an f16 key or value that
// overflowed): in the products above it reaches rows that do not attend it
// (0 * inf) and a -inf score, which weighs 0, may become NaN (hi * inf + lo *
// inf).  Lanes hold HD / 64 neighbouring dimensions.
template <int HD>
__device__ __forceinline__ void attn_row_f32(const PfAttn &a, const _Float16 *kc, const _Float16 *vc, int kvh, int client,
                                             int t, int g, int lane)
{
    constexpr int EPL = HD / EMU_WAVE;
    const int qpos = (int)a.positions[client] + t, lo = a.window > 0 && qpos + 1 > a.window ? qpos + 1 - a.window : 0;
    const size_t tok = (size_t)client * a.tc + t;
    const int head = kvh * (a.heads / a.kv_heads) + g, c = lane * EPL;
    const _Float16 *qp = a.q + (tok * a.heads + head) * 2 * HD + c;
    const float qs = a.q_scale[tok * a.heads + head];
    float q[EPL], acc[EPL], m = -INFINITY, l = 0.0f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
        q[e] = ((float)qp[e] + (float)qp[HD + e]) * qs;
        acc[e] = 0.0f;
    }
    constexpr int NP = 8; // positions whose loads are in flight together
#pragma unroll 1
    for (int p0 = lo; p0 <= qpos; p0 += NP) {
        float k[NP][EPL], v[NP][EPL], s[NP], mn = m;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const size_t at = (size_t)(p0 + i <= qpos ? p0 + i : qpos) * HD + c;
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                k[i][e] = (float)kc[at + e];
                v[i][e] = (float)vc[at + e];
            }
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            float d = 0.0f;
#pragma unroll
            for (int e = 0; e < EPL; ++e) d = __builtin_fmaf(q[e], k[i][e], d);
            d = wave_sum(d);
            d = a.score_div > 0.0f ? d / a.score_div : d * a.score_mul;
            s[i] = p0 + i <= qpos ? d : -INFINITY;
            mn = fmaxf(mn, s[i]);
        }
        const float f = m == -INFINITY ? 0.0f : expf(m - mn);
        m = mn;
        l *= f;
#pragma unroll
        for (int e = 0; e < EPL; ++e) acc[e] *= f;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const bool in = p0 + i <= qpos;
            const float w = s[i] == -INFINITY ? 0.0f : expf(s[i] - m);
            l += w;
#pragma unroll
            for (int e = 0; e < EPL; ++e) acc[e] = in ? __builtin_fmaf(w, v[i][e], acc[e]) : acc[e];
        }
    }
    float *out = a.out + tok * (size_t)(a.heads * HD) + (size_t)head * HD + c;
#pragma unroll
    for (int e = 0; e < EPL; ++e) out[e] = acc[e] / l;
}

template <int HD, int WV>
__global__ __launch_bounds__(EMU_WAVE *WV, HD > 128 ? 1 : 2) void pf_attn_kernel(PfAttn a)
{
    constexpr int NT = EMU_WAVE * WV, NS = HD / 16, ND = HD / 32;
    constexpr int KP = kAttnPos * HD / 8 / NT;     // 16-byte pieces of K per thread
    constexpr int VP = kAttnPos / 2 * HD / 8 / NT; // (position pair, 8 dims) items of V per thread
    __shared__ __align__(16) _Float16 ks[kAttnPos * HD];
    __shared__ __align__(16) _Float16 vt[HD * kVStride];
    constexpr bool kLoLds = HD > 64; // the queries' lo halves in LDS, not registers
    __shared__ __align__(16) _Float16 q_lo[kLoLds ? WV : 1][kLoLds ? NS * 64 * 8 : 8];
    __shared__ int bad_s; // a key or value of the tiles is an inf or NaN
    const int tid = threadIdx.x, lane = tid & (EMU_WAVE - 1), w = tid / EMU_WAVE;
    const int kh = lane >> 5, j32 = lane & 31;
    const int kvh = blockIdx.y, client = blockIdx.z, G = a.heads / a.kv_heads;
    const int tile = gridDim.x - 1 - blockIdx.x; // the longest first
    const int base = (int)a.positions[client];
    const int rows = a.tc * G, r0 = tile * 32 * WV;
    const int t_last = min(r0 + 32 * WV - 1, rows - 1) / G;
    const int end = base + t_last + 1; // positions [start, end)
    const int first = base + r0 / G;
    const int start = a.window > 0 && first + 1 > a.window ? (first + 1 - a.window) / kAttnPos * kAttnPos : 0;
    const int rq = r0 + 32 * w + j32, rc = rq < rows ? rq : rows - 1;
    const int t = rc / G, head = kvh * G + rc % G;
    const size_t tok = (size_t)client * a.tc + t;
    const int qpos = base + t;
    const int qlo = a.window > 0 && qpos + 1 > a.window ? qpos + 1 - a.window : 0;
    const int w_last = base + min(r0 + 32 * w + 31, rows - 1) / G; // this wavefront's last position
    const bool w_live = r0 + 32 * w < rows;
    const int w_first = base + min(r0 + 32 * w, rows - 1) / G; // and its first
    const int w_lo = a.window > 0 && w_last + 1 > a.window ? w_last + 1 - a.window : 0; // the last row's window
    const size_t cache = (((size_t)client * a.layers + a.layer) * a.kv_heads + kvh) * (size_t)a.context * HD;
    const _Float16 *kc = static_cast<const _Float16 *>(a.k_cache) + cache;
    const _Float16 *vc = static_cast<const _Float16 *>(a.v_cache) + cache;

    half8 qh[NS], ql[kLoLds ? 1 : NS];
    {
        const _Float16 *q = a.q + (tok * a.heads + head) * 2 * HD + 8 * kh;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            qh[s] = *reinterpret_cast<const half8 *>(q + 16 * s);
            const half8 lo = *reinterpret_cast<const half8 *>(q + HD + 16 * s);
            if constexpr (kLoLds)
                *reinterpret_cast<half8 *>(&q_lo[w][(s * 64 + lane) * 8]) = lo; // read back by this lane alone
            else
                ql[s] = lo;
        }
    }
    // scores in log2 units: softmax weights are exp2 of them
    const float mul = a.score_div > 0.0f ? 1.0f / a.score_div : a.score_mul;
    const float qs = a.q_scale[tok * a.heads + head] * (mul * 1.44269504088896341f);
    float16v o[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    if (tid == 0) bad_s = 0;

    uint4 kr[KP], va[VP], vb[VP];
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    auto fetch = [&](int p0) {
#pragma unroll
        for (int i = 0; i < KP; ++i) {
            const int x = tid + i * NT, p = x / (HD / 8), g = x % (HD / 8);
            kr[i] = p0 + p < end ? *reinterpret_cast<const uint4 *>(kc + (size_t)(p0 + p) * HD + 8 * g) : zero;
        }
#pragma unroll
        for (int i = 0; i < VP; ++i) { // eight threads per 128 bytes of a row, eight position pairs
            const int x = tid + i * NT, gl = x & 7, p = ((x >> 3) & 7) + 8 * ((x / 64) % 4), g = 8 * (x / 256) + gl;
            const int p1 = p0 + 2 * p;
            va[i] = p1 < end ? *reinterpret_cast<const uint4 *>(vc + (size_t)p1 * HD + 8 * g) : zero;
            vb[i] = p1 + 1 < end ? *reinterpret_cast<const uint4 *>(vc + (size_t)(p1 + 1) * HD + 8 * g) : zero;
        }
    };
    auto any_bad = [](uint4 v) { // an f16 with all exponent bits set
        const uint32_t q[4] = {v.x, v.y, v.z, v.w};
        uint32_t b = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) b |= ((q[i] & 0x7c00u) == 0x7c00u) | ((q[i] & 0x7c000000u) == 0x7c000000u);
        return b != 0;
    };
    fetch(start);
    for (int p0 = start; p0 < end; p0 += kAttnPos) {
        __syncthreads();
        bool bad = false;
#pragma unroll
        for (int i = 0; i < KP; ++i) { // operand order: position tile, 16-dim slice, lane
            const int x = tid + i * NT, p = x / (HD / 8), g = x % (HD / 8);
            *reinterpret_cast<uint4 *>(ks + ((size_t)((p >> 5) * NS + (g >> 1)) * 64 + (g & 1) * 32 + (p & 31)) * 8) = kr[i];
            bad |= any_bad(kr[i]);
        }
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int x = tid + i * NT, gl = x & 7, p = ((x >> 3) & 7) + 8 * ((x / 64) % 4), g = 8 * (x / 256) + gl;
            const uint4 u = va[i], v = vb[i];
            bad |= any_bad(u) || any_bad(v);
            const uint32_t lo[4] = {u.x, u.y, u.z, u.w}, hi[4] = {v.x, v.y, v.z, v.w};
            uint32_t *dst = reinterpret_cast<uint32_t *>(vt) + (size_t)(8 * g) * (kVStride / 2) + p;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                dst[(2 * e) * (kVStride / 2)] = (lo[e] & 0xffffu) | (hi[e] << 16);
                dst[(2 * e + 1) * (kVStride / 2)] = (lo[e] >> 16) | (hi[e] & 0xffff0000u);
            }
        }
        if (bad) bad_s = 1;
        __syncthreads();
        if (p0 + kAttnPos < end) fetch(p0 + kAttnPos);
        if (!w_live || p0 > w_last) continue; // uniform per wavefront; the barriers above are not skipped
        float16v sc[2];
#pragma unroll
        for (int pt = 0; pt < 2; ++pt) {
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[pt][i] = 0.0f;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const half8 kf = *reinterpret_cast<const half8 *>(ks + ((size_t)(pt * NS + s) * 64 + lane) * 8);
                sc[pt] = mfma(kf, qh[s], sc[pt]);
                if constexpr (kLoLds)
                    sc[pt] = mfma(kf, *reinterpret_cast<const half8 *>(&q_lo[w][(s * 64 + lane) * 8]), sc[pt]);
                else
                    sc[pt] = mfma(kf, ql[s], sc[pt]);
            }
        }
        const bool edge = p0 + kAttnPos - 1 > w_first || p0 < w_lo; // uniform per wavefront: some are masked
        float mx = -INFINITY;
#pragma unroll
        for (int pt = 0; pt < 2; ++pt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int p = p0 + 32 * pt + 8 * (i >> 2) + 4 * kh + (i & 3);
                const float s = sc[pt][i] * qs;
                sc[pt][i] = edge && (p > qpos || p < qlo) ? -INFINITY : s;
                // a NaN score reaches the row's sum through exp2 below
                mx = fmaxf(mx, sc[pt][i]);
            }
        mx = fmaxf(mx, emu_xor_get<32>(mx));
        const float mn = fmaxf(m, mx);
        const float ms = (mn == -INFINITY ? 0.0f : mn) - 15.0f; // nothing attended yet: all weights 0
        const float rs = __builtin_amdgcn_exp2f(m - 15.0f - ms);
        float ls = 0.0f;
#pragma unroll
        for (int pt = 0; pt < 2; ++pt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                sc[pt][i] = __builtin_amdgcn_exp2f(sc[pt][i] - ms);
                ls += sc[pt][i];
            }
        l = l * rs + ls;
        m = mn;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[d][i] *= rs;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float p8[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) p8[i] = sc[c >> 1][8 * (c & 1) + i];
            half8 ph, pl;
            split8(p8, ph, pl);
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                const _Float16 *vp = vt + (size_t)(32 * d + j32) * kVStride + 16 * c + 4 * kh;
                const half4 v0 = *reinterpret_cast<const half4 *>(vp), v1 = *reinterpret_cast<const half4 *>(vp + 8);
                const half8 vf = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
                o[d] = mfma(vf, ph, o[d]);
                o[d] = mfma(vf, pl, o[d]);
            }
        }
    }
    if (bad_s) { // uniform over the workgroup; the last tile's barrier stands behind the last write
        for (int i = r0 + 32 * w; i < min(r0 + 32 * (w + 1), rows); ++i)
            attn_row_f32<HD>(a, kc, vc, kvh, client, i / G, i % G, lane);
        return;
    }
    l += emu_xor_get<32>(l);
    if (rq >= rows) return;
    const float inv = 1.0f / l;
    float *out = a.out + tok * (size_t)(a.heads * HD) + (size_t)head * HD + 4 * kh;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<float4 *>(out + 32 * d + 8 * i) =
                make_float4(o[d][4 * i] * inv, o[d][4 * i + 1] * inv, o[d][4 * i + 2] * inv, o[d][4 * i + 3] * inv);
}

// The same over an f32 cache, whose keys and values are no halves: f32 fma,
// one workgroup per (token, up to GH heads of a kv head's group, client).
// LPR lanes hold a row, four values each; a wavefront takes 16 of each 64
// positions, each lane group with a softmax state of its own, merged in LDS
// (the shape of attend_rows_kernel).  511 tokens over 32 heads on 8 of 128:
// 0.23 ms per layer, bound by the L2 reads of K and V (the f16 cache's 40 us on
// the matrix cores); fed a token per step, a prompt of 256 took 447 ms on
// Qwen3-8B, and 19 so.
template <int LPR, int GH>
__global__ __launch_bounds__(kThreads) void pf_attn_f32_kernel(PfAttn a, int hd, int nhg)
{
    constexpr int V = 4, PPI = EMU_WAVE / LPR, NI = 16 / PPI, NG = kWaves * PPI;
    __shared__ float ms[NG][GH], ls[NG][GH];
    __shared__ __align__(16) float acc_s[NG][GH][LPR * V];
    const int tid = threadIdx.x, lane = tid & (EMU_WAVE - 1), w = tid / EMU_WAVE;
    const int sub = lane / LPR, piece = lane % LPR;
    const int t = gridDim.x - 1 - blockIdx.x, client = blockIdx.z; // the longest first
    const int kvh = blockIdx.y / nhg, hg = blockIdx.y % nhg, G = a.heads / a.kv_heads;
    const int h0 = kvh * G + hg * GH, nh = min(GH, G - hg * GH);
    const size_t tok = (size_t)client * a.tc + t;
    const int qpos = (int)a.positions[client] + t, n = qpos + 1;
    const int lo = a.window > 0 && n > a.window ? n - a.window : 0;
    const size_t cache = (((size_t)client * a.layers + a.layer) * a.kv_heads + kvh) * (size_t)a.context * hd;
    const float *kc = static_cast<const float *>(a.k_cache) + cache + piece * V;
    const float *vc = static_cast<const float *>(a.v_cache) + cache + piece * V;
    float qr[GH][V];
#pragma unroll
    for (int g = 0; g < GH; ++g) {
        const int head = h0 + (g < nh ? g : 0);
        const float *q = reinterpret_cast<const float *>(a.q) + (tok * a.heads + head) * hd + piece * V;
#pragma unroll
        for (int e = 0; e < V; ++e) qr[g][e] = q[e];
    }
    float m[GH], l[GH], acc[GH][V];
#pragma unroll
    for (int g = 0; g < GH; ++g) {
        m[g] = -INFINITY;
        l[g] = 0.0f;
#pragma unroll
        for (int e = 0; e < V; ++e) acc[g][e] = 0.0f;
    }
    for (int p0 = lo + 16 * w + sub; p0 - sub < n; p0 += 16 * kWaves) { // uniform per wavefront
        float4 kr[NI], vr[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int p = p0 + i * PPI < n ? p0 + i * PPI : qpos; // in-bounds; masked below
            kr[i] = *reinterpret_cast<const float4 *>(kc + (size_t)p * hd);
            vr[i] = *reinterpret_cast<const float4 *>(vc + (size_t)p * hd);
        }
        float s[NI][GH], mx[GH];
#pragma unroll
        for (int g = 0; g < GH; ++g) mx[g] = m[g];
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int g = 0; g < GH; ++g) {
                float d = qr[g][0] * kr[i].x;
                d = __builtin_fmaf(qr[g][1], kr[i].y, d);
                d = __builtin_fmaf(qr[g][2], kr[i].z, d);
                d = __builtin_fmaf(qr[g][3], kr[i].w, d);
                d = emu_group_sum<LPR>(d);
                d = a.score_div > 0.0f ? d / a.score_div : d * a.score_mul;
                s[i][g] = p0 + i * PPI < n ? d : -INFINITY;
                mx[g] = fmaxf(mx[g], s[i][g]);
            }
#pragma unroll
        for (int g = 0; g < GH; ++g) {
            const float f = m[g] == -INFINITY ? 0.0f : expf(m[g] - mx[g]);
            m[g] = mx[g];
            l[g] *= f;
#pragma unroll
            for (int e = 0; e < V; ++e) acc[g][e] *= f;
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const float v[V] = {vr[i].x, vr[i].y, vr[i].z, vr[i].w};
            const bool in = p0 + i * PPI < n;
#pragma unroll
            for (int g = 0; g < GH; ++g) {
                const float e1 = s[i][g] == -INFINITY ? 0.0f : expf(s[i][g] - m[g]);
                l[g] += e1;
#pragma unroll
                for (int e = 0; e < V; ++e) acc[g][e] = in ? __builtin_fmaf(e1, v[e], acc[g][e]) : acc[g][e];
            }
        }
    }
    const int ng = w * PPI + sub;
#pragma unroll
    for (int g = 0; g < GH; ++g) {
        if (piece == 0) {
            ms[ng][g] = m[g];
            ls[ng][g] = l[g];
        }
#pragma unroll
        for (int e = 0; e < V; ++e) acc_s[ng][g][piece * V + e] = acc[g][e];
    }
    __syncthreads();
    for (int idx = tid; idx < nh * hd; idx += kThreads) {
        const int g = idx / hd, d = idx % hd;
        float M = -INFINITY, o = 0.0f, L = 0.0f;
#pragma unroll
        for (int i = 0; i < NG; ++i) M = fmaxf(M, ms[i][g]);
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const float f = ms[i][g] == -INFINITY ? 0.0f : expf(ms[i][g] - M);
            o = __builtin_fmaf(acc_s[i][g][d], f, o);
            L = __builtin_fmaf(ls[i][g], f, L);
        }
        a.out[tok * (size_t)(a.heads * hd) + (size_t)(h0 + g) * hd + d] = o / L;
    }
}

template <int LPR> void attn_f32_launch(const PfAttn &a, int hd, int n, hipStream_t s)
{
    const int G = a.heads / a.kv_heads, gh = G >= 3 ? 4 : G, nhg = (G + gh - 1) / gh;
    const dim3 grid((unsigned)a.tc, (unsigned)(a.kv_heads * nhg), (unsigned)n);
    if (gh == 1) hipLaunchKernelGGL((pf_attn_f32_kernel<LPR, 1>), grid, dim3(kThreads), 0, s, a, hd, nhg);
    else if (gh == 2) hipLaunchKernelGGL((pf_attn_f32_kernel<LPR, 2>), grid, dim3(kThreads), 0, s, a, hd, nhg);
    else hipLaunchKernelGGL((pf_attn_f32_kernel<LPR, 4>), grid, dim3(kThreads), 0, s, a, hd, nhg);
}

// ---- routing --------------------------------------------------------------
// Router logits (partial sums) -> routes in ascending expert id, one
// wavefront per token.
__global__ __launch_bounds__(EMU_WAVE) void pf_route_kernel(const float *part, int nks, size_t ks_stride, int experts,
                                                            int k, int32_t *junk_ids, float *junk_w, int32_t *ids,
                                                            float *weights)
{
    __shared__ float p[256];
    const int r = blockIdx.x;
    for (int e = threadIdx.x; e < experts; e += EMU_WAVE) {
        float v = part[(size_t)r * experts + e];
        for (int s = 1; s < nks; ++s) v += part[s * ks_stride + (size_t)r * experts + e];
        p[e] = v;
    }
    __syncthreads();
    emu_route_token(p, experts, k, junk_ids + (size_t)r * k, junk_w + (size_t)r * k, ids + (size_t)r * k,
                    weights + (size_t)r * k);
}

// The routes sorted by expert: every expert's rows start at a multiple of 32;
// pos_of[route] is the route's row, src[row] its token (-1: padding), tiles
// the (expert, first row, rows) of the product's token tiles.  One workgroup.
__global__ __launch_bounds__(1024) void pf_group_kernel(const int32_t *ids, int routes, int k, int experts, int tile,
                                                        int32_t *pos_of, int32_t *src, int4 *tiles, int *n_tiles,
                                                        int *rows_used)
{
    __shared__ int cnt[256], base[257], tb[257], at[256];
    const int tid = threadIdx.x;
    for (int e = tid; e < 256; e += 1024) cnt[e] = at[e] = 0;
    __syncthreads();
    for (int i = tid; i < routes; i += 1024) {
        const int e = ids[i];
        if (e >= 0 && e < experts) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    if (tid == 0) {
        int b = 0, t = 0;
        for (int e = 0; e < experts; ++e) {
            base[e] = b;
            tb[e] = t;
            b += (cnt[e] + kTile - 1) / kTile * kTile;
            t += (cnt[e] + tile - 1) / tile;
        }
        *n_tiles = t;
        *rows_used = b;
    }
    __syncthreads();
    for (int e = tid; e < experts; e += 1024) {
        for (int i = 0, t = tb[e]; i < cnt[e]; i += tile, ++t) tiles[t] = make_int4(e, base[e] + i, min(tile, cnt[e] - i), 0);
        for (int i = cnt[e]; i < (cnt[e] + kTile - 1) / kTile * kTile; ++i) src[base[e] + i] = -1;
    }
    for (int i = tid; i < routes; i += 1024) {
        const int e = ids[i];
        if (e < 0 || e >= experts) continue;
        const int p = base[e] + atomicAdd(&at[e], 1);
        pos_of[i] = p;
        src[p] = i / k;
    }
}

// Token rows of the planes in route order.
__global__ __launch_bounds__(kThreads) void pf_gather_kernel(PfPlanes from, PfPlanes to, const int *rows_used,
                                                             const int32_t *src)
{
    const int r = blockIdx.x;
    if (r >= *rows_used) return;
    const int t = src[r];
    if (t < 0) return;
    for (int g = threadIdx.x; g < 2 * from.slices; g += kThreads) {
        const uint8_t *s = from.q + plane_at(t, g, from.slices);
        uint8_t *d = to.q + plane_at(r, g, to.slices);
        const uint4 hi = *reinterpret_cast<const uint4 *>(s), lo = *reinterpret_cast<const uint4 *>(s + 1024);
        *reinterpret_cast<uint4 *>(d) = hi;
        *reinterpret_cast<uint4 *>(d + 1024) = lo;
    }
    if (threadIdx.x == 0) to.scale[r] = from.scale[t];
}

// After the chunk: every client has consumed tc more tokens and is about to
// be fed the prompt's next one.
__global__ void pf_advance_kernel(uint32_t *positions, uint32_t *steps, uint32_t *tokens, const uint32_t *prompt,
                                  int stride, int t0, int tc, int n)
{
    const int c = threadIdx.x;
    if (c >= n) return;
    positions[c] += (uint32_t)tc;
    steps[c] += (uint32_t)tc;
    tokens[c] = prompt[(size_t)c * stride + t0 + tc];
}

} // namespace

int emu_pf_slices(int cols) { return (cols + kStage - 1) / kStage * (kStage / 16); }

int emu_pf_split(int rows, int nmat, int cols, int prompt)
{
    // Shares of the columns (whole 256-column spans, at most eight shares), so
    // that short matrices and short prompts still fill the chip: the count
    // with the least rounds x (stages + a start-up of about three), plus what
    // writing and reading a share's sums costs in stages.  A CU holds two
    // workgroups of the taller tiles, four of the lowest.  Not from the number
    // of clients: a client's sums keep their order in any company.
    const int spans = (cols + 255) / 256, mt = prompt <= 32 ? 1 : prompt <= 64 ? 2 : 4;
    const int tiles = nmat * ((rows + 127) / 128) * ((prompt + 32 * mt - 1) / (32 * mt));
    const int slots = 256 * (mt == 1 ? 4 : 2);
    int best = 1;
    double best_cost = 0.0;
    for (int ks = 1; ks <= kPfMaxSplit && ks <= spans; ++ks) {
        const int rounds = (tiles * ks + slots - 1) / slots;
        const double cost = rounds * (4.0 * ((spans + ks - 1) / ks) + 3.0) + ks * (1.2e-6 * prompt * rows * nmat + 0.2);
        if (ks == 1 || cost < best_cost) {
            best = ks;
            best_cost = cost;
        }
    }
    return best;
}

int emu_pf_rowscale(emu_ctx *ctx, int encoding, const uint8_t *w, size_t row_bytes, int rows, int cols, float *scale)
{
    if (rows == 0) return EMU_OK;
    const dim3 grid((unsigned)((rows + 31) / 32)), block(kThreads);
    hipStream_t s = ctx->stream;
    auto go = [&](auto enc, int nb) {
        hipLaunchKernelGGL(pf_rowscale_kernel<decltype(enc)::value>, grid, block, 0, s, w, row_bytes, rows, nb, scale);
    };
    switch (encoding) {
    case EMU_ENC_Q6_K: go(std::integral_constant<int, EMU_ENC_Q6_K>{}, cols / 256); break;
    case EMU_ENC_Q5_K: go(std::integral_constant<int, EMU_ENC_Q5_K>{}, cols / 256); break;
    case EMU_ENC_Q2_K: go(std::integral_constant<int, EMU_ENC_Q2_K>{}, cols / 256); break;
    case EMU_ENC_Q8_0: go(std::integral_constant<int, EMU_ENC_Q8_0>{}, cols / 32); break;
    case EMU_ENC_F32: go(std::integral_constant<int, EMU_ENC_F32>{}, cols); break;
    default: return EMU_E_UNSUPPORTED;
    }
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

int emu_pf_gemm(emu_ctx *ctx, int encoding, PfGemm g, int cols, int nmat, int nks, int mt)
{
    g.stages = (cols + kStage - 1) / kStage;
    const int spans = (g.stages + 3) / 4;
    g.split = 4 * ((spans + nks - 1) / nks); // stages per share: whole spans
    if (!g.tiles) g.tok_tiles = (g.n + mt * kTile - 1) / (mt * kTile);
    const dim3 grid((unsigned)(g.tok_tiles * nmat * ((g.rows + 127) / 128)), (unsigned)nks);
    switch (encoding) {
    case EMU_ENC_Q6_K: g.nb = cols / 256; gemm_launch<PfQ6K>(g, mt, grid, ctx->stream); break;
    case EMU_ENC_Q5_K: g.nb = cols / 256; gemm_launch<PfQ5K>(g, mt, grid, ctx->stream); break;
    case EMU_ENC_Q2_K: g.nb = cols / 256; gemm_launch<PfQ2K>(g, mt, grid, ctx->stream); break;
    case EMU_ENC_Q8_0: g.nb = cols / 32; gemm_launch<PfQ8_0>(g, mt, grid, ctx->stream); break;
    case EMU_ENC_F32: g.nb = cols; gemm_launch<PfF32>(g, mt, grid, ctx->stream); break;
    default: return EMU_E_UNSUPPORTED;
    }
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

int emu_pf_embed(emu_ctx *ctx, int encoding, const uint8_t *embed, size_t row_bytes, int hidden, const uint32_t *prompt,
                 int stride, int t0, int tc, int n, float *h, float scale)
{
    const dim3 grid((unsigned)(n * tc)), block(kThreads);
    hipStream_t s = ctx->stream;
    auto go = [&](auto fmt) {
        hipLaunchKernelGGL(pf_embed_kernel<decltype(fmt)>, grid, block, 0, s, embed, row_bytes, hidden, prompt, stride, t0,
                           tc, h, scale);
    };
    switch (encoding) {
    case EMU_ENC_Q6_K: go(FmtQ6K{}); break;
    case EMU_ENC_Q5_K: go(FmtQ5K{}); break;
    case EMU_ENC_Q2_K: go(FmtQ2K{}); break;
    case EMU_ENC_Q8_0: go(FmtQ8_0{}); break;
    default: return EMU_E_UNSUPPORTED;
    }
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

template <int G, int NS> static void rows_launch(const PfRows &a, int n, hipStream_t s)
{
    if (a.contrib)
        hipLaunchKernelGGL((pf_rows_kernel<G, NS, true>), dim3((unsigned)n), dim3(kRowThreads), 0, s, a);
    else
        hipLaunchKernelGGL((pf_rows_kernel<G, NS, false>), dim3((unsigned)n), dim3(kRowThreads), 0, s, a);
}

template <int G> static void rows_launch(const PfRows &a, int n, hipStream_t s)
{
    if (!a.part) rows_launch<G, 0>(a, n, s);
    else if (a.nks <= 1) rows_launch<G, 1>(a, n, s);
    else if (a.nks <= 4) rows_launch<G, 4>(a, n, s);
    else rows_launch<G, kPfMaxSplit>(a, n, s);
}

int emu_pf_rows(emu_ctx *ctx, const PfRows &a, int n)
{
    const int per = 8 * kRowThreads;
    if (a.width <= per) rows_launch<1>(a, n, ctx->stream);
    else if (a.width <= 2 * per) rows_launch<2>(a, n, ctx->stream);
    else if (a.width <= 4 * per) rows_launch<4>(a, n, ctx->stream);
    else return EMU_E_CONFIG;
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

int emu_pf_glu(emu_ctx *ctx, const float *part, int nks, size_t ks_stride, size_t mat_stride, int ff, int act,
               const PfPlanes &p, int n, const int *rows_used, const int32_t *src)
{
    auto go = [&](auto g, auto ns) {
        hipLaunchKernelGGL((pf_glu_kernel<decltype(g)::value, decltype(ns)::value>), dim3((unsigned)n), dim3(kRowThreads),
                           0, ctx->stream, part, nks, ks_stride, mat_stride, ff, act, p, rows_used, src);
    };
    auto slices = [&](auto g) {
        if (nks <= 1) go(g, std::integral_constant<int, 1>{});
        else if (nks <= 4) go(g, std::integral_constant<int, 4>{});
        else go(g, std::integral_constant<int, kPfMaxSplit>{});
    };
    const int per = 8 * kRowThreads;
    if (ff <= per) slices(std::integral_constant<int, 1>{});
    else if (ff <= 2 * per) slices(std::integral_constant<int, 2>{});
    else if (ff <= 4 * per) slices(std::integral_constant<int, 4>{});
    else return EMU_E_CONFIG;
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

template <int HD> static void heads_launch(const PfHeads &a, dim3 grid, hipStream_t s)
{
    if (a.nks <= 1) hipLaunchKernelGGL((pf_heads_kernel<HD, 1>), grid, dim3(kThreads), 0, s, a);
    else if (a.nks <= 4) hipLaunchKernelGGL((pf_heads_kernel<HD, 4>), grid, dim3(kThreads), 0, s, a);
    else hipLaunchKernelGGL((pf_heads_kernel<HD, kPfMaxSplit>), grid, dim3(kThreads), 0, s, a);
}

int emu_pf_heads(emu_ctx *ctx, const PfHeads &a, int hd, int n)
{
    const dim3 grid((unsigned)(n * a.tc), (unsigned)((a.heads + 2 * a.kv_heads + kWaves - 1) / kWaves));
    switch (hd) {
    case 64: heads_launch<64>(a, grid, ctx->stream); break;
    case 128: heads_launch<128>(a, grid, ctx->stream); break;
    case 256: heads_launch<256>(a, grid, ctx->stream); break;
    default: return EMU_E_CONFIG;
    }
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

int emu_pf_attn(emu_ctx *ctx, const PfAttn &a, int hd, int n)
{
    if (!a.kv_f16) {
        switch (hd) {
        case 64: attn_f32_launch<16>(a, hd, n, ctx->stream); break;
        case 128: attn_f32_launch<32>(a, hd, n, ctx->stream); break;
        case 256: attn_f32_launch<64>(a, hd, n, ctx->stream); break;
        default: return EMU_E_CONFIG;
        }
        EMU_LAUNCH_CHECK(ctx);
        return EMU_OK;
    }
    constexpr int WV = 4;
    const int rows = a.tc * (a.heads / a.kv_heads);
    const dim3 grid((unsigned)((rows + 32 * WV - 1) / (32 * WV)), (unsigned)a.kv_heads, (unsigned)n);
    switch (hd) {
    case 64: hipLaunchKernelGGL((pf_attn_kernel<64, WV>), grid, dim3(EMU_WAVE * WV), 0, ctx->stream, a); break;
    case 128: hipLaunchKernelGGL((pf_attn_kernel<128, WV>), grid, dim3(EMU_WAVE * WV), 0, ctx->stream, a); break;
    case 256: hipLaunchKernelGGL((pf_attn_kernel<256, WV>), grid, dim3(EMU_WAVE * WV), 0, ctx->stream, a); break;
    default: return EMU_E_CONFIG;
    }
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

int emu_pf_route(emu_ctx *ctx, const float *part, int nks, size_t ks_stride, int experts, int k, int n,
                 int32_t *junk_ids, float *junk_w, int32_t *ids, float *weights)
{
    hipLaunchKernelGGL(pf_route_kernel, dim3((unsigned)n), dim3(EMU_WAVE), 0, ctx->stream, part, nks, ks_stride, experts,
                       k, junk_ids, junk_w, ids, weights);
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

int emu_pf_group(emu_ctx *ctx, const int32_t *ids, int n, int k, int experts, int tile, const PfGroup &g)
{
    hipLaunchKernelGGL(pf_group_kernel, dim3(1), dim3(1024), 0, ctx->stream, ids, n * k, k, experts, tile, g.pos_of,
                       g.src, g.tiles, g.n_tiles, g.rows_used);
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

int emu_pf_gather(emu_ctx *ctx, const PfPlanes &from, const PfPlanes &to, const PfGroup &g, int max_rows)
{
    hipLaunchKernelGGL(pf_gather_kernel, dim3((unsigned)max_rows), dim3(kThreads), 0, ctx->stream, from, to, g.rows_used,
                       g.src);
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

int emu_pf_advance(emu_ctx *ctx, uint32_t *positions, uint32_t *steps, uint32_t *tokens, const uint32_t *prompt,
                   int stride, int t0, int tc, int n)
{
    hipLaunchKernelGGL(pf_advance_kernel, dim3(1), dim3(64), 0, ctx->stream, positions, steps, tokens, prompt, stride, t0,
                       tc, n);
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}
