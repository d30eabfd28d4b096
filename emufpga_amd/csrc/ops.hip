// ops.hip -- RMSNorm, RoPE, cached attention, MoE router and greedy selection
// as standalone entry points.  The decode step uses fused versions of the
// same arithmetic (attn.hip, qmv.hip); these are the per-function parity
// hooks and the building blocks of the MoE path.
#include "internal.hpp"

#include <algorithm>
#include <mutex>

#include <math.h>
#include <vector>

namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ float block_sum(float v, float *red)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    float s = 0.0f;
    const int nw = (blockDim.x + 63) >> 6;
    for (int i = 0; i < nw; ++i) s += red[i];
    return s;
}

// One workgroup per row of whole, aligned float4s, up to four per thread: the
// row and its gains load at once and stay in registers, so a row waits for
// memory once.  (4 rows of 4096: 5.2 us a scalar at a time in a loop, 3.2 so;
// one of 16384: 15.8, 5.4.)
__global__ __launch_bounds__(1024) void rms_norm_row_kernel(const float *x, const float *gain, int width, float eps,
                                                            float *out)
{
    __shared__ float red[16];
    constexpr int V = 4;
    const float4 *xr = reinterpret_cast<const float4 *>(x + (size_t)blockIdx.x * width);
    float4 v[V], g[V];
    const int n = width / 4;
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int i = threadIdx.x + j * blockDim.x;
        v[j] = i < n ? xr[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        g[j] = i < n ? reinterpret_cast<const float4 *>(gain)[i] : v[j];
    }
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < V; ++j)
        s = __builtin_fmaf(v[j].w, v[j].w, __builtin_fmaf(v[j].z, v[j].z, __builtin_fmaf(v[j].y, v[j].y, __builtin_fmaf(v[j].x, v[j].x, s))));
    s = block_sum(s, red);
    const float f = 1.0f / sqrtf(s / (float)width + eps);
    float4 *yr = reinterpret_cast<float4 *>(out + (size_t)blockIdx.x * width);
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int i = threadIdx.x + j * blockDim.x;
        if (i < n)
            yr[i] = make_float4(__fmul_rn(__fmul_rn(v[j].x, f), g[j].x), __fmul_rn(__fmul_rn(v[j].y, f), g[j].y),
                                __fmul_rn(__fmul_rn(v[j].z, f), g[j].z), __fmul_rn(__fmul_rn(v[j].w, f), g[j].w));
    }
}

// Any width and alignment, one workgroup per row.
__global__ __launch_bounds__(kThreads) void rms_norm_kernel(const float *x, const float *gain,
                                                            int width, float eps, float *out)
{
    __shared__ float red[4];
    const float *xr = x + (size_t)blockIdx.x * width;
    float *yr = out + (size_t)blockIdx.x * width;
    float s = 0.0f;
    for (int i = threadIdx.x; i < width; i += kThreads) s = __builtin_fmaf(xr[i], xr[i], s);
    s = block_sum(s, red);
    const float scale = 1.0f / sqrtf(s / (float)width + eps);
    for (int i = threadIdx.x; i < width; i += kThreads) yr[i] = __fmul_rn(__fmul_rn(xr[i], scale), gain[i]);
}

// Thread per (token, head, pair).  Arithmetic kept uncontracted so a table
// built with the reference's libm gives the reference's bits:
// NEOX x' = x*cos - y*sin, y' = y*cos + x*sin (spm-qwen3-slice/src/attention.rs:22-23);
// interleaved pairs (spm-granite-moe/src/attention.rs:20-23).
__global__ __launch_bounds__(kThreads) void rope_kernel(float *x, int n_tok, int heads, int hd,
                                                        const uint32_t *positions, const float2 *table,
                                                        int table_positions, int style)
{
#pragma clang fp contract(off)
    const int half = hd / 2;
    const size_t id = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (id >= (size_t)n_tok * heads * half) return;
    const int i = (int)(id % half);
    const int h = (int)((id / half) % heads);
    const int t = (int)(id / ((size_t)half * heads));
    uint32_t pos = positions[t];
    if (pos >= (uint32_t)table_positions) pos = table_positions - 1; // host validated
    const float2 cs = table[(size_t)pos * half + i];
    float *head = x + ((size_t)t * heads + h) * hd;
    const bool halves = style != EMU_ROPE_INTERLEAVED; // NEOX and its fma form pair i with i + hd/2
    const int a = halves ? i : 2 * i;
    const int b = halves ? i + half : 2 * i + 1;
    const float l = head[a], r = head[b];
    if (style == EMU_ROPE_NEOX_FMA) {
        // spm-ops/src/attention.rs:28-30: fma(x, cos, -(y*sin)), fma(x, sin, y*cos)
        head[a] = __builtin_fmaf(l, cs.x, -(r * cs.y));
        head[b] = __builtin_fmaf(l, cs.y, r * cs.x);
    } else {
        head[a] = l * cs.x - r * cs.y;
        head[b] = r * cs.x + l * cs.y;
    }
}

// attend_cached (spm-kv/src/attend.rs:37-94), the general form: any head size
// and alignment.  One workgroup per query head; threads own positions for the
// scores, then head lanes for the weighted sum.
__global__ __launch_bounds__(kThreads) void attend_kernel(const float *q, const void *keys,
                                                          const void *values, int kv_f16,
                                                          int positions, int heads, int kv_heads,
                                                          int hd, float scale, float *scores_ws,
                                                          float *out)
{
    __shared__ float red[4];
    const int head = blockIdx.x;
    const int group = heads / kv_heads;
    const int kvh = head / group;
    const int stride = kv_heads * hd;
    const float *qh = q + (size_t)head * hd;
    float *sc = scores_ws + (size_t)head * positions;
    auto kv_at = [&](const void *base, size_t idx) -> float {
        return kv_f16 ? __half2float(static_cast<const __half *>(base)[idx])
                      : static_cast<const float *>(base)[idx];
    };
    float m = -INFINITY;
    for (int p = threadIdx.x; p < positions; p += kThreads) {
        float dot = 0.0f;
        for (int i = 0; i < hd; ++i) dot = __builtin_fmaf(qh[i], kv_at(keys, (size_t)p * stride + kvh * hd + i), dot);
        const float s = dot * scale;
        sc[p] = s;
        m = fmaxf(m, s);
    }
    // block max
    m = emu_wave_reduce(m, [](float x, float y) { return fmaxf(x, y); });
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float l = 0.0f;
    for (int p = threadIdx.x; p < positions; p += kThreads) {
        const float e = expf(sc[p] - m);
        sc[p] = e;
        l += e;
    }
    l = block_sum(l, red);
    __syncthreads();
    for (int d = threadIdx.x; d < hd; d += kThreads) {
        float acc = 0.0f;
        for (int p = 0; p < positions; ++p)
            acc = __builtin_fmaf(sc[p] / l, kv_at(values, (size_t)p * stride + kvh * hd + d), acc);
        out[(size_t)head * hd + d] = acc;
    }
}

// attend_cached for whole 16-byte pieces: one workgroup per (chunk of
// positions, kv head, up to GH query heads of its group), so that a long
// prefix fills the chip (the general form has one workgroup per head: 32
// heads over 4096 positions of 8 x 128 f16 took 1520 us; this one and its
// merge 8).  LPR lanes hold a row, one 16-byte piece each, and a wavefront
// 64 / LPR rows, so every load reads whole rows; a wavefront takes 16 of each
// 64 positions and has all their K and V pieces in flight at once.  Each lane
// group keeps its own softmax state (largest score, sum, weighted values);
// they meet in LDS at the end, and the chunks' in attend_merge_kernel.
constexpr int kAttendBlock = 64;

template <class T, int LPR, int GH>
__global__ __launch_bounds__(kThreads) void attend_rows_kernel(const float *q, const T *keys, const T *values,
                                                               int positions, int heads, int kv_heads, int hd,
                                                               int chunk, int nhg, float scale, float *partial,
                                                               float *out)
{
    constexpr int V = 16 / sizeof(T), PPI = EMU_WAVE / LPR, NI = 16 / PPI, NG = 4 * PPI;
    __shared__ float ms[NG][GH], ls[NG][GH];
    __shared__ __align__(16) float acc_s[NG][GH][LPR * V];
    const int tid = threadIdx.x, lane = tid & (EMU_WAVE - 1), w = tid / EMU_WAVE;
    const int sub = lane / LPR, piece = lane % LPR;
    const int kvh = blockIdx.y / nhg, hg = blockIdx.y % nhg, group = heads / kv_heads;
    const int h0 = kvh * group + hg * GH, nh = min(GH, group - hg * GH);
    const bool live = piece * V < hd;
    const size_t stride = (size_t)kv_heads * hd, col = (size_t)kvh * hd + (live ? piece * V : 0);
    float qr[GH][V];
#pragma unroll
    for (int g = 0; g < GH; ++g) {
        const float *p = q + (size_t)(h0 + (g < nh ? g : 0)) * hd + (live ? piece * V : 0);
#pragma unroll
        for (int e = 0; e < V; e += 4) {
            const float4 f = *reinterpret_cast<const float4 *>(p + e);
            qr[g][e] = live ? f.x : 0.0f;
            qr[g][e + 1] = live ? f.y : 0.0f;
            qr[g][e + 2] = live ? f.z : 0.0f;
            qr[g][e + 3] = live ? f.w : 0.0f;
        }
    }
    auto unpack = [](uint4 raw, float (&f)[V]) {
        T t[V];
        __builtin_memcpy(t, &raw, 16);
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = (float)t[e];
    };
    float m[GH], l[GH], acc[GH][V];
#pragma unroll
    for (int g = 0; g < GH; ++g) {
        m[g] = -INFINITY;
        l[g] = 0.0f;
#pragma unroll
        for (int e = 0; e < V; ++e) acc[g][e] = 0.0f;
    }
    const int p_end = min(positions, (int)(blockIdx.x + 1) * chunk);
    for (int p0 = blockIdx.x * chunk + 16 * w + sub; p0 - sub < p_end; p0 += kAttendBlock) { // uniform per wavefront
        uint4 kr[NI], vr[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int p = p0 + i * PPI < p_end ? p0 + i * PPI : p_end - 1; // in-bounds; masked below
            kr[i] = *reinterpret_cast<const uint4 *>(keys + (size_t)p * stride + col);
            vr[i] = *reinterpret_cast<const uint4 *>(values + (size_t)p * stride + col);
        }
        float s[NI][GH], mx[GH];
#pragma unroll
        for (int g = 0; g < GH; ++g) mx[g] = m[g];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            float k[V];
            unpack(kr[i], k);
#pragma unroll
            for (int g = 0; g < GH; ++g) {
                float d = 0.0f; // idle lanes hold zero queries over another piece's key: select, 0 * inf is NaN
#pragma unroll
                for (int e = 0; e < V; ++e) d = __builtin_fmaf(qr[g][e], k[e], d);
                d = emu_group_sum<LPR>(live ? d : 0.0f) * scale;
                s[i][g] = p0 + i * PPI < p_end ? d : -INFINITY;
                mx[g] = fmaxf(mx[g], s[i][g]);
            }
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
            float v[V];
            unpack(vr[i], v);
            const bool in = p0 + i * PPI < p_end;
#pragma unroll
            for (int g = 0; g < GH; ++g) {
                // a score of -inf weighs 0 (also where nothing larger was seen yet)
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
        float M = -INFINITY;
#pragma unroll
        for (int i = 0; i < NG; ++i) M = fmaxf(M, ms[i][g]);
        float o = 0.0f, L = 0.0f;
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const float f = ms[i][g] == -INFINITY ? 0.0f : expf(ms[i][g] - M);
            o = __builtin_fmaf(acc_s[i][g][d], f, o); // a group without a position: 0 * 0
            L = __builtin_fmaf(ls[i][g], f, L);
        }
        if (partial) {
            float *pp = partial + ((size_t)(h0 + g) * gridDim.x + blockIdx.x) * (hd + 2);
            pp[d] = o;
            if (d == 0) {
                pp[hd] = M;
                pp[hd + 1] = L;
            }
        } else {
            out[(size_t)(h0 + g) * hd + d] = o / L;
        }
    }
}

// The chunks of one query head: sum of o_c * exp(m_c - M) over the same of
// l_c.  Thread (i, d): head lane d of every (kThreads / DP)-th chunk, DP the
// head size's power of two.
constexpr int kAttendMaxChunks = 256;
__global__ __launch_bounds__(kThreads) void attend_merge_kernel(const float *partial, int chunks, int hd, int dp,
                                                                float *out)
{
    __shared__ float wt[kAttendMaxChunks], red[4], sums[kThreads];
    const int tid = threadIdx.x, head = blockIdx.x;
    const float *pp = partial + (size_t)head * chunks * (hd + 2);
    const bool have = tid < chunks;
    const float mc = have ? pp[(size_t)tid * (hd + 2) + hd] : -INFINITY, lc = have ? pp[(size_t)tid * (hd + 2) + hd + 1] : 0.0f;
    float M = emu_wave_reduce(mc, [](float x, float y) { return fmaxf(x, y); });
    if ((tid & 63) == 0) red[tid >> 6] = M;
    __syncthreads();
    M = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float f = mc == -INFINITY ? 0.0f : expf(mc - M);
    wt[tid] = f;
    const float L = block_sum(lc * f, red);
    __syncthreads();
    const int rows = kThreads / dp, i0 = tid / dp, d = tid % dp;
    float o = 0.0f;
    if (d < hd) {
#pragma unroll 8
        for (int c = i0; c < chunks; c += rows) o = __builtin_fmaf(pp[(size_t)c * (hd + 2) + d], wt[c], o);
    }
    sums[tid] = o;
    __syncthreads();
    if (tid < hd) {
        for (int i = 1; i < rows; ++i) o += sums[i * dp + tid];
        out[(size_t)head * hd + tid] = o / L;
    }
}

// Rust f32::total_cmp key, as an order-preserving unsigned.
__device__ __forceinline__ uint32_t total_key_u(float f)
{
    int32_t i = __float_as_int(f);
    i ^= (int32_t)(((uint32_t)(i >> 31)) >> 1);
    return (uint32_t)i ^ 0x80000000u;
}

// Reduction key: tie_last == 0 -> greatest total-order value, lowest index;
// tie_last == 1 -> greatest value with -0 == +0, highest index.
__device__ __forceinline__ uint64_t select_key(float v, uint32_t idx, int tie_last)
{
    if (tie_last) {
        if (v == 0.0f) v = 0.0f;
        return ((uint64_t)total_key_u(v) << 32) | idx;
    }
    return ((uint64_t)total_key_u(v) << 32) | (0xffffffffu - idx);
}

__device__ __forceinline__ uint32_t key_index(uint64_t k, int tie_last)
{
    const uint32_t lo = (uint32_t)k;
    return tie_last ? lo : 0xffffffffu - lo;
}

__device__ __forceinline__ uint64_t wave_max_u64(uint64_t k)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const uint64_t o = __shfl_xor(k, off, 64);
        k = o > k ? o : k;
    }
    return k;
}

// One workgroup per (chunk of a row, row); with one chunk per row its index,
// else the chunk's key for argmax_pick_kernel.  float4s from the chunk's first
// aligned element on, four of them in flight.
__global__ __launch_bounds__(1024) void argmax_kernel(const float *x, int width, int chunk, int tie_last, uint64_t *keys,
                                                      int32_t *out)
{
    __shared__ uint64_t red[16];
    const int begin = blockIdx.x * chunk, end = min(width, begin + chunk), tid = threadIdx.x;
    const float *xr = x + (size_t)blockIdx.y * width;
    uint64_t best = 0;
    auto take = [&](float v, int i) {
        const uint64_t k = select_key(v, (uint32_t)i, tie_last);
        best = k > best ? k : best;
    };
    const int lead = min((int)(-(reinterpret_cast<uintptr_t>(xr + begin) / 4) & 3), end - begin);
    const int first = begin + lead, whole = first + (end - first) / 4 * 4;
    if (tid < lead) take(xr[begin + tid], begin + tid);
#pragma unroll 4
    for (int i = first + 4 * tid; i < whole; i += 4 * blockDim.x) {
        const float4 v = *reinterpret_cast<const float4 *>(xr + i);
        take(v.x, i);
        take(v.y, i + 1);
        take(v.z, i + 2);
        take(v.w, i + 3);
    }
    if (whole + tid < end) take(xr[whole + tid], whole + tid);
    best = wave_max_u64(best);
    if (blockDim.x > EMU_WAVE) { // uniform
        if ((tid & 63) == 0) red[tid >> 6] = best;
        __syncthreads();
        if (tid >= EMU_WAVE) return;
        best = wave_max_u64(tid < (int)(blockDim.x >> 6) ? red[tid] : 0);
    }
    if (tid != 0) return;
    if (keys) keys[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = best;
    else out[blockIdx.y] = (int32_t)key_index(best, tie_last);
}

__global__ __launch_bounds__(64) void argmax_pick_kernel(const uint64_t *keys, int chunks, int tie_last, int32_t *out)
{
    const uint64_t k = wave_max_u64((int)threadIdx.x < chunks ? keys[(size_t)blockIdx.x * chunks + threadIdx.x] : 0);
    if (threadIdx.x == 0) out[blockIdx.x] = (int32_t)key_index(k, tie_last);
}

// moe::route: one wavefront per token; n_experts <= 256, k <= 64.
__global__ __launch_bounds__(64) void route_kernel(const float *logits, int n_experts, int k,
                                                   int32_t *ids, float *weights)
{
    const int t = blockIdx.x;
    emu_route_token(logits + (size_t)t * n_experts, n_experts, k, ids + (size_t)t * k, weights + (size_t)t * k);
}

} // namespace

extern "C" int emu_rms_norm(emu_ctx *ctx, const float *d_x, const float *d_gain, uint32_t n_rows,
                            uint32_t width, float eps, float *d_out)
{
    if (!ctx || !d_x || !d_gain || !d_out || width == 0) return EMU_E_ARG;
    if (n_rows == 0) return EMU_OK;
    const auto aligned = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    // The register form where rows are few enough for the chip to wait on each
    // (8 rows of 4096: 5.8 -> 3.7 us, 512: 7.1 -> 6.0); beyond, the narrower
    // workgroups (2048 rows of 2816: 11.2 us, 13.5 with rows in registers).
    if (n_rows <= 512 && width % 4 == 0 && width <= 16384 && aligned(d_x) && aligned(d_gain) && aligned(d_out)) {
        const unsigned threads = std::min(1024u, (width / 4 + 63) / 64 * 64);
        hipLaunchKernelGGL(rms_norm_row_kernel, dim3(n_rows), dim3(threads), 0, ctx->stream, d_x, d_gain, (int)width, eps,
                           d_out);
        EMU_LAUNCH_CHECK(ctx);
        return EMU_OK;
    }
    hipLaunchKernelGGL(rms_norm_kernel, dim3(n_rows), dim3(kThreads), 0, ctx->stream, d_x, d_gain,
                       (int)width, eps, d_out);
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

// Angles as spm-qwen3-slice/src/attention.rs:14-19 computes them:
// angle = pos / theta^(2i/d), in f32 with the host libm.
int emu_build_rope_table(uint32_t positions, uint32_t head_dim, float theta, int fma_form,
                         std::vector<float> &table)
{
    const uint32_t half = head_dim / 2;
    table.resize((size_t)positions * half * 2);
    for (uint32_t pos = 0; pos < positions; ++pos) {
        for (uint32_t i = 0; i < half; ++i) {
            float angle;
            if (fma_form) {
                // spm-ops/src/attention.rs:24-27: base^(-2i/d) * pos
                volatile float e = -2.0f * (float)i;
                volatile float ex = e / (float)head_dim;
                volatile float pw = powf(theta, ex);
                angle = pw * (float)pos;
            } else {
                volatile float e = 2.0f * (float)i;
                volatile float ex = e / (float)head_dim;
                volatile float pw = powf(theta, ex);
                angle = (float)pos / pw;
            }
            table[((size_t)pos * half + i) * 2] = cosf(angle);
            table[((size_t)pos * half + i) * 2 + 1] = sinf(angle);
        }
    }
    return EMU_OK;
}

extern "C" int emu_rope_table(emu_ctx *ctx, uint32_t positions, uint32_t head_dim, float theta,
                              float *d_table)
{
    if (!ctx || !d_table || head_dim == 0 || head_dim % 2) return EMU_E_ARG;
    if (positions > 65536) return EMU_E_CONFIG; // positions fit u16 (attention.rs:14-16)
    std::vector<float> t;
    emu_build_rope_table(positions, head_dim, theta, 0, t);
    return emu_memcpy_htod(ctx, d_table, t.data(), t.size() * sizeof(float));
}

extern "C" int emu_rope_table_style(emu_ctx *ctx, int style, uint32_t positions, uint32_t head_dim, float theta,
                                    float *d_table)
{
    if (!ctx || !d_table || head_dim == 0 || head_dim % 2) return EMU_E_ARG;
    if (style != EMU_ROPE_NEOX && style != EMU_ROPE_INTERLEAVED && style != EMU_ROPE_NEOX_FMA) return EMU_E_ARG;
    if (positions > 65536) return EMU_E_CONFIG;
    std::vector<float> t;
    emu_build_rope_table(positions, head_dim, theta, style == EMU_ROPE_NEOX_FMA, t);
    return emu_memcpy_htod(ctx, d_table, t.data(), t.size() * sizeof(float));
}

extern "C" int emu_rope(emu_ctx *ctx, float *d_x, uint32_t n_tok, uint32_t heads, uint32_t head_dim,
                        const uint32_t *d_positions, const float *d_table, uint32_t table_positions,
                        int style)
{
    if (!ctx || !d_x || !d_positions || !d_table || head_dim % 2 || table_positions == 0) return EMU_E_ARG;
    if (style != EMU_ROPE_NEOX && style != EMU_ROPE_INTERLEAVED && style != EMU_ROPE_NEOX_FMA) return EMU_E_ARG;
    const size_t n = (size_t)n_tok * heads * (head_dim / 2);
    if (n == 0) return EMU_OK;
    hipLaunchKernelGGL(rope_kernel, dim3((unsigned)((n + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                       ctx->stream, d_x, (int)n_tok, (int)heads, (int)head_dim, d_positions,
                       reinterpret_cast<const float2 *>(d_table), (int)table_positions, style);
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

// ---- attend_cached ----------------------------------------------------------
// The scratch of emu_attend_cached_noalloc is this file-scope device array.
// Each device holds its own copy, at its own address, for the life of the
// process; host code reaches it only through that address (the array's name
// is not a device address on the host).  Every call on a device shares the
// device's copy, so calls that overlap on one device race; the kernels write
// everything they read, so nothing needs clearing between calls.
constexpr size_t kAttendScratchFloats = kEmuScratchFloats; // 4 MiB
static __device__ __align__(256) float scratch[kAttendScratchFloats];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float *g_scratch[kMaxDevices] = {};

// Whether the context's stream is being captured.  A graph outlives the call
// and may be replayed beside the context's own, on another stream or after its
// end: such a call leaves the context's scratch alone and runs in one launch.
bool capturing(emu_ctx *ctx)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(ctx->stream, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
}

// How a call runs, from its arguments (so the two entry points agree) and
// whether it may be split over chunks that meet in scratch.
struct AttendPlan {
    bool rows;           // attend_rows_kernel, else the general form
    int chunk, chunks;   // positions per workgroup, and how many
    int gh, nhg;         // query heads per workgroup, groups of them per kv head
    int lpr;             // lanes per row
    size_t floats;       // scratch
};

AttendPlan attend_plan(const float *q, const void *k, const void *v, int kv_f16, int positions, int heads, int kv_heads,
                       int hd, bool split)
{
    AttendPlan p{};
    const int per = kv_f16 ? 8 : 4; // values per 16-byte piece
    const auto aligned = [](const void *x) { return reinterpret_cast<uintptr_t>(x) % 16 == 0; };
    // Whole pieces, at most one per lane, a merge thread per head lane; the
    // grid's second dimension holds the head groups.
    p.rows = hd % per == 0 && hd % 4 == 0 && hd <= 64 * per && hd <= kThreads && aligned(q) && aligned(k) && aligned(v) &&
             heads <= 65535 && positions <= 1 << 30;
    if (!p.rows) {
        p.floats = (size_t)heads * positions; // its scores
        return p;
    }
    const int group = heads / kv_heads;
    p.gh = group >= 3 ? 4 : group;
    p.nhg = (group + p.gh - 1) / p.gh;
    p.lpr = 8;
    while (p.lpr * per < hd) p.lpr *= 2;
    // One 64-position block per workgroup while that makes no more than about
    // four workgroups per CU; longer prefixes take longer chunks.  Up to 192
    // positions in one workgroup cost no more than the second launch (32
    // heads on 8 of 128, f16: 6.5 us at 64 positions, 8.5 at 128, 12.7 at 256
    // against 10.2 in two launches; 9 on 3 of 64: 5.2, 6.3 and 8.5 against 8.7).
    int most = std::min(kAttendMaxChunks, std::max(1, 1024 / (kv_heads * p.nhg)));
    most = (int)std::min<size_t>((size_t)most, kAttendScratchFloats / ((size_t)heads * (hd + 2)));
    most = positions <= 3 * kAttendBlock || !split ? 1 : std::max(1, most);
    const int blocks = (positions + kAttendBlock - 1) / kAttendBlock;
    p.chunk = (blocks + most - 1) / most * kAttendBlock;
    p.chunks = (positions + p.chunk - 1) / p.chunk;
    p.floats = p.chunks > 1 ? (size_t)heads * p.chunks * (hd + 2) : 0;
    return p;
}

struct AttendCall {
    const float *q;
    const void *k, *v;
    int positions, heads, kv_heads, hd;
    float scale;
    float *ws, *out;
};

template <class T, int LPR, int GH> void attend_go(const AttendPlan &p, const AttendCall &c, hipStream_t s)
{
    hipLaunchKernelGGL((attend_rows_kernel<T, LPR, GH>), dim3((unsigned)p.chunks, (unsigned)(c.kv_heads * p.nhg)),
                       dim3(kThreads), 0, s, c.q, static_cast<const T *>(c.k), static_cast<const T *>(c.v), c.positions,
                       c.heads, c.kv_heads, c.hd, p.chunk, p.nhg, c.scale, p.chunks > 1 ? c.ws : nullptr, c.out);
}
template <class T, int LPR> void attend_go(const AttendPlan &p, const AttendCall &c, hipStream_t s)
{
    if (p.gh == 1) attend_go<T, LPR, 1>(p, c, s);
    else if (p.gh == 2) attend_go<T, LPR, 2>(p, c, s);
    else attend_go<T, LPR, 4>(p, c, s);
}
template <class T> void attend_go(const AttendPlan &p, const AttendCall &c, hipStream_t s)
{
    if (p.lpr == 8) attend_go<T, 8>(p, c, s);
    else if (p.lpr == 16) attend_go<T, 16>(p, c, s);
    else if (p.lpr == 32) attend_go<T, 32>(p, c, s);
    else attend_go<T, 64>(p, c, s);
}

int attend(emu_ctx *ctx, const AttendPlan &p, const AttendCall &c, int kv_f16)
{
    if (!p.rows) {
        hipLaunchKernelGGL(attend_kernel, dim3(c.heads), dim3(kThreads), 0, ctx->stream, c.q, c.k, c.v, kv_f16,
                           c.positions, c.heads, c.kv_heads, c.hd, c.scale, c.ws, c.out);
        EMU_LAUNCH_CHECK(ctx);
        return EMU_OK;
    }
    if (kv_f16) attend_go<_Float16>(p, c, ctx->stream);
    else attend_go<float>(p, c, ctx->stream);
    EMU_LAUNCH_CHECK(ctx);
    if (p.chunks > 1) {
        int dp = 1;
        while (dp < c.hd) dp *= 2;
        hipLaunchKernelGGL(attend_merge_kernel, dim3(c.heads), dim3(kThreads), 0, ctx->stream, c.ws, p.chunks, c.hd, dp,
                           c.out);
        EMU_LAUNCH_CHECK(ctx);
    }
    return EMU_OK;
}
} // namespace

int emu_ops_device_init(emu_ctx *ctx)
{
    if (ctx->device < 0 || ctx->device >= kMaxDevices) return EMU_E_ARG;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[ctx->device]) return EMU_OK;
    // the context's device is current (emu_ctx_create set it)
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) return emu_hip_fail(ctx, e != hipSuccess ? e : hipErrorInvalidSymbol,
                                                     "hipGetSymbolAddress(scratch)");
    g_scratch[ctx->device] = static_cast<float *>(ptr);
    return EMU_OK;
}

extern "C" int emu_attend_cached(emu_ctx *ctx, const float *d_q, const void *d_keys, const void *d_values,
                                 int kv_f16, uint32_t positions, uint32_t heads, uint32_t kv_heads,
                                 uint32_t head_dim, float scale, float *d_out)
{
    if (!ctx || !d_q || !d_keys || !d_values || !d_out || head_dim == 0) return EMU_E_ARG;
    if (kv_heads == 0 || heads % kv_heads != 0) return EMU_E_CONFIG; // attend.rs:82-85
    if (positions == 0 || heads == 0) return EMU_OK;
    const AttendPlan p = attend_plan(d_q, d_keys, d_values, kv_f16, (int)positions, (int)heads, (int)kv_heads,
                                     (int)head_dim, !capturing(ctx));
    AttendCall c{d_q, d_keys, d_values, (int)positions, (int)heads, (int)kv_heads, (int)head_dim, scale, nullptr, d_out};
    if (p.rows) { // at most kAttendScratchFloats
        c.ws = ctx->scratch;
        return attend(ctx, p, c, kv_f16);
    }
    void *ws = nullptr;
    int st = emu_malloc(ctx, sizeof(float) * p.floats, &ws);
    if (st != EMU_OK) return st;
    c.ws = static_cast<float *>(ws);
    st = attend(ctx, p, c, kv_f16);
    emu_free(ctx, ws);
    return st;
}

extern "C" int emu_attend_cached_noalloc(emu_ctx *ctx, const float *d_q, const void *d_keys, const void *d_values,
                                         int kv_f16, uint32_t positions, uint32_t heads, uint32_t kv_heads,
                                         uint32_t head_dim, float scale, float *d_out)
{
    if (!ctx || !d_q || !d_keys || !d_values || !d_out || head_dim == 0) return EMU_E_ARG;
    if (kv_heads == 0 || heads % kv_heads != 0) return EMU_E_CONFIG; // attend.rs:82-85
    if (positions == 0 || heads == 0) return EMU_OK;
    if ((uint64_t)heads * positions > kAttendScratchFloats) {
        snprintf(ctx->last_error, sizeof ctx->last_error,
                 "emu_attend_cached_noalloc: heads * positions = %llu exceeds its scratch of %zu scores",
                 (unsigned long long)heads * positions, kAttendScratchFloats);
        return EMU_E_CONFIG;
    }
    float *ws = ctx->device >= 0 && ctx->device < kMaxDevices ? g_scratch[ctx->device] : nullptr;
    if (!ws) return EMU_E_ARG; // no context set this device up
    const AttendPlan p = attend_plan(d_q, d_keys, d_values, kv_f16, (int)positions, (int)heads, (int)kv_heads,
                                     (int)head_dim, true);
    const AttendCall c{d_q, d_keys, d_values, (int)positions, (int)heads, (int)kv_heads, (int)head_dim, scale, ws, d_out};
    return attend(ctx, p, c, kv_f16);
}

extern "C" int emu_route(emu_ctx *ctx, const float *d_logits, uint32_t n_tok, uint32_t n_experts,
                         uint32_t k, int32_t *d_ids, float *d_weights)
{
    if (!ctx || !d_logits || !d_ids || !d_weights) return EMU_E_ARG;
    if (n_experts == 0 || n_experts > 256 || k == 0 || k > n_experts || k > 64) return EMU_E_CONFIG;
    if (n_tok == 0) return EMU_OK;
    hipLaunchKernelGGL(route_kernel, dim3(n_tok), dim3(64), 0, ctx->stream, d_logits, (int)n_experts,
                       (int)k, d_ids, d_weights);
    EMU_LAUNCH_CHECK(ctx);
    return EMU_OK;
}

extern "C" int emu_argmax(emu_ctx *ctx, const float *d_x, uint32_t n_rows, uint32_t width, int tie_last,
                          int32_t *d_out)
{
    if (!ctx || !d_x || !d_out || width == 0) return EMU_E_ARG;
    if (n_rows == 0) return EMU_OK;
    // Long rows, where few, are cut into up to 64 chunks of 4096 or more, whose
    // keys a second launch picks from (4 rows of 151936: 24.8 us with one
    // workgroup and scalar loads a row, 6.4 so; one of 262144: 38.3, 6.4).  Up to
    // 49152 a row takes no longer whole than the two launches (32767: 4.9
    // against 6.5), beyond 32 rows the second launch costs what the chunks save
    // (33 rows of 49155: 6.4 whole).  The keys go to the context's scratch; a
    // captured call takes whole rows.
    const uint32_t rows = std::min(n_rows, 65535u); // a grid's second dimension; the rest in further launches
    int chunks = 1;
    if (n_rows <= 32 && width > 49152 && !capturing(ctx)) chunks = (int)std::min(64u, (width + 4095) / 4096);
    const int chunk = (int)((((size_t)width + chunks - 1) / chunks + 3) / 4 * 4);
    chunks = (int)(((size_t)width + chunk - 1) / chunk);
    uint64_t *keys = chunks > 1 ? reinterpret_cast<uint64_t *>(ctx->scratch) : nullptr;
    // Four float4s per thread (1000 rows of 1000 took 9.1 us at 1024 threads
    // whatever the width, 3.7 so).
    const unsigned threads = (unsigned)std::min(1024, std::max(1, (chunk + 1023) / 1024) * EMU_WAVE);
    for (uint32_t r = 0; r < n_rows; r += rows) {
        const uint32_t n = std::min(rows, n_rows - r);
        hipLaunchKernelGGL(argmax_kernel, dim3((unsigned)chunks, n), dim3(threads), 0, ctx->stream, d_x + (size_t)r * width,
                           (int)width, chunk, tie_last ? 1 : 0, keys, d_out + r);
        EMU_LAUNCH_CHECK(ctx);
    }
    if (keys) {
        hipLaunchKernelGGL(argmax_pick_kernel, dim3(n_rows), dim3(64), 0, ctx->stream, keys, chunks, tie_last ? 1 : 0,
                           d_out);
        EMU_LAUNCH_CHECK(ctx);
    }
    return EMU_OK;
}

namespace {

// Reads every 16-byte word of the buffer once (non-temporal, as the decode
// step's weight loads), grid-stride with one load in flight per lane, so the
// grid's front is one contiguous region moving through the buffer: on this
// part that reads a 2 GiB buffer at 7.2 TB/s, against 6.0 TB/s with four
// loads per lane a grid-stride apart (four pages open per lane).  The xor of
// the words is stored only if it equals a value no input makes likely, so
// the loads are not dropped.
__global__ __launch_bounds__(256) void hbm_read_kernel(const uint8_t *buf, size_t words, uint32_t *sink)
{
    uint32_t acc = 0;
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < words; i += stride) {
        const uint4 a = ldnt16(buf + 16 * i);
        acc ^= a.x ^ a.y ^ a.z ^ a.w;
    }
    if (acc == 0x9e3779b9u) sink[0] = acc;
}

} // namespace

extern "C" int emu_hbm_read_rate(emu_ctx *ctx, const void *d_buf, size_t bytes, uint32_t passes, float *gbs)
{
    if (!ctx || !d_buf || !gbs || passes == 0 || bytes < 16) return EMU_E_ARG;
    const size_t words = bytes / 16;
    const unsigned grid = (unsigned)(ctx->cus > 0 ? ctx->cus * 8 : 2048);
    uint32_t *sink = const_cast<uint32_t *>(static_cast<const uint32_t *>(d_buf));
    const uint8_t *buf = static_cast<const uint8_t *>(d_buf);
    hipLaunchKernelGGL(hbm_read_kernel, dim3(grid), dim3(256), 0, ctx->stream, buf, words, sink); // warm
    EMU_LAUNCH_CHECK(ctx);
    int st;
    if ((st = emu_event_record(ctx, 11)) != EMU_OK) return st;
    for (uint32_t p = 0; p < passes; ++p)
        hipLaunchKernelGGL(hbm_read_kernel, dim3(grid), dim3(256), 0, ctx->stream, buf, words, sink);
    EMU_LAUNCH_CHECK(ctx);
    if ((st = emu_event_record(ctx, 12)) != EMU_OK) return st;
    float ms = 0.0f;
    if ((st = emu_event_elapsed(ctx, 11, 12, &ms)) != EMU_OK) return st;
    *gbs = ms > 0.0f ? (float)((double)words * 16.0 * passes / (ms * 1e-3) / 1e9) : 0.0f;
    return EMU_OK;
}
