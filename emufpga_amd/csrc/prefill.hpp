// prefill.hpp -- launchers of prefill.hip, for the prompt pass in model.hip.
#pragma once

#include "internal.hpp"

// A product's left operand: hi and lo half planes of rows x (16 * slices)
// columns in 32-row tiles, and per row the factor that undoes its scale.
struct PfPlanes {
    uint8_t *q;
    float *scale;
    int slices;
};
// 16-column slices of a row of `cols` columns, padded to whole stages.
int emu_pf_slices(int cols);
inline size_t emu_pf_plane_bytes(size_t rows, int slices) { return (rows + 127) / 128 * 128 * (size_t)slices * 64; }

// out[ks][mat][row][weight row] = sum over the ks-th share of the columns.
struct PfGemm {
    PfPlanes a;
    int n; // rows of a (dense form)
    const uint8_t *w0, *w1;
    const float *ws0, *ws1; // the weight rows' scales
    size_t row_bytes, expert_stride, ws_stride;
    int rows, nb, stages, split, tok_tiles;
    const int4 *tiles; // expert form: (expert, first row, rows)
    const int *n_tiles;
    float *out;
    size_t ks_stride, mat_stride;
};
// Shares of the columns a product's launch is cut into.
int emu_pf_split(int rows, int nmat, int cols, int prompt);
int emu_pf_rowscale(emu_ctx *ctx, int encoding, const uint8_t *w, size_t row_bytes, int rows, int cols, float *scale);
int emu_pf_gemm(emu_ctx *ctx, int encoding, PfGemm g, int cols, int nmat, int nks, int mt);

int emu_pf_embed(emu_ctx *ctx, int encoding, const uint8_t *embed, size_t row_bytes, int hidden, const uint32_t *prompt,
                 int stride, int t0, int tc, int n, float *h, float scale);

struct PfRows {
    const float *x; // rows x width
    float *h;       // the updated rows (null: not stored)
    int width;
    const float *part; // partial sums joining the row as x + sum * scale (null: none)
    int nks;
    size_t ks_stride;
    float scale;
    const float *contrib; // routed experts' outputs joining it (null: none)
    int k, experts;
    const int32_t *ids, *pos_of;
    const float *wts, *dscale;
    float moe_scale;
    const float *gain; // RMS gain; null: p0 gets the plain row
    float eps;
    PfPlanes p0;
    const float *rscale, *gain2; // Gemma form: also p1 (router input) and p2 (expert input)
    PfPlanes p1, p2;
};
int emu_pf_rows(emu_ctx *ctx, const PfRows &a, int n);
int emu_pf_glu(emu_ctx *ctx, const float *part, int nks, size_t ks_stride, size_t mat_stride, int ff, int act,
               const PfPlanes &p, int n, const int *rows_used, const int32_t *src);

struct PfHeads {
    const float *part; // q|k|v partial sums
    int nks;
    size_t ks_stride;
    const uint32_t *positions;
    const float2 *rope;
    const float *q_norm, *k_norm;
    float eps;
    int rope_fma, interleaved, heads, kv_heads, layers, layer, context, tc;
    void *k_cache, *v_cache; // f16 or f32
    int kv_f16;
    _Float16 *q;    // [row][head][hi, lo][head dim], or f32 [row][head][head dim] for an f32 cache
    float *q_scale; // [row][head] (f16 cache)
};
int emu_pf_heads(emu_ctx *ctx, const PfHeads &a, int hd, int n);

struct PfAttn {
    const _Float16 *q;
    const float *q_scale;
    const void *k_cache, *v_cache; // f16 or f32
    int kv_f16;
    const uint32_t *positions;
    float score_mul, score_div;
    int heads, kv_heads, layers, layer, context, tc, window;
    float *out; // [row][heads * head dim]
};
int emu_pf_attn(emu_ctx *ctx, const PfAttn &a, int hd, int n);

struct PfGroup {
    int32_t *pos_of, *src;
    int4 *tiles;
    int *n_tiles, *rows_used;
};
int emu_pf_route(emu_ctx *ctx, const float *part, int nks, size_t ks_stride, int experts, int k, int n,
                 int32_t *junk_ids, float *junk_w, int32_t *ids, float *weights);
int emu_pf_group(emu_ctx *ctx, const int32_t *ids, int n, int k, int experts, int tile, const PfGroup &g);
int emu_pf_gather(emu_ctx *ctx, const PfPlanes &from, const PfPlanes &to, const PfGroup &g, int max_rows);
int emu_pf_advance(emu_ctx *ctx, uint32_t *positions, uint32_t *steps, uint32_t *tokens, const uint32_t *prompt,
                   int stride, int t0, int tc, int n);
