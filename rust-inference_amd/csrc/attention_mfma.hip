// The matrix-core attention (attention_mfma.h) for heads of 32, 64 and 128 elements whose value heads have the same
// size: the launches.
#include "attention_mfma.h"

extern "C" int ri_attention_decode_streams(int seqs, int kv_heads, int max_chunks) {
    return stream_splits(seqs, kv_heads, max_chunks);
}

// ------------------------------------------------------------------ host side
static int check_common(const char* name, int heads, int kv_heads, int head_dim, int page_size, int q_stride,
                        int table_width) {
    RI_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "%s: heads %d, kv heads %d", name, heads, kv_heads);
    RI_REQUIRE(head_dim == 32 || head_dim == 64 || head_dim == 128,
               "%s: head_dim %d (this kernel is built for 32, 64 and 128)", name, head_dim);
    RI_REQUIRE(page_size == PAGE, "%s: pages of %d tokens (this kernel takes %d)", name, page_size, PAGE);
    RI_REQUIRE(q_stride >= heads * head_dim && q_stride % 8 == 0, "%s: q row stride %d", name, q_stride);
    RI_REQUIRE(table_width > 0, "%s: page table width %d", name, table_width);
    RI_REQUIRE(kv_heads <= 65535, "%s: %d kv heads exceed one launch", name, kv_heads);
    return 0;
}

// Column tiles per wavefront: at most 64 columns for head_dim up to 64, 32 for 128 (registers); fewer when
// that leaves the launch with less than four workgroups a compute unit (few query heads per kv head, a
// prompt of a few thousand tokens: at 32 query and 8 kv heads of 128, 2,048 tokens take 81 us with 1,024
// workgroups of half the columns against 95 us with 512; from 4,096 tokens on the full tiles win).  A
// column's arithmetic does not depend on the tile it sits in, only the grid does.
// Tiles are halved while the launch has fewer workgroups than this many for each compute unit (measured with
// 256 of them: a prompt of 3,072 tokens at Qwen3-8B sizes takes 105 us with two tiles a wavefront in 768
// workgroups, 126 us with one tile in 1,536; at 2,048 tokens one tile in 1,024 workgroups takes 57 us, two in
// 512 take 67).
// Heads of 128: the workgroups are counted by the step's tokens, and two tiles a wavefront also want sequences of twelve workgroups' tokens
// and more on average.  Below, most of what a workgroup of twice the tokens does is its start and the pages on the diagonal, which it
// walks whole.  us with one : two tiles a wavefront (heads of 128 over 8; the workgroups that two tiles make): prompts of 500, 1,500 and 900, 32
// heads (728) 60 : 82; 12 of 200 to 1,024, 16 heads (896) 44 : 53; 16 of 16 to 1,024 (1,016) 65 : 68, 32 (2,408) 127 : 133; eight of 500, 32 heads
// (1,024) 41 : 41; four of 300 to 1,800 (1,240) 150 : 141; one of 2,048 (512) 64 : 73, 3,072 (768) 140 : 122, 8,192 of 16 heads (1,024) 387 : 342.
// Single tokens beside prompts bring the average down and take longer themselves with two tiles: such a step wants a hundred workgroups' tokens
// of the sequence that a token is of on average (`weighted`, the sum of squares over the sum).  With single tokens at 1,000 keys: one of 8,192 and
// 40 (16 heads) 403 : 365, two of 4,096 and 100 (32) 475 : 446, one of 3,000 and 63 157 : 192, one of 2,048 and 256 251 : 319, eight of 1,024 and
// eight (16) 90 : 103.
#define PREFILL_MIN_WGS_PER_CU 3
#define PREFILL_MIN_WGS_PER_SEQ 12
#define PREFILL_MIN_WGS_WEIGHTED 100
static int prefill_tiles(int head_dim, int group, int max_new, int seqs, int kv_heads, int tokens, int weighted) {
    int nt = head_dim <= 64 ? 4 : 2;
    while (nt > 1 && group <= 16 * (nt / 2)) {
        const int of_wg = 4 * ((16 * nt) / group);
        const long wgs = head_dim <= 64 ? (long)((max_new + of_wg - 1) / of_wg) * seqs * kv_heads
                                        : (tokens + (long)seqs * of_wg / 2) / of_wg * kv_heads;
        if (wgs >= (long)PREFILL_MIN_WGS_PER_CU * ri_compute_units() &&
            (head_dim <= 64 || tokens >= (long)PREFILL_MIN_WGS_PER_SEQ * of_wg * seqs || weighted >= PREFILL_MIN_WGS_WEIGHTED * of_wg)) break;
        nt /= 2;
    }
    return nt;
}

// Pairs of pages a turn (attn_prefill_pairs_kernel) where a sequence brings this many tokens on average: shorter ones are mostly the start and the
// diagonal, which pairs make longer.  us, a page a turn : pairs (heads of 128 over 8): 40 of 64 (32 heads) 16.5 : 18.6, 16 of 200 (16) 15.9 : 17.2, 16 of 300
// 24.1 : 25.8, 16 of 16 to 700 27 : 30, four of 300 (32) 15.3 : 14.0, eight of 500 40.4 : 39.8, 16 of 16 to 1,024 (16) 55 : 53, two of 1,000 (32) 39 : 35.
// Two tiles a wavefront there (heads of 128) from three of their workgroups a compute unit on, for one sequence from two on, one : two tiles: 2,048 (512
// workgroups) 58 : 56, 1,792 (448) 48 : 49, 2,816 (704) 94 : 80; two of 1,500 (752) 64 : 69, 500 + 1,500 + 532 (632) 45 : 67, eight of 500 (1,024) 42 : 39, 8,192 of 64 heads
// 1,380 : 1,081.  Heads of 32 and 64: one, 2,048 of 32 heads of 64 32.5 : 38, 6,000 204 : 221 (4,096 99 : 95); more only where a key head's queries need them.
#define PAIRS_MIN_TOKENS 400
// A window or a chunk of fewer keys than this (`reach`) leaves a turn's chain too few pages: a page a turn, unless its rule takes larger tiles.  us, a
// page a turn : pairs (heads of 128 over 8; windows of 128 / 256 / 512): 8,192 of 32 heads 58 : 66 / 75 : 76 / 113 : 106, of 64 115 : 122 / 148 : 150 / 221 : 204,
// six of 700 of 16 21 : 24 / 24 : 26 / 30 : 30, of 32 35 : 39 / 41 : 41 / 49 : 48; chunks of 128 / 512, six of 700 of 32 28 : 31 / 37 : 36.  Heads of 64, four
// tiles against one: 8,192 of 32 heads 81 : 39 / 106 : 50 / 151 : 70; one against one: 2,048 11.6 : 12.5 / 15.2 : 15.8 / 21.6 : 20.0.
#define PAIRS_MIN_REACH 512
// A key head's queries that fill pairs' tiles badly (9 and 10 one tile: 0.56 and 0.63 of its columns, 17 to 21 two tiles) beside tiles of twice the size that
// they fill to 0.8 and more go a page a turn.  us, a page a turn : pairs, four key heads: 9 queries, eight of 500 35 : 39 (heads of 32), 41 : 48 (of 64), three of 1,500 92 : 97,
// 102 : 121; 17, of 32, three of 1,500 193 : 216, 6,000 948 : 1,044.  Not four tiles against one (9 and 10 queries, 6,000: 455 : 449 and 530 : 446) nor four
// of heads of 64 (17, 6,000: 1,630 : 1,138); 11 (0.69) three of 1,500 of 32 130 : 99, 22 (0.69) 283 : 217.  More than 32 queries take four tiles either way,
// for heads of 64 with some of their registers in memory: 6,000, one key head of 64 queries of 64 867 : 552, of 40 1,273 : 936, of 40 of 32 714 : 647.
#define PAIRS_MIN_FILL_TENTHS 7
#define PREFILL_MAX_LAUNCHES 65535
static int pair_tiles(int head_dim, int group, int seqs, int kv_heads, int tokens) {
    const int of_wg = 4 * (32 / (group <= 32 ? group : 32));
    const long wgs = (tokens + (long)seqs * of_wg / 2) / of_wg * kv_heads;
    if (group > 16) return group > 32 ? 4 : 2;
    return head_dim == 128 && wgs >= (seqs == 1 ? 2L : 3L) * ri_compute_units() ? 2 : 1;
}

struct PrefillPlan { bool paired; int tiles, launches; };     // tiles of columns a wavefront, workgroups of the longest sequence's tokens a key head
// pairs: 1 so, 0 not so, -1 where it pays and a launch holds it.
static PrefillPlan prefill_plan(int head_dim, int group, int max_new, int seqs, int kv_heads, int tokens, int weighted, int reach,
                                int pairs) {
    const auto plan = [&](bool paired, int nt) { const int of_wg = 4 * (group < 16 * nt ? 16 * nt / group : 1); return PrefillPlan{paired, nt, (max_new + of_wg - 1) / of_wg}; };
    const PrefillPlan one = plan(false, prefill_tiles(head_dim, group, max_new, seqs, kv_heads, tokens, weighted));
    const PrefillPlan two = plan(true, pair_tiles(head_dim, group, seqs, kv_heads, tokens));
    if (pairs >= 0) return pairs ? two : one;
    if (tokens < (long)PAIRS_MIN_TOKENS * seqs || two.launches > PREFILL_MAX_LAUNCHES) return one;
    if (reach > 0 && reach < PAIRS_MIN_REACH && one.tiles <= two.tiles) return one;
    const auto columns = [&](int nt) { return 16 * nt / group * group; };
    const bool emptier = 10 * columns(two.tiles) * one.tiles < PAIRS_MIN_FILL_TENTHS * columns(one.tiles) * two.tiles;
    return emptier && one.tiles == 2 * two.tiles && !(head_dim == 64 && one.tiles == 4) ? one : two;
}

// The tiles of columns a wavefront takes of a step that goes in pairs of pages, 0: a page a turn (host code only).
extern "C" int ri_attention_prefill_pairs(int head_dim, int group, int max_new, int seqs, int kv_heads, int tokens, int weighted, int reach) {
    const PrefillPlan plan = prefill_plan(head_dim, group, max_new, seqs, kv_heads, tokens, weighted, reach, -1);
    return plan.paired ? plan.tiles : 0;
}

// The column tiles a wavefront takes of a step with a page a turn (host code only).
extern "C" int ri_attention_prefill_tiles(int head_dim, int group, int max_new, int seqs, int kv_heads, int tokens, int weighted) {
    return prefill_tiles(head_dim, group, max_new, seqs, kv_heads, tokens, weighted);
}

extern "C" int ri_attention_prefill_kept_bf16(void* out, const void* qkv, int q_stride, const void* k_pages,
                                              const void* v_pages, const int32_t* cu_seqlens, const int32_t* tok_pos,
                                              const int32_t* page_table, int table_width, int seqs, int max_new,
                                              int heads, int kv_heads, int head_dim, int page_size, int window, int chunk,
                                              float scale, float softcap, const float* slopes, int keep_first,
                                              const float* sinks, int tokens, int weighted, int pairs, void* stream) {
    RI_REQUIRE(chunk >= 0 && (chunk == 0 || window <= 0), "attention_prefill: chunks of %d beside a window of %d", chunk, window);
    const Reach reach = {window, chunk};
    RI_REQUIRE(keep_first >= 0, "attention_prefill_bf16: %d first tokens kept", keep_first);
    const float cap_pre = softcap > 0.f ? scale / softcap : 0.f, cap_post = softcap > 0.f ? softcap / scale : 0.f;
    RI_REQUIRE(scale > 0.f, "attention_prefill_bf16: the scale %g must be positive", (double)scale);
    if (check_common("attention_prefill_bf16", heads, kv_heads, head_dim, page_size, q_stride, table_width)) return 1;
    const int group = heads / kv_heads;
    RI_REQUIRE(seqs > 0 && seqs <= 65535 && max_new > 0, "attention_prefill_bf16: seqs %d, max_new %d", seqs, max_new);
    RI_REQUIRE(pairs >= -1 && pairs <= 1, "attention_prefill_bf16: pairs %d", pairs);
    RI_REQUIRE(group <= (head_dim <= 64 ? 64 : 32), "attention_prefill_bf16: %d query heads per kv head (at most %d)", group, head_dim <= 64 ? 64 : 32);
    const PrefillPlan plan = prefill_plan(head_dim, group, max_new, seqs, kv_heads, tokens, weighted, window > 0 ? window : chunk, pairs);
    RI_REQUIRE(plan.launches <= PREFILL_MAX_LAUNCHES, "attention_prefill_bf16: %d tiles of tokens exceed one launch", plan.launches);
    int long_runs;
    const dim3 grid = prefill_grid(kv_heads, seqs, plan.launches, 4 * (16 * plan.tiles / group), tokens, long_runs);
    const float scale_log2 = scale * 1.4426950408889634f;
    hipStream_t s = (hipStream_t)stream;
    const int form = slopes ? PREFILL_ANY : cap_pre != 0.f ? PREFILL_CAPPED : PREFILL_PLAIN;
#define RI_PREFILL_ARGS                                                                                          \
    (bf16_t*)out, (const bf16_t*)qkv, q_stride, (const bf16_t*)k_pages, (const bf16_t*)v_pages, cu_seqlens,      \
        tok_pos, page_table, table_width, heads, kv_heads, reach, scale_log2, cap_pre, cap_post, slopes,         \
        1.f / scale, keep_first, sinks, seqs, long_runs
#define RI_PREFILL_GO(DH, NT, FORM)                                                                              \
    if (plan.paired) attn_prefill_pairs_kernel<DH, NT, FORM><<<grid, 256, 0, s>>>(RI_PREFILL_ARGS);                   \
    else attn_prefill_mfma_kernel<DH, NT, DH, false, FORM><<<grid, 256, 0, s>>>(RI_PREFILL_ARGS)
#define RI_PREFILL_CASE(DH, NT)                                                                                  \
    case DH * 8 + NT:                                                                                            \
        if (form == PREFILL_PLAIN) { RI_PREFILL_GO(DH, NT, PREFILL_PLAIN); }                                     \
        else if (form == PREFILL_CAPPED) { RI_PREFILL_GO(DH, NT, PREFILL_CAPPED); }                              \
        else { RI_PREFILL_GO(DH, NT, PREFILL_ANY); }                                                             \
        break;
    switch (head_dim * 8 + plan.tiles) {
        RI_PREFILL_CASE(32, 4)
        RI_PREFILL_CASE(32, 2)
        RI_PREFILL_CASE(32, 1)
        RI_PREFILL_CASE(64, 4)
        RI_PREFILL_CASE(64, 2)
        RI_PREFILL_CASE(64, 1)
        RI_PREFILL_CASE(128, 2)
        RI_PREFILL_CASE(128, 1)
    }
#undef RI_PREFILL_CASE
#undef RI_PREFILL_GO
#undef RI_PREFILL_ARGS
    RI_LAUNCH_CHECK("attention_prefill_bf16");
    return 0;
}

extern "C" int ri_attention_prefill_bf16(void* out, const void* qkv, int q_stride, const void* k_pages,
                                         const void* v_pages, const int32_t* cu_seqlens, const int32_t* tok_pos,
                                         const int32_t* page_table, int table_width, int seqs, int max_new,
                                         int heads, int kv_heads, int head_dim, int page_size, int window,
                                         float scale, float softcap, const float* slopes, void* stream) {
    return ri_attention_prefill_kept_bf16(out, qkv, q_stride, k_pages, v_pages, cu_seqlens, tok_pos, page_table, table_width,
                                          seqs, max_new, heads, kv_heads, head_dim, page_size, window, 0, scale, softcap, slopes,
                                          0, nullptr, (int)(max_new * (long)seqs < 1 << 30 ? max_new * (long)seqs : 1 << 30), max_new, -1, stream);
}

// Whether the streaming kernel ranks the step's sequences by their lengths (host code only).
extern "C" int ri_attention_decode_ranks(int seqs, int kv_heads, int max_chunks) {
    return !stream_wide(seqs, kv_heads, max_chunks) && stream_balances(seqs, kv_heads, stream_splits(seqs, kv_heads, max_chunks), max_chunks) > 0;
}

extern "C" int ri_attention_decode_chunks(int max_len) { return (max_len + DECODE_CHUNK - 1) / DECODE_CHUNK; }

// The workspace of a decode attention call has room for max_chunks times this many results a sequence and head.
extern "C" int ri_attention_decode_pieces(int seqs, int kv_heads, int heads, int max_chunks) {
    return decode_pieces(seqs, kv_heads, heads / (kv_heads > 0 ? kv_heads : 1), max_chunks);
}

// keep_first, sinks: the first keys that stay visible behind a window, and a number per head whose exponential joins
// the softmax's denominator; only the kernels that work in chunks take kept keys (where ri_attention_decode_streams says
// the step streams, the caller takes the prompt kernel).
extern "C" int ri_attention_decode_kept_bf16(void* out, float* workspace, const void* qkv, int q_stride,
                                             const void* k_pages, const void* v_pages, const int32_t* cu_seqlens,
                                             const int32_t* tok_pos, const int32_t* page_table, int table_width, int seqs,
                                             int max_chunks, int heads, int kv_heads, int head_dim, int page_size,
                                             int window, int chunk, float scale, float softcap, const float* slopes, int tiled_out,
                                             int keep_first, const float* sinks, void* stream) {
    RI_REQUIRE(chunk >= 0 && (chunk == 0 || window <= 0), "attention_decode: chunks of %d beside a window of %d", chunk, window);
    const Reach reach = {window, chunk};
    RI_REQUIRE(keep_first >= 0, "attention_decode_bf16: %d first tokens kept", keep_first);
    RI_REQUIRE(keep_first == 0 || stream_splits(seqs, kv_heads, max_chunks) == 0,
               "attention_decode_bf16: kept first tokens in a step that streams (%d sequences)", seqs);
    const float cap_pre = softcap > 0.f ? scale / softcap : 0.f, cap_post = softcap > 0.f ? softcap / scale : 0.f;
    RI_REQUIRE(scale > 0.f, "attention_decode_bf16: the scale %g must be positive", (double)scale);
    if (check_common("attention_decode_bf16", heads, kv_heads, head_dim, page_size, q_stride, table_width)) return 1;
    RI_REQUIRE(!tiled_out || (seqs <= 64 && head_dim % 32 == 0), "attention_decode_bf16: tiled rows are at most 64 (%d)", seqs);
    const int group = heads / kv_heads;
    RI_REQUIRE(group <= 16, "attention_decode_bf16: %d query heads per kv head (at most 16)", group);
    RI_REQUIRE(seqs > 0 && max_chunks > 0 && max_chunks <= 65535 && heads <= 65535,
               "attention_decode_bf16: seqs %d, chunks %d, heads %d", seqs, max_chunks, heads);
    dim3 grid(seqs, kv_heads, max_chunks);
    const float scale_log2 = scale * 1.4426950408889634f;
    hipStream_t s = (hipStream_t)stream;
    const int splits = stream_splits(seqs, kv_heads, max_chunks);
    const bool wide = stream_wide(seqs, kv_heads, max_chunks);
    if (splits > 0) {
        dim3 sgrid(seqs, kv_heads, splits);
#define RI_STREAM_CASE(DH)                                                                                        \
    case DH:                                                                                                      \
        if (wide)                                                                                                 \
            attn_decode_stream_kernel<DH, false, 8><<<sgrid, 8 * 64, 0, s>>>(                                     \
                (bf16_t*)out, workspace, (const bf16_t*)qkv, q_stride, nullptr, nullptr, 0.f, nullptr,            \
                (bf16_t*)k_pages, (bf16_t*)v_pages, tok_pos, page_table, table_width, heads, kv_heads, reach,     \
                scale_log2, splits, tiled_out, cap_pre, cap_post, slopes, 1.f / scale, sinks);                           \
        else                                                                                                      \
            attn_decode_stream_kernel<DH, false, 4><<<sgrid, 4 * 64, 0, s>>>(                                     \
                (bf16_t*)out, workspace, (const bf16_t*)qkv, q_stride, nullptr, nullptr, 0.f, nullptr,            \
                (bf16_t*)k_pages, (bf16_t*)v_pages, tok_pos, page_table, table_width, heads, kv_heads, reach,     \
                scale_log2, splits, tiled_out, cap_pre, cap_post, slopes, 1.f / scale, sinks, DH, DH,             \
                stream_balances(seqs, kv_heads, splits, max_chunks));                                                         \
        if (splits > 1)                                                                                          \
            launch_join<DH>((bf16_t*)out, workspace, tok_pos, seqs, heads, Reach{-1, 0}, splits, tiled_out, s, DECODE_CHUNK, 0, sinks); \
        break;
        switch (head_dim) {
            RI_STREAM_CASE(32)
            RI_STREAM_CASE(64)
            RI_STREAM_CASE(128)
        }
#undef RI_STREAM_CASE
        RI_LAUNCH_CHECK("attention_decode_bf16 (streaming)");
        return 0;
    }
    const int pieces = decode_pieces(seqs, kv_heads, group, max_chunks), all = max_chunks * pieces;
    const dim3 pgrid(seqs, kv_heads, all);
#define RI_DECODE_CASE(DH, CW)                                                                                    \
    case DH * 16 + CW:                                                                                            \
        attn_decode_mfma_kernel<DH, CW><<<pgrid, CW * 64, 0, s>>>(                                                \
            workspace, (const bf16_t*)qkv, q_stride, (const bf16_t*)k_pages, (const bf16_t*)v_pages,             \
            tok_pos, page_table, table_width, heads, kv_heads, reach, scale_log2, all, cap_pre, cap_post,       \
            slopes, 1.f / scale, keep_first);                                                                     \
        launch_join<DH>((bf16_t*)out, workspace, tok_pos, seqs, heads, reach, all, tiled_out, s, CW * PAGE,      \
                        keep_first, sinks);                                                                       \
        break;
    switch (head_dim * 16 + DECODE_WAVES / pieces) {
        RI_DECODE_CASE(32, 8)
        RI_DECODE_CASE(32, 4)
        RI_DECODE_CASE(32, 2)
        RI_DECODE_CASE(64, 8)
        RI_DECODE_CASE(64, 4)
        RI_DECODE_CASE(64, 2)
        RI_DECODE_CASE(128, 8)
        RI_DECODE_CASE(128, 4)
        RI_DECODE_CASE(128, 2)
    }
#undef RI_DECODE_CASE
    RI_LAUNCH_CHECK("attention_decode_bf16");
    return 0;
}

extern "C" int ri_attention_decode_bf16(void* out, float* workspace, const void* qkv, int q_stride,
                                        const void* k_pages, const void* v_pages, const int32_t* cu_seqlens,
                                        const int32_t* tok_pos, const int32_t* page_table, int table_width, int seqs,
                                        int max_chunks, int heads, int kv_heads, int head_dim, int page_size,
                                        int window, float scale, float softcap, const float* slopes, int tiled_out,
                                        void* stream) {
    return ri_attention_decode_kept_bf16(out, workspace, qkv, q_stride, k_pages, v_pages, cu_seqlens, tok_pos, page_table,
                                         table_width, seqs, max_chunks, heads, kv_heads, head_dim, page_size, window, 0, scale,
                                         softcap, slopes, tiled_out, 0, nullptr, stream);
}

// The decode attention of a layer from the raw fused projection (which is not changed): q/k norm, rotation,
// the new token's k and v into their pages and attention in chunks in one kernel, then the join.
extern "C" int ri_attention_decode_fused_bf16(void* out, float* workspace, const void* qkv, int q_stride,
                                              const float* q_gain, const float* k_gain, float eps,
                                              const float* inv_freq, void* k_pages, void* v_pages,
                                              const int32_t* tok_pos, const int32_t* page_table, int table_width,
                                              int seqs, int max_chunks, int heads, int kv_heads, int head_dim,
                                              int page_size, int window, float scale, int tiled_out, void* stream) {
    const Reach reach = {window, 0};
    if (check_common("attention_decode_fused_bf16", heads, kv_heads, head_dim, page_size, q_stride, table_width))
        return 1;
    RI_REQUIRE(!tiled_out || (seqs <= 64 && head_dim % 32 == 0), "attention_decode_fused_bf16: tiled rows are at most 64 (%d)", seqs);
    const int group = heads / kv_heads;
    RI_REQUIRE(group <= 16, "attention_decode_fused_bf16: %d query heads per kv head (at most 16)", group);
    RI_REQUIRE(seqs > 0 && max_chunks > 0 && max_chunks <= 65535 && heads <= 65535,
               "attention_decode_fused_bf16: seqs %d, chunks %d, heads %d", seqs, max_chunks, heads);
    RI_REQUIRE(q_stride >= (heads + 2 * kv_heads) * head_dim, "attention_decode_fused_bf16: qkv row stride %d",
               q_stride);
    dim3 grid(seqs, kv_heads, max_chunks);
    const float scale_log2 = scale * 1.4426950408889634f;
    hipStream_t s = (hipStream_t)stream;
    const int splits = stream_splits(seqs, kv_heads, max_chunks);
    const bool wide = stream_wide(seqs, kv_heads, max_chunks);
    if (splits > 0) {
        dim3 sgrid(seqs, kv_heads, splits);
#define RI_STREAM_CASE(DH)                                                                                        \
    case DH:                                                                                                      \
        if (wide)                                                                                                 \
            attn_decode_stream_kernel<DH, true, 8><<<sgrid, 8 * 64, 0, s>>>(                                      \
                (bf16_t*)out, workspace, (const bf16_t*)qkv, q_stride, q_gain, k_gain, eps, inv_freq,             \
                (bf16_t*)k_pages, (bf16_t*)v_pages, tok_pos, page_table, table_width, heads, kv_heads, reach,     \
                scale_log2, splits, tiled_out, 0.f, 0.f, nullptr, 0.f, nullptr);                                           \
        else                                                                                                      \
            attn_decode_stream_kernel<DH, true, 4><<<sgrid, 4 * 64, 0, s>>>(                                      \
                (bf16_t*)out, workspace, (const bf16_t*)qkv, q_stride, q_gain, k_gain, eps, inv_freq,             \
                (bf16_t*)k_pages, (bf16_t*)v_pages, tok_pos, page_table, table_width, heads, kv_heads, reach,     \
                scale_log2, splits, tiled_out, 0.f, 0.f, nullptr, 0.f, nullptr, DH, DH,                           \
                stream_balances(seqs, kv_heads, splits, max_chunks));                                                         \
        if (splits > 1) launch_join<DH>((bf16_t*)out, workspace, tok_pos, seqs, heads, Reach{-1, 0}, splits, tiled_out, s); \
        break;
        switch (head_dim) {
            RI_STREAM_CASE(32)
            RI_STREAM_CASE(64)
            RI_STREAM_CASE(128)
        }
#undef RI_STREAM_CASE
        RI_LAUNCH_CHECK("attention_decode_fused_bf16 (streaming)");
        return 0;
    }
    const int pieces = decode_pieces(seqs, kv_heads, group, max_chunks), all = max_chunks * pieces;
    const dim3 pgrid(seqs, kv_heads, all);
#define RI_FUSED_CASE(DH, CW)                                                                                     \
    case DH * 16 + CW:                                                                                            \
        attn_decode_fused_kernel<DH, CW><<<pgrid, CW * 64, 0, s>>>(                                               \
            workspace, (const bf16_t*)qkv, q_stride, q_gain, k_gain, eps, inv_freq, (bf16_t*)k_pages,             \
            (bf16_t*)v_pages, tok_pos, page_table, table_width, heads, kv_heads, reach, scale_log2, all);        \
        launch_join<DH>((bf16_t*)out, workspace, tok_pos, seqs, heads, reach, all, tiled_out, s, CW * PAGE);     \
        break;
    switch (head_dim * 16 + DECODE_WAVES / pieces) {
        RI_FUSED_CASE(32, 8)
        RI_FUSED_CASE(32, 4)
        RI_FUSED_CASE(32, 2)
        RI_FUSED_CASE(64, 8)
        RI_FUSED_CASE(64, 4)
        RI_FUSED_CASE(64, 2)
        RI_FUSED_CASE(128, 8)
        RI_FUSED_CASE(128, 4)
        RI_FUSED_CASE(128, 2)
    }
#undef RI_FUSED_CASE
    RI_LAUNCH_CHECK("attention_decode_fused_bf16");
    return 0;
}
