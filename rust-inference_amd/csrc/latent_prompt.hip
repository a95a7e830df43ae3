// Attention over a cached latent for prompts: the keys and values of all heads are made from the latents first.
//
// On the latents as they lie (latent_mfma.hip) a score costs key rows of rank + rot elements and a value product rows of rank: 1,088
// multiply-adds a (token, key, head) at 576 and 512.  With U_h c and V_h c made once a key it costs dim + rot + vdim: 320.  The products that
// make them are 2 rank (dim + vdim) operations a key and head, what about thirty tokens' scores cost more on the latents; so it pays for
// prompts, and steps of single tokens keep the latents (single tokens beside a prompt come along: below).  Three steps:
//  - ri_latent_gather: the sequences' pages side by side, sequence after sequence (a sequence begins at a multiple of 32 rows): [c | k_r] rows,
//    zeros behind a sequence's end;
//  - two products of all rows (ri_gemm_tiles_bf16 or the library's): keys U c as rows [row][heads * dim], values V c transposed, [heads * vdim][row],
//    which the value product takes as they lie;
//  - the kernel below: a workgroup of four wavefronts takes 128 tokens of one head and walks the sequence's 32-row pages through LDS, one page ahead
//    with the scores, as the paged prompt attention does (attention_mfma.h; the same masks, sums and roundings).  Its epilogue adds the sink
//    and multiplies by the head's gate before the one rounding.
// Bound by the chain of a turn, two wavefronts a SIMD (registers; four pages in LDS are half a compute unit's).  Pages come by copies straight into
// LDS, three turns ahead: through registers, a turn ahead, a turn took the time of its loads (2,048 tokens, 32 heads of 128 + 64: 131 us; so 74).
// us on the latents, with the two products per head there : these three steps; 32 heads, latents of 512 + 64: 2,048 tokens 619 : 104, 700 + 300 + 33
// 239 : 66, 512 163 : 47, 128 65 : 29, eight of 64 69 : 35, 128 after 2,000 keys 499 : 116, eight of 32 after 1,000 282 : 200; with single tokens
// beside the prompt, whose sequences' keys are made for one query each (the whole mixer, us): 2,048 and eight at 1,000 keys 1,024 : 275, 512 and eight 311 : 233,
// 1,024 and 16 at 2,000 599 : 519, 4,096 and 100 at 1,000 2,833 : 1,735, 1,024 and one at 30,000 6,510 : 1,124; error against 64 bits (2-norm)
// 3.2e-3 : 2.7e-3 (queries and results per head are no longer rounded on their way through the latents).
#include "attention_mfma.h"
#include "matrix_async.h"

// Where sequence s's rows begin, in pages of 32.
__device__ __forceinline__ int first_page_of(int s, const int32_t* __restrict__ len_after) {
    int pages = 0;
    for (int at = threadIdx.x & (RI_WAVE - 1); at < s; at += RI_WAVE) pages += (len_after[at] + PAGE - 1) / PAGE;
#pragma unroll
    for (int d = 1; d < RI_WAVE; d *= 2) pages += __shfl_xor(pages, d, RI_WAVE);
    return __builtin_amdgcn_readfirstlane(pages);
}

__global__ void __launch_bounds__(256)
latent_gather_kernel(bf16_t* __restrict__ rows, const bf16_t* __restrict__ k_pages, const int32_t* __restrict__ len_after,
                     const int32_t* __restrict__ page_table, int table_width, int seqs, int key_dim) {
    int s = -1, page = blockIdx.x;
    const int lane = threadIdx.x & (RI_WAVE - 1);
    for (int s0 = 0; s0 < seqs && s < 0; s0 += RI_WAVE) {     // a lane a sequence: whose page is it
        const int n = s0 + lane < seqs ? (len_after[s0 + lane] + PAGE - 1) / PAGE : 0;
        int upto = n;
#pragma unroll
        for (int d = 1; d < RI_WAVE; d *= 2) {
            const int before = __shfl(upto, max(lane - d, 0), RI_WAVE);
            upto += lane >= d ? before : 0;
        }
        const unsigned long long past = __ballot(upto > page);
        if (past) {
            s = s0 + __builtin_ctzll(past);
            page -= __shfl(upto - n, __builtin_ctzll(past), RI_WAVE);
        } else page -= __shfl(upto, RI_WAVE - 1, RI_WAVE);
    }
    if (s < 0) return;
    const int there = len_after[s] - page * PAGE, pieces = key_dim / 8;
    const uint4* from = reinterpret_cast<const uint4*>(k_pages + (long)page_table[(long)s * table_width + page] * PAGE * key_dim);
    uint4* to = reinterpret_cast<uint4*>(rows + (long)blockIdx.x * PAGE * key_dim);
    for (int i = threadIdx.x; i < PAGE * pieces; i += 256) to[i] = i / pieces < there ? from[i] : make_uint4(0, 0, 0, 0);
}

extern "C" int ri_latent_gather(void* rows, const void* k_pages, const int32_t* len_after, const int32_t* page_table, int table_width,
                                int seqs, int pages, int key_dim, int page_size, void* stream) {
    RI_REQUIRE(seqs > 0 && pages > 0 && table_width > 0 && page_size == PAGE && key_dim > 0 && key_dim % 8 == 0,
               "latent_gather: %d sequences, %d pages of %d rows of %d", seqs, pages, page_size, key_dim);
    RI_REQUIRE(((uintptr_t)rows | (uintptr_t)k_pages) % 16 == 0, "latent_gather: an operand is off a multiple of 16 bytes");
    latent_gather_kernel<<<pages, 256, 0, (hipStream_t)stream>>>((bf16_t*)rows, (const bf16_t*)k_pages, len_after, page_table, table_width,
                                                                  seqs, key_dim);
    RI_LAUNCH_CHECK("latent_gather");
    return 0;
}

struct LatentPrompt {
    bf16_t* out;                  // [tokens][heads * DV]
    const bf16_t* q;              // rows of q_stride, heads of KU + KR
    const bf16_t* keys;           // rows of key_stride, heads of KU
    const bf16_t* turned;         // rows of turned_stride, KR elements all heads share
    const bf16_t* values;         // [heads * DV] rows of value_stride
    const bf16_t* gates;          // rows of q_stride, one a head; NULL: none
    const float* sinks;           // one a head; NULL: none
    const int32_t *cu_seqlens, *tok_pos, *len_after;
    long value_stride;
    int q_stride, key_stride, turned_stride, seqs, heads;
    float scale_log2;
};

#define LP_SLOTS 4               // pages in LDS

template <int KU, int KR, int DV>
__global__ void __launch_bounds__(256, 2)
latent_prompt_kernel(const LatentPrompt a) {
    constexpr int DH = KU + KR, NT = 2, TOKENS = 16 * NT, OF_WG = 4 * TOKENS;
    constexpr int UK = PAGE * KU / 8, RK = PAGE * KR / 8, VK = DV * PAGE / 8, SLOT = UK + RK + VK;      // 16-byte pieces of a page
    __shared__ uint4 lds[LP_SLOTS * SLOT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), jg = lane >> 4, head = blockIdx.x;
    Run run;                                                  // the last tokens of a sequence see the most keys and go out first
    if (!run_of(blockIdx.y, a.cu_seqlens, a.seqs, 1, OF_WG, 1, run)) return;
    const int t_wg = run.start + (run.tokens - 1) / OF_WG * OF_WG - run.first, t_end = run.start + run.tokens;
    const int t0 = t_wg + wave * TOKENS, nt = max(0, min(TOKENS, t_end - t0));
    const long row0 = (long)first_page_of(run.seq, a.len_after) * PAGE;

    Columns<DH, NT, DV> c;
    init_columns<DH, NT, DV>(c);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int tl = j * 16 + (lane & 15);
        if (tl >= nt) continue;
        c.qpos[j] = a.tok_pos[t0 + tl];
        const bf16_t* qp = a.q + (long)(t0 + tl) * a.q_stride + head * DH + jg * 8;
#pragma unroll
        for (int ks = 0; ks < DH / 32; ++ks) c.q[j][ks].u = *reinterpret_cast<const uint4*>(qp + ks * 32);
    }
    const int p_last = a.tok_pos[min(t_end, t_wg + OF_WG) - 1] / PAGE;
    const int min_qpos = nt == TOKENS ? a.tok_pos[t0] : -1;  // a page is open to the wavefront when its last key is at or before it

    // A page in LDS: its keys' own parts, [32][KU] in the order of the two products' rows (row 16 h + i is key 8 (i / 4) + 4 h + i % 4), their
    // turned parts, [32][KR], and its values, [DV][32].  The pieces of a row are exchanged by the row's number so that the sixteen lanes that
    // LDS serves at once (0 to 3, 12 to 15, 20 to 27 of a fragment's, and so on) meet all its banks: rows of 256 bytes by row % 16, of 128 by
    // row % 8, of 64 by -(row / 4) % 4.  A copy of a wavefront fills a kilobyte.
    constexpr int UP = KU / 8, RP = KR / 8, UR = 64 / UP, RR = 64 / RP, UN = PAGE / UR, RN = PAGE / RR, VN = DV / 16;  // pieces a row, rows a copy, copies
    constexpr int MINE = (UN + RN + VN) / 4;
    static_assert(UN % 4 == 0 && RN % 4 == 0 && VN % 4 == 0, "every wavefront makes as many copies");
    constexpr auto exchange = [](int row, int pieces) { return pieces == 4 ? -(row >> 2) & 3 : row & (pieces - 1); };
    const auto key_of = [](int row) { return ((row & 15) >> 2) * 8 + (row >> 4) * 4 + (row & 3); };
    uint32_t off[MINE];
#pragma unroll
    for (int i = 0; i < MINE; ++i) {
        if (i < UN / 4) {
            const int row = (wave * (UN / 4) + i) * UR + lane / UP;
            off[i] = 2u * ((uint32_t)key_of(row) * (uint32_t)a.key_stride + 8u * (lane % UP ^ exchange(row, UP)));
        } else if (i < (UN + RN) / 4) {
            const int row = (wave * (RN / 4) + i - UN / 4) * RR + lane / RP;
            off[i] = 2u * ((uint32_t)key_of(row) * (uint32_t)a.turned_stride + 8u * (lane % RP ^ exchange(row, RP)));
        } else {
            const int row = (wave * (VN / 4) + i - (UN + RN) / 4) * 16 + lane / 4;
            off[i] = 2u * ((uint32_t)row * (uint32_t)a.value_stride + 8u * (lane % 4 ^ exchange(row, 4)));
        }
    }
    const bf16_t* keys = a.keys + row0 * a.key_stride + head * KU;
    const bf16_t* turned = a.turned + row0 * a.turned_stride;
    const bf16_t* values = a.values + (long)head * DV * a.value_stride + row0;
    const ma_lds_t u_at = ma_lds(lds + wave * (UK / 4)), r_at = ma_lds(lds + UK + wave * (RK / 4)), v_at = ma_lds(lds + UK + RK + wave * (VK / 4));
    auto fetch = [&](int page) {
        const int to = page % LP_SLOTS * SLOT * 16;
        const int from = min(page, p_last);                  // (past the end: the last one again, for nobody)
#pragma unroll
        for (int i = 0; i < MINE; ++i) {
            if (i < UN / 4) ma_copy16(u_at + to + i * 1024, off[i], keys + (long)from * PAGE * a.key_stride);
            else if (i < (UN + RN) / 4) ma_copy16(r_at + to + (i - UN / 4) * 1024, off[i], turned + (long)from * PAGE * a.turned_stride);
            else ma_copy16(v_at + to + (i - (UN + RN) / 4) * 1024, off[i], values + from * PAGE);
        }
    };
    const int fr = lane & 15;
    auto key_frags = [&](Frag (&kf)[2][DH / 32], int page) {
        const uint4* from = lds + page % LP_SLOTS * SLOT;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int ks = 0; ks < DH / 32; ++ks)
                kf[kt][ks].u = ks < KU / 32 ? from[(kt * 16 + fr) * UP + (4 * ks + jg ^ exchange(fr, UP))]
                                            : from[UK + (kt * 16 + fr) * RP + (4 * (ks - KU / 32) + jg ^ exchange(fr, RP))];
    };
    auto value_frags = [&](Frag (&vf)[DV / 16], int page) {
        const uint4* from = lds + page % LP_SLOTS * SLOT + UK + RK;
#pragma unroll
        for (int dt = 0; dt < DV / 16; ++dt) vf[dt].u = from[(dt * 16 + fr) * 4 + (jg ^ exchange(fr, 4))];
    };
    // Turn p takes the scores of page p + 1 and the value product of page p; page p + 3 takes the place of page p - 1.  A copy has two
    // turns to arrive, and a turn one place where the wavefronts meet.
    fetch(0);
    fetch(1);
    fetch(2);
    ma_wait_copies<2 * MINE>();
    ma_meet();
    float s_cur[NT][8], ref[NT], m_new[NT];
    {
        Frag kf[2][DH / 32];
        key_frags(kf, 0);
        scores_of<DH, NT, DV>(c, kf, s_cur, 0, lane);
        if (PAGE - 1 > min_qpos) mask_scores<DH, NT, DV>(c, s_cur, 0, lane);
        maxima_with<DH, NT, DV>(c, s_cur, m_new, a.scale_log2);
        move_reference<DH, NT, DV>(c, m_new, ref);
    }
    auto turn = [&](int p, auto masked) {                    // p: the page whose weights are due
        ma_wait_copies<MINE>();                               // page p + 1 is there,
        ma_wait_lds();                                        // page p - 1 read
        ma_meet();
        fetch(p + 3);
        Frag w[NT];
        float s_next[NT][8];
        {
            Frag kf[2][DH / 32];
            key_frags(kf, p + 1);
            scores_of<DH, NT, DV>(c, kf, s_next, p + 1, lane);
            weights_of<DH, NT, DV>(c, s_cur, ref, w, a.scale_log2);
        }
        if (decltype(masked)::value) mask_scores<DH, NT, DV>(c, s_next, p + 1, lane);
        {
            Frag vf[DV / 16];
            value_frags(vf, p);
            weighted_values<DH, NT, DV>(c, vf, w);
            maxima_with<DH, NT, DV>(c, s_next, m_new, a.scale_log2);
        }
        move_reference<DH, NT, DV>(c, m_new, ref);
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) s_cur[j][e] = s_next[j][e];
    };
    int p = 0;
    for (; p < p_last && (p + 1) * PAGE + PAGE - 1 <= min_qpos; ++p) turn(p, std::false_type());
    for (; p < p_last; ++p) turn(p, std::true_type());
    {
        Frag w[NT], vf[DV / 16];
        weights_of<DH, NT, DV>(c, s_cur, ref, w, a.scale_log2);
        value_frags(vf, p_last);
        weighted_values<DH, NT, DV>(c, vf, w);
    }
    ma_wait_copies<0>();
    finish_columns<DH, NT, DV>(c);
    const float sink = a.sinks ? a.sinks[head] * 1.4426950408889634f : -INFINITY;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int tl = j * 16 + (lane & 15);
        if (tl >= nt) continue;
        float inv = 1.0f / (c.l[j] + __builtin_amdgcn_exp2f(sink - c.m[j]));
        if (a.gates) inv /= 1.0f + expf(-bf16_to_f32(a.gates[(long)(t0 + tl) * a.q_stride + head]));
        bf16_t* op = a.out + ((long)(t0 + tl) * a.heads + head) * DV + jg * 4;
#pragma unroll
        for (int dt = 0; dt < DV / 16; ++dt)
            *reinterpret_cast<uint2*>(op + dt * 16) = uint2{pack_bf16x2(c.o[j][dt][0] * inv, c.o[j][dt][1] * inv),
                                                            pack_bf16x2(c.o[j][dt][2] * inv, c.o[j][dt][3] * inv)};
    }
}

static bool latent_prompt_heads(int dim, int rot, int vdim) {
    return (dim == 128 && rot == 64 && vdim == 128) || (dim == 64 && rot == 64 && vdim == 64);
}

// (a latent's rows are gathered, and the turned part behind `rank` elements is copied, sixteen bytes at a time)
extern "C" int ri_latent_prompt_fits(int dim, int rot, int vdim, int rank) {
    return latent_prompt_heads(dim, rot, vdim) && rank > 0 && rank % 8 == 0;
}

extern "C" int ri_latent_prompt(void* out, const void* q, int q_stride, const void* keys, int key_stride, const void* turned, int turned_stride,
                                const void* values, long value_stride, const void* gates, const float* sinks, const int32_t* cu_seqlens,
                                const int32_t* tok_pos, const int32_t* len_after, int seqs, int tokens, int heads, int dim, int rot, int vdim,
                                float scale, void* stream) {
    RI_REQUIRE(latent_prompt_heads(dim, rot, vdim), "latent_prompt: heads of %d + %d and %d", dim, rot, vdim);
    RI_REQUIRE(heads > 0 && seqs > 0 && tokens >= seqs && scale > 0.f, "latent_prompt: %d heads, %d tokens of %d sequences, scale %g", heads,
               tokens, seqs, (double)scale);
    RI_REQUIRE(q_stride >= heads * (dim + rot) && (q_stride | key_stride | turned_stride) % 8 == 0 && key_stride >= heads * dim && key_stride < (1 << 24) && turned_stride >= rot && value_stride % 8 == 0 && value_stride <= (1 << 23) && turned_stride < (1 << 24),
               "latent_prompt: rows of %d, %d, %d and %ld", q_stride, key_stride, turned_stride, value_stride);
    RI_REQUIRE(((uintptr_t)q | (uintptr_t)keys | (uintptr_t)turned | (uintptr_t)values | (uintptr_t)out) % 16 == 0,
               "latent_prompt: an operand is off a multiple of 16 bytes");
    const int runs = (tokens - seqs) / 128 + seqs;            // the most that so many tokens of so many sequences make
    RI_REQUIRE(runs <= 65535, "latent_prompt: %d runs of tokens exceed one launch", runs);
    const LatentPrompt a = {(bf16_t*)out, (const bf16_t*)q, (const bf16_t*)keys, (const bf16_t*)turned, (const bf16_t*)values,
                            (const bf16_t*)gates, sinks, cu_seqlens, tok_pos, len_after, value_stride, q_stride, key_stride, turned_stride, seqs, heads,
                            scale * 1.4426950408889634f};
    const dim3 grid(heads, runs);
    if (dim == 128) latent_prompt_kernel<128, 64, 128><<<grid, 256, 0, (hipStream_t)stream>>>(a);
    else latent_prompt_kernel<64, 64, 64><<<grid, 256, 0, (hipStream_t)stream>>>(a);
    RI_LAUNCH_CHECK("latent_prompt");
    return 0;
}
