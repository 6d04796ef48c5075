// Paged softmax attention in 32 bits on the matrix cores: scores and weighted sums by v_mfma_f32_16x16x4_f32 (fused multiply-adds of
// 32-bit operands), softmax in 32 bits. For what the 32-bit engine asks for most (a softmax over a head's own values, one head size of
// 32 to 128 in steps of 32, up to 16 query heads a key/value head, windows and masking chunks); everything else goes the plain way
// (attention_generic.hip), one wave a (token, head) with a serial sum over its keys.
//
// A wave owns up to 16 columns: the query heads of one key/value head for a few consecutive tokens of one request. With
// S^T[key, col] = K Q^T and O^T[dim, col] += V^T P^T every operand is 16 consecutive bytes a lane where it lies in memory (values are
// kept transposed inside their page), in an order of k that leaves the probabilities in the registers where the second product wants
// them: nothing passes through LDS and no wave waits for another. A step's 128 matrix instructions (head size 64) are 4,096 cycles
// for 32 KB of keys and values, which the waves of a block share in L1; what bounds it is the trips to memory of the few waves that such
// calls have, so keys are dealt to as many waves as there are chunks. 700 tokens of the 0.5B shape: 34 us a layer and 6 for the merge where
// the plain kernel took 623; a decode step of 8 requests of 100 to 1,000 tokens 10 us and 5 where it took 320.
//
// A token's result depends on its request's cache alone: keys are taken in chunks of 128 by absolute position, a chunk in steps of
// KEYS keys with a running maximum, and the chunks' results are put together one after the other. Whether one wave walks all chunks or
// each is a wave of its own (few columns: the keys are dealt over blockIdx.z) changes no bit of it, since the merge kernel adds chunks with the
// walk's own operations; chunks and steps that a column does not see leave what it holds as it is.
#include "attention_internal.h"
#include "common.h"

typedef float floatx4 __attribute__((ext_vector_type(4)));

#define F32_CHUNK 128
#define F32_NONE (-1.0e30f)          // the maximum of no keys

__device__ __forceinline__ float pick(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// One more chunk (m, l) behind (M, L): the factors of what was and of what comes.
__device__ __forceinline__ void join(float& M, float& L, float m, float l, float& was, float& now) {
    const float mn = fmaxf(M, m);
    was = expf(M - mn);
    now = expf(m - mn);
    L = fmaf(L, was, l * now);
    M = mn;
}

// ND: head size / 16; KT: tiles of 16 keys of a step. SPLIT: chunk blockIdx.z alone, (maximum, sum, output) into `partial`.
template <int ND, int KT, bool SPLIT>
__global__ __launch_bounds__(256) void attn_f32_kernel(
    const float* __restrict__ q, int ldq, const float* __restrict__ kc, const float* __restrict__ vc, int kvw,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ token_slot, const int* __restrict__ positions,
    const int* __restrict__ q_start, int n_seqs, float* __restrict__ out, int ldo, float* __restrict__ partial, int H, int psh, int window,
    int mask_chunk, float scale, int tpt, int cpt, int one_tile_each, int n_chunks) {
    constexpr int D = ND * 16, KEYS = KT * 16;
    const int lane = threadIdx.x & (WAVE - 1), col = lane & 15, quarter = lane >> 4;
    const int g = blockIdx.y, P = 1 << psh;
    int tile = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE, t0 = -1, t_end = 0;
    if (one_tile_each) {
        if (tile < n_seqs) {
            t0 = q_start[tile];
            t_end = q_start[tile + 1];
        }
    } else {
        for (int s = 0; s < n_seqs; s++) {
            const int a = q_start[s], b = q_start[s + 1], nt = (b - a + tpt - 1) / tpt;
            if (tile < nt) {
                t0 = a + tile * tpt;
                t_end = t0 + tpt < b ? t0 + tpt : b;
                break;
            }
            tile -= nt;
        }
    }
    if (t0 < 0 || t_end <= t0) return;                     // the grid is an upper bound on the tiles
    const bool col_ok = col < (t_end - t0) * cpt;
    const int tok = col_ok ? t0 + col / cpt : t0, head = g * cpt + (col_ok ? col % cpt : 0);
    const int pos = positions[tok], lo = first_visible(pos, window, mask_chunk);
    const int hi = positions[t_end - 1], pos_first = positions[t0];
    const int first = first_visible(pos_first, window, mask_chunk), lo_last = first_visible(hi, window, mask_chunk);   // first .. hi: seen by some column
    const int c_first = SPLIT ? (int)blockIdx.z : first / F32_CHUNK, c_last = SPLIT ? c_first : hi / F32_CHUNK;
    if (SPLIT && (c_first > hi / F32_CHUNK || c_first < first / F32_CHUNK)) return;
    const int* bt = block_table + (size_t)token_slot[t0] * max_blocks;

    float4 qf[ND];
#pragma unroll
    for (int s = 0; s < ND; s++)
        qf[s] = col_ok ? *reinterpret_cast<const float4*>(q + (size_t)tok * ldq + head * D + s * 16 + quarter * 4) : make_float4(0.f, 0.f, 0.f, 0.f);

    // Keys outside [first, hi] are not read: rows that nobody has written yet, pages that were given back. Their lanes read a key at
    // the end of that range instead, and their values are zero in the second product.
    int pages = 0, row[KT];                                // lane i: the i-th page of the chunk (at most 64: a page holds 2 tokens or more)
    auto pages_of = [&](int c) {
        const int b = ((c * F32_CHUNK) >> psh) + lane, b0 = first >> psh, b1 = hi >> psh;
        pages = bt[b < b0 ? b0 : b > b1 ? b1 : b];
    };
    auto rows_of = [&](int j0, int chunk_begin) {
#pragma unroll
        for (int t = 0; t < KT; t++) {
            int j = j0 + t * 16 + col;
            j = j < first ? first : j > hi ? hi : j;
            row[t] = (__shfl(pages, (j >> psh) - (chunk_begin >> psh), WAVE) << psh) + (j & (P - 1));
        }
    };
    float4 kf[KT][ND], vf[KT][ND];
    auto load_keys = [&]() {
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int s = 0; s < ND; s++)
                kf[t][s] = *reinterpret_cast<const float4*>(kc + (size_t)row[t] * kvw + g * D + s * 16 + quarter * 4);
    };
    auto load_values = [&](int j0) {
#pragma unroll
        for (int t = 0; t < KT; t++) {
            // the four keys that follow `quarter`'s first: their page is that of a row some lane holds
            const int r = __shfl(row[t], quarter * 4 + 3, WAVE), j = j0 + t * 16 + quarter * 4;
            int k4 = __shfl(row[t], quarter * 4, WAVE);
            if (j < first) k4 = r;                          // the group's first key lies before the range, its last one may lie in it
            const float* base = vc + (size_t)(k4 >> psh) * P * kvw + (size_t)(g * D + col) * P + ((k4 & (P - 1)) & ~3);
#pragma unroll
            for (int s = 0; s < ND; s++) vf[t][s] = *reinterpret_cast<const float4*>(base + (size_t)s * 16 * P);
        }
    };
    // (apart from the loads: a condition between them would have each wait for the one before)
    auto clear_unseen = [&](int j0) {
#pragma unroll
        for (int t = 0; t < KT; t++) {
            const int j = j0 + t * 16 + quarter * 4;
            const bool b0 = j >= first && j <= hi, b1 = j + 1 >= first && j + 1 <= hi, b2 = j + 2 >= first && j + 2 <= hi, b3 = j + 3 >= first && j + 3 <= hi;
#pragma unroll
            for (int s = 0; s < ND; s++) {
                vf[t][s].x = b0 ? vf[t][s].x : 0.f;
                vf[t][s].y = b1 ? vf[t][s].y : 0.f;
                vf[t][s].z = b2 ? vf[t][s].z : 0.f;
                vf[t][s].w = b3 ? vf[t][s].w : 0.f;
            }
        }
    };

    float M = F32_NONE, L = 0.f;
    floatx4 O[ND];
#pragma unroll
    for (int s = 0; s < ND; s++) O[s] = floatx4{0.f, 0.f, 0.f, 0.f};
    pages_of(c_first);
    for (int c = c_first; c <= c_last; c++) {
        const int begin = c * F32_CHUNK > first / KEYS * KEYS ? c * F32_CHUNK : first / KEYS * KEYS;
        const int end = c * F32_CHUNK + F32_CHUNK - 1 < hi ? c * F32_CHUNK + F32_CHUNK - 1 : hi;
        float m = F32_NONE, l = 0.f;
        floatx4 o[ND];
#pragma unroll
        for (int s = 0; s < ND; s++) o[s] = floatx4{0.f, 0.f, 0.f, 0.f};
        rows_of(begin, c * F32_CHUNK);
        load_keys();
        for (int j0 = begin; j0 <= end; j0 += KEYS) {
            load_values(j0);
            floatx4 sc[KT];
#pragma unroll
            for (int t = 0; t < KT; t++) sc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < ND; s++)
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int t = 0; t < KT; t++) sc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(pick(kf[t][s], e), pick(qf[s], e), sc[t], 0, 0, 0);
            if (j0 + KEYS <= end) {                         // the next step's keys travel from here on
                rows_of(j0 + KEYS, c * F32_CHUNK);
                load_keys();
            } else if (c < c_last) {
                pages_of(c + 1);
            }
            float top = F32_NONE;
#pragma unroll
            for (int t = 0; t < KT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int j = j0 + t * 16 + quarter * 4 + r;
                    sc[t][r] = j >= lo && j <= pos ? sc[t][r] * scale : -INFINITY;
                    top = fmaxf(top, sc[t][r]);
                }
            top = fmaxf(top, __shfl_xor(top, 16, WAVE));
            top = fmaxf(top, __shfl_xor(top, 32, WAVE));
            const float mn = fmaxf(m, top), corr = expf(m - mn);
            m = mn;
            float sum = 0.f;
#pragma unroll
            for (int t = 0; t < KT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    sc[t][r] = expf(sc[t][r] - mn);
                    sum += sc[t][r];
                }
            sum += __shfl_xor(sum, 16, WAVE);
            sum += __shfl_xor(sum, 32, WAVE);
            l = fmaf(l, corr, sum);
#pragma unroll
            for (int s = 0; s < ND; s++) o[s] *= corr;
            if (j0 < first || j0 + KEYS - 1 > hi) clear_unseen(j0);
            // A key that only some of the tile's tokens see has weight zero in the others' columns, which is not nothing if its value is
            // infinite or no number: such steps go token by token.
            bool odd = false;
            if (t_end - t0 > 1 && (j0 < lo_last || j0 + KEYS - 1 > pos_first)) {
#pragma unroll
                for (int t = 0; t < KT; t++)
#pragma unroll
                    for (int s = 0; s < ND; s++)
#pragma unroll
                        for (int r = 0; r < 4; r++) odd |= !(fabsf(pick(vf[t][s], r)) < INFINITY);
                odd = __any(odd);
            }
            if (!odd) {
#pragma unroll
                for (int t = 0; t < KT; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int s = 0; s < ND; s++) o[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(pick(vf[t][s], r), sc[t][r], o[s], 0, 0, 0);
            } else {
                for (int one = t0; one < t_end; one++) {
                    const int p1 = positions[one], l1 = first_visible(p1, window, mask_chunk);
#pragma unroll
                    for (int s = 0; s < ND; s++) {
                        floatx4 sum1 = o[s];
#pragma unroll
                        for (int t = 0; t < KT; t++)
#pragma unroll
                            for (int r = 0; r < 4; r++) {
                                const int j = j0 + t * 16 + quarter * 4 + r;
                                sum1 = __builtin_amdgcn_mfma_f32_16x16x4f32(j >= l1 && j <= p1 ? pick(vf[t][s], r) : 0.f, sc[t][r], sum1, 0, 0, 0);
                            }
                        o[s] = tok == one ? sum1 : o[s];
                    }
                }
            }
        }
        if (SPLIT) {
            if (!col_ok) return;
            float* dst = partial + ((size_t)(tok * H + head) * n_chunks + c) * (D + 2);
            if (quarter == 0) {
                dst[0] = m;
                dst[1] = l;
            }
#pragma unroll
            for (int s = 0; s < ND; s++) {                  // (rows of D + 2 numbers are 8-byte aligned)
                *reinterpret_cast<float2*>(dst + 2 + s * 16 + quarter * 4) = make_float2(o[s][0], o[s][1]);
                *reinterpret_cast<float2*>(dst + 4 + s * 16 + quarter * 4) = make_float2(o[s][2], o[s][3]);
            }
            return;
        }
        float was, now;
        join(M, L, m, l, was, now);
#pragma unroll
        for (int s = 0; s < ND; s++)
#pragma unroll
            for (int r = 0; r < 4; r++) O[s][r] = fmaf(O[s][r], was, o[s][r] * now);
    }
    if (!col_ok) return;
    const float inv = 1.0f / L;
#pragma unroll
    for (int s = 0; s < ND; s++)
        *reinterpret_cast<float4*>(out + (size_t)tok * ldo + head * D + s * 16 + quarter * 4) =
            make_float4(O[s][0] * inv, O[s][1] * inv, O[s][2] * inv, O[s][3] * inv);
}

// The chunks of a (token, head) one after the other, as the walk puts them together. A lane owns two neighbouring dimensions; the
// chunks' numbers are asked for MERGE_F32 at a time.
#define MERGE_F32 8
__global__ __launch_bounds__(WAVE) void attn_f32_merge_kernel(const float* __restrict__ partial, const int* __restrict__ positions,
                                                              float* __restrict__ out, int ldo, int H, int D, int n_chunks, int window,
                                                              int mask_chunk) {
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const int pos = positions[t], c0 = first_visible(pos, window, mask_chunk) / F32_CHUNK, c1 = pos / F32_CHUNK;
    const size_t rec = D + 2;
    const float* src = partial + (size_t)(t * H + h) * n_chunks * rec;
    const int d = 2 * lane < D ? 2 * lane : 0;
    float M = F32_NONE, L = 0.f, ox = 0.f, oy = 0.f;
    for (int c = c0; c <= c1; c += MERGE_F32) {
        float2 ml[MERGE_F32], v[MERGE_F32];
#pragma unroll
        for (int i = 0; i < MERGE_F32; i++) {
            const float* r = src + (size_t)(c + i <= c1 ? c + i : c1) * rec;
            ml[i] = *reinterpret_cast<const float2*>(r);
            v[i] = *reinterpret_cast<const float2*>(r + 2 + d);
        }
#pragma unroll
        for (int i = 0; i < MERGE_F32; i++) {
            if (c + i > c1) break;
            float was, now;
            join(M, L, ml[i].x, ml[i].y, was, now);
            ox = fmaf(ox, was, v[i].x * now);
            oy = fmaf(oy, was, v[i].y * now);
        }
    }
    const float inv = 1.0f / L;
    if (2 * lane < D) *reinterpret_cast<float2*>(out + (size_t)t * ldo + h * D + d) = make_float2(ox * inv, oy * inv);
}

static int shift_of(int n) {
    int s = 0;
    while ((1 << s) < n) s++;
    return (1 << s) == n ? s : -1;
}

bool attn_f32_supports(const AttnArgs& a) {
    const int dv = a.v_head_dim > 0 ? a.v_head_dim : a.head_dim, vw = a.v_width > 0 ? a.v_width : a.kv_width;
    return a.weights == 0 && !attn_shaped_scores(a) && !a.sink && !a.rel && a.keep_first == 0 && a.v_share <= 1 && !a.gate && a.out_mul == 1.f &&
           a.v_rot == 0 && dv == a.head_dim && vw == a.kv_width && a.head_dim % 32 == 0 && a.head_dim <= 128 && a.n_heads / a.n_kv_heads <= 16 &&
           a.page_tokens >= 4 && shift_of(a.page_tokens) >= 0 && a.q_start != nullptr && a.n_seqs > 0 && a.max_q_len > 0 && a.max_seq_len > 0 &&
           a.n_kv_heads <= 65535 && a.n_heads <= 65535 && a.ldq % 4 == 0 && a.ldo % 4 == 0 && a.kv_width % 4 == 0 && ((uintptr_t)a.q & 15) == 0 &&
           ((uintptr_t)a.out & 15) == 0 && ((uintptr_t)a.k_cache & 15) == 0 && ((uintptr_t)a.v_cache & 15) == 0;
}

template <int ND, int KT>
static int launch(const AttnArgs& a) {
    const int cpt = a.n_heads / a.n_kv_heads, tpt = 16 / cpt, one = a.max_q_len <= tpt ? 1 : 0;
    const long tiles = one ? a.n_seqs : (long)(a.n_tokens + tpt - 1) / tpt + a.n_seqs;
    const int n_chunks = (a.max_seq_len + F32_CHUNK - 1) / F32_CHUNK;
    // Fewer waves than SIMDs: every chunk of keys becomes a wave of its own, if the workspace holds their results.
    const bool split = tiles * a.n_kv_heads < 1024 && n_chunks > 1 && n_chunks <= 65535 && a.workspace != nullptr && ((uintptr_t)a.workspace & 7) == 0 &&
                       (size_t)a.n_tokens * a.n_heads * n_chunks * (a.head_dim + 2) * sizeof(float) <= a.workspace_bytes;
    // single waves as blocks of their own where there are few (they then land on different CUs)
    const int waves = tiles * a.n_kv_heads * (split ? n_chunks : 1) <= 1024 ? 1 : 4;
    const dim3 grid((unsigned)((tiles + waves - 1) / waves), a.n_kv_heads, split ? n_chunks : 1);
    if (split) {
        attn_f32_kernel<ND, KT, true><<<grid, waves * WAVE, 0, a.stream>>>(
            (const float*)a.q, a.ldq, (const float*)a.k_cache, (const float*)a.v_cache, a.kv_width, a.block_table, a.max_blocks, a.token_slot,
            a.positions, a.q_start, a.n_seqs, (float*)a.out, a.ldo, (float*)a.workspace, a.n_heads, shift_of(a.page_tokens), a.window, a.mask_chunk,
            a.scale, tpt, cpt, one, n_chunks);
        HFA_LAUNCH_CHECK("attn_f32");
        attn_f32_merge_kernel<<<dim3(a.n_tokens, a.n_heads), WAVE, 0, a.stream>>>((const float*)a.workspace, a.positions, (float*)a.out, a.ldo, a.n_heads,
                                                                                 a.head_dim, n_chunks, a.window, a.mask_chunk);
    } else {
        attn_f32_kernel<ND, KT, false><<<grid, waves * WAVE, 0, a.stream>>>(
            (const float*)a.q, a.ldq, (const float*)a.k_cache, (const float*)a.v_cache, a.kv_width, a.block_table, a.max_blocks, a.token_slot,
            a.positions, a.q_start, a.n_seqs, (float*)a.out, a.ldo, nullptr, a.n_heads, shift_of(a.page_tokens), a.window, a.mask_chunk,
            a.scale, tpt, cpt, one, n_chunks);
    }
    HFA_LAUNCH_CHECK("attn_f32");
    return 0;
}

int attn_f32_launch(const AttnArgs& a) {
    switch (a.head_dim / 32) {
        case 1: return launch<2, 4>(a);
        case 2: return launch<4, 4>(a);
        case 3: return launch<6, 2>(a);
        default: return launch<8, 2>(a);
    }
}
