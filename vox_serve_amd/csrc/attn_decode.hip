// Decode attention over long contexts: one query row per request, its new token's K / V among the rows it sees.  Rows of short prompts: the same with q prepared and every
// token's K / V in the pages.
#include "vox_internal.h"
#include "vox_attn.h"

__device__ u32 dec_zero_row[64];      // a V row behind a chunk's last token

template <int OFF>
__device__ __forceinline__ float xor_max(float s) {
    if constexpr (OFF == 32) {
        const vox_u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false);
        return fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
    } else if constexpr (OFF == 16) {
        const vox_u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s), false, false);
        return fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
    } else {
        static_assert(OFF == 8, "rows of 16 lanes");
        return fmaxf(s, vox_dpp<0x128, 0xF>(s, s));      // row_ror:8
    }
}
// One block of NWV waves per (row, G heads of a kv head): a wave takes the chunks w, w + NWV, .. of 32 tokens by itself, from memory to its partial output, without LDS
// and without a barrier; the partial outputs stay in LDS until the block merges them.  The arithmetic is k_attn_partial<D, true>'s and k_attn_merge's.
//  - K: 16 bytes a lane, whole rows per request, straight into the registers that are multiplied (lane = token and piece of 8 dims: the order of the scores' sums);
//  - the scores go through a row of LDS per head, after which a lane has one token's of one head (G = 4: of two) for the exponential;
//  - V: a lane has two dims (D = 64: one) of every token; p comes by v_readlane as a scalar operand.
// The next chunk's K rows are in flight under the softmax and P.V, its V rows under the next scores.  us a Qwen3-TTS layer of 32 rows, before and now: 2000 tokens (262 MB) 91, 55.8
// (4.7 TB/s), 325 tokens (43 MB) 18.3, 14.8 (one chunk of a wave: the trip of its rows, 750 vector instructions, the merge).
// PREP: a decode row, whose q and newest k and v come from the projection (norm, RoPE and append here); else a.q and the pages hold them.
template <int D, int G, int NWV, bool PREP>
__global__ __launch_bounds__(64 * NWV, PREP ? 1 : 4) void k_attn_decode(AttnArgs a, int nchunk) {
    touch_args(a);
    constexpr int LPT = D / 8, TPW = 64 / LPT, NP = VOX_TC / TPW, NS = G * NP, E = (G + 1) / 2;
    extern __shared__ __attribute__((aligned(16))) char dec_lds[];      // partial outputs [nchunk][G][D] | (m, l) [nchunk][G] | weights [nchunk][G]
    __shared__ __attribute__((aligned(16))) uint4 Qs[G * LPT];
    __shared__ float S[NWV][G * VOX_TC];
    __shared__ float Sh[(G + 1) * D];
    __shared__ __attribute__((aligned(16))) bf16_t Knew[D];
    float* const Po = reinterpret_cast<float*>(dec_lds);
    float2* const Pml = reinterpret_cast<float2*>(Po + (size_t)nchunk * G * D);
    float* const Wm = reinterpret_cast<float*>(Pml + (size_t)nchunk * G);
    const int HS = gridDim.x / a.Hkv, hk = blockIdx.x / HS, hs = blockIdx.x - hk * HS, row = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane % LPT, tg = lane / LPT;
    const int* const pages = a.ptab ? a.ptab + (size_t)row * a.pt_stride : a.indices + a.indptr[a.q_req[row]];
    // (a row longer than its call says ends with the chunks that LDS was asked for)
    const int Lr = a.q_kvlen[row], L = Lr < nchunk * VOX_TC ? Lr : nchunk * VOX_TC, pg_new = PREP ? a.page[row] : -1, sl_new = PREP ? a.slot[row] : 0;
    const int nc = (L + VOX_TC - 1) / VOX_TC, Gf = a.Hq / a.Hkv, h0 = hk * Gf + hs * G;
    const size_t trow = (size_t)a.Hkv * D, ps = (size_t)2 * a.page_size * trow;
    const bf16_t* const raw = PREP ? a.qkv + (size_t)row * (a.Hq + 2 * a.Hkv) * D : a.q + ((size_t)row * a.Hq + h0) * D;
    const bf16_t* const vnew = PREP ? raw + (size_t)(a.Hq + a.Hkv + hk) * D : nullptr;
    uint4 k[NP];
    u32 v[VOX_TC];                // D = 128: dims 2 lane, 2 lane + 1 of token t; D = 64: dim lane
    const u32 k_at = tg * (u32)trow + j * 8, v_at = lane * (D / 64);      // elements
    // (a chunk lies in one page; what the page holds behind the row's cached tokens is read and not used.  Scalar bases, one 32-bit offset a lane)
    auto k_rows = [&](int c) {
        const int tok = c * VOX_TC, pi = page_of(a, tok);
        // (a chunk of the newest token alone reads page 0 for nothing: its entry of the table may not be there yet, and a padding row has none)
        const int pg = !PREP || tok < L - 1 ? __builtin_amdgcn_readfirstlane(pages[pi]) : 0;
        return a.kv + (size_t)pg * ps + ((size_t)(tok - pi * a.page_size) * a.Hkv + hk) * D;
    };
    auto fetch_k = [&](const bf16_t* kb) {
#pragma unroll
        for (int n = 0; n < NP; ++n, kb += TPW * trow) k[n] = *reinterpret_cast<const uint4*>(kb + k_at);
    };
    auto fetch_v = [&](int c, const bf16_t* vb) {
        vb += (size_t)a.page_size * trow;
        auto dims = [&](const bf16_t* r) { return D == 128 ? *reinterpret_cast<const u32*>(r + v_at) : (u32)r[v_at]; };
        if (c < nc - 1) {
#pragma unroll
            for (int t = 0; t < VOX_TC; ++t, vb += trow) v[t] = dims(vb);
        } else {                  // the newest token's row is the projection's, zeros behind it
            const int last = L - 1 - c * VOX_TC;
#pragma unroll
            for (int t = 0; t < VOX_TC; ++t, vb += trow) v[t] = dims(t < last + !PREP ? vb : PREP && t == last ? vnew : reinterpret_cast<const bf16_t*>(dec_zero_row));
        }
    };
    float* const Sw = S[wave];
    int c = wave;
    PrepOps po;
    uint4 qv[G];
    int p = PREP ? a.pos[row] : 0;
    p = p < 0 ? 0 : (p >= a.table_max_pos ? a.table_max_pos - 1 : p);
    const float* const cs_row = PREP && a.cs ? a.cs + (size_t)p * (a.rot >> 1) * 2 : nullptr;
    const bf16_t* const nw = wave == G ? a.kn : a.qn;
    if (!PREP) {
#pragma unroll
        for (int g = 0; g < G; ++g) qv[g] = reinterpret_cast<const uint4*>(raw)[g * LPT + j];
    } else if (wave <= G) po = prep_head_load<D>(wave == G ? raw + (size_t)(a.Hq + hk) * D : raw + (size_t)(h0 + wave) * D, nw, cs_row, a.rot, lane);
    const bf16_t* kb = a.kv;
    if (c < nc) {
        kb = k_rows(c);
        fetch_k(kb);
        fetch_v(c, kb);
    }
    if (PREP && wave <= G) prep_head_apply<D>(po, nw, a.eps, cs_row, a.rot, a.interleave, Sh + wave * D, wave == G ? Knew : reinterpret_cast<bf16_t*>(Qs) + (size_t)wave * D, lane);
    if (PREP) __syncthreads();
    float qf[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const uint4 q = PREP ? Qs[g * LPT + j] : qv[g];
        const u32 w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) { qf[g][2 * e] = bflo(w[e]); qf[g][2 * e + 1] = bfhi(w[e]); }
    }
    while (c < nc) {
        const int nt = L - c * VOX_TC < VOX_TC ? L - c * VOX_TC : VOX_TC;
        if (PREP && c == nc - 1) {        // the row's newest token is the last one
            const uint4 kn = reinterpret_cast<const uint4*>(Knew)[j];
#pragma unroll
            for (int n = 0; n < NP; ++n)
                if (n == (nt - 1) / TPW && tg == (nt - 1) % TPW) k[n] = kn;
            if (hs == 0 && pg_new >= 0 && lane < LPT) {        // append it to the cache (page < 0: graph padding row)
                bf16_t* const base = a.kv_w + (size_t)pg_new * ps + ((size_t)sl_new * a.Hkv + hk) * D;
                reinterpret_cast<uint4*>(base)[lane] = kn;
                reinterpret_cast<uint4*>(base + (size_t)a.page_size * trow)[lane] = reinterpret_cast<const uint4*>(vnew)[lane];
            }
        }
        float s[NS];
#pragma unroll
        for (int n = 0; n < NP; ++n) {
            if (n % 2 == 0) __builtin_amdgcn_sched_barrier(0);
            const u32 w[4] = {k[n].x, k[n].y, k[n].z, k[n].w};
            float kf[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) { kf[2 * e] = bflo(w[e]); kf[2 * e + 1] = bfhi(w[e]); }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                float d = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) d = __fmaf_rn(qf[g][e], kf[e], d);
                if constexpr (LPT == 16) {      // (behind the first step a value repeats every 8 lanes: lane ^ 4 and lane + 4 hold the same)
                    d = xor_add<8>(d);
                    d = d + vox_dpp<0x124, 0xF>(d, d);
                    d = xor_add<1>(xor_add<2>(d));
                } else {
                    d = butterfly<LPT>(d);
                }
                s[g * NP + n] = d * a.scale;
            }
        }
        const int cc = c;
        c += NWV;
        if (PREP && c < nc) {     // (the next chunk's K rows under this one's outputs, its V rows under its scores)
            kb = k_rows(c);
            fetch_k(kb);
        }
        if (j == 0)
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int n = 0; n < NP; ++n) Sw[g * VOX_TC + n * TPW + tg] = s[g * NP + n];
        __builtin_amdgcn_wave_barrier();
        float m[E], pe[E];        // lane: token lane % 32 of head e * 2 + lane / 32 (G = 1: both halves the same)
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float x = (lane & 31) < nt ? Sw[G == 1 ? lane & 31 : e * 64 + lane] : -INFINITY;
            float mm = xor_max<8>(xor_max<16>(x));
            mm = fmaxf(mm, vox_dpp<0x124, 0xF>(mm, mm));
            mm = fmaxf(mm, vox_dpp<0x122, 0xF>(mm, mm));
            m[e] = fmaxf(mm, vox_dpp<0x121, 0xF>(mm, mm));
            pe[e] = exp2_flat((x - m[e]) * VOX_LOG2E);        // (0 for the masked ones)
        }
        __builtin_amdgcn_wave_barrier();
        float o0[G], o1[G], l[G];
#pragma unroll
        for (int g = 0; g < G; ++g) o0[g] = o1[g] = l[g] = 0.0f;
#pragma unroll
        for (int t = 0; t < VOX_TC; ++t) {
            if (t % 4 == 0) __builtin_amdgcn_sched_barrier(0);      // (a few tokens' operands at a time)
            const float v0 = bflo(v[t]), v1 = bfhi(v[t]);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const float pt = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(pe[g / 2]), (g & 1) * 32 + t));
                l[g] = l[g] + pt;
                o0[g] = __fmaf_rn(pt, v0, o0[g]);
                if constexpr (D == 128) o1[g] = __fmaf_rn(pt, v1, o1[g]);
            }
        }
        if (PREP && c < nc) fetch_v(c, kb);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float* const o = Po + ((size_t)cc * G + g) * D;
            if constexpr (D == 128) reinterpret_cast<float2*>(o)[lane] = make_float2(o0[g], o1[g]);
            else o[lane] = o0[g];
            if (lane == (g & 1) * 32) Pml[cc * G + g] = make_float2(m[g / 2], l[g]);
        }
        if (!PREP) break;         // (a chunk a wave)
    }
    __syncthreads();
    if (wave < G) {               // the chunks' weights against the largest of their maxima
        float M = -INFINITY;
        for (int i = lane; i < nc; i += 64) M = fmaxf(M, Pml[i * G + wave].x);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, VOX_WAVE));
        for (int i = lane; i < nc; i += 64) Wm[i * G + wave] = exp2_flat((Pml[i * G + wave].x - M) * VOX_LOG2E);
    }
    __syncthreads();
    if (tid >= G * D) return;
    const int g = tid / D, d = tid % D;
    float Ls = 0.0f, O = 0.0f;
#pragma unroll 8
    for (int i = 0; i < nc; ++i) {
        const float w = Wm[i * G + g];
        Ls = __fmaf_rn(Pml[i * G + g].y, w, Ls);
        O = __fmaf_rn(Po[((size_t)i * G + g) * D + d], w, O);
    }
    const bf16_t r = f2bf(O / Ls);
    a.out[((size_t)row * a.Hq + h0 + g) * D + d] = r;
    if (a.out_frag) a.out_frag[frag_off(row, (h0 + g) * D + d, a.Hq * D)] = r;
}

// Heads of a block, 0: not a call for this kernel.  One head and sixteen waves (128 registers) while that is no more than a block per CU, else two heads, which share the K and
// V rows, and eight waves.  More than eight chunks (k_attn_decode8 takes the others: one request of 128 tokens of GLM-4-Voice 3592 / 3528 us a frame there and here, eight
// 3714 / 3792; Qwen3-TTS 8 x 100 3015 / 3032), and enough blocks for the rounds of a block's waves over its chunks, where k_attn_partial has a block per chunk.  us a frame,
// k_attn_partial + merge (up to 512 tokens from 16 rows on k_attn_decode8) and this kernel, rows x tokens, Qwen3-TTS: 2 x 300 2799 / 2838, 4 x 300 3137 / 3092, 4 x 1000 3217 / 3317,
// 8 x 600 3382 / 3231, 8 x 2000 3765 / 3818, 12 x 1400 3957 / 3607, 16 x 2000 4327 / 4137, 32 x 325 3749 / 3646, 32 x 600 4552 / 3822, 32 x 2000 5742 / 4766; CSM 4 x 1000 4335 / 4363,
// 8 x 600 4490 / 4419, 16 x 1000 4701 / 4631; sixteen heads on a kv head (GLM-4-Voice), whose chunk blocks are long: 1 x 300 3897 / 3591, 1 x 1000 3954 / 3783, 8 x 1000 4261 / 4169.
// LDS and the estimate go by the call's bound, which a graph's rows may be far below: a layer of 32 rows of Qwen3-TTS in calls of 2048 with 2000 / 1030 tokens 118 / 87, 106 / 65, of 4096 with 4000
// / 2100 196 / 138, 151 / 93 (134 KB of LDS: a block to a CU); 24 rows of 4000 157 / 120, 12 of 1000 42 / 39, of 2000 58 / 54.  Sixteen heads: a chunk's K and V are fetched by eight blocks of two
// heads here and by one there, which pays while no CU has two of them: a layer of 16 rows of 300 38.8 / 33.2, of 1000 46.2 / 46.1, 24 of 300 53.0 / 53.3, of 1000 69 / 78, 64 of 2000 157 / 208.
static int decode_heads(const AttnCall& c) {
    const int G = c.Hkv > 0 ? c.Hq / c.Hkv : 0, nchunk = (c.max_kvlen + VOX_TC - 1) / VOX_TC;
    const size_t at = (size_t)c.qkv | (size_t)c.kv | (size_t)c.qn | (size_t)c.kn;
    if (!c.qkv || !c.out || c.identity_pages || c.fixed_kvlen > 0 || !c.page || !c.slot || c.Nq < 1 || c.Hq != G * c.Hkv || c.page_size % VOX_TC || nchunk <= 8 ||
        nchunk > 128 || (at & 15) || ((size_t)c.cs & 7)) return 0;
    if (!((c.D == 128 && (G == 2 || G == 16)) || (c.D == 64 && G == 4))) return 0;
    if (G == 16 ? nchunk > 32 || c.Nq * c.Hkv > 32 : 2 * c.Nq * c.Hkv < 3 * nchunk) return 0;
    return c.Hq * c.Nq <= 256 ? 1 : 2;
}
bool vox_attn_decode_supported(const AttnCall& c) { return decode_heads(c) > 0; }
template <int D, int G, int NWV, bool PREP>
static int launch_decode(hipStream_t st, const AttnArgs& a, int Nq, int nchunk) {
    const int lds = nchunk * G * (D * 4 + 8 + 4);
    const auto kern = k_attn_decode<D, G, NWV, PREP>;
    if (lds > 60 * 1024) VOX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));
    hipLaunchKernelGGL(kern, dim3(a.Hq / G, Nq), dim3(64 * NWV), lds, st, a, nchunk);
    return VOX_OK;
}
int vox_launch_attn_decode(hipStream_t st, const AttnCall& c) {
    AttnArgs a{};
    a.q_req = c.q_req; a.q_kvlen = c.q_kvlen; a.indptr = c.indptr; a.indices = c.indices; a.scale = c.scale; a.kv = (const bf16_t*)c.kv;
    a.Hq = c.Hq; a.Hkv = c.Hkv; set_page_size(a, c.page_size); a.max_chunks = c.max_chunks;
    a.qkv = (const bf16_t*)c.qkv; a.kv_w = (bf16_t*)const_cast<void*>(c.kv); a.qn = (const bf16_t*)c.qn; a.kn = (const bf16_t*)c.kn; a.cs = c.cs;
    a.pos = c.pos; a.page = c.page; a.slot = c.slot; a.eps = c.eps; a.rot = c.rot; a.interleave = c.interleave; a.table_max_pos = c.table_max_pos;
    a.ptab = c.ptab; a.pt_stride = c.pt_stride; a.out = (bf16_t*)c.out; a.out_frag = (bf16_t*)c.out_frag;
    const int G = decode_heads(c), nchunk = (c.max_kvlen + VOX_TC - 1) / VOX_TC;
    if (c.D == 128) return G == 1 ? launch_decode<128, 1, 16, true>(st, a, c.Nq, nchunk) : launch_decode<128, 2, 8, true>(st, a, c.Nq, nchunk);
    return G == 1 ? launch_decode<64, 1, 16, true>(st, a, c.Nq, nchunk) : launch_decode<64, 2, 8, true>(st, a, c.Nq, nchunk);
}

// Rows of up to eight chunks that read q and their pages, a wave per chunk (108 registers, D = 64: 90, since no wave goes on to a next chunk), four waves a block for up to four
// chunks.  One launch of short trips instead of k_attn_partial's barriers and a merge, but every row fetches its own K and V, where k_attn_prompt's tiles share them: by estimates
// fitted to 2 to 250 rows behind 0 to 190 tokens.  us, k_attn_partial + merge or k_attn_prompt / this kernel, 16 heads on 8, D = 128, no context: 33 rows 7.4 / 5.1, 64 8.4 / 5.2,
// 75 9.4 / 6.5, 96 11.6 / 6.5, 128 11.0 / 8.1, 144 13.1 / 13.5 (eight waves), 250 14.1 / 21.8; behind 100: 8 rows 7.4 / 5.1, 64 13.4 / 7.7, 128 14.1 / 14.5; 32 heads on 8, D = 64:
// 48 7.2 / 4.7, 96 9.4 / 8.5, 128 9.7 / 9.8; 32 heads on 2: 48 10.5 / 5.4, 96 11.0 / 10.7, behind 190 24 13.6 / 9.2, 64 13.9 / 15.2.
static bool rows_pay(const AttnCall& c, int nchunk) {
    const float seen = vox_attn_seen(c, nchunk);
    const int blocks = c.Nq * c.Hq / 2, slots = nchunk > 4 ? 512 : c.D == 64 ? 1280 : 1024, rounds = (blocks + slots - 1) / slots;
    const float waves = (float)blocks * nchunk * seen, round = c.D == 64 ? 1.7f : nchunk > 4 ? 1.9f : 2.0f;
    const float wave = nchunk > 4 ? (c.D == 64 ? 0.0008f : 0.00105f) : c.D == 64 ? 0.00135f : 0.00155f, base = nchunk > 4 ? (c.D == 64 ? 3.2f : 4.0f) : c.D == 64 ? 1.8f : 2.1f;
    float parts, prompt;
    vox_attn_prompt_us(c, nchunk, parts, prompt);
    return base + round * rounds + wave * waves < (parts < prompt ? parts : prompt);
}
// (one row is no prompt: it stays with k_attn_partial, the form that tests hold this one and k_attn_prompt to)
bool vox_attn_rows_supported(const AttnCall& c) {
    const int G = c.Hkv > 0 ? c.Hq / c.Hkv : 0, nchunk = (c.max_kvlen + VOX_TC - 1) / VOX_TC;
    const size_t at = (size_t)c.q | (size_t)c.kv;
    return c.q && !c.qkv && c.out && !c.ptab && !c.identity_pages && c.fixed_kvlen <= 0 && c.Nq > 1 && c.Hq == G * c.Hkv && G >= 2 && G <= 16 && G % 2 == 0 && (c.D == 128 || c.D == 64) &&
           c.page_size % VOX_TC == 0 && nchunk > 1 && nchunk <= 8 && (at & 15) == 0 && rows_pay(c, nchunk);
}
int vox_launch_attn_rows(hipStream_t st, const AttnCall& c) {
    AttnArgs a{};
    a.q = (const bf16_t*)c.q; a.q_req = c.q_req; a.q_kvlen = c.q_kvlen; a.indptr = c.indptr; a.indices = c.indices; a.scale = c.scale; a.kv = (const bf16_t*)c.kv;
    a.Hq = c.Hq; a.Hkv = c.Hkv; set_page_size(a, c.page_size); a.max_chunks = c.max_chunks; a.out = (bf16_t*)c.out; a.out_frag = (bf16_t*)c.out_frag;
    const int nchunk = (c.max_kvlen + VOX_TC - 1) / VOX_TC;
    if (c.D == 128) return nchunk <= 4 ? launch_decode<128, 2, 4, false>(st, a, c.Nq, nchunk) : launch_decode<128, 2, 8, false>(st, a, c.Nq, nchunk);
    return nchunk <= 4 ? launch_decode<64, 2, 4, false>(st, a, c.Nq, nchunk) : launch_decode<64, 2, 8, false>(st, a, c.Nq, nchunk);
}
