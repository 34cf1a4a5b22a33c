// Prompt attention: many query rows of a request against the request's K / V pages.
#include "vox_internal.h"
#include "vox_attn.h"

typedef float f32x16_t __attribute__((ext_vector_type(16)));

struct PromptAttnArgs {
    const bf16_t *q, *kv;
    const int *q_req, *q_kvlen, *indptr, *indices;
    float* scores;           // [Nq][Hq][max_chunks][32]
    bf16_t *out, *out_frag;
    float scale;
    int Nq, Hq, Hkv, G, rows, page_size, page_shift, max_chunks;      // G: q heads per kv head; rows: query rows of a tile (16 / G)
};

// One block per (16 columns = `rows` query rows x G heads of a kv head), NWV waves, over the rows' whole context: the outputs of k_attn_partial and k_attn_merge to
// the bit.  Their sums are chains of fp32 fused multiply-adds, and an MFMA with K = 1 is exactly one link of such a chain for a whole tile: D[i][j] = fma(A[i], B[j],
// C[i][j]) (rounding, denormals and infinities as v_fma_f32: 524 288 chains of 32 compared).  v_mfma_f32_16x16x1_4b takes four tiles at once (lane = tile and row or
// column of it; register i of an output: tile i / 4, row lane / 16 * 4 + i % 4, column lane % 16), 32 multiply-adds a clock and SIMD where the vector units take 16
// beside their unpacking, LDS reads and cross-lane adds, and a chunk's K / V come once per tile instead of once per row:
//  - scores: rows = tokens (two tiles of 16), columns = (query row, head); tiles 0, 1 take piece j and tiles 2, 3 piece j + D / 16 of the head (8 elements, one chain
//    each), which are each other's first partners in the butterfly over the pieces; the rest of it is adds between registers of a lane;
//  - P.V: rows = dims (D = 128: the even ones in one instruction, the odd ones in the next), columns as before, k = token in ascending order.
// Wave w takes chunks w, w + NWV, ..  First all scores and the chunks' maxima (the merge wants the largest of all before it weighs any); the scores go through the
// workspace (32 per column and chunk, a quarter of a partial output), everything else stays on the CU: round by round P.V, whose 16 x D partial outputs meet in LDS, where
// every thread adds its dims over the round's chunks in ascending order.
// K comes by global_load_lds in whole rows (the lanes of a fragment read 16 bytes of 32 rows each: from memory those are 64 cache lines a request, which took four times as
// long as the products), pieces at piece ^ (row & 7).  The next chunk's K rows and the next round's V rows are in flight under this one's products.  Tiles of the longest
// rows come first.  A kv head's blocks follow each other modulo their number: with eight heads an XCD's L2 holds one head's K / V.
// Rows of several requests in a tile: one request after the other, the other columns masked.
// A column's tokens past its own length have p = 0 and, in k_attn_partial, a zero V row; here the V row may be a later token's, so where such a row holds an infinity or
// NaN (0 times it is no zero) the columns of each length go through P.V by themselves, with zero rows behind that length.
// us with the merge, 16 heads on 8, D = 128, k_attn_partial + merge and now: 96 rows 12.0, 11.0, 128 18.8, 11.2, 256 53, 14.3, 450 92, 33, 640 185,
// 43, 1000 704, 91 (the products alone 27: the rest are the trips and the barriers of the rounds, two waves a SIMD).
__device__ __forceinline__ f32x16_t prompt_fma(float x, float y, f32x16_t c) { return __builtin_amdgcn_mfma_f32_16x16x1f32(x, y, c, 0, 0, 0); }
template <int D, int NWV>
__global__ __launch_bounds__(64 * NWV, 2) void k_attn_prompt(PromptAttnArgs a, int nchunk) {
    touch_args(a);
    typedef f32x16_t acc_t;
    constexpr int NC = 16, NJ = D / 16, NS = 8, ROWB = 2 * D, REG = 8192, NK = 32 * ROWB / 1024;
    extern __shared__ __attribute__((aligned(1024))) char pa_lds[];      // [NWV][2][8 KB] | q [16][ROWB] | (l, w) [NWV][16] | maxima [nchunk][16]
    char* const qs = pa_lds + 2 * NWV * REG;
    float2* const lw = reinterpret_cast<float2*>(qs + 16 * ROWB);
    float* const mx = reinterpret_cast<float*>(lw + NWV * 16);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, quad = lane >> 4, half = lane >> 5, tl = lane & 31;
    const int hk = blockIdx.x, row0 = (int)(gridDim.y - 1 - blockIdx.y) * a.rows;
    auto column = [&](int c, int& row, int& head) {      // false: no such column (row and head are the tile's first then)
        const int rr = c / a.G;
        const bool own = rr < a.rows && row0 + rr < a.Nq;
        row = own ? row0 + rr : row0;
        head = hk * a.G + (own ? c - rr * a.G : 0);
        return own;
    };
    int row, head;
    const bool own = column(col, row, head);
    const int L = own ? a.q_kvlen[row] : 0, req = a.q_req[row];
    // the column this thread adds up, pieces md, md + TC, .. of four dims
    constexpr int TC = 4 * NWV, PC = D / 4, NP = (PC + TC - 1) / TC;
    const int mcol = tid / TC, md = tid % TC;
    int mrow, mhead;
    const bool mown = column(mcol, mrow, mhead) && md < PC;
    const int mL = mown ? a.q_kvlen[mrow] : 0, mreq = a.q_req[mrow];
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)pa_lds;
    if (wave < 16 * ROWB / 1024) {      // q: piece p of column c at p ^ (c & 7)
        constexpr int CPI = 1024 / ROWB;      // columns of a request
        const int qc = wave * CPI + lane / (ROWB / 16), pc = (lane % (ROWB / 16)) ^ (qc & 7);
        int r, h;
        column(qc, r, h);
        lds_dma16(a.q + ((size_t)r * a.Hq + h) * D + pc * 8, __builtin_amdgcn_readfirstlane(lds0 + 2 * NWV * REG + wave * 1024));
    }
    const size_t trow = (size_t)a.Hkv * D;      // elements of a token's row; V rows lie page_size rows behind the K rows
    const bf16_t *kvh = a.kv + (size_t)hk * D, *vh = kvh + (size_t)a.page_size * trow;
    const unsigned mine_lds = __builtin_amdgcn_readfirstlane(lds0 + wave * (2 * REG));
    char* const mine_reg = pa_lds + wave * (2 * REG);
    float* const sws = a.scores + ((size_t)row * a.Hq + head) * a.max_chunks * VOX_TC + quad * 4;      // this lane's scores: chunk c at c * 32, + 16
    auto token = [&](int i) { return (i >> 2) * 16 + quad * 4 + (i & 3); };
    auto across = [&](float x, float (&y)[4]) {      // y[n]: quad n's value, in all four of the column
        const vox_u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        const vox_u2 e = __builtin_amdgcn_permlane32_swap(r.x, r.x, false, false), o = __builtin_amdgcn_permlane32_swap(r.y, r.y, false, false);
        y[0] = __uint_as_float(e.x); y[1] = __uint_as_float(o.x); y[2] = __uint_as_float(e.y); y[3] = __uint_as_float(o.y);
    };
    acc_t zero;
#pragma unroll
    for (int i = 0; i < 16; ++i) zero[i] = 0.0f;
    auto store = [&](int u, uint2 y) {
        const int d = mhead * D + (md + u * TC) * 4, K = a.Hq * D;
        *reinterpret_cast<uint2*>(a.out + (size_t)mrow * K + d) = y;
        if (a.out_frag) *reinterpret_cast<uint2*>(a.out_frag + frag_off(mrow, d, K)) = y;
    };
    bool todo = L > 0;
    for (unsigned long long open; (open = __ballot(todo)) != 0;) {      // (the same in every wave)
        const int r0 = __builtin_amdgcn_readlane(req, (int)__builtin_ctzll(open));
        const bool mine = todo && req == r0;
        todo = todo && !mine;
        int Lmax = mine ? L : 0;
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) {
            const int o = __shfl_xor(Lmax, off, VOX_WAVE);
            Lmax = o > Lmax ? o : Lmax;
        }
        Lmax = __builtin_amdgcn_readfirstlane(Lmax);
        int nct = (Lmax + VOX_TC - 1) / VOX_TC;
        nct = nct < nchunk ? nct : nchunk;
        const int* const pages = a.indices + a.indptr[r0];
        // this lane's token of a chunk (those past the last one repeat it), counted in token rows of the cache
        auto place = [&](int c) {
            int tok = c * VOX_TC + tl;
            tok = tok < Lmax ? tok : Lmax - 1;
            const int pi = a.page_shift >= 0 ? tok >> a.page_shift : tok / a.page_size;
            return (u32)pages[pi] * (u32)(2 * a.page_size) + (u32)(tok - pi * a.page_size);
        };
        const u32 first = place(wave < nct ? wave : 0);
        auto request = [&](u32 at, int reg) {
            constexpr int TPI = 1024 / ROWB;      // tokens of a request
#pragma unroll
            for (int n = 0; n < NK; ++n) {
                const int t = n * TPI + lane / (ROWB / 16), pc = (lane % (ROWB / 16)) ^ (t & 7);
                lds_dma16(kvh + (size_t)(u32)__shfl((int)at, t, VOX_WAVE) * trow + pc * 8, __builtin_amdgcn_readfirstlane(mine_lds + reg * REG + n * 1024));
            }
        };
        if (wave < nct) request(first, 0);
        u32 next = wave + NWV < nct ? place(wave + NWV) : 0;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();      // (q is there)
        int reg = 0;
        for (int c = wave; c < nct; c += NWV) {
            if (c > wave) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (c + NWV < nct) request(next, reg ^ 1);      // (in flight under this chunk's products)
            if (c + 2 * NWV < nct) next = place(c + 2 * NWV);
            const char* const kr = mine_reg + reg * REG;
            reg ^= 1;
            // (opaque: sixteen addresses kept across the loops would be spilled)
            u32 kx = (u32)(tl * ROWB + ((NJ * half) ^ (tl & 7)) * 16), qx = (u32)(col * ROWB + ((NJ * half) ^ (col & 7)) * 16);
            asm volatile("" : "+v"(kx), "+v"(qx));
            auto pairs = [&](int j, float (&y)[NS]) {      // pieces j and j + NJ / 2 (the next partners), two chains at a time
                const uint4 k0 = *reinterpret_cast<const uint4*>(kr + (kx ^ (j << 4))), k1 = *reinterpret_cast<const uint4*>(kr + (kx ^ ((j + NJ / 2) << 4)));
                const uint4 q0 = *reinterpret_cast<const uint4*>(qs + (qx ^ (j << 4))), q1 = *reinterpret_cast<const uint4*>(qs + (qx ^ ((j + NJ / 2) << 4)));
                const u32 kw[8] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w}, qw[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
                acc_t d0 = zero, d1 = zero;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    d0 = prompt_fma(bflo(kw[e]), bflo(qw[e]), d0);
                    d1 = prompt_fma(bflo(kw[4 + e]), bflo(qw[4 + e]), d1);
                    d0 = prompt_fma(bfhi(kw[e]), bfhi(qw[e]), d0);
                    d1 = prompt_fma(bfhi(kw[4 + e]), bfhi(qw[4 + e]), d1);
                }
#pragma unroll
                for (int i = 0; i < NS; ++i) y[i] = (d0[i] + d0[NS + i]) + (d1[i] + d1[NS + i]);
            };
            auto add = [&](float (&x)[NS], const float (&y)[NS]) {
#pragma unroll
                for (int i = 0; i < NS; ++i) x[i] = x[i] + y[i];
            };
            float s[NS], w[NS];
            if constexpr (D == 128) {
                float u[NS], x[NS];
                pairs(0, s); pairs(2, u); add(s, u);
                pairs(1, w); pairs(3, x); add(w, x);
            } else {
                pairs(0, s); pairs(1, w);
            }
            add(s, w);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the rows are read: the next ones may land)
            const int nt = mine ? L - c * VOX_TC : 0;
            float mm = -INFINITY, y[4];
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                s[i] = token(i) < nt ? s[i] * a.scale : -INFINITY;
                mm = fmaxf(mm, s[i]);
            }
            across(mm, y);
            if (quad == 0) mx[c * 16 + col] = fmaxf(fmaxf(y[0], y[1]), fmaxf(y[2], y[3]));
            if (mine) {
                float4* const sp = reinterpret_cast<float4*>(sws + c * VOX_TC);
                sp[0] = make_float4(s[0], s[1], s[2], s[3]);
                sp[4] = make_float4(s[4], s[5], s[6], s[7]);
            }
        }
        u32 v[VOX_TC];                // token t of the chunk, dims 2 * lane, + 1 (D = 64: lane & 31)
        auto rows = [&](u32 at) {
#pragma unroll
            for (int t = 0; t < VOX_TC; ++t)
                v[t] = reinterpret_cast<const u32*>(vh + (size_t)(u32)__builtin_amdgcn_readlane((int)at, t) * trow)[D == 128 ? lane : lane & 31];
        };
        float4 s0, s1;                // ... and its scores
        auto scores = [&](int c) {
            const float4* const sp = reinterpret_cast<const float4*>(sws + c * VOX_TC);
            s0 = sp[0]; s1 = sp[4];
        };
        if (wave < nct) { scores(wave); rows(first); }
        next = wave + NWV < nct ? place(wave + NWV) : 0;
        __syncthreads();
        float M = -INFINITY;
        const int ncol = mine ? (L + VOX_TC - 1) / VOX_TC : 0;
        for (int c = 0; c < nct; ++c) {
            const float x = mx[c * 16 + col];
            if (c < ncol) M = fmaxf(M, x);
        }
        const int mnc = mown && mL > 0 && mreq == r0 ? (mL + VOX_TC - 1) / VOX_TC : 0;
        float O[NP][4], Ls = 0.0f;
#pragma unroll
        for (int u = 0; u < NP; ++u) O[u][0] = O[u][1] = O[u][2] = O[u][3] = 0.0f;
        for (int c0 = 0; c0 < nct; c0 += NWV) {
            const int c = c0 + wave;
            if (c < nct) {
                const int left_t = L - c * VOX_TC, nt = mine && left_t > 0 ? (left_t < VOX_TC ? left_t : VOX_TC) : 0;
                const int ntile = Lmax - c * VOX_TC < VOX_TC ? Lmax - c * VOX_TC : VOX_TC;
                float s[NS] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
                const float m = mx[c * 16 + col];
#pragma unroll
                for (int i = 0; i < NS; ++i) s[i] = token(i) < nt ? exp2_flat((s[i] - m) * VOX_LOG2E) : 0.0f;
                const float w = exp2_flat((m - M) * VOX_LOG2E);
                const bool ragged = __any(nt > 0 && nt < VOX_TC);      // (rows past the last token repeat it)
                bool special = false;
                if (ragged) {
#pragma unroll
                    for (int t = 0; t < VOX_TC; ++t) special = special || (v[t] & 0x7f80u) == 0x7f80u || (v[t] & 0x7f800000u) == 0x7f800000u;
                    special = __any(special);
                }
                unsigned long long left = __ballot(nt > 0);
                while (left) {
                    const int lim = special ? __builtin_amdgcn_readlane(nt, (int)__builtin_ctzll(left)) : ntile;
                    const bool sel = nt > 0 && (!special || nt == lim);
                    if (special) rows(place(c));
                    if (ragged)
#pragma unroll
                        for (int t = 0; t < VOX_TC; ++t) v[t] = t < lim ? v[t] : 0u;
                    acc_t o0 = zero, o1 = zero;
                    float l = 0.0f;
#pragma unroll
                    for (int g = 0; g < 2; ++g) {
                        float p[4][4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) across(s[g * 4 + i], p[i]);
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            const float pt = p[i & 3][i >> 2];
                            const u32 vt = v[16 * g + i];
                            l = l + pt;
                            if constexpr (D == 128) {
                                o0 = prompt_fma(bflo(vt), pt, o0);
                                o1 = prompt_fma(bfhi(vt), pt, o1);
                            } else {
                                o0 = prompt_fma(half ? bfhi(vt) : bflo(vt), pt, o0);
                            }
                        }
                    }
                    left &= ~__ballot(sel);
                    if (!sel) continue;
                    constexpr int PER = D == 128 ? 16 : 8;      // registers that hold even dims
#pragma unroll
                    for (int i0 = 0; i0 < PER; i0 += 4) {
                        float y[8];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            y[2 * i] = o0[i0 + i];
                            y[2 * i + 1] = D == 128 ? o1[i0 + i] : o0[PER + i0 + i];
                        }
                        const int p4 = 2 * (i0 + quad);         // 16-byte pieces of the column's D sums, at piece ^ (column & 7)
                        float* const ob = reinterpret_cast<float*>(mine_reg) + col * D;
                        *reinterpret_cast<float4*>(ob + ((p4 ^ (col & 7)) << 2)) = make_float4(y[0], y[1], y[2], y[3]);
                        *reinterpret_cast<float4*>(ob + (((p4 + 1) ^ (col & 7)) << 2)) = make_float4(y[4], y[5], y[6], y[7]);
                    }
                    if (quad == 0) lw[wave * 16 + col] = make_float2(l, w);
                }
                if (c + NWV < nct) { scores(c + NWV); rows(next); }      // (in flight while the round is added up)
                if (c + 2 * NWV < nct) next = place(c + 2 * NWV);
            }
            __syncthreads();
#pragma unroll
            for (int w = 0; w < NWV; ++w) {
                if (c0 + w >= mnc) continue;
                const float2 f = lw[w * 16 + mcol];
                Ls = __fmaf_rn(f.x, f.y, Ls);
#pragma unroll
                for (int u = 0; u < NP; ++u) {
                    const float4 o = *reinterpret_cast<const float4*>(pa_lds + w * (2 * REG) + mcol * (4 * D) + (((md + u * TC) ^ (mcol & 7)) << 4));
                    O[u][0] = __fmaf_rn(o.x, f.y, O[u][0]);
                    O[u][1] = __fmaf_rn(o.y, f.y, O[u][1]);
                    O[u][2] = __fmaf_rn(o.z, f.y, O[u][2]);
                    O[u][3] = __fmaf_rn(o.w, f.y, O[u][3]);
                }
            }
            __syncthreads();
        }
        if (mnc > 0)
#pragma unroll
            for (int u = 0; u < NP; ++u) store(u, make_uint2(pack_bf2(O[u][0] / Ls, O[u][1] / Ls), pack_bf2(O[u][2] / Ls, O[u][3] / Ls)));
    }
    if (mown && mL <= 0) {      // a row without tokens: 0 / 0, as the merge leaves it
        const float z = 0.0f, y = z / z;
#pragma unroll
        for (int u = 0; u < NP; ++u) store(u, make_uint2(pack_bf2(y, y), pack_bf2(y, y)));
    }
}

template <int D, int NWV>
static int launch_prompt_t(hipStream_t st, const PromptAttnArgs& a, int nchunk) {
    const int lds = NWV * 16384 + 16 * 2 * D + NWV * 16 * 8 + nchunk * 16 * 4;
    const auto kern = k_attn_prompt<D, NWV>;
    VOX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    hipLaunchKernelGGL(kern, dim3(a.Hkv, (a.Nq + a.rows - 1) / a.rows), dim3(64 * NWV), lds, st, a, nchunk);
    return VOX_OK;
}
static int prompt_blocks(const AttnCall& c) {
    const int rows = 16 / (c.Hq / c.Hkv);
    return c.Hkv * ((c.Nq + rows - 1) / rows);
}
static int requests(const AttnCall& c) { return c.n_req < 1 || c.n_req > c.Nq ? c.Nq : c.n_req; }
float vox_attn_seen(const AttnCall& c, int nchunk) {      // (a prompt's rows alone see half of it on average)
    const float own = (float)c.Nq / (64.0f * nchunk * requests(c));
    return own < 0.5f ? 1.0f - own : 0.5f;
}
static bool four_waves(const AttnCall& c) { return prompt_blocks(c) > (c.D == 64 ? 256 : 512); }
// What k_attn_partial and k_attn_merge take and what this kernel takes, us, fitted to 2 to 1000 rows behind 0 to 1500 tokens, 1 to 8 kv heads of 1 to 16 q heads.  The
// former by blocks (row, kv head, chunk; a prompt's rows see half of it), the latter by rounds of eight chunks (a last one of up to four is shorter), of which a tile's block goes
// through one after the other while the chip may be idle.  A tile takes its rows' requests one after the other: at most as many as it has rows, and since no request has more rows than the call
// has tokens, at most two beyond those that the call's rows leave over.  Measured, former / latter: 16 heads on 8, D = 128, no context: 64 rows 8.6 / 10.8, 96 12.0 / 11.0; behind 1500 tokens: 2 rows 12 / 59,
// 32 48 / 60, 64 84 / 65, 128 152 / 67; 32 heads on 8, D = 64, behind 700: 16 rows 17 / 24, 48 35 / 25; 32 heads on 2: 48 rows 14.0 / 9.5, behind 1500: 32 48 / 60, 64 81 / 65; 14 on 2, D = 64, behind 200:
// 30 rows 8.6 / 11.4, 128 17.1 / 15.8; 24 on 8, D = 128: 96 rows 13.4 / 11.4.
// One row a request (one per tile and pass), 16 heads on 8, D = 128: 64 rows of 1500 tokens 115 / 516, 128 of 600 93 / 234; 32 heads on 8, D = 64: 128 of 600 71 / 93; 32 heads on 2 (a row
// a tile) 65 / 37.  16 heads on 8: a prompt of 75 rows beside 31 of one row behind 300 tokens 25 / 149, eight prompts of 128 rows 105 / 28, four of 250 189 / 44.
void vox_attn_prompt_us(const AttnCall& c, int nchunk, float& parts, float& prompt) {
    const float G = (float)(c.Hq / c.Hkv), seen = vox_attn_seen(c, nchunk);
    parts = 6.3f + 0.3f * G * c.D / 128 + (float)c.Nq * c.Hkv * nchunk * seen * (0.00195f + 0.0000053f * G * c.D);
    const int req = requests(c), rows = 16 / (c.Hq / c.Hkv), tiles = (c.Nq + rows - 1) / rows;
    int passes = 1;
    if (req > 1) {
        const int whole = c.Nq > rows ? (c.Nq - rows + c.max_kvlen - 1) / c.max_kvlen : 0, left = req - whole + 2;
        passes = left < 1 ? 1 : left;
        if (passes > rows) passes = rows;
        if (passes > req) passes = req;
    }
    const bool four = passes > 1 && four_waves(c);
    const float round = c.D == 64 ? 6.8f : 9.5f, half = c.D == 64 ? 2.1f : 3.2f;
    const float pass = four ? round * ((nchunk + 3) / 4) : round * ((nchunk + 7) / 8) - ((nchunk - 1) % 8 < 4 ? half : 0.0f);
    const float longest = passes * pass, all = round * c.Hkv * (tiles + req - 1) * seen * nchunk / 2048.0f;
    prompt = 4.7f + (longest > all ? longest : all);
}
static bool prompt_pays(const AttnCall& c, int nchunk) {
    float parts, prompt;
    vox_attn_prompt_us(c, nchunk, parts, prompt);
    return prompt < parts;
}
bool vox_attn_prompt_supported(const AttnCall& c) {
    const int G = c.Hkv > 0 ? c.Hq / c.Hkv : 0, nchunk = (c.max_kvlen + VOX_TC - 1) / VOX_TC;
    const size_t at = (size_t)c.q | (size_t)c.kv | (size_t)c.part_o | (size_t)c.out | (size_t)c.out_frag;
    return c.Nq > 0 && c.out && !c.qkv && !c.ptab && !c.identity_pages && c.fixed_kvlen <= 0 && (c.D == 128 || c.D == 64) && G >= 1 && G <= 16 && c.Hq == G * c.Hkv &&
           (at & 15) == 0 && nchunk > 1 && nchunk <= c.max_chunks && nchunk <= 256 && prompt_pays(c, nchunk);
}
int vox_launch_attn_prompt(hipStream_t st, const AttnCall& c) {
    PromptAttnArgs a{};
    a.q = (const bf16_t*)c.q; a.kv = (const bf16_t*)c.kv; a.q_req = c.q_req; a.q_kvlen = c.q_kvlen; a.indptr = c.indptr; a.indices = c.indices;
    a.scores = c.part_o; a.out = (bf16_t*)c.out; a.out_frag = (bf16_t*)c.out_frag; a.scale = c.scale; a.Nq = c.Nq; a.Hq = c.Hq; a.Hkv = c.Hkv; a.G = c.Hq / c.Hkv;
    a.rows = 16 / a.G; a.page_size = c.page_size; a.page_shift = -1; a.max_chunks = c.max_chunks;
    if ((c.page_size & (c.page_size - 1)) == 0) a.page_shift = __builtin_ctz((unsigned)c.page_size);
    const int nchunk = (c.max_kvlen + VOX_TC - 1) / VOX_TC;
    // four waves and two blocks to a CU where there are blocks for it (one's trips behind the other's products, shorter last rounds), else eight.  us, eight / four: 16 heads on
    // 8, D = 128: 256 rows (256 blocks) 14.3 / 18.2, 450 (456) 32.7 / 34.3, 640 (640) 52.2 / 42.8, 1000 101 / 91; 32 heads on 8, D = 64: 128 rows (256) 10.7 / 10.9, 160 (320)
    // 17.2 / 14.1, 1000 148 / 120
    const bool four = four_waves(c);
    if (c.D == 128) return four ? launch_prompt_t<128, 4>(st, a, nchunk) : launch_prompt_t<128, 8>(st, a, nchunk);
    return four ? launch_prompt_t<64, 4>(st, a, nchunk) : launch_prompt_t<64, 8>(st, a, nchunk);
}
