// What the decode and prompt attention kernels share: their arguments, and a head's norm and RoPE.
#pragma once
#include "vox_device.h"

// element offset of (row r, column k) of a [*, K] matrix in fragment-major form
__device__ __forceinline__ size_t frag_off(int r, int k, int K) {
    return ((size_t)(r >> 4) * (K >> 5) + (k >> 5)) * 512 + (size_t)(((r & 15) + 16 * ((k & 31) >> 3)) * 8 + (k & 7));
}

struct AttnArgs {
    const bf16_t *q, *kv;
    const int *q_req, *q_kvlen, *indptr, *indices;
    float *part_o, *part_ml;
    float scale;
    int Hq, Hkv, page_size, max_chunks;
    int hnd_probe;      // development builds only (VOX_ATTN_HND_PROBE=1)
    int page_shift;     // log2(page_size) when it is a power of two (set_page_size), else -1: token -> (page, slot) by shift / mask instead of
                        // an integer division per K/V element (no divide instruction: ~40 VALU each; 8..16 of them per thread stood in
                        // front of the K/V requests of every decode attention)
    // fused decode mode: q/k/v of each row's own (newest) token come straight from the projection output;
    // per-head norm + RoPE happen here and the block owning the last chunk appends K/V to the cache.
    const bf16_t* qkv;      // [N, (Hq+2Hkv)*D]
    bf16_t* kv_w;           // writable alias of kv
    const bf16_t *qn, *kn;
    const float* cs;
    const int *pos, *page, *slot;
    float eps;
    int rot, interleave, table_max_pos;
    // shortcuts that cut the dependent-load chain in front of the K/V tile loads:
    const int* ptab;     // optional per-row page table [rows][pt_stride] (else indices[indptr[q_req[row]] + j])
    int pt_stride;
    int fixed_kvlen;     // > 0: every row sees exactly this many tokens (depth loop: known on the host)
    int fixed_pos;       // >= 0: every row's RoPE position
    int identity_pages;  // 1: request r owns the single page r and q_req[row] == row (depth loop)
    bf16_t* out;   // single-chunk launches write the final bf16 output here (merge of one chunk == o/l)
    bf16_t* out_frag;   // optional fragment-major copy of the output (see LinearCall)
    int hoist;          // 1: page ids requested before the row length is known (k_attn_decode8 with a per-row page table)
};
static inline void set_page_size(AttnArgs& a, int page_size) {
    a.page_size = page_size;
    a.page_shift = -1;
    if (page_size > 0 && (page_size & (page_size - 1)) == 0) { a.page_shift = 0; while ((1 << a.page_shift) < page_size) ++a.page_shift; }
}
__device__ __forceinline__ int page_of(const AttnArgs& a, int tok) { return a.page_shift >= 0 ? tok >> a.page_shift : tok / a.page_size; }
__device__ __forceinline__ int slot_of(const AttnArgs& a, int tok) { return a.page_shift >= 0 ? tok & (a.page_size - 1) : tok % a.page_size; }

// norm (optional) + rope of one head held as one 16-byte chunk per lane (lanes < LPT); result as bf16 bits in
// `out` (LDS, D elements).  sh: LDS scratch of D floats.  All 64 lanes of the wave must call this.
struct PrepOps { u32x4_t v, g; float csx, csy; };
// the three operands (head row, norm weight, this lane's RoPE table entry) are requested together: one exposed L2 latency instead
// of three dependent ones.  Branch-free (every lane requests something in range, prep_head_apply selects): a conditional load
// would be joined with its default by a copy behind a wait, in front of whatever the caller requests next.
template <int D>
__device__ __forceinline__ PrepOps prep_head_load(const bf16_t* src, const bf16_t* nw, const float* cs_row, int rot, int lane) {
    constexpr int LPT = D / 8;
    PrepOps o;
    const int l = lane < LPT ? lane : 0;
    o.v = reinterpret_cast<const u32x4_t*>(src)[l];
    o.g = reinterpret_cast<const u32x4_t*>(nw ? nw : src)[l];
    const float2 c = *reinterpret_cast<const float2*>((cs_row ? cs_row : reinterpret_cast<const float*>(src)) + 2 * (lane < (rot >> 1) ? lane : 0));
    o.csx = c.x; o.csy = c.y;
    return o;
}
// ... the head row staged in LDS by the caller (q | k | v of the new token gathered from hand-off granules: k_talker_layers); norm weight and
// RoPE table must exist (no pointer selects between LDS and global memory)
template <int D>
__device__ __forceinline__ PrepOps prep_head_load_lds(const bf16_t* src_lds, const bf16_t* nw, const float* cs_row, int rot, int lane) {
    constexpr int LPT = D / 8;
    PrepOps o;
    const int l = lane < LPT ? lane : 0;
    o.v = reinterpret_cast<const u32x4_t*>(src_lds)[l];
    o.g = *((const VOX_GLOBAL_AS u32x4_t*)nw + l);
    const VOX_GLOBAL_AS float* cp = (const VOX_GLOBAL_AS float*)cs_row + 2 * (lane < (rot >> 1) ? lane : 0);
    o.csx = cp[0]; o.csy = cp[1];
    return o;
}
// the operands are in registers from here on (the caller's own wait may already have covered them)
__device__ __forceinline__ void prep_head_arrived(PrepOps& o) { asm volatile("" : "+v"(o.v), "+v"(o.g), "+v"(o.csx), "+v"(o.csy)); }
template <int D>
__device__ __forceinline__ void prep_head_apply(const PrepOps& o, const bf16_t* nw, float eps, const float* cs_row,
                                                int rot, int interleave, float* sh, bf16_t* out, int lane) {
    constexpr int LPT = D / 8;
    const int half = rot >> 1;
    const bool own = lane < LPT;
    const uint4 v = own ? as_uint4(o.v) : make_uint4(0, 0, 0, 0), g = own && nw ? as_uint4(o.g) : make_uint4(0, 0, 0, 0);
    const float2 cs0 = cs_row && lane < half ? make_float2(o.csx, o.csy) : make_float2(1.0f, 0.0f);
    float e[8] = {bflo(v.x), bfhi(v.x), bflo(v.y), bfhi(v.y), bflo(v.z), bfhi(v.z), bflo(v.w), bfhi(v.w)};
    if (nw) {
        float s = sq8(v, 0.0f);
        s = butterfly<64>(s);
        const float rinv = 1.0f / sqrtf(s / (float)D + eps);
        if (lane < LPT) {
            const float gw[8] = {bflo(g.x), bfhi(g.x), bflo(g.y), bfhi(g.y), bflo(g.z), bfhi(g.z), bflo(g.w), bfhi(g.w)};
#pragma unroll
            for (int i = 0; i < 8; ++i) e[i] = bfround((e[i] * rinv) * gw[i]);
        }
    }
    if (lane < LPT) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            sh[lane * 8 + i] = e[i];
            out[lane * 8 + i] = f2bf(e[i]);
        }
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    if (cs_row) {
        for (int i = lane; i < half; i += 64) {
            const int ia = interleave ? 2 * i : i, ib = interleave ? 2 * i + 1 : i + half;
            const float x = sh[ia], y = sh[ib], c = i == lane ? cs0.x : cs_row[2 * i], sn = i == lane ? cs0.y : cs_row[2 * i + 1];
            const float xc = x * c, yc = y * c;
            out[ia] = f2bf(__fmaf_rn(-y, sn, xc));
            out[ib] = f2bf(__fmaf_rn(x, sn, yc));
        }
    }
}
template <int D>
__device__ __forceinline__ void prep_head(const bf16_t* src, const bf16_t* nw, float eps, const float* cs_row,
                                          int rot, int interleave, float* sh, bf16_t* out, int lane) {
    const PrepOps o = prep_head_load<D>(src, nw, cs_row, rot, lane);
    prep_head_apply<D>(o, nw, eps, cs_row, rot, interleave, sh, out, lane);
}
