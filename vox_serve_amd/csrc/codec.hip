// Qwen3-TTS 12 Hz codec decoder (token -> waveform), streaming, for gfx950.
// Replaces Qwen3TTSTokenizerV2Decoder.forward_chunk (vox_serve/tokenizer/qwen3_codec.py:1541-1666) and the
// per-request DecoderCache cat / copy-in / copy-out of CudaGraphWorker.run_detokenize
// (worker/cuda_graph_worker.py:1217-1241: ~57 MiB per request per chunk) with in-place per-slot state
// (conv tails + a 72-slot bf16 KV ring: ~2.6 MiB per request).
//
// Layout: activations fp32, time-major [rows = (request, t)][channels] so that
//   * every conv / transposed conv / linear is ONE implicit GEMM  out[t, n] = sum_tap sum_c A[t - off_tap, c] * W[tap][n][c]
//     on the matrix cores.  The waveform parity bar of 1e-4 RMS is not reachable with bf16-rounded activations, so the
//     fp32 activation is split EXACTLY into three bf16 terms when it is staged (x = h + m + l, 24 mantissa bits) and each
//     term meets the (already bf16) weight in v_mfma_f32_16x16x32_bf16: products exact, fp32 accumulation — the result
//     of an fp32-input MFMA at 3/16 of its issue cost (the fp32 16x16x4 form made these kernels MFMA-bound per CU);
//   * a transposed conv with stride r writes r*Cout contiguous values per input row = r output rows: no scatter;
//   * LayerNorm / RMSNorm / depthwise conv run over the contiguous channel axis.
// Weights stay bf16 in HBM ([tap][N][Cin], packed once on the host side) and are widened when staged to LDS.
#include "vox_internal.h"
#include <type_traits>

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 cbf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ cbf16x8 as_cbf8(uint4 v) {
    union { uint4 u; cbf16x8 b; } c;
    c.u = v;
    return c.b;
}
// exact three-way split of 8 fp32 values into bf16 planes: x = h + m + l (each subtraction is exact in fp32)
__device__ __forceinline__ void split3(const float4 lo4, const float4 hi4, uint4& h, uint4& m, uint4& l) {
    const float x[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
    unsigned short hb[8], mb[8], lb[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        hb[i] = f2bf(x[i]);
        const float r1 = x[i] - bf2f(hb[i]);
        mb[i] = f2bf(r1);
        const float r2 = r1 - bf2f(mb[i]);
        lb[i] = f2bf(r2);
    }
    h = make_uint4(hb[0] | (unsigned)hb[1] << 16, hb[2] | (unsigned)hb[3] << 16, hb[4] | (unsigned)hb[5] << 16, hb[6] | (unsigned)hb[7] << 16);
    m = make_uint4(mb[0] | (unsigned)mb[1] << 16, mb[2] | (unsigned)mb[3] << 16, mb[4] | (unsigned)mb[5] << 16, mb[6] | (unsigned)mb[7] << 16);
    l = make_uint4(lb[0] | (unsigned)lb[1] << 16, lb[2] | (unsigned)lb[3] << 16, lb[4] | (unsigned)lb[5] << 16, lb[6] | (unsigned)lb[7] << 16);
}

// ================================================================================================
// implicit-GEMM convolution on the matrix cores (fp32 activations split 3-way into bf16).  Block 256 threads = 2x2 waves.
// ================================================================================================
#define CG_BM 64
#define CG_BN 64
#define CG_BK 32            // smallest K chunk (Cin granularity); 64-wide chunks are used where Cin allows
#define CG_MAXTAPS 24          // (HiFT: 11-tap dilated convs with fp32 weights carried as two bf16 planes)

struct ConvGemmArgs {
    const float* x;        // [n*L, Cin] current-chunk input rows
    const float* state;    // [slots, P, Cin] history rows (NULL when no tap looks back)
    const int* slots;      // [n] state slot of each request in this batch
    const bf16_t* w;       // [taps][N][Cin]
    const float* bias;     // [bias_mod] or NULL
    const float* res;      // [M, N] residual or NULL
    const float* scale;    // [N] multiplier applied before the residual add, or NULL
    const float* rscale;   // [M] per-row multiplier applied before the residual add, or NULL (SNAC NoiseBlock: x + noise[t] * Wx)
    int planes;            // 3: exact products (fp32 activation = three bf16 terms); 1: activations rounded to bf16 (the reference's
                           // own serving precision: its decoder runs in bf16, qwen3_tts.py:1061-1064) at a third of the MFMA issue
    float* out;            // [M, N]
    int M, N, Cin, L, P, n_taps, bias_mod, gelu;
    int off[CG_MAXTAPS];   // row look-back of each tap (negative: look-ahead)
    // fused SnakeBeta of the NEXT layer's input: out2[m][n] = v + inv_beta[c] * sin(v * alpha[c])^2, c = n % sn_mod, beside
    // (out != NULL) or instead of (out == NULL) the plain output — the arithmetic of k_snake, one elementwise pass less
    float* out2;
    const float *sn_alpha, *sn_invb;
    int sn_mod;
    // LayerNorm of the input rows fused into the A-operand staging (few-row kernel, one tap): x <- (x - mean) * rstd * ln_w + ln_b
    const float *ln_w, *ln_b;
    float ln_eps;
    // "S2" rows: an activation row of Cin values stored as its two leading bf16 terms, [Cin x bf16 h][Cin x bf16 m] (x ~ h + m, 16
    // significand bits; the same 4 * Cin bytes as the fp32 row, so buffers, history state and k_state_update are format-agnostic).
    // The producing epilogue splits each value ONCE (out2_s2); the consumers (k_conv_dma, k_conv_unit) read plain bf16 — the per-tap
    // split of fp32 rows made the many-row decoder convs VALU-bound (MFMA 16 % busy).
    // NP = 3: "S3" rows, [h][m][l], 6 * Cin bytes, the value itself.
    int out2_s2;
    // k_rows_gemm: x / (Cin / 32) and x / L as the high word of a product (div_inverse); 0: by division
    unsigned kpt_inv, len_inv;
    int dev;               // development builds (-DVOX_DEV_KNOBS, VOX_CODEC_DEV): 1 skip the K loop, 2 no out2 stores, 4 no out stores, 8 no residual loads
};
#ifdef VOX_DEV_KNOBS
#define CG_DEV(a, bit) ((a).dev & (bit))
#else
#define CG_DEV(a, bit) 0
#endif
// sin for the fused epilogues: explicit reduction to revolutions + the hardware v_sin_f32 (absolute error ~1e-6 on [-1, 1]:
// far inside the 1e-4 waveform bar, and sin^2 enters scaled by 1/beta ~ 1).  The libm sinf (argument-reduction table,
// private array) cannot be inlined into a GEMM epilogue without spilling the accumulators to scratch.
__device__ __forceinline__ float snake_f(float v, float alpha, float invb) {
    const float r = (v * alpha) * 0.15915494309189535f;
    const float s_ = __builtin_amdgcn_sinf(r - floorf(r));
    return v + invb * (s_ * s_);
}

// The same with the sine right to fp32, for one conv's epilogue (no room for libm's table there): revolutions, the nearest half turn and its
// Taylor series in fp64, remainder below (pi / 2)^17 / 17! = 6e-12.
__device__ __forceinline__ float snake_exact(float v, float alpha, float invb) {
    const double r = (double)(v * alpha) * 0.15915494309189533577;
    double q = r - rint(r);
    if (fabs(q) > 0.25) q = copysign(0.5, q) - q;
    const double t = q * 6.28318530717958647693, t2 = t * t;
    double s = -1.0 / 1307674368000.0;
    s = fma(s, t2, 1.0 / 6227020800.0);
    s = fma(s, t2, -1.0 / 39916800.0);
    s = fma(s, t2, 1.0 / 362880.0);
    s = fma(s, t2, -1.0 / 5040.0);
    s = fma(s, t2, 1.0 / 120.0);
    s = fma(s, t2, -1.0 / 6.0);
    const float s_ = (float)fma(t * t2, s, t);
    return v + invb * (s_ * s_);
}

// GELU in its exact form.  (As v Phi(v) with log2 Phi by a polynomial and no branch: k_tb_ff, 896 rows, 9.9 us for 10.5, and 3.4e-8 from 64 bits over normal inputs
// for 3.9e-8, relative 2-norm; but every codec's samples move by it, a flow's by 4e-4 once ten solver steps and the vocoder's source phase have carried it on.)
__device__ __forceinline__ float gelu_f(float v) { return 0.5f * v * (1.0f + erff(v * 0.70710678118654752440f)); }

// Epilogue of the tiled conv GEMMs (2 x 2 waves, WM x WN 16x16 tiles per wave)
template <int WM, int WN>
__device__ __forceinline__ void conv_epilogue(const ConvGemmArgs& a, f32x4 (&acc)[WM][WN], int m0, int n0, int wm, int wn, int lane) {
    // epilogue.  D layout of a 16x16 tile: col = lane & 15, row = (lane >> 4) * 4 + reg.  The per-column constants are fetched once and
    // the residual values of a whole row fragment are requested together, ahead of the arithmetic: an epilogue that interleaves loads,
    // stores and integer divisions element by element serialises on memory latency (the compiler must keep every load behind the
    // previous store) — the 1-tap conv2 of a residual unit took longer than its 7-tap conv1 (485 vs 365 us at 614 k rows).
    const int l15 = lane & 15, rg = (lane >> 4) * 4;
    float cb[WN], cs[WN], ca[WN], ci[WN];
    int cn[WN], cj[WN], cc[WN];
#pragma unroll
    for (int j = 0; j < WN; ++j) {
        const int n = n0 + wn + j * 16 + l15, nn = n < a.N ? n : a.N - 1;
        cn[j] = n;
        cb[j] = a.bias ? a.bias[nn % a.bias_mod] : 0.0f;
        cs[j] = a.scale ? a.scale[nn] : 1.0f;
        ca[j] = ci[j] = 0.0f; cj[j] = cc[j] = 0;
        if (a.out2) {
            cj[j] = nn / a.sn_mod; cc[j] = nn - cj[j] * a.sn_mod;      // (a transposed conv's N = r * sn_mod outputs: r consumer rows)
            ca[j] = a.sn_alpha[cc[j]]; ci[j] = a.sn_invb[cc[j]];
        }
    }
#pragma unroll
    for (int i = 0; i < WM; ++i) {
        const int mb = m0 + wm + i * 16 + rg;
        float rs[WN][4], rsc[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) rsc[r] = (a.rscale && mb + r < a.M) ? a.rscale[mb + r] : 1.0f;
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                rs[j][r] = (a.res && !CG_DEV(a, 8) && mb + r < a.M && cn[j] < a.N) ? a.res[(size_t)(mb + r) * a.N + cn[j]] : 0.0f;
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = mb + r;
                const bool ok = m < a.M && cn[j] < a.N;
                float v = acc[i][j][r] + cb[j];
                if (a.gelu) v = gelu_f(v);
                if (a.rscale) v = rsc[r] * v;
                if (a.res) v = rs[j][r] + cs[j] * v;
                else if (a.scale) v = cs[j] * v;
                const size_t o = (size_t)m * a.N + cn[j];
                if (a.out && ok && !CG_DEV(a, 4)) a.out[o] = v;
                if (a.out2 && !CG_DEV(a, 2)) {
                    const float sv2 = snake_f(v, ca[j], ci[j]);
                    if (ok) a.out2[o] = sv2;
                }
            }
    }
}

// WM x WN 16x16 MFMA tiles per wave, 2 x 2 waves: block tile (32 WM) x (32 WN).  Smaller tiles are used when the
// 64 x 64 grid would leave most of the 256 CUs idle (the mid-size decoder stages are MFMA-bound per CU).
template <int BK, int WM, int WN, bool UNR = false>
__global__ __launch_bounds__(256, (WM * WN > 12 ? 3 : 4)) void k_conv_gemm(ConvGemmArgs a) {
    touch_args(a);
    constexpr int BM = 32 * WM, BN = 32 * WN;
    constexpr int LD = BK + 8;          // LDS row stride in bf16 elements (+16 B: the 16 rows of a fragment read hit distinct banks)
    constexpr int SEG = BK / 8;         // 8-element segments per row
    constexpr int NA = (BM * SEG + 255) / 256, NB = (BN * SEG + 255) / 256;
    __shared__ __attribute__((aligned(16))) bf16_t As[3][BM * LD];     // the h / m / l planes of the activation tile
    __shared__ __attribute__((aligned(16))) bf16_t Bs[BN * LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int wm = (wave >> 1) * 16 * WM, wn = (wave & 1) * 16 * WN;

    f32x4 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int nck = a.Cin / BK, nit = CG_DEV(a, 1) ? 0 : a.n_taps * nck;

    // staging slots of this thread: (row, segment) pairs of the A and B tiles
    int a_b[NA], a_t[NA];
    bool a_ok[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int idx = tid + 256 * i, am = m0 + idx / SEG;
        a_ok[i] = idx < BM * SEG && am < a.M;
        a_b[i] = a_ok[i] ? am / a.L : 0;
        a_t[i] = a_ok[i] ? am % a.L : 0;
    }
    // the operands of step it+1 are requested before the MFMAs of step it
    float4 v0[NA], v1[NA];
    uint4 wv[NB];
    auto fetch = [&](int it) {
        const int tap = it / nck, c0 = (it - tap * nck) * BK;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int seg = (tid + 256 * i) % SEG;
            v0[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            v1[i] = v0[i];
            if (a_ok[i]) {
                const int st = a_t[i] - a.off[tap];      // (off < 0: the tap looks ahead; rows past the request's end read as zero)
                const float* arow = nullptr;
                if (st >= a.L) arow = nullptr;
                else if (st >= 0) arow = a.x + ((size_t)a_b[i] * a.L + st) * a.Cin;
                else if (a.state && a.P + st >= 0) arow = a.state + ((size_t)a.slots[a_b[i]] * a.P + (a.P + st)) * a.Cin;
                if (arow) {
                    v0[i] = *reinterpret_cast<const float4*>(arow + c0 + seg * 8);
                    v1[i] = *reinterpret_cast<const float4*>(arow + c0 + seg * 8 + 4);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int idx = tid + 256 * i, bn = n0 + idx / SEG;
            wv[i] = make_uint4(0, 0, 0, 0);
            if (idx < BN * SEG && bn < a.N)
                wv[i] = *reinterpret_cast<const uint4*>(a.w + ((size_t)tap * a.N + bn) * a.Cin + c0 + (idx % SEG) * 8);
        }
    };
    fetch(0);
    // UNR (few-block launches of the small tiles: one request's chunk): the plane count (1 .. 3 bf16 terms per activation) is a compile-time
    // constant inside the loop.  As a run-time trip count the term loop is not unrolled and every MFMA sits behind its own ds_read + wait —
    // 12 dependent LDS round trips per K step of the 32 x 32 tile; unrolled, a k-block's operand reads go out together (one-request chunk
    // 1.76 -> 1.72 ms).  Many-block launches keep the run-time count: the unrolled reads cost 30 registers, i.e. a wave per SIMD, and
    // there the other waves hide the round trips (8-request chunk 3.34 -> 3.36 ms unrolled).
    auto kloop = [&](auto np_tag) {
    constexpr int NP = decltype(np_tag)::value;
    for (int it = 0; it < nit; ++it) {
        __syncthreads();   // previous tile fully consumed
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int idx = tid + 256 * i;
            if (idx < BM * SEG) {
                const int o = (idx / SEG) * LD + (idx % SEG) * 8;
                uint4 h, m, l;
                split3(v0[i], v1[i], h, m, l);
                *reinterpret_cast<uint4*>(&As[0][o]) = h;
                if ((NP ? NP : a.planes) > 1) *reinterpret_cast<uint4*>(&As[1][o]) = m;
                if ((NP ? NP : a.planes) > 2) *reinterpret_cast<uint4*>(&As[2][o]) = l;
            }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int idx = tid + 256 * i;
            if (idx < BN * SEG) *reinterpret_cast<uint4*>(&Bs[(idx / SEG) * LD + (idx % SEG) * 8]) = wv[i];
        }
        __syncthreads();
        if (it + 1 < nit) fetch(it + 1);
        // lane (fr, g) holds 8 consecutive k of row fr of every 32-wide K block: one 16-byte LDS read per operand
        const int fr = lane & 15, fk = (lane >> 4) * 8;
#pragma unroll
        for (int kb = 0; kb < BK; kb += 32) {
            uint4 bfr[WN];
#pragma unroll
            for (int j = 0; j < WN; ++j) bfr[j] = *reinterpret_cast<const uint4*>(&Bs[(wn + j * 16 + fr) * LD + kb + fk]);
            // (NP = 0: the run-time count — the 128-row tiles run 3 .. 4 blocks per CU on a register budget the unrolled reads do not fit)
#pragma unroll
            for (int t = (NP ? NP : a.planes) - 1; t >= 0; --t) {      // smallest term first
#pragma unroll
                for (int i = 0; i < WM; ++i) {
                    const uint4 afr = *reinterpret_cast<const uint4*>(&As[t][(wm + i * 16 + fr) * LD + kb + fk]);
#pragma unroll
                    for (int j = 0; j < WN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_cbf8(afr), as_cbf8(bfr[j]), acc[i][j], 0, 0, 0);
                }
            }
        }
    }
    };
    if constexpr (!UNR) kloop(std::integral_constant<int, 0>{});
    else if (a.planes >= 3) kloop(std::integral_constant<int, 3>{});
    else if (a.planes == 2) kloop(std::integral_constant<int, 2>{});
    else kloop(std::integral_constant<int, 1>{});
    conv_epilogue<WM, WN>(a, acc, m0, n0, wm, wn, lane);
}

// LayerNorm row statistics by the 16 lanes l16 = 0..15 of a row group (two passes over float4 chunks, butterfly inside the group).
// Shared by the GEMM with the fused LayerNorm and by k_flow_ln, so a row normalises to the same bits on either path (a request's output
// must not depend on how many requests share its batch).
__device__ __forceinline__ void ln_row_stats(const float* row, int C, int l16, float eps, float& mean, float& rstd) {
    const float4* xr = reinterpret_cast<const float4*>(row);
    float sm = 0.0f;
    for (int c = l16; c < C / 4; c += 16) { const float4 v = xr[c]; sm += (v.x + v.y) + (v.z + v.w); }
    sm = butterfly<16>(sm);
    mean = sm / (float)C;
    float vs = 0.0f;
    for (int c = l16; c < C / 4; c += 16) {
        const float4 v = xr[c];
        const float d0 = v.x - mean, d1 = v.y - mean, d2 = v.z - mean, d3 = v.w - mean;
        vs += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
    }
    vs = butterfly<16>(vs);
    rstd = rsqrtf(vs / (float)C + eps);
}

// ================================================================================================
// Convolutions over S2 (NP = 1: their first terms; 2) and S3 (NP = 3) rows through LDS DMA.  BM x BN outputs per block of WM x WN x WK waves; K is walked tap by tap in steps of BK
// channels.  A step's NP x BM activation rows (a row may lie in the chunk, in the history or in neither) and BN weight rows go from memory
// straight into one of S LDS stages (global_load_lds, 1 KB per wave instruction); S - 1 steps are in flight and no register holds them.
// One wait + barrier per step: every wave's part of the step has landed, and nobody reads the stage of the step before any more.  16-byte
// pieces lie swizzled by row (in the address that each lane reads), so the fragment reads of 16 rows do not meet in a bank.
// WP = 1: every output adds its products tap by tap, 32 channels at a time in ascending order, the lowest term first, in whatever tile the
// rows pick, so a request's samples do not depend on its batch.  WK > 1: WM * WN * (WK - 1) further waves only load.  In a small tile the
// few waves that multiply are a serial chain (barrier, LDS reads, dependent MFMAs), and their share of the requests stood in it (10 rows, 20
// and 40 rows, us, 4 or 8 waves that share K / one such wave with loads / with loaders: 3072 x 512 6.5 / 6.9 / 5.5, 1024 x 4096 8.7 / 11.3 / 9.6,
// 1536 x 7 x 1024 14.4 / 18.1 / 14.5, 6144 x 2 x 1536 14.7 / 16.9 / 13.1).
// WP = 2: every tap has two weight planes (n_taps * N rows apart; fp32 weights as two terms) that share the tap's rows; WK waves share the
// 32-channel slices of a step and add their sums through LDS at the end (hift_conv keeps one such order for all its tiles).
// EPI: 0, CONV_GELU, CONV_GLU: columns come in pairs (n, N + n) of w, out2 <- S2 of silu(v[n]) * v[N + n], N columns; or CONV_CHUNKS.
// The weights are the MFMA's first operand, so a lane ends with 4 (8) neighbouring channels of one row: the residual, the constants and both
// outputs move in 16-byte accesses without a lane exchange.  With a lane per column the same epilogue cost more than the products of the
// one-tap convs (us, rows x channels, residual + h + activation: 51 200 x 384 134 -> 67, 204 800 x 192 240 -> 175 = 3.6 TB/s).
// Bound: few rows, the chain of steps (one L2 trip for the first, ~0.2 us for each further); many rows, the L2 -> LDS path beside the
// matrix cores (1.27 PFLOP/s at 10 240 rows, 768 x 7 x 768, one 128 x 256 tile per CU).
// Extra blocks behind the tiles write a history that an earlier launch was the last to read (ConvDmaArgs::job).
// ================================================================================================
struct ConvJob {           // history rows <- the last P rows of [history ++ x], n requests of L rows; C: floats per row
    float* state;
    const float* x;
    int L, P, C, n;
};
// new history = last P rows of [history ++ x].  A chunk of at least P rows replaces it: 16 bytes a thread and turn, four turns (the 54 rows
// of a dilated conv, row by row in one thread, outlasted the launch they rode on: 15 us against 9).  A shorter one shifts it: one thread per
// (request, channel), rows ascending (in place).
__host__ __device__ __forceinline__ bool conv_job_whole(const ConvJob& j) { return j.L >= j.P && j.C % 4 == 0; }
__host__ __device__ __forceinline__ int conv_job_per(const ConvJob& j, int threads) {      // blocks of a request
    return conv_job_whole(j) ? (j.P * (j.C / 4) + 4 * threads - 1) / (4 * threads) : (j.C + threads - 1) / threads;
}
__device__ __forceinline__ void conv_job(const ConvJob& j, const int* slots, int block, int threads) {
    const int per = conv_job_per(j, threads), b = block / per, e0 = block % per;
    float* s = j.state + (size_t)slots[b] * j.P * j.C;
    const float* x = j.x + (size_t)b * j.L * j.C;
    if (conv_job_whole(j)) {
        const float4* src = reinterpret_cast<const float4*>(x + (size_t)(j.L - j.P) * j.C);
        const int n4 = j.P * (j.C / 4);
        const int e1 = e0 * 4 * threads + (int)threadIdx.x;
        float4 v[4];      // (requested together: a condition around each would make four trips of them)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = ldg_f4(reinterpret_cast<const float*>(src + (e1 + i * threads < n4 ? e1 + i * threads : n4 - 1)));
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (e1 + i * threads < n4) reinterpret_cast<float4*>(s)[e1 + i * threads] = v[i];
        return;
    }
    const int c = e0 * threads + (int)threadIdx.x;
    if (c >= j.C) return;
    for (int i0 = 0; i0 < j.P; i0 += 8) {      // (rows are read ahead of where they are written: L > 0)
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int e = j.L + (i0 + i < j.P ? i0 + i : j.P - 1);
            v[i] = ldg(e < j.P ? s + (size_t)e * j.C + c : x + (size_t)(e - j.P) * j.C + c);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i0 + i < j.P) s[(size_t)(i0 + i) * j.C + c] = v[i];
    }
}
static int conv_job_blocks(const ConvJob& j, int threads) { return j.state ? j.n * conv_job_per(j, threads) : 0; }
// what is left at the end of a chunk: two histories (state NULL: none) and the slots' positions
__global__ __launch_bounds__(256) void k_conv_jobs(ConvJob a, ConvJob b, int na, int nb, const int* slots, long* pos, int n, int T) {
    const int i = (int)blockIdx.x;
    if (i < na) conv_job(a, slots, i, 256);
    else if (i < na + nb) conv_job(b, slots, i - na, 256);
    else
        for (int k = threadIdx.x; k < n; k += 256) pos[slots[k]] += T;
}
struct ConvDmaArgs : ConvGemmArgs {
    int tm, tn, tiles8, mfast;      // tiles along M and N; their number rounded up to 8; 1: the blocks of an XCD walk the rows first
    int tdiv;              // tiles of the direction walked first, and div_inverse of it
    unsigned tdiv_inv;
    const float* rms_x;    // fp32 rows [M, Cin] whose 1 / rms scales the sums of row m (the rows' RMSNorm, its weight already in x), or NULL
    float rms_eps;
    const float* nw;       // out2 <- terms of v * nw[n] (no activation), or NULL
    int elu;               // out2 <- ELU of v
    int parts;             // three-term rows: sums start anew every 256 channels (conv_long_sums)
    ConvJob job;
};
__device__ uint4 g_conv_zero_row[1];        // what a tap reads outside the chunk and its history
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));       // (per-channel constants are where the caller's tensors have them)
// W neighbouring channels of a row as its T terms
template <int T, int W>
__device__ __forceinline__ void conv_put_terms(bf16_t* row, int width, int c, const float (&v)[W]) {
    float r[W];
#pragma unroll
    for (int e = 0; e < W; ++e) r[e] = v[e];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        unsigned h[W / 2];
#pragma unroll
        for (int e = 0; e < W / 2; ++e) {
            h[e] = pack_bf2(r[2 * e], r[2 * e + 1]);
            r[2 * e] -= bflo(h[e]);
            r[2 * e + 1] -= bfhi(h[e]);
        }
        if constexpr (W == 8) *reinterpret_cast<uint4*>(row + (size_t)t * width + c) = make_uint4(h[0], h[1], h[2], h[3]);
        else *reinterpret_cast<uint2*>(row + (size_t)t * width + c) = make_uint2(h[0], h[1]);
    }
}
#define CONV_GELU 1
#define CONV_GLU 2
#define CONV_CHUNKS 3      // 0, with K in k_conv_unit's order: 32 channels at a time, all taps of them (a step of 64: two such slices)
#define CONV_SINE 4        // 0, with snake_exact for SnakeBeta
// The epilogue of W neighbouring channels (n ..) of MT rows (m, m + 16, ..) that one lane holds: constants once, every row's residual
// requested ahead of the first store, 16-byte accesses throughout.
template <int W>
__device__ __forceinline__ void conv_get(float (&d)[W], const float* p) {
#pragma unroll
    for (int q = 0; q < W / 4; ++q) {
        const f32x4 t = *reinterpret_cast<const f32x4_a4*>(p + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; ++e) d[4 * q + e] = t[e];
    }
}
// the consumer row and the bias of channel n (no division where there is one row, one bias a channel)
__device__ __forceinline__ int conv_row_of(const ConvDmaArgs& a, int n) { return !a.out2 || a.sn_mod >= a.N ? 0 : n / a.sn_mod; }
__device__ __forceinline__ int conv_bias_at(const ConvDmaArgs& a, int n) { return a.bias_mod >= a.N ? n : n % a.bias_mod; }
template <int W, int MT>
struct conv_consts {
    float b[W], s[W], al[W], ib[W], nw[W], rs[MT][W];
    int cj, cc;      // (a transposed conv's N = r * sn_mod outputs: r consumer rows)
};
// What the epilogue reads, asked for ahead of the K loop.  (Kernels whose waves have no registers for it read it in the epilogue: through this
// struct the 256 x 192 tile spilled 36 bytes a lane there, 146 -> 165 us at 51 200 rows of 384 channels, 7 taps.)
template <int W, int MT>
__device__ __forceinline__ void conv_fetch(conv_consts<W, MT>& k, const ConvDmaArgs& a, int m, int n) {
    if (n >= a.N) return;
    k.cj = conv_row_of(a, n);
    k.cc = n - k.cj * a.sn_mod;
    if (a.bias) conv_get<W>(k.b, a.bias + conv_bias_at(a, n));
    if (a.scale) conv_get<W>(k.s, a.scale + n);
    if (a.sn_alpha) { conv_get<W>(k.al, a.sn_alpha + k.cc); conv_get<W>(k.ib, a.sn_invb + k.cc); }
    if (a.nw) conv_get<W>(k.nw, a.nw + n);
    if (a.res)
#pragma unroll
        for (int i = 0; i < MT; ++i) conv_get<W>(k.rs[i], a.res + (size_t)(m + 16 * i < a.M ? m + 16 * i : a.M - 1) * a.N + n);
}
template <int T, int EPI, int W, int MT, bool FETCHED = false>
__device__ __forceinline__ void conv_dma_out(const ConvDmaArgs& a, const f32x4 (&acc)[MT][W / 4], const float* rms, int m, int n,
                                             const f32x4* res_ready = nullptr, const conv_consts<W, MT>& early = conv_consts<W, MT>{}) {
    if (n >= a.N) return;          // (N and the group width are multiples of W)
    float b[W], s[W], al[W], ib[W], nw[W], rs[MT][W];
    int cj, cc;      // (a transposed conv's N = r * sn_mod outputs: r consumer rows)
    if constexpr (FETCHED) {
        cj = early.cj;
        cc = early.cc;
#pragma unroll
        for (int e = 0; e < W; ++e) {
            b[e] = early.b[e]; s[e] = early.s[e]; al[e] = early.al[e]; ib[e] = early.ib[e]; nw[e] = early.nw[e];
#pragma unroll
            for (int i = 0; i < MT; ++i) rs[i][e] = early.rs[i][e];
        }
    } else {
        cj = conv_row_of(a, n);
        cc = n - cj * a.sn_mod;
        if (a.bias) conv_get<W>(b, a.bias + conv_bias_at(a, n));
        if (a.scale) conv_get<W>(s, a.scale + n);
        if (a.sn_alpha) { conv_get<W>(al, a.sn_alpha + cc); conv_get<W>(ib, a.sn_invb + cc); }
        if (a.nw) conv_get<W>(nw, a.nw + n);
        if (res_ready) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int e = 0; e < W; ++e) rs[i][e] = res_ready[i * (W / 4) + e / 4][e % 4];
        } else if (a.res)
#pragma unroll
            for (int i = 0; i < MT; ++i)
                if (m + 16 * i < a.M) conv_get<W>(rs[i], a.res + (size_t)(m + 16 * i) * a.N + n);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const size_t o = (size_t)(m + 16 * i) * a.N + n;
        if (m + 16 * i >= a.M) continue;
        const float rr = rms ? rms[16 * i] : 1.0f;
        float v[W];
#pragma unroll
        for (int e = 0; e < W; ++e) {
            v[e] = acc[i][e / 4][e % 4];
            if (rms) v[e] *= rr;
            if (a.bias) v[e] += b[e];
            if (EPI == CONV_GELU) v[e] = gelu_f(v[e]);
            if (a.scale) v[e] = s[e] * v[e];
            if (a.res) v[e] = rs[i][e] + v[e];
        }
        if (a.out)
#pragma unroll
            for (int q = 0; q < W / 4; ++q) *reinterpret_cast<float4*>(a.out + o + 4 * q) = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
        if (!a.out2) continue;
#pragma unroll
        for (int e = 0; e < W; ++e) {
            if (a.sn_alpha) v[e] = EPI == CONV_SINE ? snake_exact(v[e], al[e], ib[e]) : snake_f(v[e], al[e], ib[e]);
            else if (a.elu) v[e] = v[e] > 0.0f ? v[e] : expm1f(v[e]);
            else if (a.nw) v[e] *= nw[e];
        }
        if (a.out2_s2) {
            conv_put_terms<T>(reinterpret_cast<bf16_t*>(a.out2) + ((size_t)(m + 16 * i) * a.N + (size_t)cj * a.sn_mod) * T, a.sn_mod, cc, v);
        } else {
#pragma unroll
            for (int q = 0; q < W / 4; ++q) *reinterpret_cast<float4*>(a.out2 + o + 4 * q) = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
        }
    }
}
__device__ __forceinline__ void conv_dma_glu(const ConvDmaArgs& a, f32x4 g, f32x4 u, float rms, int m, int n) {
    if (n >= a.N || m >= a.M) return;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float gv = g[e] * rms, uv = u[e] * rms;
        v[e] = (gv / (1.0f + expf(-gv))) * uv;
    }
    conv_put_terms<2>(reinterpret_cast<bf16_t*>(a.out2) + (size_t)m * a.N * 2, a.N, n, v);
}
// A conv of few rows is one dependent chain, 4 - 6 us of it for 1 - 2 us of bytes, so what stands in front of the first request and behind the
// last product counts as much as the products: arguments in one trip (touch_args), tile and request numbers by host-made inverses, the
// slots of all of a wave's rows and the epilogue's constants asked for together and early.  us a launch, one request of 2 frames, before / so:
// 3072 x 512 (16 x 32 tiles) 6.8 / 5.4, 512 x 1024 5.4 / 4.9; the decoder's 84 launches 665 / 594, of 10 frames 829 / 795.
template <int BM, int BN, int WM, int WN, int WK, int BK, int S, int NP, int EPI, int WP = 1>
__global__ __launch_bounds__(64 * WM * WN * WK) void k_conv_dma(ConvDmaArgs a) {
    constexpr int NWV = WM * WN * WK, MT = BM / WM / 16, NT = BN / WN / 16, KS = BK / 32, PPR = BK / 8, KW = WP == 2 ? WK : 1;
    constexpr int SA = NP * BM * BK * 2, SB = WP * BN * BK * 2, ST = SA + SB, CA = SA / 1024, CB = SB / 1024;
    constexpr bool PAIR = EPI != CONV_GLU && NT % 2 == 0;
    constexpr int NC = WM * WN, NLD = KW == 1 && WK > 1 ? NWV - NC : NWV;      // waves that multiply one part of K; waves that load
    constexpr int NA = (CA + NLD - 1) / NLD, NB = (CB + NLD - 1) / NLD;      // (where the waves do not divide them some chunks are asked for twice)
    static_assert(SA % 1024 == 0 && SB % 1024 == 0 && KS % KW == 0 && (BM * PPR) % 64 == 0, "whole wave instructions");
    static_assert(KW == 1 || NWV * MT * NT * 1024 <= S * ST, "partial sums");
    static_assert((BK & (BK - 1)) == 0 && (EPI != CONV_GLU || NT % 2 == 0), "swizzle; gate and up columns in one lane");
    extern __shared__ __attribute__((aligned(1024))) char conv_lds[];
    __shared__ float rms_s[BM];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    touch_args(a);
    if ((int)blockIdx.x >= a.tiles8) {
        conv_job(a.job, a.slots, (int)blockIdx.x - a.tiles8, 64 * NWV);
        return;
    }
    const int t = ((int)blockIdx.x & 7) * (a.tiles8 >> 3) + ((int)blockIdx.x >> 3);
    if (t >= a.tm * a.tn) return;
    const int tq = a.tdiv_inv ? (int)__umulhi((unsigned)t, a.tdiv_inv) : a.tdiv == 1 ? t : t / a.tdiv, tr = t - tq * a.tdiv;
    const int m0 = (a.mfast ? tr : tq) * BM, n0 = (a.mfast ? tq : tr) * BN;      // (glu: n0 counts gate and up columns)
    const int wk = wv / NC, wmn = wv % NC, wm = wmn / WN, wn = wmn % WN, fr = lane & 15, fk = lane >> 4, lw = NLD < NWV ? wv - NC : wv;
    const bool loads = NLD == NWV || lw >= 0, multiplies = NLD == NWV || lw < 0;
    const int rl = wm * MT * 16 + fr, nl = n0 + wn * NT * 16;
    // Waves that only multiply have nothing in flight: they ask for the epilogue's constants and residual now, not in a trip of their own behind the last step
    constexpr int P = PAIR ? 2 : 1;
    constexpr bool EARLY = NLD < NWV && EPI != CONV_GLU;
    conv_consts<4 * P, MT> kc[EARLY ? NT / P : 1];
    if constexpr (EARLY)
        if (multiplies)
#pragma unroll
            for (int j = 0; j < NT; j += P) conv_fetch(kc[j / P], a, m0 + rl, nl + j * 16 + fk * 4 * P);
    const int rb = a.Cin * (NP == 3 ? 6 : 4);
    // The weights are the first operand of the MFMA: a lane's four sums are neighbouring channels of one row.  PAIR: tiles j and j + 1 take the
    // weight rows 8 q + 0..3 and 8 q + 4..7 (q = 0..3), so that they hold eight neighbouring channels together.
    const auto wswz = [](int r) {
        if (PAIR) return BK == 32 ? ((r >> 1) & 1) | ((r >> 2) & 2) : (r & 3) | ((r >> 1) & 4);
        return BK == 32 ? (r >> 1) & 3 : r & 7;
    };
    // per DMA instruction of the wave: the lane's row of the chunk (its time), that row in x and the row that time 0 would have in the history
    const char *xp[NA], *sp[NA], *cur[NA], *wp[NB], *wbase[EPI == CONV_CHUNKS ? NB : 1];
    int ts[NA], step[NA];
    bool half_a = false, half_b[EPI == CONV_CHUNKS ? NB : 1];      // (the lane's piece is of the step's second slice)
    static_assert(EPI != CONV_CHUNKS || BK == 64, "two slices a step");
    if (loads) {
        int slot[NA];      // (asked for together, in front of everything else)
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            int m = m0 + ((i * NLD + lw) % CA * 64 + lane) / PPR % BM;
            m = m < a.M ? m : a.M - 1;                  // (rows past the end repeat the last one: nothing of them is stored)
            const int b = a.len_inv ? (int)__umulhi((unsigned)m, a.len_inv) : a.L == 1 ? m : m / a.L;
            ts[i] = m - b * a.L;
            slot[i] = ldg(a.state ? a.slots + b : reinterpret_cast<const int*>(g_conv_zero_row));
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int q = (i * NLD + lw) % CA * 64 + lane, pl = q / (BM * PPR), r = q / PPR % BM, pc8 = (q % PPR) ^ (BK == 32 ? (r >> 1) & 3 : r & 7);
            const int pc = EPI == CONV_CHUNKS ? pc8 & 3 : pc8;
            if (EPI == CONV_CHUNKS) half_a = pc8 > 3;      // (the same for every i: whole rows of eight pieces apart)
            const int m = m0 + r < a.M ? m0 + r : a.M - 1;
            xp[i] = reinterpret_cast<const char*>(a.x) + (size_t)m * rb + pl * a.Cin * 2 + pc * 16;
            sp[i] = reinterpret_cast<const char*>(a.state) + ((size_t)slot[i] * a.P + a.P + ts[i]) * rb + pl * a.Cin * 2 + pc * 16;      // (read where there is a state)
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int q = (i * NLD + lw) % CB * 64 + lane, r = q / PPR % BN, pl = q / (BN * PPR), pc8 = (q % PPR) ^ wswz(r);
            const int pc = EPI == CONV_CHUNKS ? pc8 & 3 : pc8;
            int n = n0 + r;
            if (EPI == CONV_GLU) {
                n = (n0 >> 1) + (r >> 5) * 16 + (r & 15);
                n = (n < a.N ? n : a.N - 1) + ((r >> 4) & 1) * a.N;
            } else {
                n = n < a.N ? n : a.N - 1;
            }
            wp[i] = reinterpret_cast<const char*>(a.w) + (((size_t)pl * a.n_taps * a.N + n) * a.Cin + pc * 8) * 2;
            if constexpr (EPI == CONV_CHUNKS) {
                wbase[i] = wp[i];
                half_b[i] = pc8 > 3;
            }
        }
    }
    const int nck = a.Cin / BK, nit = a.n_taps * nck;
    const size_t wtap = (size_t)(EPI == CONV_GLU ? 2 * a.N : a.N) * a.Cin * 2 - (size_t)a.Cin * 2;      // from the end of one tap's row to the next tap's
    const unsigned sbase = (unsigned)(size_t)(__attribute__((address_space(3))) char*)conv_lds;
    auto row_of = [&](int i, int off) {
        const int e = ts[i] - off;
        const bool in = e >= 0 && e < a.L, hist = e < 0 && a.state && a.P + e >= 0;
        cur[i] = in ? xp[i] - (ptrdiff_t)off * rb : hist ? sp[i] - (ptrdiff_t)off * rb : reinterpret_cast<const char*>(g_conv_zero_row);
        step[i] = in || hist ? BK * 2 : 0;
    };
    auto tap_rows = [&](int tap) {
        const int off = a.off[tap];
#pragma unroll
        for (int i = 0; i < NA; ++i) row_of(i, off);
    };
    int rt = 0, rc = 0, rq = 0;      // tap, chunk and number of the next request
    int t0 = 0, c0 = 0, t1 = 1, c1 = 0;      // CONV_CHUNKS: tap and chunk of the step's two slices; a lane holds a piece of one of them
    const int off0 = a.off[0], dil = EPI == CONV_CHUNKS ? off0 - a.off[1] : 0;
    auto slices = [&]() {
        const int o0 = off0 - t0 * dil, o1 = off0 - t1 * dil;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            row_of(i, half_a ? o1 : o0);
            cur[i] += step[i] ? (half_a ? c1 : c0) * 64 : 0;
        }
        const ptrdiff_t w0 = ((ptrdiff_t)t0 * a.N * a.Cin + c0 * 32) * 2, w1 = ((ptrdiff_t)t1 * a.N * a.Cin + c1 * 32) * 2;
#pragma unroll
        for (int i = 0; i < NB; ++i) wp[i] = wbase[i] + (half_b[i] ? w1 : w0);
        t0 += 2; t1 += 2;
        if (t0 >= a.n_taps) { t0 -= a.n_taps; ++c0; }
        if (t1 >= a.n_taps) { t1 -= a.n_taps; ++c1; }
    };
    auto request = [&](int stage) {
        const unsigned ls = __builtin_amdgcn_readfirstlane(sbase + stage * ST);
#pragma unroll
        for (int i = 0; i < NA; ++i) lds_dma16(cur[i], ls + (i * NLD + lw) % CA * 1024);
#pragma unroll
        for (int i = 0; i < NB; ++i) lds_dma16(wp[i], ls + SA + (i * NLD + lw) % CB * 1024);
        if (++rq >= nit) return;     // (past the last step the same one is asked for again: the count in flight stays the same)
        if (EPI == CONV_CHUNKS) {
            slices();
            return;
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) cur[i] += step[i];
#pragma unroll
        for (int i = 0; i < NB; ++i) wp[i] += BK * 2;
        if (++rc == nck) {
            rc = 0;
            tap_rows(++rt);
#pragma unroll
            for (int i = 0; i < NB; ++i) wp[i] += wtap;
        }
    };
    if (loads) {
        if (EPI == CONV_CHUNKS) slices();
        else tap_rows(0);
#pragma unroll
        for (int s = 0; s < S - 1; ++s) request(s);
    }
    if (EPI != CONV_CHUNKS && a.rms_x) {      // (CONV_CHUNKS has no such rows)
        for (int r = wv; r < BM && m0 + r < a.M; r += NWV) {
            const float* x = a.rms_x + (size_t)(m0 + r) * a.Cin;
            float s = 0.0f;
            for (int c0 = lane * 4; c0 < a.Cin; c0 += 1024) {      // (four requests together; what is past the end adds nothing)
                float4 v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = ldg_f4(x + (c0 + k * 256 < a.Cin ? c0 + k * 256 : c0));
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float q = v[k].x * v[k].x + v[k].y * v[k].y + v[k].z * v[k].z + v[k].w * v[k].w;
                    s += c0 + k * 256 < a.Cin ? q : 0.0f;
                }
            }
            for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
            if (lane == 0) rms_s[r] = rsqrtf(s / (float)a.Cin + a.rms_eps);
        }
    }
    int stage = 0;
    auto landed = [&]() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * (NA + NB)) : "memory"); };
    if (!multiplies) {
        for (int it = 0; it < nit; ++it) {
            landed();
            request(stage == 0 ? S - 1 : stage - 1);
            stage = stage == S - 1 ? 0 : stage + 1;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return;
    }
    constexpr bool PARTS = NP == 3 && WP == 1 && BK >= 64;      // tiles that know ConvDmaArgs::parts
    f32x4 acc[MT][NT], done[PARTS ? MT : 1][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
            if (PARTS) done[i][j] = acc[i][j];
        }
    auto part_done = [&]() {
        if constexpr (PARTS)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    done[i][j] += acc[i][j];
                    acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
                }
    };
    const int wfr = PAIR ? (fr >> 2) * 8 + (fr & 3) : fr;
    for (int it = 0; it < nit; ++it) {
        if (loads) {
            landed();
            request(stage == 0 ? S - 1 : stage - 1);
        } else {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        if (PARTS && a.parts && it % (256 / BK) == 0) part_done();
        const char *as = conv_lds + stage * ST + (wm * MT * 16 + fr) * BK * 2, *bs = conv_lds + stage * ST + SA + (wn * NT * 16 + wfr) * BK * 2;
#pragma unroll
        for (int k = 0; k < KS / KW; ++k) {
            const int piece = (((wk * (KS / KW) + k) * 4 + fk) ^ (BK == 32 ? (fr >> 1) & 3 : fr & 7)) * 16;
            const int wpiece = (((wk * (KS / KW) + k) * 4 + fk) ^ wswz(wfr)) * 16;
            cbf16x8 bf[WP][NT];
#pragma unroll
            for (int w = 0; w < WP; ++w)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    bf[w][j] = *reinterpret_cast<const cbf16x8*>(bs + (w * BN + (PAIR ? (j >> 1) * 32 + (j & 1) * 4 : j * 16)) * BK * 2 + wpiece);
#pragma unroll
            for (int p = NP - 1; p >= 0; --p) {
                cbf16x8 af[MT];
#pragma unroll
                for (int i = 0; i < MT; ++i) af[i] = *reinterpret_cast<const cbf16x8*>(as + (p * BM + i * 16) * BK * 2 + piece);
#pragma unroll
                for (int w = WP - 1; w >= 0; --w)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
#pragma unroll
                        for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[w][j], af[i], acc[i][j], 0, 0, 0);
            }
        }
        stage = stage == S - 1 ? 0 : stage + 1;
    }
    if (KW > 1) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");        // (the repeated last steps: nothing may land any more)
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (PARTS)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = done[i][j] + acc[i][j];
    constexpr int FR = MT * NT;
    f32x4* part = reinterpret_cast<f32x4*>(conv_lds) + (size_t)wmn * KW * FR * 64 + lane;
    if (KW > 1) {
#pragma unroll
        for (int f = 0; f < FR; ++f) part[(wk * FR + f) * 64] = acc[f / NT][f % NT];
        __syncthreads();
    }
    auto sum = [&](int f) {
        if (KW == 1) return acc[f / NT][f % NT];
        f32x4 v = part[f * 64];
#pragma unroll
        for (int k = 1; k < KW; ++k) v += part[(k * FR + f) * 64];
        return v;
    };
    if constexpr (EPI == CONV_GLU) {
#pragma unroll
        for (int f = 0; f < FR; f += 2)
            if (KW == 1 || (f / 2) % KW == wk)
                conv_dma_glu(a, sum(f), sum(f + 1), rms_s[rl + f / NT * 16], m0 + rl + f / NT * 16, (nl >> 1) + f % NT * 8 + fk * 4);
    } else {
        const float* rms = a.rms_x ? rms_s + rl : nullptr;
#pragma unroll
        for (int j = 0; j < NT; j += P) {
            const int n = nl + j * 16 + fk * 4 * P;
            if constexpr (KW == 1) {
                f32x4 v[MT][P];
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int q = 0; q < P; ++q) v[i][q] = acc[i][j + q];
                if constexpr (EARLY) conv_dma_out<NP == 3 ? 3 : 2, EPI, 4 * P, MT, true>(a, v, rms, m0 + rl, n, nullptr, kc[j / P]);
                else conv_dma_out<NP == 3 ? 3 : 2, EPI, 4 * P, MT>(a, v, rms, m0 + rl, n);
            } else {
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    if ((i * (NT / P) + j / P) % KW == wk) {
                        f32x4 v[1][P];
#pragma unroll
                        for (int q = 0; q < P; ++q) v[0][q] = sum(i * NT + j + q);
                        conv_dma_out<NP == 3 ? 3 : 2, EPI, 4 * P, 1>(a, v, rms ? rms + i * 16 : nullptr, m0 + rl + i * 16, n);
                    }
            }
        }
    }
}

// A whole residual unit of a decoder:  h += conv2(act2(conv1(x)))  and  out2 = act_next(h);  conv1: TAPS taps C -> CH, conv2: one tap CH -> C;
// T = 2: SnakeBeta over two-term rows (Qwen3 codec: 7 taps, dilated, CH = C), T = 3: ELU over three-term rows (Mimi: 3 taps, CH = C / 2).
// A block takes 16 MT NW rows of one request and ALL C channels of them; a wave takes 16 MT rows.  conv1 walks K in 32-channel chunks: a
// chunk's rows with their look-back (up to HP) are staged once for all taps (two buffers, the next chunk's requests spread over the
// taps of this one), the weights are a stream of C x 32 slices through S stages.  What the lanes then hold, eight neighbouring channels
// of a row, is after SnakeBeta and the two-term split the activation operand of conv2 as it stands: conv2 is C / 32 further slices of the
// same stream, and the intermediate never leaves the registers.  x, the history and the weights arrive by LDS DMA as in k_conv_dma.
// Bound: memory (x, h read, h, out2 written: 944 MB at 614 400 rows x 96) beside the matrix cores and the activations' VALU work: 335 us on
// average there within a chunk, 2.8 TB/s; the staged form of this kernel, with the intermediate through LDS, took 461 - 498.  (Against 309 when
// timed alone: 326 with the residual asked for in the epilogue, 311 - 332 with four stages or 64-row blocks.)
template <int C, int CH, int TAPS, int T, int HP, int NW, int MT, int S>
__global__ __launch_bounds__(64 * NW, C == 192 ? 2 : C == 128 ? 3 : 4) void k_conv_unit(ConvDmaArgs a1, ConvDmaArgs a2, int H) {
    touch_args(a1);
    touch_args(a2);
    constexpr int BM = 16 * MT * NW, R = BM + HP, NT = CH / 16, NP = CH / 32, NT2 = C / 16, NCK = C / 32;
    constexpr int SA = T * R * 64, CA = SA / 1024, NA = (CA + NW - 1) / NW, CW1 = CH / 16, CW2 = C / 16, SW = (C > CH ? C : CH) * 64;
    constexpr int NB = ((C > CH ? CW2 : CW1) + NW - 1) / NW;       // requests of a wave per slice (the smaller kind repeats some)
    constexpr int AT = (NA + TAPS - S + 1) / (TAPS - S + 2), AN = (NA + AT - 1) / AT;      // requests for rows per tap, taps that make them
    static_assert(AN <= TAPS - S + 2, "a chunk's rows are asked for by the taps that the next chunk's first wait covers");
    extern __shared__ __attribute__((aligned(1024))) char conv_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    if ((int)blockIdx.x >= a1.tiles8) {
        conv_job(a1.job, a1.slots, (int)blockIdx.x - a1.tiles8, 64 * NW);
        return;
    }
    const int t = ((int)blockIdx.x & 7) * (a1.tiles8 >> 3) + ((int)blockIdx.x >> 3);
    if (t >= a1.tm) return;
    const int m0 = t * BM, fr = lane & 15, fk = lane >> 4;
    const int b = m0 / a1.L, t0 = m0 - b * a1.L;
    constexpr int rb = C * (T == 3 ? 6 : 4);
    // rows t0 - H .. t0 + BM - 1 at LDS rows 0 .. (the buffer's last rows repeat the tile's last one: no tap reads them)
    const char* xp[NA];
    int step[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int q = (i * NW + wv) % CA * 64 + lane, pl = q / (R * 4), r = q / 4 % R, pc = (q & 3) ^ ((r >> 1) & 3);
        int e = t0 - H + r;
        e = e < t0 + BM ? e : t0 + BM - 1;
        const bool hist = e < 0 && a1.state && a1.P + e >= 0;
        const char* p = e >= 0 ? reinterpret_cast<const char*>(a1.x) + ((size_t)b * a1.L + e) * rb
                               : reinterpret_cast<const char*>(a1.state) + ((size_t)a1.slots[b] * a1.P + a1.P + e) * rb;
        xp[i] = e >= 0 || hist ? p + pl * C * 2 + pc * 16 : reinterpret_cast<const char*>(g_conv_zero_row);
        step[i] = e >= 0 || hist ? 64 : 0;
    }
    const auto wswz = [](int r) { return ((r >> 1) & 1) | ((r >> 2) & 2); };      // (rows are read as in k_conv_dma's PAIR order)
    unsigned wo1[NB], wo2[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int c1 = (i * NW + wv) % CW1 * 16 + (lane >> 2), c2 = (i * NW + wv) % CW2 * 16 + (lane >> 2);
        wo1[i] = (unsigned)(c1 * C + ((lane & 3) ^ wswz(c1)) * 8) * 2;
        wo2[i] = (unsigned)(c2 * CH + ((lane & 3) ^ wswz(c2)) * 8) * 2;
    }
    // the residual rows: asked for first where registers allow (their wait is the first rows' own)
    constexpr bool EARLY = C <= 128 && MT == 1;
    f32x4 res[EARLY ? NT2 / 2 : 1][2];
    if (EARLY) {
#pragma unroll
        for (int p = 0; p < NT2 / 2; ++p)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                res[p][q] = *reinterpret_cast<const f32x4*>(a2.res + (size_t)(m0 + wv * 16 + fr) * C + p * 32 + fk * 8 + 4 * q);
    }
    const unsigned sbase = (unsigned)(size_t)(__attribute__((address_space(3))) char*)conv_lds;
    auto rows = [&](int i, int buf) {
        lds_dma16(xp[i], __builtin_amdgcn_readfirstlane(sbase + buf * SA + (i * NW + wv) % CA * 1024));
        xp[i] += step[i];
    };
    int rt = 0, rc = 0, rs = 0;      // tap, chunk and stage of the next slice; past conv1's chunks: conv2's
    auto slice = [&]() {
        const bool second = rc >= NCK;
        const int kc = second ? (rt < NP ? rt : NP - 1) : rc;      // (past the last slice it is asked for again)
        const size_t at = reinterpret_cast<size_t>(second ? a2.w : a1.w) + ((second ? 0 : rt * C * CH) + kc * 32) * 2;
        const char* base = reinterpret_cast<const char*>((size_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32 |
                                                         (unsigned)__builtin_amdgcn_readfirstlane((int)at));
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int c = i * NW + wv;
            const unsigned ld = __builtin_amdgcn_readfirstlane(sbase + 2 * SA + rs * SW + (second ? c % CW2 : c % CW1) * 1024);
            const unsigned off = second ? wo2[i] : wo1[i];
            lds_dma16(base, off, ld);
        }
        rs = rs == S - 1 ? 0 : rs + 1;
        if (++rt == TAPS && !second) {
            rt = 0;
            ++rc;
        }
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NA; ++i) rows(i, 0);
#pragma unroll
    for (int i = 0; i < S - 1; ++i) slice();
    const int wfr = (fr >> 2) * 8 + (fr & 3), wpiece = (fk ^ wswz(wfr)) * 16;
    int ws = 0;      // stage of the slice being multiplied
    auto weights = [&](auto& wf) {
        const char* p = conv_lds + 2 * SA + ws * SW + wfr * 64 + wpiece;
#pragma unroll
        for (int j = 0; j < (int)(sizeof(wf) / sizeof(wf[0])); ++j) wf[j] = *reinterpret_cast<const cbf16x8*>(p + ((j >> 1) * 32 + (j & 1) * 4) * 64);
        ws = ws == S - 1 ? 0 : ws + 1;
    };
    auto chunk = [&](int ck, auto last_tag) {
        constexpr bool LAST = decltype(last_tag)::value;
        const char* As = conv_lds + (ck & 1) * SA;
        auto tap = [&](auto tap_tag) {
            constexpr int TP = decltype(tap_tag)::value;
            // requests younger than this tap's slice: S - 2 slices and what the taps since then asked of the next chunk's rows
            constexpr int lo = TP - S + 2 > 0 ? (TP - S + 2) * AT : 0, hi = TP * AT < NA ? TP * AT : NA, young = (S - 2) * NB + (!LAST && hi > lo ? hi - lo : 0);
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(young) : "memory");
#pragma unroll
            for (int q = TP * AT; q < (TP + 1) * AT; ++q)
                if (!LAST && q < NA) rows(q, (ck + 1) & 1);
            slice();
            const int r0 = wv * MT * 16 + fr + H - a1.off[TP];
            cbf16x8 wf[NT];
            weights(wf);
#pragma unroll
            for (int p = T - 1; p >= 0; --p)
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    const int r = r0 + i * 16;
                    const cbf16x8 af = *reinterpret_cast<const cbf16x8*>(As + (p * R + r) * 64 + (fk ^ ((r >> 1) & 3)) * 16);
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], af, acc[i][j], 0, 0, 0);
                }
        };
        tap(std::integral_constant<int, 0>{}); tap(std::integral_constant<int, 1>{}); tap(std::integral_constant<int, 2>{});
        if constexpr (TAPS == 7) {
            tap(std::integral_constant<int, 3>{}); tap(std::integral_constant<int, 4>{}); tap(std::integral_constant<int, 5>{});
            tap(std::integral_constant<int, 6>{});
        }
    };
    static_assert(TAPS == 3 || TAPS == 7, "tap list");
    for (int ck = 0; ck + 1 < NCK; ++ck) chunk(ck, std::false_type{});
    chunk(NCK - 1, std::true_type{});
    // act2 of the sums, split: the operand of conv2 (channels 32 p + 8 fk + 0..7 of the lane's row)
    cbf16x8 y[MT][NP][T];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int c = p * 32 + fk * 8;
        float bi[8], al[8], ib[8];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const f32x4 tb = a1.bias ? *reinterpret_cast<const f32x4_a4*>(a1.bias + c + 4 * q) : (f32x4){0.f, 0.f, 0.f, 0.f};
            f32x4 ta = tb, ti = tb;
            if constexpr (T == 2) {
                ta = *reinterpret_cast<const f32x4_a4*>(a1.sn_alpha + c + 4 * q);
                ti = *reinterpret_cast<const f32x4_a4*>(a1.sn_invb + c + 4 * q);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) { bi[4 * q + e] = tb[e]; al[4 * q + e] = ta[e]; ib[4 * q + e] = ti[e]; }
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] = acc[i][2 * p + e / 4][e % 4] + bi[e];
                if constexpr (T == 2) v[e] = snake_f(v[e], al[e], ib[e]);
                else v[e] = v[e] > 0.0f ? v[e] : expm1f(v[e]);
            }
#pragma unroll
            for (int t3 = 0; t3 < T; ++t3) {
                unsigned h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    h[e] = pack_bf2(v[2 * e], v[2 * e + 1]);
                    v[2 * e] -= bflo(h[e]);
                    v[2 * e + 1] -= bfhi(h[e]);
                }
                y[i][p][t3] = as_cbf8(make_uint4(h[0], h[1], h[2], h[3]));
            }
        }
    }
    f32x4 out[MT][NT2];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT2; ++j) out[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * NB) : "memory");
        slice();
        cbf16x8 wf[NT2];
        weights(wf);
#pragma unroll
        for (int p = T - 1; p >= 0; --p)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT2; ++j) out[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], y[i][k][p], out[i][j], 0, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // (the repeated last slices: nothing may land after the block has ended)
#pragma unroll
    for (int p = 0; p < NT2 / 2; ++p) {
        f32x4 v[MT][2];
#pragma unroll
        for (int i = 0; i < MT; ++i) { v[i][0] = out[i][2 * p]; v[i][1] = out[i][2 * p + 1]; }
        conv_dma_out<T, 0, 8, MT>(a2, v, nullptr, m0 + wv * MT * 16 + fr, p * 32 + fk * 8, EARLY ? res[EARLY ? p : 0] : nullptr);
    }
}

// Few-row variant (M <= 48: the transformer and the first upsampling stages of a single request's chunk): tile
// 16(M) x 64(N), one n-tile per wave, K walked in BK-wide chunks (128 where Cin allows) with the same one-step
// register prefetch.  These stages run a handful of blocks: time = number of dependent K steps, so the steps are wide.
template <int BK, bool LN = false>
__global__ __launch_bounds__(256) void k_conv_gemm_skinny(ConvGemmArgs a) {
    touch_args(a);
    constexpr int LD = BK + 8;                      // bf16 elements
    constexpr int NA = (16 * BK / 4 + 255) / 256;   // float4 per thread (activations)
    constexpr int NB = 64 * BK / 8 / 256;           // uint4 per thread (weights)
    constexpr int SEGA = BK / 4, SEGB = BK / 8;
    __shared__ __attribute__((aligned(16))) bf16_t As[3][16 * LD];
    __shared__ __attribute__((aligned(16))) bf16_t Bs[64 * LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * 16, n0 = blockIdx.x * 64;
    f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int nck = a.Cin / BK, nit = a.n_taps * nck;
    float4 av[NA];
    uint4 bv[NB];
    auto fetch = [&](int it) {
        const int tap = it / nck, c0 = (it - tap * nck) * BK;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int idx = tid + 256 * i, r = idx / SEGA, seg = idx % SEGA;
            av[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            const int am = m0 + r;
            if (idx < 16 * SEGA && am < a.M) {
                const int ab = am / a.L, st = am % a.L - a.off[tap];
                const float* arow = nullptr;
                if (st >= a.L) arow = nullptr;
                else if (st >= 0) arow = a.x + ((size_t)ab * a.L + st) * a.Cin;
                else if (a.state && a.P + st >= 0) arow = a.state + ((size_t)a.slots[ab] * a.P + (a.P + st)) * a.Cin;
                if (arow) av[i] = *reinterpret_cast<const float4*>(arow + c0 + seg * 4);
            }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int idx = tid + 256 * i, r = idx / SEGB, seg = idx % SEGB;
            const int bn = n0 + r;
            bv[i] = make_uint4(0, 0, 0, 0);
            if (bn < a.N) bv[i] = *reinterpret_cast<const uint4*>(a.w + ((size_t)tap * a.N + bn) * a.Cin + c0 + seg * 8);
        }
    };
    fetch(0);
    __shared__ float ln_stat[LN ? 32 : 1];
    if (LN) {      // row statistics of the block's 16 rows (two passes, 16 lanes per row), while the first operands are in flight
        const int r = tid >> 4, l16 = tid & 15, am = m0 + r;
        float mean = 0.0f, rstd = 0.0f;
        if (am < a.M) ln_row_stats(a.x + (size_t)am * a.Cin, a.Cin, l16, a.ln_eps, mean, rstd);
        if (l16 == 0) { ln_stat[2 * r] = mean; ln_stat[2 * r + 1] = rstd; }
    }
    auto kloop = [&](auto np_tag) {       // (the plane count as a compile-time constant: see k_conv_gemm)
    constexpr int NP = decltype(np_tag)::value;
    for (int it = 0; it < nit; ++it) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int idx = tid + 256 * i;
            if (idx < 16 * SEGA) {      // 4 fp32 -> 4 bf16 per plane (8 bytes)
                float x4[4] = {av[i].x, av[i].y, av[i].z, av[i].w};
                if (LN) {
                    const int r = idx / SEGA, c = (it % nck) * BK + (idx % SEGA) * 4;
                    const float mean = ln_stat[2 * r], rstd = ln_stat[2 * r + 1];
                    const float4 w4 = *reinterpret_cast<const float4*>(a.ln_w + c), b4 = *reinterpret_cast<const float4*>(a.ln_b + c);
                    x4[0] = (x4[0] - mean) * rstd * w4.x + b4.x; x4[1] = (x4[1] - mean) * rstd * w4.y + b4.y;
                    x4[2] = (x4[2] - mean) * rstd * w4.z + b4.z; x4[3] = (x4[3] - mean) * rstd * w4.w + b4.w;
                }
                unsigned short hb[4], mb[4], lb[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    hb[e] = f2bf(x4[e]);
                    const float r1 = x4[e] - bf2f(hb[e]);
                    mb[e] = f2bf(r1);
                    lb[e] = f2bf(r1 - bf2f(mb[e]));
                }
                const int o = (idx / SEGA) * LD + (idx % SEGA) * 4;
                *reinterpret_cast<uint2*>(&As[0][o]) = make_uint2(hb[0] | (unsigned)hb[1] << 16, hb[2] | (unsigned)hb[3] << 16);
                *reinterpret_cast<uint2*>(&As[1][o]) = make_uint2(mb[0] | (unsigned)mb[1] << 16, mb[2] | (unsigned)mb[3] << 16);
                *reinterpret_cast<uint2*>(&As[2][o]) = make_uint2(lb[0] | (unsigned)lb[1] << 16, lb[2] | (unsigned)lb[3] << 16);
            }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int idx = tid + 256 * i;
            *reinterpret_cast<uint4*>(&Bs[(idx / SEGB) * LD + (idx % SEGB) * 8]) = bv[i];
        }
        __syncthreads();
        if (it + 1 < nit) fetch(it + 1);
        const int fr = lane & 15, fk = (lane >> 4) * 8;
#pragma unroll
        for (int kb = 0; kb < BK; kb += 32) {
            const uint4 bfr = *reinterpret_cast<const uint4*>(&Bs[(wave * 16 + fr) * LD + kb + fk]);
#pragma unroll
            for (int t = NP - 1; t >= 0; --t) {
                const uint4 afr = *reinterpret_cast<const uint4*>(&As[t][fr * LD + kb + fk]);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_cbf8(afr), as_cbf8(bfr), acc, 0, 0, 0);
            }
        }
    }
    };
    if (a.planes >= 3) kloop(std::integral_constant<int, 3>{});
    else if (a.planes == 2) kloop(std::integral_constant<int, 2>{});
    else kloop(std::integral_constant<int, 1>{});
    const int n = n0 + wave * 16 + (lane & 15);
    if (n >= a.N) return;
    const float bvv = a.bias ? a.bias[n % a.bias_mod] : 0.0f;
    const float sv = a.scale ? a.scale[n] : 1.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = m0 + (lane >> 4) * 4 + r;
        if (m >= a.M) continue;
        float v = acc[r] + bvv;
        if (a.gelu) v = gelu_f(v);
        if (a.rscale) v = a.rscale[m] * v;
        const size_t o = (size_t)m * a.N + n;
        if (a.res) v = a.res[o] + sv * v;
        else if (a.scale) v = sv * v;
        if (a.out) a.out[o] = v;
        if (a.out2) {
            const float sv2 = snake_f(v, a.sn_alpha[n % a.sn_mod], a.sn_invb[n % a.sn_mod]);
            a.out2[o] = sv2;
        }
    }
}

// Few-row GEMM with no dependent K steps ("rows" kernel; the flow detokenizers' 56..2752-row linears and causal convs: thousands of
// launches per chunk whose time is exposed memory latency, not arithmetic).  A block owns 16 MT rows x 16 NT columns; its WV waves split
// the n_taps * Cin reduction into WV runs of KB 32-wide k-blocks and each lane requests ALL its operands up front, straight in the
// layout an MFMA operand register holds (A: 8 consecutive fp32 of row lane % 16; B: 8 consecutive bf16 of weight row lane % 16) — one
// exposed round trip per launch, no LDS staging, no barrier until the cross-wave sum (fixed order w0 + w1 + ... ).  With the fused
// LayerNorm the row statistics come from the operand registers while the weights are in flight.  A row's result depends on that row only
// and on (K, WV) — never on MT / NT, which the launcher picks from the row count: more rows per block when the call is large enough
// that the operand traffic from L2 (12 KB per 16 x 16 output tile at MT = 1, NT = 4, K = 256) is what bounds it.  WV is a function of K
// alone (8 waves from K = 512 on: half the serial work per wave), so a request's output does not depend on what shares its batch.
template <int KB, int NT, bool LN, int MT, int WV>
__global__ __launch_bounds__(64 * WV) void k_rows_gemm(ConvGemmArgs a) {
    touch_args(a);
    __shared__ float red[WV][MT * NT][256];
    __shared__ float ln_stat[LN ? 2 * WV * 16 * MT : 1];
    // (the wave index provably uniform: the tap of a k-block, and with it a.off[tap], is then a scalar — read per lane from the argument
    // block it was a dependent vector load, one round trip in front of every operand row's address)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, kq = lane >> 4;
    const int m0 = blockIdx.y * 16 * MT, n0 = blockIdx.x * 16 * NT;
    const int kpt = a.Cin >> 5;                     // k-blocks per tap
    float4 av[MT][KB][2];
    uint4 bv[NT][KB];
    float4 lw[LN ? KB : 1][2], lb[LN ? KB : 1][2];
    // No load stands behind a branch of its own: rows and columns beyond the last read that one (nothing stores them), rows outside a request read the
    // lane's own row and are zeroed in the registers (`out_of`).  The history's slot is asked for by the waves that have such a row, ahead of everything.
    int col[KB], off[KB], tap_of[KB];
    {
        int tap = a.kpt_inv ? (int)__umulhi((unsigned)(wave * KB), a.kpt_inv) : wave * KB / kpt, kc = wave * KB - tap * kpt;
#pragma unroll
        for (int j = 0; j < KB; ++j) {
            tap_of[j] = tap; col[j] = kc * 32; off[j] = a.off[tap];
            if (++kc == kpt) { kc = 0; ++tap; }
        }
    }
    int back = off[0];
#pragma unroll
    for (int j = 1; j < KB; ++j) back = back > off[j] ? back : off[j];
    const int first = a.state ? -a.P : 0;      // rows of a request and its history: first .. L - 1
    const unsigned span = (unsigned)(a.L - first);
    const float *row[MT], *hist[MT];
    int al[MT];
    unsigned out_of = 0;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = m0 + mt * 16 + fr, am = m < a.M ? m : a.M - 1, ab = a.len_inv ? (int)__umulhi((unsigned)am, a.len_inv) : am / a.L;
        al[mt] = am - ab * a.L;
        row[mt] = hist[mt] = a.x + (size_t)am * a.Cin + kq * 8;
        if (a.state && __ballot(al[mt] < back)) hist[mt] = a.state + ((size_t)a.slots[ab] * a.P + (a.P + al[mt])) * a.Cin + kq * 8;
    }
    auto load_rows = [&] {
#pragma unroll
        for (int j = 0; j < KB; ++j)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int st = al[mt] - off[j];
                const bool none = (unsigned)(st - first) >= span;
                out_of |= none ? 1u << (mt * KB + j) : 0u;
                const float* p = (st < 0 ? hist[mt] : row[mt]) + (none ? (ptrdiff_t)col[j] : (ptrdiff_t)col[j] - (ptrdiff_t)off[j] * a.Cin);
                av[mt][j][0] = ldg_f4(p);
                av[mt][j][1] = ldg_f4(p + 4);
            }
    };
    if (LN) load_rows();      // (their statistics come first)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int n = n0 + t * 16 + fr;
        const unsigned wo = (unsigned)(n < a.N ? n : a.N - 1) * (unsigned)a.Cin + kq * 8;
#pragma unroll
        for (int j = 0; j < KB; ++j) bv[t][j] = *reinterpret_cast<const uint4*>(a.w + ((size_t)tap_of[j] * a.N * a.Cin + col[j]) + wo);
    }
    if (LN)
#pragma unroll
        for (int j = 0; j < KB; ++j) {
            const int c0 = col[j] + kq * 8;
            lw[j][0] = *reinterpret_cast<const float4*>(a.ln_w + c0); lw[j][1] = *reinterpret_cast<const float4*>(a.ln_w + c0 + 4);
            lb[j][0] = *reinterpret_cast<const float4*>(a.ln_b + c0); lb[j][1] = *reinterpret_cast<const float4*>(a.ln_b + c0 + 4);
        }
    else load_rows();
    const bool zeroes = __ballot(out_of != 0);
    float mean[MT], rstd[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) mean[mt] = rstd[mt] = 0.0f;
    if (LN) {
        // Row statistics from the operand registers (one tap: the block's WV KB k-blocks are exactly the row): lane (fr, kq) of wave w
        // holds 8 KB values of row fr; two passes (mean, then centred squares), each = lane sum -> the row's four k groups by two
        // butterfly steps -> the waves in the fixed order w0 + w1 + ...  No second trip to memory for the centred pass.
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < KB; ++j)
                s += ((av[mt][j][0].x + av[mt][j][0].y) + (av[mt][j][0].z + av[mt][j][0].w)) + ((av[mt][j][1].x + av[mt][j][1].y) + (av[mt][j][1].z + av[mt][j][1].w));
            s = xor_add<32>(xor_add<16>(s));
            if (kq == 0) ln_stat[(mt * WV + wave) * 16 + fr] = s;
        }
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            float tot = ln_stat[mt * WV * 16 + fr];
#pragma unroll
            for (int w = 1; w < WV; ++w) tot += ln_stat[(mt * WV + w) * 16 + fr];
            mean[mt] = tot / (float)a.Cin;
            float vs = 0.0f;
#pragma unroll
            for (int j = 0; j < KB; ++j) {
                const float d0 = av[mt][j][0].x - mean[mt], d1 = av[mt][j][0].y - mean[mt], d2 = av[mt][j][0].z - mean[mt], d3 = av[mt][j][0].w - mean[mt];
                const float d4 = av[mt][j][1].x - mean[mt], d5 = av[mt][j][1].y - mean[mt], d6 = av[mt][j][1].z - mean[mt], d7 = av[mt][j][1].w - mean[mt];
                vs += ((d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3)) + ((d4 * d4 + d5 * d5) + (d6 * d6 + d7 * d7));
            }
            vs = xor_add<32>(xor_add<16>(vs));
            if (kq == 0) ln_stat[(MT * WV + mt * WV + wave) * 16 + fr] = vs;
        }
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            float tot = ln_stat[(MT * WV + mt * WV) * 16 + fr];
#pragma unroll
            for (int w = 1; w < WV; ++w) tot += ln_stat[(MT * WV + mt * WV + w) * 16 + fr];
            rstd[mt] = rsqrtf(tot / (float)a.Cin + a.ln_eps);
        }
    }
    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[mt][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < KB; ++j) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            float x8[8] = {av[mt][j][0].x, av[mt][j][0].y, av[mt][j][0].z, av[mt][j][0].w, av[mt][j][1].x, av[mt][j][1].y, av[mt][j][1].z, av[mt][j][1].w};
            if (LN) {
                const float w8[8] = {lw[j][0].x, lw[j][0].y, lw[j][0].z, lw[j][0].w, lw[j][1].x, lw[j][1].y, lw[j][1].z, lw[j][1].w};
                const float b8[8] = {lb[j][0].x, lb[j][0].y, lb[j][0].z, lb[j][0].w, lb[j][1].x, lb[j][1].y, lb[j][1].z, lb[j][1].w};
#pragma unroll
                for (int e = 0; e < 8; ++e) x8[e] = (x8[e] - mean[mt]) * rstd[mt] * w8[e] + b8[e];
            }
            if (zeroes) {
                const bool z = out_of >> (mt * KB + j) & 1;
#pragma unroll
                for (int e = 0; e < 8; ++e) x8[e] = z ? 0.0f : x8[e];
            }
            u32 h[3][4];
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    h[p][e] = pack_bf2(x8[2 * e], x8[2 * e + 1]);
                    if (p < 2) { x8[2 * e] -= bflo(h[p][e]); x8[2 * e + 1] -= bfhi(h[p][e]); }
                }
#pragma unroll
            for (int t = 0; t < NT; ++t)      // plane order of the staged kernels: low terms first
#pragma unroll
                for (int p = 2; p >= 0; --p)
                    acc[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_cbf8(make_uint4(h[p][0], h[p][1], h[p][2], h[p][3])), as_cbf8(bv[t][j]), acc[mt][t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][mt * NT + t][r * 64 + lane] = acc[mt][t][r];
    __syncthreads();
    // work item e = (tile, accumulator component r): row m0 + 16 mt + 4 (lane / 16) + r, column n0 + 16 t + lane % 16; wave w takes
    // the items w, w + WV, ...  Two passes: every operand of every item of this wave (bias, scale, row scale, residual)
    // is requested first, branch-free (clamped indices), THEN the arithmetic and the stores — item by item the loads of item i + 1 could not
    // move above the stores of item i (the residual may alias the output), and an item cost up to three dependent round trips: the
    // epilogue was most of this kernel's time.  Per element the operations and their order are unchanged.
    constexpr int NE = (MT * NT * 4 + WV - 1) / WV;
    float e_b[NE], e_s[NE], e_rs[NE], e_res[NE];
    const int Mc = a.M - 1, Nc = a.N - 1;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const int e = wave + i * WV, tile = (e >> 2) < MT * NT ? (e >> 2) : 0, r = e & 3, mt = tile / NT, t = tile - mt * NT;
        int m = m0 + mt * 16 + kq * 4 + r, n = n0 + t * 16 + fr;
        m = m < Mc ? m : Mc; n = n < Nc ? n : Nc;
        e_b[i] = a.bias ? a.bias[a.bias_mod >= a.N ? n : n % a.bias_mod] : 0.0f;
        e_s[i] = a.scale ? a.scale[n] : 1.0f;
        e_rs[i] = a.rscale ? a.rscale[m] : 1.0f;
        e_res[i] = a.res ? a.res[(size_t)m * a.N + n] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const int e = wave + i * WV;
        if (e >= MT * NT * 4) continue;
        const int tile = e >> 2, r = e & 3, mt = tile / NT, t = tile - mt * NT;
        const int m = m0 + mt * 16 + kq * 4 + r, n = n0 + t * 16 + fr;
        if (m >= a.M || n >= a.N) continue;
        const int idx = r * 64 + lane;
        float v = red[0][tile][idx];
#pragma unroll
        for (int w = 1; w < WV; ++w) v += red[w][tile][idx];
        v += e_b[i];
        const float sv = e_s[i];
        if (a.gelu) v = gelu_f(v);
        if (a.rscale) v = e_rs[i] * v;
        const size_t o = (size_t)m * a.N + n;
        if (a.res) v = e_res[i] + sv * v;
        else if (a.scale) v = sv * v;
        a.out[o] = v;
    }
}

// ================================================================================================
// small kernels
// ================================================================================================
// element c of row `row` of a C-wide activation: fp32 (terms == 0), or the two / three terms of an S2 / S3 row
__device__ __forceinline__ void put_row(float* y, size_t row, int C, int c, float v, int terms) {
    if (terms == 0) {
        y[row * C + c] = v;
        return;
    }
    bf16_t* r16 = reinterpret_cast<bf16_t*>(y) + row * C * terms + c;
    for (int t = 0; t < terms; ++t) {
        const bf16_t h = f2bf(v);
        r16[(size_t)t * C] = h;
        v -= bf2f(h);
    }
}
// RVQ decode: q0 = emb[0][code0], qr = sum_{k>=1} emb[k][code_k] (sequential in k)      qwen3_codec.py:1204-1210
__global__ __launch_bounds__(256) void k_rvq(const int* codes, int code_stride, const float* emb, int Q, int bins, int vq,
                                             float* q0, float* qr, int terms) {
    const int row = blockIdx.x;
    const int* cr = codes + (size_t)row * code_stride;
    for (int d = threadIdx.x; d < vq; d += 256) {
        int c0 = cr[0];
        c0 = c0 < 0 ? 0 : (c0 >= bins ? bins - 1 : c0);          // postprocess clamps to [0, bins-1] (qwen3_tts.py:2027)
        put_row(q0, row, vq, d, emb[((size_t)c0) * vq + d], terms);
        float s = 0.0f;
        for (int k0 = 1; k0 < Q; k0 += 8) {      // (asked for eight at a time: 16 codes, 2 rows 6.8 -> 4.1 us)
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int k = k0 + u < Q ? k0 + u : Q - 1;
                int c = cr[k];
                c = c < 0 ? 0 : (c >= bins ? bins - 1 : c);
                v[u] = ldg(emb + ((size_t)k * bins + c) * vq + d);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) s = k0 + u < Q ? s + v[u] : s;
        }
        put_row(qr, row, vq, d, s, terms);
    }
}

// new_state = last P rows of [state ++ x]; one thread per (request, channel), ascending rows (in-place safe)
__global__ __launch_bounds__(256) void k_state_update(float* state, const int* slots, const float* x, int L, int P, int C) {
    const int b = blockIdx.y;
    float* s = state + (size_t)slots[b] * P * C;
    const float* xb = x + (size_t)b * L * C;
    for (int c = blockIdx.x * 256 + threadIdx.x; c < C; c += gridDim.x * 256)
        for (int j = 0; j < P; ++j) {
            const int e = L + j;   // index into ext = [state(P) ++ x(L)]
            s[(size_t)j * C + c] = e < P ? s[(size_t)e * C + c] : xb[(size_t)(e - P) * C + c];
        }
}

// SnakeBeta: y = x + inv_beta[c] * sin(x * alpha[c])^2          qwen3_codec.py:1004-1018 (alpha/beta pre-exponentiated)
__global__ __launch_bounds__(256) void k_snake(const float* x, const float* alpha, const float* inv_beta, float* y,
                                               size_t total, int C, int terms) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % C);
        const float v = x[i];
        const float s = sinf(v * alpha[c]);
        put_row(y, i / C, C, (int)(i % C), v + inv_beta[c] * (s * s), terms);
    }
}

__device__ __forceinline__ float block_sum(float v, float* red) {
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    const int wave = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[wave] = v;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

// codec RMSNorm: y = w * (x * rsqrt(mean(x^2) + eps))       qwen3_codec.py:713-718
__global__ __launch_bounds__(256) void k_rmsnorm_f32(const float* x, const float* w, float* y, int C, float eps) {
    __shared__ float red[4];
    const float* xr = x + (size_t)blockIdx.x * C;
    float s = 0.0f;
    for (int c = threadIdx.x; c < C; c += 256) s += xr[c] * xr[c];
    s = block_sum(s, red);
    const float r = rsqrtf(s / (float)C + eps);
    for (int c = threadIdx.x; c < C; c += 256) y[(size_t)blockIdx.x * C + c] = w[c] * (xr[c] * r);
}

// RoPE (NeoX halves) on q in place; k rotated and v written to the bf16 KV ring.   qwen3_codec.py:212-236, 614-631
// qkv [rows, 3*HD]; ring [slots][Wn][2][HD] bf16; pos[slot] = tokens already in the window's history.
__global__ __launch_bounds__(256) void k_codec_rope_kv(float* qkv, bf16_t* ring, const int* slots, const long* pos, int T,
                                                       int H, int D, int Wn, const float* inv_freq) {
    const int row = blockIdx.x, b = row / T, t = row % T;
    const int HD = H * D, half = D / 2;
    const long p = pos[slots[b]] + t;
    float* q = qkv + (size_t)row * 3 * HD;
    float* k = q + HD;
    const float* v = q + 2 * HD;
    bf16_t* rk = ring + (((size_t)slots[b] * Wn + (p % Wn)) * 2) * HD;
    bf16_t* rv = rk + HD;
    for (int e = threadIdx.x; e < H * half; e += 256) {
        const int h = e / half, i = e % half;
        const float ang = (float)p * inv_freq[i];
        const float c = cosf(ang), s = sinf(ang);
        const int ia = h * D + i, ib = ia + half;
        const float qa = q[ia], qb = q[ib], ka = k[ia], kb = k[ib];
        q[ia] = qa * c - qb * s;
        q[ib] = qb * c + qa * s;
        rk[ia] = f2bf(ka * c - kb * s);
        rk[ib] = f2bf(kb * c + ka * s);
    }
    for (int e = threadIdx.x; e < HD; e += 256) rv[e] = f2bf(v[e]);
}

// windowed attention over the ring.  Query i (absolute position p0+i) sees absolute positions
// [p0+T-Wn, p0+i]; positions < 0 are the reference's never-written zero slots, which stay visible.
// One block per (head, request): K/V ring tile in LDS (row stride D+1: conflict-free both for "lane = key" in the
// scores and "lane = dim" in PV), the T queries of the chunk spread over the four waves.
__global__ __launch_bounds__(256) void k_codec_attn(const float* qkv, const bf16_t* ring, const int* slots, const long* pos,
                                                    float* out, int T, int H, int D, int Wn, int terms) {
    extern __shared__ float sm[];   // K [Wn][D+1], V [Wn][D+1], Q [T][D], P [4][Wn]
    const int LD = D + 1;
    float* Ks = sm;
    float* Vs = Ks + (size_t)Wn * LD;
    float* Qs = Vs + (size_t)Wn * LD;
    float* Ps = Qs + (size_t)T * D;
    const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int HD = H * D;
    const int slot = slots[b];
    const long p0 = pos[slot];
    const long lo = p0 + T - Wn;   // absolute position of logical slot 0
    for (int e = tid; e < Wn * D; e += 256) {
        const int j = e / D, d = e % D;
        const long ap = lo + j;
        float kv = 0.0f, vv = 0.0f;
        if (ap >= 0) {
            const bf16_t* r = ring + (((size_t)slot * Wn + (ap % Wn)) * 2) * HD + (size_t)h * D + d;
            kv = bf2f(r[0]);
            vv = bf2f(r[HD]);
        }
        Ks[j * LD + d] = kv;
        Vs[j * LD + d] = vv;
    }
    for (int e = tid; e < T * D; e += 256) Qs[e] = qkv[((size_t)(b * T + e / D)) * 3 * HD + (size_t)h * D + e % D];
    __syncthreads();
    const float scale = rsqrtf((float)D);
    float* P = Ps + (size_t)wave * Wn;
    for (int i = wave; i < T; i += 4) {
        const float* q = Qs + (size_t)i * D;
        const int nvis = Wn - T + i + 1;
        float mx = -INFINITY;
        for (int j = lane; j < Wn; j += 64) {
            float sc = -INFINITY;
            if (j < nvis) {
                sc = 0.0f;
                for (int d = 0; d < D; ++d) sc = fmaf(q[d], Ks[j * LD + d], sc);
                sc *= scale;
            }
            P[j] = sc;
            mx = fmaxf(mx, sc);
        }
        for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        float ls = 0.0f;
        for (int j = lane; j < Wn; j += 64) {
            const float pj = j < nvis ? expf(P[j] - mx) : 0.0f;
            P[j] = pj;
            ls += pj;
        }
        for (int off = 32; off >= 1; off >>= 1) ls += __shfl_xor(ls, off, 64);
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        for (int d = lane; d < D; d += 64) {
            float o = 0.0f;
            for (int j = 0; j < nvis; ++j) o = fmaf(P[j], Vs[j * LD + d], o);
            put_row(out, (size_t)(b * T + i), HD, h * D + d, o / ls, terms);
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
}

// k_codec_rope_kv + k_codec_attn as ONE launch per layer, head dim as a compile-time constant: block (head, request) rotates its
// head's T new q / k rows (q stays in LDS), writes the new K / V rows of its head to the ring and keeps their bf16 values in the LDS
// tile next to the history rows (16-byte ring loads, one 64-bit modulo per row chunk instead of one per element); the T x Wn scores are
// spread over all 256 threads as (query, key) pairs — the old form gave a wave one query at a time and left 56 lanes idle in the second
// key pass — and the per-query softmax + P.V keep their wave-per-query form.  Every output's arithmetic (the fma chain over d of a
// score, the lane sums and butterfly of the softmax, the fma chain over the keys of P.V, the bf16 rounding of the ring rows) is the
// chain of the two kernels above: bit-identical (waveform digests equal).  Chunk of 1 / 8 / 32 requests: 1.95 -> 1.76, 3.53 -> 3.34, 7.70 -> 7.47 ms
// (profiles/round4_codec_attn_ab.txt).
// A launch of few requests is its chain of trips, so all that can be asked for early is: the new rows' first values in front of slot and
// position, the history four chunks a thread at once, its ring rows from one modulo; scores and weights are read 16 bytes at a time, the
// softmax's sums go by DPP.  10 frames, us a launch before / so: one
// request 8.4 / 7.5, 32 requests 13.2 / 10.8.
template <int D>
__global__ __launch_bounds__(1024) void k_codec_attn2(const float* qkv, bf16_t* ring, const int* slots, const long* pos, float* out, int T,
                                                     int H, int Wn, const float* inv_freq, int terms) {
    extern __shared__ __attribute__((aligned(16))) float sm[];   // K [Wn][D+4], V [Wn][D], Q [T][D], P [T][Wp]
    constexpr int LK = D + 4, half = D / 2, CH = D / 8, HB = 4;
    const int Wp = (Wn + 3) & ~3;
    float* Ks = sm;
    float* Vs = Ks + (size_t)Wn * LK;
    float* Qs = Vs + (size_t)Wn * D;
    float* Ps = Qs + (size_t)T * D;
    const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = blockDim.x;
    const int HD = H * D;
    const float* qr = qkv + (size_t)b * T * 3 * HD + (size_t)h * D;
    const auto rope_in = [&](int e, float (&v)[5]) {
        const int t = e / half, i = e % half;
        const float* q = qr + (size_t)t * 3 * HD + i;
        v[0] = ldg(q); v[1] = ldg(q + half); v[2] = ldg(q + HD); v[3] = ldg(q + HD + half); v[4] = ldg(inv_freq + i);
    };
    const auto value_in = [&](int e) { return ldg(qr + (size_t)(e / D) * 3 * HD + 2 * HD + e % D); };
    float rv[5];
    rope_in(tid < T * half ? tid : 0, rv);
    float vv = value_in(tid < T * D ? tid : 0);
    const int slot = slots[b];
    const long p0 = pos[slot];
    const int first = p0 + T < Wn ? (int)(Wn - T - p0) : 0;      // logical slots before it lie in front of the stream: zero rows
    const int r0 = (int)((p0 + T) % Wn);                       // ring row of logical slot 0 (absolute position p0 + T - Wn)
    const auto ring_row = [&](int j) { const int r = r0 + j; return (size_t)(r < Wn ? r : r - Wn) * 2 * HD; };
    bf16_t* rbase = ring + (size_t)slot * Wn * 2 * HD + (size_t)h * D;
    // history rows: logical slots 0 .. Wn - T - 1
    const int nh = (Wn - T) * CH;
    for (int c0 = tid; c0 < nh; c0 += HB * nt) {
        uint4 kq[HB], vq[HB];
#pragma unroll
        for (int u = 0; u < HB; ++u) {
            const int c = c0 + u * nt < nh ? c0 + u * nt : c0, j = c / CH;
            const uint4* r = reinterpret_cast<const uint4*>(rbase + ring_row(j) + (c % CH) * 8);
            kq[u] = ldg(r);
            vq[u] = ldg(r + HD / 8);
        }
#pragma unroll
        for (int u = 0; u < HB; ++u) {
            const int c = c0 + u * nt, j = c / CH, d0 = (c % CH) * 8;
            if (c >= nh) break;
            const bool in = j >= first;
            const unsigned kw[4] = {in ? kq[u].x : 0u, in ? kq[u].y : 0u, in ? kq[u].z : 0u, in ? kq[u].w : 0u};
            const unsigned vw[4] = {in ? vq[u].x : 0u, in ? vq[u].y : 0u, in ? vq[u].z : 0u, in ? vq[u].w : 0u};
            float4 *kd = reinterpret_cast<float4*>(Ks + j * LK + d0), *vd = reinterpret_cast<float4*>(Vs + j * D + d0);
            kd[0] = make_float4(bflo(kw[0]), bfhi(kw[0]), bflo(kw[1]), bfhi(kw[1]));
            kd[1] = make_float4(bflo(kw[2]), bfhi(kw[2]), bflo(kw[3]), bfhi(kw[3]));
            vd[0] = make_float4(bflo(vw[0]), bfhi(vw[0]), bflo(vw[1]), bfhi(vw[1]));
            vd[1] = make_float4(bflo(vw[2]), bfhi(vw[2]), bflo(vw[3]), bfhi(vw[3]));
        }
    }
    // the chunk's T new rows: RoPE (NeoX halves) on q and k, k / v rounded to bf16 for the ring — and for this launch's own tile
    for (int e = tid; e < T * half; e += nt) {
        if (e != tid) rope_in(e, rv);
        const int t = e / half, i = e % half, j = Wn - T + t;
        const float ang = (float)(p0 + t) * rv[4];
        const float c = cosf(ang), s = sinf(ang);
        Qs[t * D + i] = rv[0] * c - rv[1] * s;
        Qs[t * D + i + half] = rv[1] * c + rv[0] * s;
        const bf16_t k0 = f2bf(rv[2] * c - rv[3] * s), k1 = f2bf(rv[3] * c + rv[2] * s);
        bf16_t* rk = rbase + ring_row(j);
        rk[i] = k0;
        rk[i + half] = k1;
        Ks[j * LK + i] = bf2f(k0);
        Ks[j * LK + i + half] = bf2f(k1);
    }
    for (int e = tid; e < T * D; e += nt) {
        if (e != tid) vv = value_in(e);
        const int t = e / D, d = e % D, j = Wn - T + t;
        const bf16_t v16 = f2bf(vv);
        rbase[ring_row(j) + HD + d] = v16;
        Vs[j * D + d] = bf2f(v16);
    }
    __syncthreads();
    const float scale = rsqrtf((float)D);
    for (int pr = tid; pr < T * Wn; pr += nt) {
        const int i = pr / Wn, j = pr - i * Wn;
        const int nvis = Wn - T + i + 1;
        float sc = -INFINITY;
        if (j < nvis) {
            const float4* q = reinterpret_cast<const float4*>(Qs + (size_t)i * D);
            const float4* kr = reinterpret_cast<const float4*>(Ks + (size_t)j * LK);
            sc = 0.0f;
#pragma unroll
            for (int d = 0; d < D / 4; ++d) {
                const float4 a = q[d], k = kr[d];
                sc = fmaf(a.x, k.x, sc); sc = fmaf(a.y, k.y, sc); sc = fmaf(a.z, k.z, sc); sc = fmaf(a.w, k.w, sc);
            }
            sc *= scale;
        }
        Ps[i * Wp + j] = sc;
    }
    __syncthreads();
    for (int i = wave; i < T; i += nt >> 6) {
        float* P = Ps + (size_t)i * Wp;
        const int nvis = Wn - T + i + 1;
        float mx = -INFINITY;
        for (int j = lane; j < Wn; j += 64) mx = fmaxf(mx, P[j]);
        for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        float ls = 0.0f;
        for (int j = lane; j < Wn; j += 64) {
            const float pj = j < nvis ? expf(P[j] - mx) : 0.0f;
            P[j] = pj;
            ls += pj;
        }
        ls = butterfly<64>(ls);
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        for (int d = lane; d < D; d += 64) {
            float o = 0.0f;
            int j = 0;
#pragma unroll 3
            for (; j + 8 <= nvis; j += 8) {
                const float4 pa = *reinterpret_cast<const float4*>(P + j), pb = *reinterpret_cast<const float4*>(P + j + 4);
                const float pv[8] = {pa.x, pa.y, pa.z, pa.w, pb.x, pb.y, pb.z, pb.w};
                float x[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) x[u] = Vs[(j + u) * D + d];
#pragma unroll
                for (int u = 0; u < 8; ++u) o = fmaf(pv[u], x[u], o);
            }
            if (j < nvis) {      // (read together: what is past the last visible key is not added)
                float pv[8], x[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int k = j + u < nvis ? j + u : nvis - 1;
                    pv[u] = P[k];
                    x[u] = Vs[k * D + d];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) o = j + u < nvis ? fmaf(pv[u], x[u], o) : o;
            }
            put_row(out, (size_t)(b * T + i), HD, h * D + d, o / ls, terms);
        }
    }
}

__global__ __launch_bounds__(256) void k_pos_advance(long* pos, const int* slots, int n, int T) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b < n) pos[slots[b]] += T;
}

// h[m][i] = silu(gu[m][i]) * gu[m][I+i]
__global__ __launch_bounds__(256) void k_silu_mul_f32(const float* gu, float* h, size_t rows, int I) {
    const size_t total = rows * I;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t)gridDim.x * 256) {
        const size_t m = e / I;
        const int i = (int)(e % I);
        const float g = gu[m * 2 * I + i], u = gu[m * 2 * I + I + i];
        h[e] = (g / (1.0f + expf(-g))) * u;
    }
}

// ConvNeXt front: causal depthwise conv k=7 (+bias) then LayerNorm over channels.   qwen3_codec.py:447-450
__global__ __launch_bounds__(256) void k_dwconv_ln(const float* x, const float* state, const int* slots, const float* w,
                                                   const float* wb, const float* lnw, const float* lnb, float* y, int L,
                                                   int C, float eps, int terms) {
    __shared__ float red[4];
    extern __shared__ float ybuf[];   // [C]
    const int row = blockIdx.x, b = row / L, t = row % L;
    const float* st = state + (size_t)slots[b] * 6 * C;
    float s1 = 0.0f;
#pragma unroll 4
    for (int c = threadIdx.x; c < C; c += 256) {
        float acc = wb[c], v[7], wk[7];
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            const int e = t + k;   // index into ext = [state(6) ++ x]
            v[k] = ldg(e < 6 ? st + (size_t)e * C + c : x + ((size_t)b * L + (e - 6)) * C + c);
            wk[k] = ldg(w + c * 7 + k);
        }
#pragma unroll
        for (int k = 0; k < 7; ++k) acc += wk[k] * v[k];
        ybuf[c] = acc;
        s1 += acc;
    }
    const float mean = block_sum(s1, red) / (float)C;
    float sq = 0.0f;
    for (int c = threadIdx.x; c < C; c += 256) {
        const float d = ybuf[c] - mean;
        sq += d * d;
    }
    const float rstd = rsqrtf(block_sum(sq, red) / (float)C + eps);
    for (int c = threadIdx.x; c < C; c += 256) put_row(y, (size_t)row, C, c, (ybuf[c] - mean) * rstd * lnw[c] + lnb[c], terms);
}

// final causal conv k=7, C -> 1, + clamp(-1,1).  One wave per output sample group.
__global__ __launch_bounds__(256) void k_final_conv(const float* x, const float* state, const int* slots, const float* w,
                                                    float bias, float* out, int L, int C) {
    const int b = blockIdx.y;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= L) return;
    const float* st = state + (size_t)slots[b] * 6 * C;
    float acc = 0.0f;
    for (int e = lane; e < 7 * C; e += 64) {
        const int k = e / C, c = e % C;
        const int r = t + k;
        const float v = r < 6 ? st[(size_t)r * C + c] : x[((size_t)b * L + (r - 6)) * C + c];
        acc += w[c * 7 + k] * v;
    }
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) out[(size_t)b * L + t] = fminf(1.0f, fmaxf(-1.0f, acc + bias));
}

// The last conv of a decoder (K taps, C = 32 V channels -> 1), every row read once: out[t] = bias + sum_k (w_k . x[t - (K-1) + k]).  Eight lanes
// hold a row in V 16-byte pieces each and make its K products together (the weights stay in their registers); the K sums of a row go to
// LDS, an output adds K of them.  32 IT rows per block, the first K - 1 of them only for their products.  Rows before the chunk come from
// the history (NULL: zero).  Memory bound: 614 400 rows of 96 channels 155 -> 72 us, 307 200 of 64 (K = 3) 88 -> 24 (one output per lane
// out of LDS rows, and one wave per output, before).
template <int K, int V, int IT, bool CLAMP>
__global__ __launch_bounds__(256) void k_final_taps(const float* x, const float* state, const int* slots, const float* w, float bias, float* out, int L) {
    constexpr int C = 32 * V, ROWS = 32 * IT, OUT = ROWS - (K - 1);
    __shared__ __attribute__((aligned(16))) float ws[K * C];
    __shared__ float part[ROWS * K];
    const int b = blockIdx.y, t0 = blockIdx.x * OUT, tid = threadIdx.x, l8 = tid & 7, rg = tid >> 3;
    const float* xb = x + (size_t)b * L * C;
    const float* sb = state ? state + (size_t)slots[b] * (K - 1) * C : nullptr;
    for (int e = tid; e < K * C; e += 256) ws[e % K * C + e / K] = w[e];
    float4 v[IT < 4 ? IT : 4][V];
    const auto fetch = [&](int it0) {
#pragma unroll
        for (int i = 0; i < (IT < 4 ? IT : 4); ++i) {
            const int r = t0 - (K - 1) + (it0 + i) * 32 + rg;
            const float* p = r >= 0 ? (r < L ? xb + (size_t)r * C : nullptr) : (sb ? sb + (size_t)(K - 1 + r) * C : nullptr);
#pragma unroll
            for (int q = 0; q < V; ++q) v[i][q] = p ? *reinterpret_cast<const float4*>(p + (q * 8 + l8) * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    fetch(0);
    __syncthreads();
    float4 wr[K][V];
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
        for (int q = 0; q < V; ++q) wr[k][q] = *reinterpret_cast<const float4*>(ws + k * C + (q * 8 + l8) * 4);
#pragma unroll
    for (int it0 = 0; it0 < IT; it0 += 4) {
        if (it0) fetch(it0);
#pragma unroll
        for (int i = 0; i < (IT < 4 ? IT : 4); ++i) {
            float s[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                s[k] = 0.0f;
                if (k < K) {
#pragma unroll
                    for (int q = 0; q < V; ++q) {
                        s[k] = __fmaf_rn(wr[k][q].x, v[i][q].x, s[k]); s[k] = __fmaf_rn(wr[k][q].y, v[i][q].y, s[k]);
                        s[k] = __fmaf_rn(wr[k][q].z, v[i][q].z, s[k]); s[k] = __fmaf_rn(wr[k][q].w, v[i][q].w, s[k]);
                    }
                }
            }
            // the eight lanes' sums: halves are exchanged, so that lane k ends with tap k
#pragma unroll
            for (int o = 4; o >= 1; o >>= 1)
#pragma unroll
                for (int k = 0; k < o; ++k) {
                    const bool up = l8 & o;
                    const float keep = up ? s[k + o] : s[k], give = up ? s[k] : s[k + o];
                    s[k] = keep + __shfl_xor(give, o, 64);
                }
            if (l8 < K) part[((it0 + i) * 32 + rg) * K + l8] = s[0];
        }
    }
    __syncthreads();
    const int t = t0 + tid;
    if (tid >= OUT || t >= L) return;
    float o = 0.0f;
#pragma unroll
    for (int k = 0; k < K; ++k) o += part[(tid + k) * K + k];
    o += bias;
    out[(size_t)b * L + t] = CLAMP ? fminf(1.0f, fmaxf(-1.0f, o)) : o;
}
// few outputs: 64-row blocks, so that one request still fills the chip
template <int K, bool CLAMP>
static bool final_taps(hipStream_t st, const float* x, const float* state, const int* slots, const float* w, float bias, float* out, int n, int L, int C) {
    const bool few = (long)n * ((L + 255) / 256) < 512;
#define VOX_FT(V_) \
    case V_: \
        if (few) hipLaunchKernelGGL((k_final_taps<K, V_, 2, CLAMP>), dim3((L + 64 - K) / (65 - K), n), dim3(256), 0, st, x, state, slots, w, bias, out, L); \
        else hipLaunchKernelGGL((k_final_taps<K, V_, 8, CLAMP>), dim3((L + 256 - K) / (257 - K), n), dim3(256), 0, st, x, state, slots, w, bias, out, L); \
        return true;
    if (C % 32 == 0) switch (C / 32) { VOX_FT(1) VOX_FT(2) VOX_FT(3) VOX_FT(4) }
#undef VOX_FT
    return false;
}

// ================================================================================================
// engine
// ================================================================================================
#include <vector>

struct vox_codec {
    vox_ctx* ctx;
    vox_codec_config cfg;
    vox_codec_weights w;
    int max_batch, max_slots, T;
    int planes = 2;     // operand planes of the conv GEMMs (vox_codec_set_operand_planes)
    bool decoded = false;   // a chunk has run: the slots' streaming history is stored in the format `planes` implies
    // state (per slot)
    // (one or two operand planes: all but st_dw and st_final hold the two bf16 terms that the conv which reads them would make of a row, 4 bytes a value)
    float *st_pre, *st_dw[2], *st_dec0, *st_tc[4], *st_ru[4][3], *st_final;
    bf16_t* ring;   // [layers][slots][Wn][2][HD]
    long* pos;      // [slots]
    // work buffers
    float* buf[4];
    size_t buf_floats;
    float *q0, *qr;
};

// operand planes of the conv GEMMs launched by the current decode call (set by the entry points from their object's setting)
static thread_local int g_conv_planes = 3;
// rows up to which the few-row GEMM variant (16-row tiles, wide K steps) is used: the flow's GEMMs have 56..450 rows and K <= 2048, their
// time is the number of dependent K steps, not MFMA issue
static thread_local int g_conv_skinny_rows = 48;
// k_rows_gemm for eligible shapes: the flows only (their row bound is unbounded, so one kernel serves a shape at every batch size; the
// codecs' and HiFT's few-row stages become many-row stages as the batch grows and must keep one summation order)
static thread_local bool g_conv_rows_gemm = false;
// few-row GEMMs walk K in 256-wide steps where Cin allows (half the dependent steps of the 128-wide walk; same accumulation order, so
// the results are bit-identical).  VOX_SKINNY_BK256=0 keeps the 128-wide walk (A/B timing).
static bool skinny_wide() {
    static const bool on = [] { const char* e = getenv("VOX_SKINNY_BK256"); return !(e && e[0] == '0'); }();
    return on;
}
// VOX_ROWS_GEMM=0: the LDS-staged few-row kernel instead of k_rows_gemm (A/B timing)
static bool rows_gemm_on() {
    static const bool on = [] { const char* e = getenv("VOX_ROWS_GEMM"); return !(e && e[0] == '0'); }();
    return on;
}
// VOX_ROWS_WV8=0: four waves per k_rows_gemm block at every K (A/B timing; changes the summation order of the K >= 512 linears)
static bool rows_wv8_on() {
    static const bool on = [] { const char* e = getenv("VOX_ROWS_WV8"); return !(e && e[0] == '0'); }();
    return on;
}
// blocks from which k_rows_gemm takes two 16-row tiles per block (VOX_ROWS_MT2=<blocks>; 0 = never)
static int rows_mt2_blocks() {
    static const int v = [] { const char* e = getenv("VOX_ROWS_MT2"); const int x = e ? atoi(e) : 1024; return x > 0 ? x : (1 << 30); }();
    return v;
}
// 16 x 16 output tiles above which a k_rows_gemm block takes 2 / 4 column tiles where a call has 256 rows and more (VOX_ROWS_NT2; VOX_ROWS_NT4: at every row
// count; 0: by the rule in conv_gemm)
static int rows_nt_tiles(int which) {
    static const int v2 = [] { const char* e = getenv("VOX_ROWS_NT2"); return e ? atoi(e) : 256; }();
    static const int v4 = [] { const char* e = getenv("VOX_ROWS_NT4"); return e ? atoi(e) : 0; }();
    return which ? v4 : v2;
}
// x / d = umulhi(x, inverse) for 0 <= x < n: with inverse = (2^32 + r) / d, 0 <= r < d, exact while x r < 2^32.  0 where that does not hold (and for d = 1)
static unsigned div_inverse(int d, int n) {
    return d > 1 && (uint64_t)d * (uint64_t)n < 1ull << 32 ? (unsigned)(((1ull << 32) + (unsigned)d - 1) / (unsigned)d) : 0u;
}
static int conv_gemm(hipStream_t st, const vox_conv_w& w, const float* x, const float* state, const int* slots, int n,
                     int L, int P, const int* offs, float* out, const float* res, const float* scale, int gelu,
                     float* out2 = nullptr, const vox_snake_w* sn = nullptr, int sn_mod = 0, const float* rscale = nullptr,
                     const float* ln_w = nullptr, const float* ln_b = nullptr, float ln_eps = 0.0f) {
    if (w.cin % CG_BK) return vox_fail(VOX_ERR_INVALID, "codec gemm: Cin %d %% %d != 0", w.cin, CG_BK);
    if (w.n_taps > CG_MAXTAPS) return vox_fail(VOX_ERR_INVALID, "codec gemm: too many taps");
    ConvGemmArgs a{};
    a.x = x; a.state = state; a.slots = slots; a.w = (const bf16_t*)w.w; a.bias = w.bias; a.res = res; a.scale = scale;
    a.out = out; a.M = n * L; a.N = w.n; a.Cin = w.cin; a.L = L; a.P = P; a.n_taps = w.n_taps; a.rscale = rscale;
    a.planes = g_conv_planes;
#ifdef VOX_DEV_KNOBS
    { static const int dv = [] { const char* e = getenv("VOX_CODEC_DEV"); return e ? atoi(e) : 0; }(); a.dev = dv; }
#endif
    a.bias_mod = w.bias_mod > 0 ? w.bias_mod : w.n; a.gelu = gelu;
    if (out2 && sn) { a.out2 = out2; a.sn_alpha = sn->alpha; a.sn_invb = sn->inv_beta; a.sn_mod = sn_mod > 0 ? sn_mod : w.n; }
    for (int k = 0; k < w.n_taps; ++k) a.off[k] = offs ? offs[k] : 0;
    if (g_conv_rows_gemm && a.planes == 3 && rows_gemm_on() && out && !out2 && a.M <= g_conv_skinny_rows && w.cin % 32 == 0 && (long)w.n * w.cin < 1l << 31 && (w.n_taps * w.cin) % 128 == 0 && (!ln_w || (w.n_taps == 1 && a.off[0] == 0))) {
        // every operand requested up front, K split over the block's waves (k_rows_gemm): 8 waves from K = 512 on
        const int K = w.n_taps * w.cin, wv = (K >= 512 && K % 256 == 0 && rows_wv8_on()) ? 8 : 4, kb = K / (32 * wv);
        const int tiles = ((w.n + 15) / 16) * ((a.M + 15) / 16);
        // column tiles per block: one while the call is a handful of row tiles (latency: more blocks in flight), two from 256 tiles on
        // once there are >= 16 row tiles (every block re-loads and re-splits its A rows: at 448+ rows that traffic and VALU work
        // outweigh the extra blocks — CosyVoice2 chunk 49.7 -> 46.6 ms at B=8, 36.6 -> 35.2 at B=4, unchanged at B=1), four above 512
        // (above 2048, and this: 8 requests of 28 tokens, 896 rows, 28.61 and 28.16 ms; 4 of 20 22.60, 22.54; 1 of 28 20.58 both; nowhere
        // slower at 40 shapes of CosyVoice2's flow and 24 of GLM-4-Voice's), but above 2048 below those 16 row tiles and from 1025 rows on (GLM-4-Voice's flow with 512 there too, 1032 rows 53.7 and 54.2 ms, 1376 rows 57.3, 57.8)
        const int four = rows_nt_tiles(1) ? rows_nt_tiles(1) : a.M >= 256 && a.M <= 1024 ? 512 : 2048;
        int nt = tiles > four ? 4 : tiles > (a.M >= 256 ? rows_nt_tiles(0) : 1024) ? 2 : 1;
        while (nt > 1 && nt * kb > 16) nt >>= 1;
        const int mt = (tiles / nt >= rows_mt2_blocks() && kb <= 4 && (wv == 4 || nt <= 2)) ? 2 : 1;      // (the 8-wave sum buffer: MT NT <= 4)
        if (ln_w) { a.ln_w = ln_w; a.ln_b = ln_b; a.ln_eps = ln_eps; }
        a.kpt_inv = div_inverse(w.cin / 32, K / 32);
        a.len_inv = div_inverse(L, a.M);
        const dim3 g((w.n + 16 * nt - 1) / (16 * nt), (a.M + 16 * mt - 1) / (16 * mt));
#define VOX_ROWS1(KB_, NT_, MT_, WV_)                                                                              \
        if (kb == KB_ && nt == NT_ && mt == MT_ && wv == WV_) {                                                        \
            if (ln_w) hipLaunchKernelGGL((k_rows_gemm<KB_, NT_, true, MT_, WV_>), g, dim3(64 * WV_), 0, st, a);        \
            else hipLaunchKernelGGL((k_rows_gemm<KB_, NT_, false, MT_, WV_>), g, dim3(64 * WV_), 0, st, a);            \
            return VOX_OK;                                                                                             \
        }
#define VOX_ROWS(KB_, WV_) VOX_ROWS1(KB_, 1, 1, WV_) VOX_ROWS1(KB_, 2, 1, WV_) VOX_ROWS1(KB_, 4, 1, WV_) VOX_ROWS1(KB_, 1, 2, WV_) \
                           VOX_ROWS1(KB_, 2, 2, WV_)
        VOX_ROWS(2, 4) VOX_ROWS(4, 4) VOX_ROWS(2, 8) VOX_ROWS(3, 8) VOX_ROWS(4, 8) VOX_ROWS1(2, 4, 2, 4) VOX_ROWS1(4, 4, 2, 4)
        VOX_ROWS1(6, 1, 1, 4) VOX_ROWS1(6, 2, 1, 4) VOX_ROWS1(8, 1, 1, 4) VOX_ROWS1(8, 2, 1, 4) VOX_ROWS1(12, 1, 1, 4) VOX_ROWS1(16, 1, 1, 4)
        VOX_ROWS1(6, 1, 1, 8) VOX_ROWS1(6, 2, 1, 8) VOX_ROWS1(8, 1, 1, 8) VOX_ROWS1(8, 2, 1, 8)
#undef VOX_ROWS
#undef VOX_ROWS1
        a.ln_w = a.ln_b = nullptr;      // no variant for this K: the staged kernels below
    }
    if (ln_w) {      // fused input LayerNorm: few-row kernel, one plain tap, the row statistics need the whole row in one K walk
        if (a.M > g_conv_skinny_rows || w.n_taps != 1 || a.off[0] != 0)
            return vox_fail(VOX_ERR_INVALID, "codec gemm: fused LayerNorm needs the few-row one-tap path");
        a.ln_w = ln_w; a.ln_b = ln_b; a.ln_eps = ln_eps;
        const dim3 g((w.n + 63) / 64, (a.M + 15) / 16);
        if (w.cin % 256 == 0 && skinny_wide()) hipLaunchKernelGGL((k_conv_gemm_skinny<256, true>), g, dim3(256), 0, st, a);
        else if (w.cin % 128 == 0) hipLaunchKernelGGL((k_conv_gemm_skinny<128, true>), g, dim3(256), 0, st, a);
        else if (w.cin % 64 == 0) hipLaunchKernelGGL((k_conv_gemm_skinny<64, true>), g, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((k_conv_gemm_skinny<32, true>), g, dim3(256), 0, st, a);
        return VOX_OK;
    }
    if (a.M <= g_conv_skinny_rows) {
        const dim3 g((w.n + 63) / 64, (a.M + 15) / 16);
        if (w.cin % 256 == 0 && skinny_wide()) hipLaunchKernelGGL(k_conv_gemm_skinny<256>, g, dim3(256), 0, st, a);
        else if (w.cin % 128 == 0) hipLaunchKernelGGL(k_conv_gemm_skinny<128>, g, dim3(256), 0, st, a);
        else if (w.cin % 64 == 0) hipLaunchKernelGGL(k_conv_gemm_skinny<64>, g, dim3(256), 0, st, a);
        else hipLaunchKernelGGL(k_conv_gemm_skinny<32>, g, dim3(256), 0, st, a);
        return VOX_OK;
    }
    // many-row stages (batched chunks, the late upsampling stages): 128-row tiles, 64 x (48|64) per wave — each LDS
    // fragment read then feeds 3-4 MFMAs instead of 2 (the 64 x 64 tile is LDS-read bound with the 3-term split)
    {
        const int wnb = (w.n % 128 == 0 || w.n >= 256) ? 4 : ((w.n > 64 && w.n <= 96) || w.n % 96 == 0) ? 3 : 0;
        if (wnb && ((w.n + 32 * wnb - 1) / (32 * wnb)) * ((a.M + 127) / 128) >= 256) {
            const dim3 gb((w.n + 32 * wnb - 1) / (32 * wnb), (a.M + 127) / 128);
            if (wnb == 4) hipLaunchKernelGGL((k_conv_gemm<32, 4, 4>), gb, dim3(256), 0, st, a);
            else hipLaunchKernelGGL((k_conv_gemm<32, 4, 3>), gb, dim3(256), 0, st, a);
            return VOX_OK;
        }
    }
    // tile: 64 x 64 unless that leaves most CUs idle (these GEMMs are MFMA-bound per CU)
    const int b64 = ((w.n + 63) / 64) * ((a.M + 63) / 64);
    const int wm = b64 >= 192 ? 2 : 1, wn = (b64 >= 192 || 2 * b64 >= 192) ? 2 : 1;
    const dim3 grid((w.n + 32 * wn - 1) / (32 * wn), (a.M + 32 * wm - 1) / (32 * wm));
    const bool few = grid.x * grid.y <= 512;       // at most two blocks per CU: nothing else hides a block's LDS round trips
#define VOX_CG(K_, M_, N_) if (wm == M_ && wn == N_) { \
        if (few && M_ * N_ <= 2) hipLaunchKernelGGL((k_conv_gemm<K_, M_, N_, (M_ * N_ <= 2)>), grid, dim3(256), 0, st, a); \
        else hipLaunchKernelGGL((k_conv_gemm<K_, M_, N_>), grid, dim3(256), 0, st, a); \
        return VOX_OK; }
    // few blocks, long K (HiFT's resblock convs of one request: 112 blocks x 88 K steps of 64): 128-wide K steps halve the dependent
    // stage-and-barrier rounds; the k order is unchanged, so the results are bit-identical (VOX_CG_BK128=0: 64-wide steps)
    static const bool bk128 = [] { const char* e = getenv("VOX_CG_BK128"); return !(e && e[0] == '0'); }();
    if (w.cin % 128 == 0 && bk128) { VOX_CG(128, 1, 1) }
    if (w.cin % 64 == 0) { VOX_CG(64, 2, 2) VOX_CG(64, 1, 2) VOX_CG(64, 1, 1) }
    VOX_CG(32, 2, 2) VOX_CG(32, 1, 2) VOX_CG(32, 1, 1)
#undef VOX_CG
    return vox_fail(VOX_ERR_INVALID, "codec gemm: no tile variant");
}

// a wave per query of a (head, request): the rounds of a wave are a serial chain of a few thousand clocks each
static int attn_threads(int L) { return 64 * (L < 4 ? 4 : L > 16 ? 16 : L); }
static void state_update(hipStream_t st, float* state, const int* slots, const float* x, int n, int L, int P, int C) {
    hipLaunchKernelGGL(k_state_update, dim3((C + 255) / 256, n), dim3(256), 0, st, state, slots, x, L, P, C);
}

// ---- convolutions over S2 rows (k_conv_dma) ----
template <int BM, int BN, int WM, int WN, int WK, int BK, int S, int NP, int EPI, int WP = 1>
static int conv_dma_launch(hipStream_t st, ConvDmaArgs& a) {
    constexpr int lds = S * (NP * BM + WP * BN) * BK * 2, threads = 64 * WM * WN * WK;
    static_assert(lds + BM * 4 <= 160 * 1024, "LDS of a CU");
    const auto kern = k_conv_dma<BM, BN, WM, WN, WK, BK, S, NP, EPI, WP>;
    if (lds > 64 * 1024) VOX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    a.tm = (a.M + BM - 1) / BM;
    a.tn = ((EPI == CONV_GLU ? 2 * a.N : a.N) + BN - 1) / BN;
    a.tiles8 = (a.tm * a.tn + 7) & ~7;
    a.mfast = (size_t)a.n_taps * a.N > (size_t)a.M * 2;      // weights larger than rows: each XCD reads its own columns of them
    a.tdiv = a.mfast ? a.tm : a.tn;
    a.tdiv_inv = div_inverse(a.tdiv, a.tiles8);
    hipLaunchKernelGGL(kern, dim3(a.tiles8 + conv_job_blocks(a.job, threads)), dim3(threads), lds, st, a);
    return VOX_OK;
}
// The smallest tile that leaves no CU a second round: a call of few rows is a chain of dependent steps, and more blocks, fewer columns and
// deeper steps each shorten it.  Past one 64 x 64 tile per CU the waves all load and multiply; past two the tile grows (fewer bytes through
// LDS per product).  us, against the staged kernels, two-term rows (M rows, N x taps x Cin):
//   M = 10: 3072 x 512 7.1 -> 5.4, 512 x 1024 10.4 -> 5.7 | 20: 4096 x 1024 5.7, 1024 x 4096 9.6 | 40: 1536 x 7 x 1024 58 -> 14.5, 6144 x 2 x 1536 31 -> 13.1
//   M = 320: 768 x 7 x 768 48 -> 15.2, 1920 x 2 x 768 22 -> 11.3 | 1600: 384 x 7 x 384 36 -> 16.4 | 6400: 192 x 7 x 192 30 -> 19
//   M = 1280: 1536 x 7 x 1024 157 -> 72, 6144 x 2 x 1536 157 -> 84 | 10240: 768 x 7 x 768 194 -> 134, 1920 x 2 x 768 168 -> 131
//   three-term rows: M = 320: 1024 x 7 x 512 18.8, 4096 x 2 x 1024 45 -> 28 | 2560: 256 x 3 x 512 14.4 | 76 800: 256 x 2 x 128 67 (128 x 128)
//   M = 51200: 384 x 7 x 384 250 -> 193 (rounds of 256 tiles decide: 128 x 256 leaves a quarter of its columns empty there, > 245)
// Two multiplying waves and eight that load beat one of either kind in 16 x 32 tiles (10 rows, 3072 x 512: 5.4; four loaders 5.9; 16 x 16 with
// one and four: 5.8).
// Three-term rows carry the fp32 values, so the order of a long sum is what is left of the error: from 768 products on an output adds parts of
// 256 channels (a property of the layer, as the order has to be).  Mimi against 64 bits, 16 requests of 10 frames: 1.26e-6 in one run, 6.6e-7 so.
// Their many-row tile is 64 x 128; 128 x 128 has no registers for the parts (15 360 rows, 640 x 2 x 256: 46 us, with parts 57).
static bool conv_long_sums(int taps, int cin) { return cin % 64 == 0 && taps * cin >= 768; }
template <int NP, int EPI>
static int conv_dma_pick(hipStream_t st, ConvDmaArgs& a) {
    const int n2 = EPI == CONV_GLU ? 2 * a.N : a.N;
    const auto tiles = [&](int bm, int bn) { return (long)((a.M + bm - 1) / bm) * ((n2 + bn - 1) / bn); };
    const bool k64 = a.Cin % 64 == 0, k128 = a.Cin % 128 == 0;      // (other Cin: 32-channel steps)
    a.parts = NP == 3 && conv_long_sums(a.n_taps, a.Cin);
    if (k128) {
        if constexpr (EPI == CONV_GLU) {      // (gate and up columns in one wave; 10 rows, 2048 x 512: 16 x 32 5.9, 16 x 64 6.4)
            if (a.Cin % 256 == 0 && tiles(16, 32) <= 256) return conv_dma_launch<16, 32, 1, 1, 9, 256, 4, NP, EPI>(st, a);
            if (tiles(16, 64) <= 256) return conv_dma_launch<16, 64, 1, 2, 5, 128, 5, NP, EPI>(st, a);
        } else {
            if (tiles(16, 32) <= 256) {
                if (a.Cin % 256 == 0) return conv_dma_launch<16, 32, 1, 2, 5, 256, 3, NP, EPI>(st, a);
                return conv_dma_launch<16, 32, 1, 2, 5, 128, 6, NP, EPI>(st, a);
            }
            if (tiles(16, 64) <= 256) return conv_dma_launch<16, 64, 1, 4, 2, 128, 3, NP, EPI>(st, a);
        }
        if (tiles(32, 64) <= 256) return conv_dma_launch<32, 64, 2, 2, 3, 128, 3, NP, EPI>(st, a);
    }
    if (k64) {
        if (tiles(32, 64) <= 256) {
            if constexpr (EPI == CONV_GLU) return conv_dma_launch<32, 64, 2, 2, 2, 64, 6, NP, EPI>(st, a);
            else return conv_dma_launch<32, 64, 2, 4, 1, 64, 6, NP, EPI>(st, a);
        }
        if (tiles(64, 64) <= 256) return conv_dma_launch<64, 64, 4, 2, 2, 64, 4, NP, EPI>(st, a);
        if constexpr (NP == 3) {
            if (tiles(64, 128) <= 256 || a.parts) return conv_dma_launch<64, 128, 2, 4, 2, 64, 2, NP, EPI>(st, a);
        } else if (tiles(64, 64) <= 512) {
            return conv_dma_launch<64, 64, 2, 2, 1, 64, 3, NP, EPI>(st, a);
        }
    }
    // what the busiest CU multiplies, weighted by how well each tile does it
    const auto cost = [&](int bm, int bn, double w) { return (double)((tiles(bm, bn) + 255) / 256) * bm * bn * w; };
    const auto least = [](const double* c, int n) {
        int best = 0;
        for (int i = 1; i < n; ++i) best = c[i] < c[best] ? i : best;
        return best;
    };
    if constexpr (NP == 3 && EPI == 0) {
        const double c[6] = {cost(128, 192, 1.0), cost(128, 128, 1.1), cost(64, 128, 1.25), cost(64, 96, 1.35), cost(64, 64, 1.45), cost(128, 32, 1.7)};
        switch (least(c, 6)) {
            case 0: return conv_dma_launch<128, 192, 4, 2, 1, 32, 2, NP, EPI>(st, a);
            case 1: return conv_dma_launch<128, 128, 4, 2, 1, 32, 2, NP, EPI>(st, a);
            case 2: return conv_dma_launch<64, 128, 4, 2, 1, 32, 3, NP, EPI>(st, a);
            case 3: return conv_dma_launch<64, 96, 4, 1, 1, 32, 4, NP, EPI>(st, a);
            case 4: return conv_dma_launch<64, 64, 2, 2, 1, 32, 4, NP, EPI>(st, a);
            default: return conv_dma_launch<128, 32, 8, 1, 1, 32, 3, NP, EPI>(st, a);
        }
    } else if constexpr (EPI == 0) {
        // (128 x 128: two blocks a CU in step, so past 512 tiles it is pairs of rounds that count: 51 200 x 384 206 us for 193 of 256 x 192)
        const double two = tiles(128, 128) > 512 && (tiles(128, 128) + 255) / 256 % 2 ? 16384 * 1.07 : 0.0;
        const double c[7] = {cost(128, 256, 1.0), cost(256, 192, 1.0),  cost(128, 192, 1.08), cost(128, 128, 1.07) + two,
                             cost(64, 128, 1.25), cost(64, 96, 1.4), cost(128, 96, 1.3)};
        switch (least(c, 7)) {
            case 0: return conv_dma_launch<128, 256, 4, 4, 1, 32, 3, NP, EPI>(st, a);
            case 1: return conv_dma_launch<256, 192, 8, 2, 1, 32, 3, NP, EPI>(st, a);
            case 2: return conv_dma_launch<128, 192, 4, 2, 1, 32, 2, NP, EPI>(st, a);
            case 3: return conv_dma_launch<128, 128, 4, 2, 1, 32, 3, NP, EPI>(st, a);
            case 4:
                if (k64) return conv_dma_launch<64, 128, 2, 2, 1, 64, 2, NP, EPI>(st, a);
                return conv_dma_launch<64, 128, 2, 2, 1, 32, 4, NP, EPI>(st, a);
            case 5: return conv_dma_launch<64, 96, 4, 1, 1, 32, 4, NP, EPI>(st, a);
            default: return conv_dma_launch<128, 96, 4, 1, 1, 32, 2, NP, EPI>(st, a);
        }
    } else if constexpr (NP == 3) {
        return conv_dma_launch<64, 128, 4, 2, 1, 32, 3, NP, EPI>(st, a);
    } else {
        if (k64) return conv_dma_launch<64, 128, 2, 2, 1, 64, 2, NP, EPI>(st, a);
        return conv_dma_launch<64, 64, 2, 2, 1, 32, 6, NP, EPI>(st, a);
    }
}
// The operands and the shape of a conv over S2 rows; the caller adds the epilogue (out / out2 / ...) and hands it to conv_s2.
static ConvDmaArgs conv_s2_args(const vox_conv_w& w, const float* x, const float* state, const int* slots, int n, int L, int P, const int* offs) {
    ConvDmaArgs a{};
    a.x = x; a.state = state; a.slots = slots; a.w = (const bf16_t*)w.w; a.bias = w.bias;
    a.M = n * L; a.N = w.n; a.Cin = w.cin; a.L = L; a.P = P; a.n_taps = w.n_taps;
    a.bias_mod = w.bias_mod > 0 ? w.bias_mod : w.n;
    a.sn_mod = w.n;
    for (int k = 0; k < w.n_taps && k < CG_MAXTAPS; ++k) a.off[k] = offs ? offs[k] : 0;
    return a;
}
// The first conv of a 192-channel unit of few rows (conv_unit).  us beside the tap-major walk: 640 rows 10.5 / 9.7, 1 280 10.7 / 9.9, 2 560 12.2 / 10.1,
// 5 120 15.8 / 11.8, 6 400 18.8 / 18.9 — a step's two slices are of two taps, so every lane has its addresses worked out anew each step.
static int conv_dma_chunks(hipStream_t st, ConvDmaArgs& a) {
    const auto tiles = [&](int bm, int bn) { return (long)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn); };
    if (tiles(16, 64) <= 256) return conv_dma_launch<16, 64, 1, 4, 2, 64, 6, 2, CONV_CHUNKS>(st, a);
    if (tiles(32, 64) <= 256) return conv_dma_launch<32, 64, 2, 4, 2, 64, 6, 2, CONV_CHUNKS>(st, a);
    if (tiles(64, 64) <= 256) return conv_dma_launch<64, 64, 4, 2, 2, 64, 4, 2, CONV_CHUNKS>(st, a);
    return conv_dma_launch<64, 96, 4, 2, 2, 64, 3, 2, CONV_CHUNKS>(st, a);
}
static int conv_s2(hipStream_t st, ConvDmaArgs& a, int epi = 0) {
    if (a.Cin % CG_BK) return vox_fail(VOX_ERR_INVALID, "codec conv: Cin %d %% %d != 0", a.Cin, CG_BK);
    if (a.n_taps > CG_MAXTAPS) return vox_fail(VOX_ERR_INVALID, "codec conv: too many taps");
    if (a.N % 16 || a.sn_mod % 8 || a.bias_mod % 8) return vox_fail(VOX_ERR_INVALID, "codec conv: %d channels (groups of %d)", a.N, a.sn_mod);
    a.planes = g_conv_planes;
    a.len_inv = div_inverse(a.L, a.M);
    if (epi == CONV_GLU) {
        a.N /= 2;
        a.sn_mod = a.N;
        return a.planes == 2 ? conv_dma_pick<2, CONV_GLU>(st, a) : conv_dma_pick<1, CONV_GLU>(st, a);
    }
    if (epi == CONV_CHUNKS) return conv_dma_chunks(st, a);
    if (epi == CONV_SINE) return a.planes == 2 ? conv_dma_pick<2, CONV_SINE>(st, a) : conv_dma_pick<1, CONV_SINE>(st, a);
    if (epi == CONV_GELU)
        return a.planes == 3 ? conv_dma_pick<3, CONV_GELU>(st, a) : a.planes == 2 ? conv_dma_pick<2, CONV_GELU>(st, a) : conv_dma_pick<1, CONV_GELU>(st, a);
    return a.planes == 3 ? conv_dma_pick<3, 0>(st, a) : a.planes == 2 ? conv_dma_pick<2, 0>(st, a) : conv_dma_pick<1, 0>(st, a);
}

// A residual unit as ONE launch (k_conv_unit) where its tile can cover all channels and the rows fill the chip (*fused = 1); otherwise nothing
// is launched and the caller runs the two convs, the first in k_conv_unit's order when *fused = CONV_CHUNKS.  a1: conv1 with act2 (sn_*), a2: conv2 with res, out and the NEXT consumer's
// activation, whose rows must not be a1's: a neighbouring tile still reads its look-back there.  (a1.job is done by extra blocks.)
template <int C, int CH, int TAPS, int T, int HP, int NW, int MT, int S>
static int conv_unit_launch(hipStream_t st, ConvDmaArgs& a1, ConvDmaArgs& a2, int H) {
    constexpr int BM = 16 * MT * NW, lds = 2 * T * (BM + HP) * 64 + S * (C > CH ? C : CH) * 64;
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    const auto kern = k_conv_unit<C, CH, TAPS, T, HP, NW, MT, S>;
    if (lds > 64 * 1024) VOX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    a1.tm = a1.M / BM;
    a1.tiles8 = (a1.tm + 7) & ~7;
    hipLaunchKernelGGL(kern, dim3(a1.tiles8 + conv_job_blocks(a1.job, 64 * NW)), dim3(64 * NW), lds, st, a1, a2, H);
    return VOX_OK;
}
static int conv_unit(hipStream_t st, ConvDmaArgs& a1, ConvDmaArgs& a2, int* fused) {
    *fused = 0;
    const int C = a1.N;
    if (g_conv_planes != 2 || a1.n_taps != 7 || a2.n_taps != 1 || a1.Cin != C || a2.Cin != C || a2.N != C || (C != 96 && C != 192) ||
        a2.out2 == a1.x || a1.bias_mod != C || a2.bias_mod != C || !a1.sn_alpha)
        return VOX_OK;
    int H = 0, omin = 0;
    for (int k = 0; k < a1.n_taps; ++k) { H = a1.off[k] > H ? a1.off[k] : H; omin = a1.off[k] < omin ? a1.off[k] : omin; }
    for (int k = 2; k < a1.n_taps; ++k)
        if (a1.off[k - 1] - a1.off[k] != a1.off[0] - a1.off[1]) return VOX_OK;
    // 96 channels: always (within a chunk: one request, 19 200 rows 27 -> 20 us, 614 400 rows 600 -> 335).  192 channels: from 8192 rows on (12 800
    // rows two launches 48 us, one 32; 204 800: 412 and 327 timed alone, 424 and 382 within a chunk); below, two launches that add in the same
    // order (6 400 rows 27 and 30, 1 280: 16 and 29)
    if (omin < 0 || H > 64 || a1.L % 64 || !a2.res) return VOX_OK;
    if (C == 192 && a1.M <= 8192) {
        *fused = CONV_CHUNKS;
        return VOX_OK;
    }
    *fused = 1;
    if (C == 192) return conv_unit_launch<192, 192, 7, 2, 64, 4, 1, 3>(st, a1, a2, H);
    if (a1.L % 128 == 0 && a1.M / 128 >= 256) return conv_unit_launch<96, 96, 7, 2, 64, 8, 1, 3>(st, a1, a2, H);
    return conv_unit_launch<96, 96, 7, 2, 64, 4, 1, 3>(st, a1, a2, H);
}

// The same for Mimi's units (3 taps C -> C / 2, ELU, one tap back to C, three-term rows): the last two stages.  307 200 rows x 64: 145 us
// in two launches -> 86 (276 MB: 3.2 TB/s), 76 800 x 128: 78 -> 65.
static int conv_unit_elu(hipStream_t st, ConvDmaArgs& a1, ConvDmaArgs& a2, int* fused) {
    *fused = 0;
    const int C = a2.N;
    if (a1.n_taps != 3 || a2.n_taps != 1 || a1.Cin != C || a1.N * 2 != C || a2.Cin * 2 != C || (C != 64 && C != 128) || a1.bias_mod != a1.N ||
        a2.bias_mod != C || a2.out2 == a1.x || !a2.res || !a1.elu)
        return VOX_OK;
    int H = 0, omin = 0;
    for (int k = 0; k < 3; ++k) { H = a1.off[k] > H ? a1.off[k] : H; omin = a1.off[k] < omin ? a1.off[k] : omin; }
    if (omin < 0 || H > 16 || a1.L % 64) return VOX_OK;
    *fused = 1;
    if (C == 64) {
        if (a1.L % 128 == 0 && a1.M / 128 >= 256) return conv_unit_launch<64, 32, 3, 3, 16, 8, 1, 3>(st, a1, a2, H);
        return conv_unit_launch<64, 32, 3, 3, 16, 4, 1, 3>(st, a1, a2, H);
    }
    return conv_unit_launch<128, 64, 3, 3, 16, 4, 1, 3>(st, a1, a2, H);
}

static void snake(hipStream_t st, const float* x, const vox_snake_w& s, float* y, size_t rows, int C, int terms = 0) {
    const size_t total = rows * C;
    int grid = (int)((total + 255) / 256);
    if (grid > 4096) grid = 4096;
    hipLaunchKernelGGL(k_snake, dim3(grid), dim3(256), 0, st, x, s.alpha, s.inv_beta, y, total, C, terms);
}

extern "C" {

int vox_codec_create(vox_ctx* ctx, const vox_codec_config* cfg, const vox_codec_weights* w, int max_batch, int max_slots,
                     int frames_per_chunk, vox_codec** out) {
    if (!ctx || !cfg || !w || !out) return vox_fail(VOX_ERR_INVALID, "codec_create: NULL");
    if (cfg->n_blocks != 4 || cfg->n_upsample != 2 || cfg->num_layers > 16)
        return vox_fail(VOX_ERR_INVALID, "codec_create: expects 4 decoder blocks, 2 upsample stages");
    vox_codec* m = new vox_codec();
    m->ctx = ctx; m->cfg = *cfg; m->w = *w; m->max_batch = max_batch; m->max_slots = max_slots; m->T = frames_per_chunk;
    const int S = max_slots, HD = cfg->num_heads * cfg->head_dim;
    size_t L = frames_per_chunk;
    auto zalloc = [&](float** p, size_t n) { return hipMalloc((void**)p, n * 4) == hipSuccess && hipMemset(*p, 0, n * 4) == hipSuccess; };
    bool ok = zalloc(&m->st_pre, (size_t)S * 2 * cfg->codebook_dim);
    for (int u = 0; u < 2; ++u) ok = ok && zalloc(&m->st_dw[u], (size_t)S * 6 * cfg->latent_dim);
    ok = ok && zalloc(&m->st_dec0, (size_t)S * 6 * cfg->latent_dim);
    size_t maxf = (size_t)L * (4 * cfg->latent_dim) * 4;   // ConvNeXt hidden at 4L rows
    L *= 4;
    for (int b = 0; b < 4; ++b) {
        const int cin = cfg->decoder_dim >> b, cout = cfg->decoder_dim >> (b + 1);
        ok = ok && zalloc(&m->st_tc[b], (size_t)S * cin);
        L *= cfg->rates[b];
        for (int u = 0; u < 3; ++u) {
            const int d = u == 0 ? 1 : (u == 1 ? 3 : 9);
            ok = ok && zalloc(&m->st_ru[b][u], (size_t)S * 6 * d * cout);
        }
        if (L * cout > maxf) maxf = L * cout;
        if ((L / cfg->rates[b]) * cin > maxf) maxf = (L / cfg->rates[b]) * cin;
    }
    ok = ok && zalloc(&m->st_final, (size_t)S * 6 * (cfg->decoder_dim >> 4));
    const size_t ring_elems = (size_t)cfg->num_layers * S * cfg->window * 2 * HD;
    ok = ok && hipMalloc((void**)&m->ring, ring_elems * 2) == hipSuccess && hipMemset(m->ring, 0, ring_elems * 2) == hipSuccess;
    ok = ok && hipMalloc((void**)&m->pos, (size_t)S * 8) == hipSuccess && hipMemset(m->pos, 0, (size_t)S * 8) == hipSuccess;
    m->buf_floats = maxf * max_batch;
    for (int i = 0; i < 4; ++i) ok = ok && hipMalloc((void**)&m->buf[i], m->buf_floats * 4) == hipSuccess;
    ok = ok && hipMalloc((void**)&m->q0, (size_t)max_batch * frames_per_chunk * cfg->vq_dim * 4) == hipSuccess;
    ok = ok && hipMalloc((void**)&m->qr, (size_t)max_batch * frames_per_chunk * cfg->vq_dim * 4) == hipSuccess;
    if (!ok) return vox_fail(VOX_ERR_NOMEM, "codec_create: hipMalloc failed");
    *out = m;
    return VOX_OK;
}

int vox_codec_set_operand_planes(vox_codec* m, int planes) {
    if (!m || planes < 1 || planes > 3) return vox_fail(VOX_ERR_INVALID, "codec_set_operand_planes: 1, 2 or 3");
    // the slots' history rows are kept in the operand format (two-term rows vs fp32 rows): switching with history in place would
    // make the convs misread it, so the mode is fixed once the first chunk has been decoded
    if (planes != m->planes && m->decoded)
        return vox_fail(VOX_ERR_INVALID, "codec_set_operand_planes: %d -> %d after a chunk was decoded (set it before the first chunk)", m->planes, planes);
    m->planes = planes;
    return VOX_OK;
}
void vox_codec_destroy(vox_codec* m) {
    if (!m) return;
    (void)hipFree(m->st_pre); (void)hipFree(m->st_dec0); (void)hipFree(m->st_final); (void)hipFree(m->ring);
    (void)hipFree(m->pos); (void)hipFree(m->q0); (void)hipFree(m->qr);
    for (int u = 0; u < 2; ++u) (void)hipFree(m->st_dw[u]);
    for (int b = 0; b < 4; ++b) {
        (void)hipFree(m->st_tc[b]);
        for (int u = 0; u < 3; ++u) (void)hipFree(m->st_ru[b][u]);
    }
    for (int i = 0; i < 4; ++i) (void)hipFree(m->buf[i]);
    delete m;
}

int64_t vox_codec_state_bytes(vox_codec* m) {
    if (!m) return 0;
    const vox_codec_config& c = m->cfg;
    int64_t f = 2 * c.codebook_dim + 6 * c.latent_dim * 3 + 6 * (c.decoder_dim >> 4);
    for (int b = 0; b < 4; ++b) f += (c.decoder_dim >> b) + 6 * 13 * (c.decoder_dim >> (b + 1));
    return f * 4 + (int64_t)c.num_layers * c.window * 2 * c.num_heads * c.head_dim * 2 + 8;
}

// Zero the streaming state of one slot (a new request takes it over).  Replaces audio_decoder_initial_cache
// (model/qwen3_tts.py:1243-1260).
int vox_codec_reset_slot(vox_codec* m, void* stream, int slot) {
    if (!m || slot < 0 || slot >= m->max_slots) return vox_fail(VOX_ERR_INVALID, "codec_reset_slot: bad slot");
    hipStream_t st = (hipStream_t)stream;
    const vox_codec_config& c = m->cfg;
    auto z = [&](float* p, size_t per) { return hipMemsetAsync(p + (size_t)slot * per, 0, per * 4, st); };
    VOX_HIP(z(m->st_pre, (size_t)2 * c.codebook_dim));
    for (int u = 0; u < 2; ++u) VOX_HIP(z(m->st_dw[u], (size_t)6 * c.latent_dim));
    VOX_HIP(z(m->st_dec0, (size_t)6 * c.latent_dim));
    for (int b = 0; b < 4; ++b) {
        VOX_HIP(z(m->st_tc[b], (size_t)(c.decoder_dim >> b)));
        for (int u = 0; u < 3; ++u) VOX_HIP(z(m->st_ru[b][u], (size_t)6 * (u == 0 ? 1 : (u == 1 ? 3 : 9)) * (c.decoder_dim >> (b + 1))));
    }
    VOX_HIP(z(m->st_final, (size_t)6 * (c.decoder_dim >> 4)));
    const size_t HD = (size_t)c.num_heads * c.head_dim, per = (size_t)c.window * 2 * HD;
    for (int l = 0; l < c.num_layers; ++l)
        VOX_HIP(hipMemsetAsync(m->ring + ((size_t)l * m->max_slots + slot) * per, 0, per * 2, st));
    VOX_HIP(hipMemsetAsync(m->pos + slot, 0, 8, st));
    return VOX_OK;
}

// codes: int32 [n, T, code_stride] (first num_quantizers columns used); slots: int32 [n]; out: fp32 [n, T*hop]
}  // extern "C"

// RoPE, the ring's new rows and the attention of layer l: qkv fp32 [nL, 3 HD] -> out [nL, HD] (fp32 or S2 rows)
static int codec_attention(vox_codec* m, hipStream_t st, int l, const int32_t* slots, int n, int L, float* qkv, float* out, int terms) {
    const vox_codec_config& c = m->cfg;
    const int HD = c.num_heads * c.head_dim;
    bf16_t* ring = m->ring + (size_t)l * m->max_slots * c.window * 2 * HD;
    // (VOX_CODEC_ATTN2=0: RoPE / ring write and the attention as two launches — A/B timing; bit-identical)
    static const bool attn2 = [] { const char* e = getenv("VOX_CODEC_ATTN2"); return !(e && e[0] == '0'); }();
    // One launch up to a tile of 64 KB; with its rows on 16 bytes it takes up to 2 % more, two blocks of which still share a CU's LDS
    const size_t tile = (size_t)(2 * c.window * (c.head_dim + 1) + L * c.head_dim + L * c.window) * 4;
    if (attn2 && c.head_dim == 64 && L <= c.window && tile <= 64 * 1024) {
        const size_t lds = tile + (size_t)(2 * c.window + L * (-c.window & 3)) * 4;
        if (lds > 64 * 1024) VOX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_codec_attn2<64>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(k_codec_attn2<64>, dim3(c.num_heads, n), dim3(attn_threads(L)), lds, st, qkv, ring, slots, m->pos, out, L, c.num_heads, c.window,
                           m->w.inv_freq, terms);
    } else {
        hipLaunchKernelGGL(k_codec_rope_kv, dim3(n * L), dim3(256), 0, st, qkv, ring, slots, m->pos, L, c.num_heads, c.head_dim, c.window,
                           m->w.inv_freq);
        hipLaunchKernelGGL(k_codec_attn, dim3(c.num_heads, n), dim3(256),
                           (size_t)(2 * c.window * (c.head_dim + 1) + L * c.head_dim + 4 * c.window) * 4, st, qkv, ring, slots, m->pos, out, L,
                           c.num_heads, c.head_dim, c.window, terms);
    }
    return VOX_OK;
}
// the final conv over x (fp32 rows, activated), its history, a history still due and the slots' positions (T codec frames on)
static void codec_final(vox_codec* m, hipStream_t st, const float* x, const int32_t* slots, int n, int T, int L, float* out, const ConvJob& pending = ConvJob{}) {
    const vox_codec_weights& w = m->w;
    const int cl = m->cfg.decoder_dim >> 4;
    if (!final_taps<7, true>(st, x, m->st_final, slots, w.final_w, w.final_b, out, n, L, cl))
        hipLaunchKernelGGL(k_final_conv, dim3((L + 3) / 4, n), dim3(256), 0, st, x, m->st_final, slots, w.final_w, w.final_b, out, L, cl);
    const ConvJob last{m->st_final, x, L, 6, cl, n};
    const int na = conv_job_blocks(pending, 256), nb = conv_job_blocks(last, 256);
    hipLaunchKernelGGL(k_conv_jobs, dim3(na + nb + 1), dim3(256), 0, st, pending, last, na, nb, slots, m->pos, n, T);
}
// One chunk with fp32 activations, split three ways inside each conv (planes == 3).
static int codec_chunk_f32(vox_codec* m, hipStream_t st, const int32_t* codes, int code_stride, const int32_t* slots, int n, int T, float* out) {
    const vox_codec_config& c = m->cfg;
    const vox_codec_weights& w = m->w;
    const int H = c.hidden, LD = c.latent_dim;
    float *A = m->buf[0], *B = m->buf[1], *C = m->buf[2], *D = m->buf[3];
    const int off0[1] = {0};
    int L = T;

    hipLaunchKernelGGL(k_rvq, dim3(n * L), dim3(256), 0, st, codes, code_stride, w.emb, c.num_quantizers, c.codebook_size,
                       c.vq_dim, m->q0, m->qr, 0);
    VOX_TRY(conv_gemm(st, w.rvq_first_out, m->q0, nullptr, slots, n, L, 0, off0, A, nullptr, nullptr, 0));
    VOX_TRY(conv_gemm(st, w.rvq_rest_out, m->qr, nullptr, slots, n, L, 0, off0, B, A, nullptr, 0));      // B = A + rest
    const int off3[3] = {2, 1, 0};
    VOX_TRY(conv_gemm(st, w.pre_conv, B, m->st_pre, slots, n, L, 2, off3, A, nullptr, nullptr, 0));      // [nL, latent]
    state_update(st, m->st_pre, slots, B, n, L, 2, c.codebook_dim);
    // ---- transformer (hidden H) ----
    VOX_TRY(conv_gemm(st, w.in_proj, A, nullptr, slots, n, L, 0, off0, B, nullptr, nullptr, 0));          // h = B [nL,H]
    for (int l = 0; l < c.num_layers; ++l) {
        const vox_codec_layer_w& lw = w.layers[l];
        hipLaunchKernelGGL(k_rmsnorm_f32, dim3(n * L), dim3(256), 0, st, B, lw.ln1, C, H, c.rms_eps);
        VOX_TRY(conv_gemm(st, lw.qkv, C, nullptr, slots, n, L, 0, off0, D, nullptr, nullptr, 0));        // D [nL,3HD]
        VOX_TRY(codec_attention(m, st, l, slots, n, L, D, C, 0));                                                 // C [nL,HD]
        VOX_TRY(conv_gemm(st, lw.o, C, nullptr, slots, n, L, 0, off0, B, B, lw.scale1, 0));              // h += s1*o(attn)
        hipLaunchKernelGGL(k_rmsnorm_f32, dim3(n * L), dim3(256), 0, st, B, lw.ln2, C, H, c.rms_eps);
        VOX_TRY(conv_gemm(st, lw.gate_up, C, nullptr, slots, n, L, 0, off0, D, nullptr, nullptr, 0));    // D [nL,2I]
        hipLaunchKernelGGL(k_silu_mul_f32, dim3((n * L * c.intermediate + 255) / 256), dim3(256), 0, st, D, C,
                           (size_t)n * L, c.intermediate);
        VOX_TRY(conv_gemm(st, lw.down, C, nullptr, slots, n, L, 0, off0, B, B, lw.scale2, 0));           // h += s2*down
    }
    hipLaunchKernelGGL(k_rmsnorm_f32, dim3(n * L), dim3(256), 0, st, B, w.final_norm, C, H, c.rms_eps);
    VOX_TRY(conv_gemm(st, w.out_proj, C, nullptr, slots, n, L, 0, off0, A, nullptr, nullptr, 0));         // A [nL,latent]
    // ---- upsample x2 x2 with ConvNeXt ----
    for (int u = 0; u < 2; ++u) {
        const vox_codec_up_w& uw = w.up[u];
        VOX_TRY(conv_gemm(st, uw.tconv, A, nullptr, slots, n, L, 0, off0, B, nullptr, nullptr, 0));      // B [n*2L, latent]
        L *= 2;
        hipLaunchKernelGGL(k_dwconv_ln, dim3(n * L), dim3(256), (size_t)LD * 4, st, B, m->st_dw[u], slots, uw.dw_w, uw.dw_b,
                           uw.ln_w, uw.ln_b, C, L, LD, 1e-6f, 0);
        state_update(st, m->st_dw[u], slots, B, n, L, 6, LD);
        VOX_TRY(conv_gemm(st, uw.pw1, C, nullptr, slots, n, L, 0, off0, D, nullptr, nullptr, 1));        // GELU
        VOX_TRY(conv_gemm(st, uw.pw2, D, nullptr, slots, n, L, 0, off0, A, B, uw.gamma, 0));             // A = B + gamma*pw2
    }
    // ---- decoder ----
    const int off7[7] = {6, 5, 4, 3, 2, 1, 0};
    VOX_TRY(conv_gemm(st, w.dec0, A, m->st_dec0, slots, n, L, 6, off7, B, nullptr, nullptr, 0));          // B [nL, decoder_dim]
    state_update(st, m->st_dec0, slots, A, n, L, 6, LD);
    // SnakeBeta is fused into the epilogue of the conv that produces its input: a conv whose output is only ever consumed
    // through a snake (conv1 of a residual unit) writes just the activated tensor, the others write both (the plain tensor
    // is the residual branch).  t1 always holds the activated input of the next conv.
    float* h = B;      // current activations
    float* t1 = A;
    float* t2 = C;
    float* t3 = D;
    snake(st, h, w.blocks[0].snake0, t1, (size_t)n * L, c.decoder_dim);      // (dec0's input A is t1: no room for a fused second output)
    for (int b = 0; b < 4; ++b) {
        const vox_codec_block_w& bw = w.blocks[b];
        const int cin = c.decoder_dim >> b, cout = c.decoder_dim >> (b + 1), r = c.rates[b];
        const int offt[2] = {0, 1};
        // t2 [n*L*r, cout] = tconv(t1); t3 = act1 of unit 0 applied to it (t1 is still being read by other blocks)
        VOX_TRY(conv_gemm(st, bw.tconv, t1, m->st_tc[b], slots, n, L, 1, offt, t2, nullptr, nullptr, 0, t3, &bw.res[0].act1, cout));
        state_update(st, m->st_tc[b], slots, t1, n, L, 1, cin);
        L *= r;
        { float* x = h; h = t2; t2 = x; }
        { float* x = t1; t1 = t3; t3 = x; }             // t1 = act1(h)
        for (int u = 0; u < 3; ++u) {
            const vox_codec_res_w& rw = bw.res[u];
            const int d = u == 0 ? 1 : (u == 1 ? 3 : 9);
            const int offd[7] = {6 * d, 5 * d, 4 * d, 3 * d, 2 * d, d, 0};
            const vox_snake_w* nx = u < 2 ? &bw.res[u + 1].act1 : (b < 3 ? &w.blocks[b + 1].snake0 : &w.final_snake);
            // t3 = act2(conv1(t1))   (the plain conv1 output has no other consumer)
            VOX_TRY(conv_gemm(st, rw.conv1, t1, m->st_ru[b][u], slots, n, L, 6 * d, offd, nullptr, nullptr, nullptr, 0, t3, &rw.act2, cout));
            state_update(st, m->st_ru[b][u], slots, t1, n, L, 6 * d, cout);
            // h += conv2(t3); t1 = the next consumer's activation of the new h
            VOX_TRY(conv_gemm(st, rw.conv2, t3, nullptr, slots, n, L, 0, off0, h, h, nullptr, 0, t1, nx, cout));
        }
    }
    codec_final(m, st, t1, slots, n, T, L, out);
    return VOX_OK;
}

// One chunk with S2 activations (planes 1 and 2): every tensor that only convs read is written as S2 rows by whatever produces it, and what
// stood between two convs (RMSNorm, SiLU, SnakeBeta) is in the epilogue of the first: 86 launches of 134.  The SnakeBeta behind dec0 is the one
// that planes == 3 takes on its own (libm's sine): snake_exact.  RMSNorm: the producer writes h * w
// beside h, the consumer scales its sums by the rows' 1 / rms.
static int codec_chunk_s2(vox_codec* m, hipStream_t st, const int32_t* codes, int code_stride, const int32_t* slots, int n, int T, float* out) {
    const vox_codec_config& c = m->cfg;
    const vox_codec_weights& w = m->w;
    const int LD = c.latent_dim;
    float *A = m->buf[0], *B = m->buf[1], *C = m->buf[2], *D = m->buf[3];
    const int off3[3] = {2, 1, 0}, off7[7] = {6, 5, 4, 3, 2, 1, 0};
    int L = T;
    // A conv's history is rewritten after the conv has read it: by extra blocks of the next launch (its output must not be the history's
    // source); the last one's with the final conv's.
    ConvJob job{};
    auto later = [&](float* state, const float* x, int P, int ch) { job = ConvJob{state, x, L, P, ch, n}; };
    auto conv = [&](const vox_conv_w& cw, const float* x, const float* state, int P, const int* offs) { return conv_s2_args(cw, x, state, slots, n, L, P, offs); };
    auto run = [&](ConvDmaArgs& a, int epi = 0) {
        a.job = job;
        job = ConvJob{};
        return conv_s2(st, a, epi);
    };
    auto s2_out = [](ConvDmaArgs& a, float* y, const float* nw = nullptr) { a.out2 = y; a.out2_s2 = 1; a.nw = nw; };
    auto act_out = [](ConvDmaArgs& a, float* y, const vox_snake_w& sn, int ch, int s2 = 1) {
        a.out2 = y; a.out2_s2 = s2; a.sn_alpha = sn.alpha; a.sn_invb = sn.inv_beta; a.sn_mod = ch;
    };
    auto rms_in = [&](ConvDmaArgs& a, const float* h) { a.rms_x = h; a.rms_eps = c.rms_eps; };

    hipLaunchKernelGGL(k_rvq, dim3(n * L), dim3(256), 0, st, codes, code_stride, w.emb, c.num_quantizers, c.codebook_size, c.vq_dim, m->q0, m->qr, 2);
    { ConvDmaArgs a = conv(w.rvq_first_out, m->q0, nullptr, 0, nullptr); a.out = A; VOX_TRY(run(a)); }
    { ConvDmaArgs a = conv(w.rvq_rest_out, m->qr, nullptr, 0, nullptr); a.res = A; s2_out(a, B); VOX_TRY(run(a)); }
    { ConvDmaArgs a = conv(w.pre_conv, B, m->st_pre, 2, off3); s2_out(a, A); VOX_TRY(run(a)); }             // A [nL, latent]
    later(m->st_pre, B, 2, c.codebook_dim);
    // ---- transformer: h = C (fp32), D = S2 of h * the next norm's weight ----
    { ConvDmaArgs a = conv(w.in_proj, A, nullptr, 0, nullptr); a.out = C; s2_out(a, D, c.num_layers ? w.layers[0].ln1 : w.final_norm); VOX_TRY(run(a)); }
    for (int l = 0; l < c.num_layers; ++l) {
        const vox_codec_layer_w& lw = w.layers[l];
        { ConvDmaArgs a = conv(lw.qkv, D, nullptr, 0, nullptr); rms_in(a, C); a.out = A; VOX_TRY(run(a)); }
        VOX_TRY(codec_attention(m, st, l, slots, n, L, A, B, 2));
        { ConvDmaArgs a = conv(lw.o, B, nullptr, 0, nullptr); a.res = C; a.scale = lw.scale1; a.out = C; s2_out(a, D, lw.ln2); VOX_TRY(run(a)); }
        { ConvDmaArgs a = conv(lw.gate_up, D, nullptr, 0, nullptr); rms_in(a, C); s2_out(a, A); VOX_TRY(run(a, CONV_GLU)); }
        { ConvDmaArgs a = conv(lw.down, A, nullptr, 0, nullptr); a.res = C; a.scale = lw.scale2; a.out = C;
          s2_out(a, D, l + 1 < c.num_layers ? w.layers[l + 1].ln1 : w.final_norm); VOX_TRY(run(a)); }
    }
    { ConvDmaArgs a = conv(w.out_proj, D, nullptr, 0, nullptr); rms_in(a, C); s2_out(a, A); VOX_TRY(run(a)); }      // A [nL, latent]
    // ---- upsample x2 x2 with ConvNeXt ----
    for (int u = 0; u < 2; ++u) {
        const vox_codec_up_w& uw = w.up[u];
        { ConvDmaArgs a = conv(uw.tconv, A, nullptr, 0, nullptr); a.out = B; VOX_TRY(run(a)); }                     // B [n*2L, latent]
        L *= 2;
        hipLaunchKernelGGL(k_dwconv_ln, dim3(n * L), dim3(256), (size_t)LD * 4, st, B, m->st_dw[u], slots, uw.dw_w, uw.dw_b, uw.ln_w, uw.ln_b, C, L, LD,
                           1e-6f, 2);
        later(m->st_dw[u], B, 6, LD);
        { ConvDmaArgs a = conv(uw.pw1, C, nullptr, 0, nullptr); s2_out(a, D); VOX_TRY(run(a, CONV_GELU)); }
        { ConvDmaArgs a = conv(uw.pw2, D, nullptr, 0, nullptr); a.res = B; a.scale = uw.gamma; s2_out(a, A); VOX_TRY(run(a)); }
    }
    // ---- decoder.  SnakeBeta is in the epilogue of the conv that produces its input; h stays fp32 and is written only where a residual
    // branch reads it.  free: the two buffers that hold neither h nor x (job.x may still be one of them). ----
    { ConvDmaArgs a = conv(w.dec0, A, m->st_dec0, 6, off7); act_out(a, C, w.blocks[0].snake0, c.decoder_dim); VOX_TRY(run(a, CONV_SINE)); }
    later(m->st_dec0, A, 6, LD);
    float *h = B, *x = C, *free_[2] = {A, D};
    auto take = [&](float* avoid) {          // a free buffer other than `avoid`; its place is left empty (NULL)
        float** f = free_[0] && free_[0] != avoid ? &free_[0] : &free_[1];
        float* p = *f;
        *f = nullptr;
        return p;
    };
    auto put = [&](float* p) { (free_[0] ? free_[1] : free_[0]) = p; };
    for (int b = 0; b < 4; ++b) {
        const vox_codec_block_w& bw = w.blocks[b];
        const int cin = c.decoder_dim >> b, cout = c.decoder_dim >> (b + 1);
        const int offt[2] = {0, 1};
        {   // h' [n*L*r, cout] = tconv(x), x' = act1 of unit 0 applied to it.  The old h is dead: three buffers to choose from
            float *old_x = x, *xn = take(const_cast<float*>(job.x)), *hn = h;
            ConvDmaArgs a = conv(bw.tconv, x, m->st_tc[b], 1, offt);
            a.out = hn;
            act_out(a, xn, bw.res[0].act1, cout);
            VOX_TRY(run(a));
            later(m->st_tc[b], old_x, 1, cin);
            x = xn;
            put(old_x);
        }
        L *= c.rates[b];
        for (int u = 0; u < 3; ++u) {
            const vox_codec_res_w& rw = bw.res[u];
            const int d = u == 0 ? 1 : (u == 1 ? 3 : 9), last = b == 3 && u == 2;
            const int offd[7] = {6 * d, 5 * d, 4 * d, 3 * d, 2 * d, d, 0};
            const vox_snake_w* nx = u < 2 ? &bw.res[u + 1].act1 : (b < 3 ? &w.blocks[b + 1].snake0 : &w.final_snake);
            float *y = take(const_cast<float*>(job.x)), *ho = u < 2 ? h : nullptr;      // (after unit 2 only the activation of h goes on)
            ConvDmaArgs a1 = conv(rw.conv1, x, m->st_ru[b][u], 6 * d, offd);      // y = act2(conv1(x))
            act_out(a1, y, rw.act2, cout);
            ConvDmaArgs a2 = conv(rw.conv2, y, nullptr, 0, nullptr);               // h += conv2(y), and the next consumer's activation of it
            a2.res = h;
            a2.out = ho;
            act_out(a2, y, *nx, cout, !last);                                      // (the final conv reads fp32 rows)
            int fused = 0;
            a1.job = job;
            VOX_TRY(conv_unit(st, a1, a2, &fused));
            if (fused == 1) {
                later(m->st_ru[b][u], x, 6 * d, cout);
                put(x);
                x = y;
                continue;
            }
            VOX_TRY(run(a1, fused));
            later(m->st_ru[b][u], x, 6 * d, cout);
            float* z = take(nullptr);
            a2.out2 = z;
            VOX_TRY(run(a2));
            put(x);
            put(y);
            x = z;
        }
    }
    codec_final(m, st, x, slots, n, T, L, out, job);
    return VOX_OK;
}

extern "C" {

int vox_codec_decode_chunk(vox_codec* m, void* stream, const int32_t* codes, int code_stride, const int32_t* slots, int n,
                           int T, float* out) {
    if (!m || !codes || !slots || !out) return vox_fail(VOX_ERR_INVALID, "codec_decode_chunk: NULL");
    if (n < 1 || n > m->max_batch || T < 1 || T > m->T) return vox_fail(VOX_ERR_INVALID, "codec_decode_chunk: n=%d T=%d out of range", n, T);
    m->decoded = true;
    hipStream_t st = (hipStream_t)stream;
    struct PlanesGuard { int saved; explicit PlanesGuard(int p) : saved(g_conv_planes) { g_conv_planes = p; } ~PlanesGuard() { g_conv_planes = saved; } } pg(m->planes);
    return m->planes <= 2 ? codec_chunk_s2(m, st, codes, code_stride, slots, n, T, out) : codec_chunk_f32(m, st, codes, code_stride, slots, n, T, out);
}

}  // extern "C"

// ================================================================================================
// Mimi decoder (CSM's codec), stateless per chunk.  Same building blocks: implicit-GEMM convolutions on split-fp32
// MFMA (look-back rows before the chunk start read as zero = the reference's constant padding of a fresh state),
// transposed conv with stride r = 2-tap GEMM writing r*Cout contiguous values per input row (the reference trims the
// K-S rightmost samples: exactly the part the second tap of the NEXT chunk would add).
// ================================================================================================
// y[b, 2t+j, c] = x[b,t,c] * w[c][j] + x[b,t-1,c] * w[c][j+2]        (ConvTrUpsample1d, mimi.py:2272-2323)
// state (streaming): [slots][1][C] = the previous chunk's last input row; NULL = fresh state (zeros)
__global__ __launch_bounds__(256) void k_mimi_upsample(const float* x, const float* w, float* y, int L, int C, size_t total,
                                                        const float* state, const int* slots) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % C);
        const size_t row = i / C;                     // output row = b*2L + 2t + j
        const int tj = (int)(row % (2 * (size_t)L)), t = tj >> 1, j = tj & 1;
        const size_t b = row / (2 * (size_t)L);
        const float cur = x[(b * L + t) * C + c];
        const float prev = t > 0 ? x[(b * L + t - 1) * C + c] : (state ? state[(size_t)slots[b] * C + c] : 0.0f);
        y[i] = cur * w[c * 4 + j] + prev * w[c * 4 + j + 2];
    }
}
__global__ __launch_bounds__(256) void k_layernorm_f32(const float* x, const float* w, const float* b, float* y, int C, float eps, int terms = 0) {
    __shared__ float red[8];
    const float* xr = x + (size_t)blockIdx.x * C;
    float s = 0.0f;
    for (int i = threadIdx.x; i < C; i += 256) s += xr[i];
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float mean = (red[0] + red[1] + red[2] + red[3]) / (float)C;
    float v = 0.0f;
    for (int i = threadIdx.x; i < C; i += 256) { const float d = xr[i] - mean; v += d * d; }
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) red[4 + (threadIdx.x >> 6)] = v;
    __syncthreads();
    const float rstd = rsqrtf((red[4] + red[5] + red[6] + red[7]) / (float)C + eps);
    for (int i = threadIdx.x; i < C; i += 256) put_row(y, blockIdx.x, C, i, (xr[i] - mean) * rstd * w[i] + b[i], terms);
}
__global__ __launch_bounds__(256) void k_elu(const float* x, float* y, size_t total) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const float v = x[i];
        y[i] = v > 0.0f ? v : expm1f(v);
    }
}
// causal attention inside one chunk of L <= 64 tokens with RoPE on interleaved pairs at positions 0..L-1
// (apply_rope mimi.py:874-931; offset 0: stateless).  qkv rows [3][H][D]; one block per (head, request).
// DC: the head dim where it is known when compiled (0: it is not), so that the products of a score are not one LDS trip each: 16 requests of 20
// rows, head dim 64: 8.0 -> 7.5 us.
template <int DC>
__global__ __launch_bounds__(1024) void k_mimi_attn(const float* qkv, float* out, int L, int H, int D_, int context, float max_period) {
    const int D = DC ? DC : D_;
    extern __shared__ float sm[];   // Q [L][D], K [L][D+1], V [L][D+1], P [waves][L]
    const int LD = D + 1;
    float* Qs = sm;
    float* Ks = Qs + (size_t)L * D;
    float* Vs = Ks + (size_t)L * LD;
    float* Ps = Vs + (size_t)L * LD;
    const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = blockDim.x;
    const int HD = H * D;
    for (int e = tid; e < L * (D / 2); e += nt) {
        const int t = e / (D / 2), i = e % (D / 2);
        const float* r = qkv + ((size_t)(b * L + t)) * 3 * HD + (size_t)h * D + 2 * i;
        const float freq = expf((float)i * (-logf(max_period) * 2.0f / (float)D));
        const float ang = freq * (float)t;
        const float cr = cosf(ang), ci = sinf(ang);
        const float qr = r[0], qi = r[1], kr = r[HD], ki = r[HD + 1];
        Qs[t * D + 2 * i] = qr * cr - qi * ci;
        Qs[t * D + 2 * i + 1] = qr * ci + qi * cr;
        Ks[t * LD + 2 * i] = kr * cr - ki * ci;
        Ks[t * LD + 2 * i + 1] = kr * ci + ki * cr;
        Vs[t * LD + 2 * i] = r[2 * HD];
        Vs[t * LD + 2 * i + 1] = r[2 * HD + 1];
    }
    __syncthreads();
    const float scale = rsqrtf((float)D);
    float* P = Ps + (size_t)wave * L;
    for (int i = wave; i < L; i += nt >> 6) {
        const float* q = Qs + (size_t)i * D;
        const int j = lane;
        const bool vis = j < L && j <= i && (i - j) < context;
        float sc = -INFINITY;
        if (vis) {
            sc = 0.0f;
            if constexpr (DC > 0) {
#pragma unroll
                for (int d = 0; d < DC; ++d) sc = fmaf(q[d], Ks[j * LD + d], sc);
            } else {
                for (int d = 0; d < D; ++d) sc = fmaf(q[d], Ks[j * LD + d], sc);
            }
            sc *= scale;
        }
        float mx = sc;
        for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        const float pj = vis ? expf(sc - mx) : 0.0f;
        const float ls = butterfly<64>(pj);
        if (j < L) P[j] = pj;
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        for (int d = lane; d < D; d += 64) {
            float o = 0.0f;
            for (int j0 = 0; j0 <= i; j0 += 8) {      // (read together: what is past row i is not added)
                float pv[8], x[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int k = j0 + u <= i ? j0 + u : i;
                    pv[u] = P[k];
                    x[u] = Vs[k * LD + d];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) o = j0 + u <= i ? fmaf(pv[u], x[u], o) : o;
            }
            put_row(out, (size_t)(b * L + i), HD, h * D + d, o / ls, 3);
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
}
// Streaming variant: queries = the L new rows at absolute positions pos0 .. pos0+L-1 of the slot, keys = the slot's K/V ring
// (post-RoPE K) + the new rows; visibility 0 <= p_q - p_k < context.  Ring capacity RC >= context + L - 1 so that a new key
// never overwrites one an earlier query of the same chunk still sees.  One block per (head, request): the visible K window
// (<= context + L - 1 rows) sits in LDS (row stride D+1), V is read from the ring (coalesced rows, L2-resident).
__global__ __launch_bounds__(256) void k_mimi_attn_stream(const float* qkv, float* out, float* kring, float* vring, const long* pos,
                                                           const int* slots, int L, int H, int D, int context, int RC, float max_period) {
    extern __shared__ float sm[];   // Q [L][D], K [context+L][D+1], P [4][context+L]
    const int LD = D + 1, W = context + L;
    float* Qs = sm;
    float* Ks = Qs + (size_t)L * D;
    float* Ps = Ks + (size_t)W * LD;
    const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int HD = H * D;
    const long p0 = pos[slots[b]];
    float* kr = kring + (size_t)slots[b] * RC * HD + (size_t)h * D;     // row stride HD
    float* vr = vring + (size_t)slots[b] * RC * HD + (size_t)h * D;
    for (int e = tid; e < L * (D / 2); e += 256) {       // RoPE the new q / k at their absolute positions, append k / v
        const int t = e / (D / 2), i = e % (D / 2);
        const float* r = qkv + ((size_t)(b * L + t)) * 3 * HD + (size_t)h * D + 2 * i;
        const float freq = expf((float)i * (-logf(max_period) * 2.0f / (float)D));
        const float ang = freq * (float)(p0 + t);
        const float cr = cosf(ang), ci = sinf(ang);
        const float qr = r[0], qi = r[1], k0 = r[HD], k1 = r[HD + 1];
        Qs[t * D + 2 * i] = qr * cr - qi * ci;
        Qs[t * D + 2 * i + 1] = qr * ci + qi * cr;
        const size_t ro = (size_t)((p0 + t) % RC) * HD + 2 * i;
        kr[ro] = k0 * cr - k1 * ci;
        kr[ro + 1] = k0 * ci + k1 * cr;
        vr[ro] = r[2 * HD];
        vr[ro + 1] = r[2 * HD + 1];
    }
    __syncthreads();                                       // (block-scope: this block is the only reader of its ring rows)
    const long lo = (p0 - context + 1) > 0 ? (p0 - context + 1) : 0;     // oldest position any query of the chunk sees
    const int nk = (int)(p0 + L - lo);                     // window rows [lo, p0+L)
    for (int e = tid; e < nk * D; e += 256) {
        const int j = e / D, d = e % D;
        Ks[j * LD + d] = kr[(size_t)((lo + j) % RC) * HD + d];
    }
    __syncthreads();
    const float scale = rsqrtf((float)D);
    float* P = Ps + (size_t)wave * W;
    for (int i = wave; i < L; i += 4) {
        const float* q = Qs + (size_t)i * D;
        const long pq = p0 + i;
        float mx = -INFINITY;
        for (int j = lane; j < nk; j += 64) {
            const long pk = lo + j;
            float sc = -INFINITY;
            if (pk <= pq && (pq - pk) < context) {
                sc = 0.0f;
                for (int d = 0; d < D; ++d) sc = fmaf(q[d], Ks[j * LD + d], sc);
                sc *= scale;
            }
            P[j] = sc;
            mx = fmaxf(mx, sc);
        }
        for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        float ls = 0.0f;
        for (int j = lane; j < nk; j += 64) {
            const float pj = P[j] == -INFINITY ? 0.0f : expf(P[j] - mx);
            P[j] = pj;
            ls += pj;
        }
        for (int off = 32; off >= 1; off >>= 1) ls += __shfl_xor(ls, off, 64);
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        const int jlo = (int)((pq - context + 1 > lo ? pq - context + 1 : lo) - lo), jhi = (int)(pq - lo);
        for (int d = lane; d < D; d += 64) {
            float o = 0.0f;
            for (int jj = jlo; jj <= jhi; ++jj) o = fmaf(P[jj], vr[(size_t)((lo + jj) % RC) * HD + d], o);
            put_row(out, (size_t)(b * L + i), HD, h * D + d, o / ls, 3);
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
}
// last conv: C -> 1 channel, kernel K, zero history
__global__ __launch_bounds__(256) void k_mimi_final(const float* x, const float* w, float bias, float* out, int L, int C, int K,
                                                     const float* state, const int* slots) {
    const int b = blockIdx.y;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= L) return;
    float acc = 0.0f;
    for (int e = lane; e < K * C; e += 64) {
        const int k = e / C, c = e % C;
        const int r = t - (K - 1) + k;
        if (r >= 0) acc += w[c * K + k] * x[((size_t)b * L + r) * C + c];
        else if (state) acc += w[c * K + k] * state[((size_t)slots[b] * (K - 1) + (K - 1 + r)) * C + c];   // streaming history
    }
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) out[(size_t)b * L + t] = acc + bias;
}

struct vox_mimi {
    vox_ctx* ctx;
    vox_mimi_config cfg;
    vox_mimi_weights w;
    int max_batch, max_frames;
    float *q0, *qr, *buf[4];
    int32_t* zero_slots;
    // streaming state (vox_mimi_stream_enable), per slot: the look-back rows of every causal conv / transposed conv input,
    // a K/V ring per transformer layer and the number of transformer-rate rows seen so far
    int max_slots = 0, ring_cap = 0;
    float *st_up = nullptr, *st_dec0 = nullptr, *st_tc[4] = {nullptr, nullptr, nullptr, nullptr},
          *st_c1[4] = {nullptr, nullptr, nullptr, nullptr}, *st_final = nullptr, *kring = nullptr, *vring = nullptr;
    long* pos = nullptr;
};

// fp32 rows as S3 rows
__global__ __launch_bounds__(256) void k_terms3(const float* x, float* y, int C) {
    for (int c = threadIdx.x; c < C; c += 256) put_row(y, blockIdx.x, C, c, x[(size_t)blockIdx.x * C + c], 3);
}
static void elu(hipStream_t st, const float* x, float* y, size_t total) {
    int grid = (int)((total + 255) / 256);
    if (grid > 4096) grid = 4096;
    hipLaunchKernelGGL(k_elu, dim3(grid), dim3(256), 0, st, x, y, total);
}

extern "C" {

int vox_mimi_create(vox_ctx* ctx, const vox_mimi_config* cfg, const vox_mimi_weights* w, int max_batch, int max_frames,
                    vox_mimi** out) {
    if (!ctx || !cfg || !w || !out) return vox_fail(VOX_ERR_INVALID, "mimi_create: NULL");
    if (cfg->num_layers > 16 || cfg->dim % cfg->num_heads || 2 * max_frames > 64)
        return vox_fail(VOX_ERR_INVALID, "mimi_create: <= 16 layers, <= 32 frames per chunk");
    vox_mimi* m = new vox_mimi();
    m->ctx = ctx; m->cfg = *cfg; m->w = *w; m->max_batch = max_batch; m->max_frames = max_frames;
    // largest activation: rows x channels is the same (2T * 16 n_filters * prod so far / 2^i) at every SEANet stage up to
    // the ratio products; bound it by the widest of each stage
    size_t L = (size_t)2 * max_frames, ch = (size_t)16 * cfg->n_filters, maxf = L * ch;
    for (int i = 0; i < 4; ++i) {
        L *= cfg->ratios[i];
        ch /= 2;
        maxf = maxf > L * ch ? maxf : L * ch;
    }
    const size_t tr = (size_t)2 * max_frames * (3 * cfg->dim > cfg->ffn ? 3 * cfg->dim : cfg->ffn);
    maxf = (maxf > tr ? maxf : tr) * max_batch;
    // (6 bytes an element: a buffer holds fp32 or S3 rows)
    bool ok = hipMalloc((void**)&m->q0, (size_t)max_batch * max_frames * cfg->vq_dim * 6) == hipSuccess &&
              hipMalloc((void**)&m->qr, (size_t)max_batch * max_frames * cfg->vq_dim * 6) == hipSuccess &&
              hipMalloc((void**)&m->zero_slots, (size_t)max_batch * 4) == hipSuccess;
    for (int i = 0; i < 4; ++i) ok = ok && hipMalloc((void**)&m->buf[i], maxf * 6) == hipSuccess;
    if (!ok) return vox_fail(VOX_ERR_NOMEM, "mimi_create: hipMalloc failed");
    VOX_HIP(hipMemset(m->zero_slots, 0, (size_t)max_batch * 4));
    *out = m;
    return VOX_OK;
}
void vox_mimi_destroy(vox_mimi* m) {
    if (!m) return;
    (void)hipFree(m->q0); (void)hipFree(m->qr); (void)hipFree(m->zero_slots);
    (void)hipFree(m->st_up); (void)hipFree(m->st_dec0); (void)hipFree(m->st_final); (void)hipFree(m->kring); (void)hipFree(m->vring); (void)hipFree(m->pos);
    for (int b = 0; b < 4; ++b) { (void)hipFree(m->st_tc[b]); (void)hipFree(m->st_c1[b]); }
    for (int i = 0; i < 4; ++i) (void)hipFree(m->buf[i]);
    delete m;
}
}  // extern "C"

// LayerNorm of 512-wide fp32 rows and the linear behind it (one tap, three-term rows, EPI as k_conv_dma's) in one launch: k_layernorm_f32's sums and k_conv_dma's products to the
// bit.  The launch between them wrote three terms of every row for 12 to 16 column blocks to read back; here each of those norms its 16 rows itself (a wave
// per row: two of k_layernorm_f32's four waves in the halves of the wave, the other two behind them), while the weights of its columns, all of K, are on their way into
// registers: one trip, one barrier, no step behind another.  W of the eight waves multiply, 16 columns each.  us, both launches
// before and now: 8 rows, q | k | v 3.9 + 4.8, 6.9, with GELU 3.9 + 6.0, 8.2 (eight waves); 320 rows 4.9 + 7.8, 9.2 and 4.9 + 11.4, 14.8.
template <int W, int EPI>
__global__ __launch_bounds__(512) void k_ln_linear(ConvDmaArgs a, const float* x, const float* lw, const float* lb, float eps) {
    touch_args(a);
    constexpr int C = 512, KS = C / 32;
    __shared__ uint4 lnl_rows[3 * 16 * (C / 8)];      // [3 terms][16 rows][C / 8 pieces], piece c of row r at c ^ (r & 7)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, fk = lane >> 4;
    const int t = (int)blockIdx.x, m0 = t / a.tn * 16, n0 = (t % a.tn * W + wave) * 16;
    const bool multiplies = W == 8 || wave < W;
    const int j = lane & 31, hw = lane >> 5;
    float2 v[2][2][2], w2[2][2], b2[2][2];      // [row of the wave][wave hw or hw + 2 of the norm][first or second of its two columns]
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int m = m0 + wave * 2 + i;
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int u = 0; u < 2; ++u) v[i][p][u] = *reinterpret_cast<const float2*>(x + (size_t)(m < a.M ? m : a.M - 1) * C + 256 * u + 64 * (hw + 2 * p) + 2 * j);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            w2[p][u] = *reinterpret_cast<const float2*>(lw + 256 * u + 64 * (hw + 2 * p) + 2 * j);
            b2[p][u] = *reinterpret_cast<const float2*>(lb + 256 * u + 64 * (hw + 2 * p) + 2 * j);
        }
    uint4 wf[KS];
    if (multiplies) {
        const int n = n0 + fr;
        const uint4* wr = reinterpret_cast<const uint4*>(a.w + (size_t)(n < a.N ? n : a.N - 1) * C) + fk;
#pragma unroll
        for (int k = 0; k < KS; ++k) wf[k] = ldg(wr + k * 4);
    }
    // the sum of one of the four waves' 64 values, two to a lane: partners 32 .. 2 in other lanes, 1 in this one
    auto wave_sum = [](float s0, float s1) {
        s0 = xor_add<1>(xor_add<2>(xor_add<4>(xor_add<8>(xor_add<16>(s0)))));
        s1 = xor_add<1>(xor_add<2>(xor_add<4>(xor_add<8>(xor_add<16>(s1)))));
        return s0 + s1;
    };
    auto four = [&](float r0, float r1) {       // waves hw, hw + 2 -> ((0 + 1) + 2) + 3
        const vox_u2 a0 = __builtin_amdgcn_permlane32_swap(__float_as_uint(r0), __float_as_uint(r0), false, false);
        const vox_u2 a1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(r1), __float_as_uint(r1), false, false);
        return __uint_as_float(a0.x) + __uint_as_float(a0.y) + __uint_as_float(a1.x) + __uint_as_float(a1.y);
    };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        float r[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) r[p] = wave_sum(v[i][p][0].x + v[i][p][1].x, v[i][p][0].y + v[i][p][1].y);
        const float mean = four(r[0], r[1]) / (float)C;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            float s[2] = {0.0f, 0.0f};
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                v[i][p][u].x -= mean;
                v[i][p][u].y -= mean;
                s[0] += v[i][p][u].x * v[i][p][u].x;
                s[1] += v[i][p][u].y * v[i][p][u].y;
            }
            r[p] = wave_sum(s[0], s[1]);
        }
        const float rstd = rsqrtf(four(r[0], r[1]) / (float)C + eps);
        const int row = wave * 2 + i;
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                float y0 = v[i][p][u].x * rstd * w2[p][u].x + b2[p][u].x, y1 = v[i][p][u].y * rstd * w2[p][u].y + b2[p][u].y;
                const int c = 256 * u + 64 * (hw + 2 * p) + 2 * j;
                u32* const d = reinterpret_cast<u32*>(lnl_rows + row * (C / 8) + ((c >> 3) ^ (row & 7))) + (j & 3);
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const u32 h = pack_bf2(y0, y1);
                    d[q * (16 * C / 2)] = h;
                    y0 -= bflo(h);
                    y1 -= bfhi(h);
                }
            }
    }
    __syncthreads();
    if (!multiplies) return;
    f32x4 acc[1][1] = {{(f32x4){0.f, 0.f, 0.f, 0.f}}};
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int p = 2; p >= 0; --p) {
            union { uint4 u; cbf16x8 b; } wa, xa;
            wa.u = wf[k];
            xa.u = lnl_rows[(p * 16 + fr) * (C / 8) + ((k * 4 + fk) ^ (fr & 7))];
            acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa.b, xa.b, acc[0][0], 0, 0, 0);
        }
    conv_dma_out<3, EPI, 4, 1>(a, acc, nullptr, m0 + fr, n0 + fk * 4);
}
template <int W, int EPI>
static int ln_linear_launch(hipStream_t st, ConvDmaArgs& a, const float* x, const float* lw, const float* lb, float eps) {
    a.tn = (a.N + 16 * W - 1) / (16 * W);
    hipLaunchKernelGGL((k_ln_linear<W, EPI>), dim3((a.M + 15) / 16 * a.tn), dim3(512), 0, st, a, x, lw, lb, eps);
    return VOX_OK;
}
// a: the linear's arguments, whose rows are LayerNorm(x); buf: rows for the two launches where the one does not apply
template <int EPI>
static int ln_linear(hipStream_t st, ConvDmaArgs& a, const float* x, const float* lw, const float* lb, float eps, float* buf) {
    const size_t at = (size_t)a.w | (size_t)x, at8 = (size_t)lw | (size_t)lb;
    if (a.M <= 640 && a.Cin == 512 && a.n_taps == 1 && !a.state && !a.job.state && a.N % 16 == 0 && a.sn_mod % 8 == 0 && a.bias_mod % 8 == 0 && (at & 15) == 0 && (at8 & 7) == 0) {
        // (More than 640 rows fill the chip with larger tiles, and these norm and fetch weights too often: launch pairs / eight waves 400 1078 / 1079, 640 1476 / 1466, 960 1935 / 1961,
        // 1280 2465 / 2515.)  Up to 64 rows two waves multiply (all eight norm): four times the CUs fetch the weights.  Mimi chunks, us, rows of the transformer, launch pairs / two / eight waves:
        // 2 371 / 344 / 349, 20 429 / 396 / 408, 32 422 / 389 / 401, 64 460 / 423 / 433, 80 514 / 494 / 487, 128 529 / 523 / 497, 160 627 / 638 / 583, 320 916 / 983 / 877
        return a.M <= 64 ? ln_linear_launch<2, EPI>(st, a, x, lw, lb, eps) : ln_linear_launch<8, EPI>(st, a, x, lw, lb, eps);
    }
    hipLaunchKernelGGL(k_layernorm_f32, dim3(a.M), dim3(256), 0, st, x, lw, lb, buf, a.Cin, eps, 3);
    return conv_s2(st, a, EPI);
}


// slots == NULL: stateless chunk (fresh state: the reference's MimiDecoder.decode); else streaming on the given state slots.
// Activations that only convs read are S3 rows (three bf16 terms: the fp32 value), written by whatever produces them; ELU is in the
// epilogue of the conv in front of it, a conv's history in extra blocks of the next launch (as in codec_chunk_s2).
static int mimi_run(vox_mimi* m, hipStream_t st, const int32_t* codes, int code_stride, const int32_t* slots, int n, int T, float* out) {
    const vox_mimi_config& c = m->cfg;
    const vox_mimi_weights& w = m->w;
    const int C = c.dim, H = c.num_heads, D = c.dim / c.num_heads;
    const bool S = slots != nullptr;
    const int* sl = S ? slots : m->zero_slots;
    struct PlanesGuard { int saved; PlanesGuard() : saved(g_conv_planes) { g_conv_planes = 3; } ~PlanesGuard() { g_conv_planes = saved; } } pg;
    float *A = m->buf[0], *B = m->buf[1], *Cb = m->buf[2], *Db = m->buf[3];
    int L = T;
    ConvJob job{};
    auto later = [&](float* state, const float* x, int P, int ch) {
        if (S) job = ConvJob{state, x, L, P, ch / 2 * 3, n};
    };
    auto conv = [&](const vox_conv_w& cw, const float* x, const float* state, int P, const int* offs) {
        return conv_s2_args(cw, x, S ? state : nullptr, sl, n, L, S ? P : 0, offs);
    };
    auto run = [&](ConvDmaArgs& a, int epi = 0) {
        a.job = job;
        job = ConvJob{};
        return conv_s2(st, a, epi);
    };
    auto terms = [](ConvDmaArgs& a, float* y) { a.out2 = y; a.out2_s2 = 1; };
    auto elu_out = [](ConvDmaArgs& a, float* y, int ch, int t = 1) { a.out2 = y; a.out2_s2 = t; a.elu = 1; a.sn_mod = ch; };
    hipLaunchKernelGGL(k_rvq, dim3(n * L), dim3(256), 0, st, codes, code_stride, w.emb, c.n_q, c.bins, c.vq_dim, m->q0, m->qr, 3);
    { ConvDmaArgs a = conv(w.rvq_first_out, m->q0, nullptr, 0, nullptr); a.out = A; VOX_TRY(run(a)); }
    { ConvDmaArgs a = conv(w.rvq_rest_out, m->qr, nullptr, 0, nullptr); a.res = A; a.out = B; VOX_TRY(run(a)); }            // B [nL, dim]
    {
        const size_t total = (size_t)n * 2 * L * C;
        int grid = (int)((total + 255) / 256);
        if (grid > 4096) grid = 4096;
        hipLaunchKernelGGL(k_mimi_upsample, dim3(grid), dim3(256), 0, st, B, w.up_w, A, L, C, total, S ? m->st_up : nullptr, sl);   // A [n*2L, dim]
        if (S) state_update(st, m->st_up, sl, B, n, L, 1, C);
    }
    L *= 2;
    for (int l = 0; l < c.num_layers; ++l) {                                                                 // h = A
        const vox_mimi_layer_w& lw = w.layers[l];
        { ConvDmaArgs a = conv(lw.qkv, Cb, nullptr, 0, nullptr); a.out = Db; VOX_TRY(ln_linear<0>(st, a, A, lw.ln1_w, lw.ln1_b, c.ln_eps, Cb)); }              // Db [nL, 3*dim]
        if (S) {
            const size_t ring = (size_t)m->max_slots * m->ring_cap * C;
            const size_t smem = ((size_t)L * D + (size_t)(c.context + L) * (D + 1) + 4 * (size_t)(c.context + L)) * 4;
            hipLaunchKernelGGL(k_mimi_attn_stream, dim3(H, n), dim3(256), smem, st, Db, Cb, m->kring + l * ring, m->vring + l * ring,
                               m->pos, sl, L, H, D, c.context, m->ring_cap, c.max_period);
        } else {
            hipLaunchKernelGGL(D == 64 ? k_mimi_attn<64> : k_mimi_attn<0>, dim3(H, n), dim3(attn_threads(L)), (size_t)(L * D + 2 * L * (D + 1) + attn_threads(L) / 64 * L) * 4, st, Db, Cb, L, H, D,
                               c.context, c.max_period);
        }
        { ConvDmaArgs a = conv(lw.o, Cb, nullptr, 0, nullptr); a.res = a.out = A; a.scale = lw.scale1; VOX_TRY(run(a)); }   // h += s1 * o(attn)
        { ConvDmaArgs a = conv(lw.fc1, Cb, nullptr, 0, nullptr); terms(a, Db); VOX_TRY(ln_linear<CONV_GELU>(st, a, A, lw.ln2_w, lw.ln2_b, c.ln_eps, Cb)); }
        { ConvDmaArgs a = conv(lw.fc2, Db, nullptr, 0, nullptr); a.res = a.out = A; a.scale = lw.scale2;                    // h += s2 * mlp
          if (l == c.num_layers - 1) terms(a, Cb);
          VOX_TRY(run(a)); }
    }
    if (S) hipLaunchKernelGGL(k_pos_advance, dim3((n + 255) / 256), dim3(256), 0, st, m->pos, sl, n, L);
    if (!c.num_layers) hipLaunchKernelGGL(k_terms3, dim3(n * L), dim3(256), 0, st, A, Cb, C);
    // ---- SEANet decoder: x = the activated rows of the next conv; h only where a residual reads it ----
    int offk[CG_MAXTAPS];
    for (int k = 0; k < c.kernel_size && k < CG_MAXTAPS; ++k) offk[k] = c.kernel_size - 1 - k;
    const int Pk = c.kernel_size - 1;
    int ch = 16 * c.n_filters;
    { ConvDmaArgs a = conv(w.dec0, Cb, m->st_dec0, Pk, offk); elu_out(a, B, ch); VOX_TRY(run(a)); }           // B [nL, 16 nf]
    later(m->st_dec0, Cb, Pk, C);
    float *x = B, *h = A, *f0 = Db, *f1 = Cb;      // (f1 may be the pending history's source: the next launch must not write it)
    for (int b = 0; b < 4; ++b) {
        const vox_mimi_block_w& bw = w.blocks[b];
        const int offt[2] = {0, 1}, off3[3] = {2, 1, 0};
        { ConvDmaArgs a = conv(bw.tconv, x, m->st_tc[b], 1, offt); a.out = h; elu_out(a, f0, ch / 2); VOX_TRY(run(a)); }     // h [n*L*r, ch/2]
        later(m->st_tc[b], x, 1, ch);
        { float* o = x; x = f0; f0 = f1; f1 = o; }
        L *= c.ratios[b];
        ch /= 2;
        ConvDmaArgs a1 = conv(bw.conv1, x, m->st_c1[b], 2, off3), a2 = conv(bw.conv2, f0, nullptr, 0, nullptr);
        elu_out(a1, f0, ch / 2);                                  // f0 [nL, ch/2]
        a2.res = h;
        elu_out(a2, f0, ch, b < 3);                               // h + conv2(f0), activated (the final conv reads fp32 rows)
        int fused = 0;
        a1.job = job;
        VOX_TRY(conv_unit_elu(st, a1, a2, &fused));
        if (fused) {
            job = ConvJob{};
            later(m->st_c1[b], x, 2, ch);
            { float* o = x; x = f0; f0 = f1; f1 = o; }
            continue;
        }
        VOX_TRY(run(a1));
        later(m->st_c1[b], x, 2, ch);
        a2.out2 = f1;
        VOX_TRY(run(a2));
        { float* o = x; x = f1; f1 = o; }
    }
    if (c.last_kernel_size != 3 || !final_taps<3, false>(st, x, S ? m->st_final : nullptr, sl, w.final_w, w.final_b, out, n, L, ch))
        hipLaunchKernelGGL(k_mimi_final, dim3((L + 3) / 4, n), dim3(256), 0, st, x, w.final_w, w.final_b, out, L, ch, c.last_kernel_size,
                           S ? m->st_final : nullptr, sl);
    if (S) {
        if (job.state) state_update(st, job.state, sl, job.x, n, job.L, job.P, job.C);
        state_update(st, m->st_final, sl, x, n, L, c.last_kernel_size - 1, ch);
    }
    return VOX_OK;
}

extern "C" {

int vox_mimi_decode(vox_mimi* m, void* stream, const int32_t* codes, int code_stride, int n, int T, float* out) {
    if (!m || !codes || !out) return vox_fail(VOX_ERR_INVALID, "mimi_decode: NULL");
    if (n < 1 || n > m->max_batch || T < 1 || T > m->max_frames) return vox_fail(VOX_ERR_INVALID, "mimi_decode: n=%d T=%d out of range", n, T);
    return mimi_run(m, (hipStream_t)stream, codes, code_stride, nullptr, n, T, out);
}

int vox_mimi_stream_enable(vox_mimi* m, int max_slots) {
    if (!m || max_slots < 1 || m->max_slots) return vox_fail(VOX_ERR_INVALID, "mimi_stream_enable: bad argument or already enabled");
    const vox_mimi_config& c = m->cfg;
    if (c.kernel_size - 1 > 8 || c.last_kernel_size < 2) return vox_fail(VOX_ERR_INVALID, "mimi_stream_enable: unsupported kernel sizes");
    const size_t S = max_slots, C = c.dim;
    m->ring_cap = c.context + 2 * m->max_frames;           // >= context + L - 1
    bool ok = hipMalloc((void**)&m->st_up, S * C * 4) == hipSuccess && hipMalloc((void**)&m->st_dec0, S * (c.kernel_size - 1) * C * 6) == hipSuccess &&
              hipMalloc((void**)&m->kring, (size_t)c.num_layers * S * m->ring_cap * C * 4) == hipSuccess &&
              hipMalloc((void**)&m->vring, (size_t)c.num_layers * S * m->ring_cap * C * 4) == hipSuccess &&
              hipMalloc((void**)&m->pos, S * sizeof(long)) == hipSuccess;
    size_t ch = (size_t)16 * c.n_filters;
    for (int b = 0; ok && b < 4; ++b) {
        ok = hipMalloc((void**)&m->st_tc[b], S * ch * 6) == hipSuccess && hipMalloc((void**)&m->st_c1[b], S * 2 * (ch / 2) * 6) == hipSuccess;
        ch /= 2;
    }
    ok = ok && hipMalloc((void**)&m->st_final, S * (c.last_kernel_size - 1) * ch * 4) == hipSuccess;
    if (!ok) return vox_fail(VOX_ERR_NOMEM, "mimi_stream_enable: hipMalloc failed");
    m->max_slots = max_slots;
    for (int sl = 0; sl < max_slots; ++sl) VOX_TRY(vox_mimi_reset_slot(m, nullptr, sl));
    VOX_HIP(hipDeviceSynchronize());
    return VOX_OK;
}

int vox_mimi_reset_slot(vox_mimi* m, void* stream, int slot) {
    if (!m || slot < 0 || slot >= m->max_slots) return vox_fail(VOX_ERR_INVALID, "mimi_reset_slot: slot %d out of range", slot);
    hipStream_t st = (hipStream_t)stream;
    const vox_mimi_config& c = m->cfg;
    const size_t C = c.dim;
    VOX_HIP(hipMemsetAsync(m->st_up + (size_t)slot * C, 0, C * 4, st));
    const auto zero6 = [&](float* p, size_t elems) { return hipMemsetAsync(reinterpret_cast<char*>(p) + (size_t)slot * elems * 6, 0, elems * 6, st); };      // (S3 rows)
    VOX_HIP(zero6(m->st_dec0, (c.kernel_size - 1) * C));
    size_t ch = (size_t)16 * c.n_filters;
    for (int b = 0; b < 4; ++b) {
        VOX_HIP(zero6(m->st_tc[b], ch));
        VOX_HIP(zero6(m->st_c1[b], 2 * (ch / 2)));
        ch /= 2;
    }
    VOX_HIP(hipMemsetAsync(m->st_final + (size_t)slot * (c.last_kernel_size - 1) * ch, 0, (c.last_kernel_size - 1) * ch * 4, st));
    VOX_HIP(hipMemsetAsync(m->pos + slot, 0, sizeof(long), st));     // (the K/V ring needs no clearing: only positions < pos are read)
    return VOX_OK;
}

int vox_mimi_decode_chunk(vox_mimi* m, void* stream, const int32_t* codes, int code_stride, const int32_t* slots, int n, int T, float* out) {
    if (!m || !codes || !out || !slots) return vox_fail(VOX_ERR_INVALID, "mimi_decode_chunk: NULL");
    if (!m->max_slots) return vox_fail(VOX_ERR_INVALID, "mimi_decode_chunk: call vox_mimi_stream_enable first");
    if (n < 1 || n > m->max_batch || T < 1 || T > m->max_frames) return vox_fail(VOX_ERR_INVALID, "mimi_decode_chunk: n=%d T=%d out of range", n, T);
    return mimi_run(m, (hipStream_t)stream, codes, code_stride, slots, n, T, out);
}

}  // extern "C"


// ====================================================================================================================
// SNAC decoder (Orpheus): SNAC.decode of /root/reference/vox_serve/tokenizer/snac.py:438-441, stateless per window.
// Layout as above (fp32, time-major rows).  A transposed conv with stride r, kernel 2r, padding r/2 is the 2-tap GEMM
//   G[q][j*Cout + co] = x[q] . W[:, co, j] + x[q-1] . W[:, co, j + r],   q = 0..Tin  (x[-1] = x[Tin] = 0),
// and the conv's output row o is row o + r/2 of G seen as [(Tin + 1) * r][Cout].  Instead of copying, every later kernel
// of the block works on that padded block (Lb = (Tin + 1) r rows per request, valid rows [v0, v0 + Lv)): the 1x1 GEMMs run
// on all rows (rows never mix), the depthwise convs read zeros outside the valid range, and the next block's Snake
// compacts the valid rows again (plus the zero row x[Tin]).
// ====================================================================================================================
struct SnacGeo { int B, Lb, v0, Lv, C; };

__device__ __forceinline__ float snake_a(float v, float alpha, float invb) { return snake_f(v, alpha, invb); }

// z[b][t][c] = sum_i tab_i[code_i[b][t / stride_i]][c]  (sequential in i; from_codes: snac.py:350-357)
__global__ __launch_bounds__(256) void k_snac_embed(const int* codes, int code_row, const float* t0, const float* t1, const float* t2,
                                                     const float* t3, int n_levels, int s0, int s1, int s2, int s3, int bins, int T,
                                                     int C, float* z) {
    const int b = blockIdx.z, t = blockIdx.y;
    const float* tabs[4] = {t0, t1, t2, t3};
    const int st[4] = {s0, s1, s2, s3};
    const int* cr = codes + (size_t)b * code_row;
    int id[4], off = 0;
    for (int i = 0; i < n_levels; ++i) {
        int v = cr[off + t / st[i]];
        id[i] = v < 0 ? 0 : (v >= bins ? bins - 1 : v);
        off += T / st[i];
    }
    for (int c = blockIdx.x * 256 + threadIdx.x; c < C; c += gridDim.x * 256) {
        float acc = tabs[0][(size_t)id[0] * C + c];
        for (int i = 1; i < n_levels; ++i) acc = acc + tabs[i][(size_t)id[i] * C + c];
        z[((size_t)b * T + t) * C + c] = acc;
    }
}

// depthwise conv k = 7, dilation d, "same" zero padding inside the valid rows, optional Snake on the input taps and on
// the output:  y[t][c] = post( bias[c] + sum_j w[c][j] * pre(x[t + (j - 3) d][c]) )      (ResidualUnit: snac.py:160-176)
__global__ __launch_bounds__(256) void k_snac_dw(const float* x, const float* w, const float* bias, const float* pa, const float* pib,
                                                  const float* qa, const float* qib, float* y, SnacGeo g, int dil) {
    const size_t total = (size_t)g.B * g.Lb * g.C;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % g.C);
        const size_t row = i / g.C;
        const int t = (int)(row % g.Lb) - g.v0;
        float v = 0.0f;
        if (t >= 0 && t < g.Lv) {
            const float a = pa ? pa[c] : 0.0f, ib = pa ? pib[c] : 0.0f;
            v = bias[c];
#pragma unroll
            for (int j = 0; j < 7; ++j) {
                const int tt = t + (j - 3) * dil;
                if (tt >= 0 && tt < g.Lv) {
                    float xv = x[(row + (size_t)((j - 3) * dil)) * g.C + c];
                    if (pa) xv = snake_a(xv, a, ib);
                    v = fmaf(w[c * 7 + j], xv, v);
                }
            }
            if (qa) v = snake_a(v, qa[c], qib[c]);
        }
        y[i] = v;
    }
}

// Snake of the valid rows -> compact [B][Lv + 1][C] with a trailing zero row (the x[Tin] = 0 of the transposed conv)
__global__ __launch_bounds__(256) void k_snac_snake_pack(const float* x, const float* alpha, const float* invb, float* y, SnacGeo g) {
    const size_t total = (size_t)g.B * (g.Lv + 1) * g.C;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % g.C);
        const size_t row = i / g.C;
        const int b = (int)(row / (g.Lv + 1)), t = (int)(row % (g.Lv + 1));
        y[i] = t < g.Lv ? snake_a(x[((size_t)b * g.Lb + g.v0 + t) * g.C + c], alpha[c], invb[c]) : 0.0f;
    }
}

__device__ __forceinline__ void philox4(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1, uint32_t* o0,
                                        uint32_t* o1) {
#pragma unroll
    for (int i = 0; i < 10; ++i) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0, n1 = (uint32_t)p1, n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1, n3 = (uint32_t)p0;
        c0 = n0; c1 = n1; c2 = n2; c3 = n3;
        k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
    }
    *o0 = c0; *o1 = c1;
}
// per-row NoiseBlock multiplier in the padded geometry (junk rows 0): given noise [B][Lv] or the seeded Philox stream
__global__ __launch_bounds__(256) void k_snac_noise(const float* noise, uint64_t seed, const uint32_t* stream_base, int stage, int n_stages,
                                                     float* rs, SnacGeo g) {
    const size_t total = (size_t)g.B * g.Lb;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int b = (int)(i / g.Lb), t = (int)(i % g.Lb) - g.v0;
        float v = 0.0f;
        if (t >= 0 && t < g.Lv) {
            if (noise) v = noise[(size_t)b * g.Lv + t];
            else {
                const uint32_t stream = (stream_base ? stream_base[b] : (uint32_t)(b * n_stages)) + (uint32_t)stage;
                uint32_t w0, w1;
                philox4((uint32_t)t, stream, 0u, 0u, (uint32_t)seed, (uint32_t)(seed >> 32), &w0, &w1);
                const float u1 = ((float)(w0 >> 8) + 1.0f) * (1.0f / 16777216.0f), u2 = (float)(w1 >> 8) * (1.0f / 16777216.0f);
                v = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
            }
        }
        rs[i] = v;
    }
}

// final Snake -> conv k7 (C -> 1) -> tanh, samples [out_off, out_off + out_len) of the valid rows; one wave per sample
__global__ __launch_bounds__(256) void k_snac_final(const float* x, const float* alpha, const float* invb, const float* w, float bias,
                                                     float* out, SnacGeo g, int out_off, int out_len) {
    const int lane = threadIdx.x & 63;
    const size_t s = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (s >= (size_t)g.B * out_len) return;
    const int b = (int)(s / out_len), t = out_off + (int)(s % out_len);
    float acc = 0.0f;
    for (int c = lane; c < g.C; c += 64) {
        const float a = alpha[c], ib = invb[c];
#pragma unroll
        for (int j = 0; j < 7; ++j) {
            const int tt = t + j - 3;
            if (tt >= 0 && tt < g.Lv) acc = fmaf(w[c * 7 + j], snake_a(x[((size_t)b * g.Lb + g.v0 + tt) * g.C + c], a, ib), acc);
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) out[s] = tanhf(acc + bias);
}

// Snake of the valid rows, zeros elsewhere (same padded geometry): the input of a DENSE k7 conv, whose taps must read zeros
// outside the sequence                                                                        (ResidualUnit with groups = 1)
__global__ __launch_bounds__(256) void k_snac_snake_mask(const float* x, const float* alpha, const float* invb, float* y, SnacGeo g) {
    const size_t total = (size_t)g.B * g.Lb * g.C;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % g.C);
        const int t = (int)((i / g.C) % g.Lb) - g.v0;
        y[i] = (t >= 0 && t < g.Lv) ? snake_a(x[i], alpha[c], invb[c]) : 0.0f;
    }
}

// LocalMHA core (snac.py:33-47, 76-90): one block per (window, head, request).  qkv rows [T][3C] (q | k | v, heads of 64 inside
// each), window = ws consecutive frames; q and k get the rotary embedding of their position INSIDE the window (no xpos: scale 1),
// full (non-causal) softmax over the window, scale 1/8.  out rows [T][C].
__global__ __launch_bounds__(256) void k_snac_local_attn(const float* qkv, float* out, int T, int C, int ws) {
    constexpr int DH = 64;
    __shared__ float q[32 * DH], k[32 * DH], v[32 * DH], sc[32 * 65];      // ws <= 32 (vox_snac_create)
    const int w = blockIdx.x, h = blockIdx.y, b = blockIdx.z, tid = threadIdx.x;
    const float* base = qkv + ((size_t)b * T + (size_t)w * ws) * 3 * C + h * DH;
    for (int e = tid; e < ws * DH; e += 256) {
        const int n = e / DH, d = e % DH, dp = d < DH / 2 ? d + DH / 2 : d - DH / 2;
        const float* row = base + (size_t)n * 3 * C;
        const float inv_freq = 1.0f / powf(10000.0f, (float)(2 * (d % (DH / 2))) / (float)DH);
        const float fr = (float)n * inv_freq, cs = cosf(fr), sn = sinf(fr);
        const float sgn = d < DH / 2 ? -1.0f : 1.0f;                      // rotate_half: (-x2, x1)
        q[e] = row[d] * cs + sgn * row[dp] * sn;
        k[e] = row[C + d] * cs + sgn * row[C + dp] * sn;
        v[e] = row[2 * C + d];
    }
    __syncthreads();
    for (int e = tid; e < ws * ws; e += 256) {
        const int i = e / ws, j = e % ws;
        float s = 0.0f;
        for (int d = 0; d < DH; ++d) s = fmaf(q[i * DH + d], k[j * DH + d], s);
        sc[i * 65 + j] = s * 0.125f;
    }
    __syncthreads();
    if (tid < ws) {
        float mx = -INFINITY, l = 0.0f;
        for (int j = 0; j < ws; ++j) mx = fmaxf(mx, sc[tid * 65 + j]);
        for (int j = 0; j < ws; ++j) { const float p = expf(sc[tid * 65 + j] - mx); sc[tid * 65 + j] = p; l += p; }
        const float il = 1.0f / l;
        for (int j = 0; j < ws; ++j) sc[tid * 65 + j] *= il;
    }
    __syncthreads();
    for (int e = tid; e < ws * DH; e += 256) {
        const int i = e / DH, d = e % DH;
        float o = 0.0f;
        for (int j = 0; j < ws; ++j) o = fmaf(sc[i * 65 + j], v[j * DH + d], o);
        out[((size_t)b * T + (size_t)w * ws + i) * C + h * DH + d] = o;
    }
}

struct vox_snac {
    vox_ctx* ctx;
    vox_snac_config cfg;
    vox_snac_weights w;
    int max_batch, max_T, n_stages;
    float *buf[4], *rs;
    size_t buf_floats;
};

static inline int ew_grid(size_t total) {
    size_t g = (total + 255) / 256;
    return (int)(g > 8192 ? 8192 : (g < 1 ? 1 : g));
}

extern "C" {

int vox_snac_create(vox_ctx* ctx, const vox_snac_config* cfg, const vox_snac_weights* w, int max_batch, int max_T, vox_snac** out) {
    if (!ctx || !cfg || !w || !out) return vox_fail(VOX_ERR_INVALID, "snac_create: NULL");
    if (cfg->n_levels < 1 || cfg->n_levels > 4 || max_batch < 1 || max_T < 1) return vox_fail(VOX_ERR_INVALID, "snac_create: bad config");
    vox_snac* m = new vox_snac();
    m->ctx = ctx; m->cfg = *cfg; m->w = *w; m->max_batch = max_batch; m->max_T = max_T;
    m->n_stages = 0;
    int ch = cfg->decoder_dim;
    if (cfg->attn_window < 0 || cfg->attn_window > 32 || (cfg->attn_window && cfg->decoder_dim % 64))
        return vox_fail(VOX_ERR_INVALID, "snac_create: attention window 1..32, decoder_dim a multiple of 64");
    size_t worst = (size_t)max_T * (cfg->latent_dim > cfg->decoder_dim ? cfg->latent_dim : cfg->decoder_dim) * (cfg->attn_window ? 3 : 1);
    size_t T = max_T, rs_rows = 0;
    for (int i = 0; i < 4 && cfg->rates[i] > 0; ++i) {
        const int r = cfg->rates[i];
        if (r % 2 || ch % 2) { delete m; return vox_fail(VOX_ERR_INVALID, "snac_create: rates must be even"); }
        const size_t Lb = (T + 1) * r;
        if (Lb * (ch / 2) > worst) worst = Lb * (ch / 2);
        if ((T + 1) * ch > worst) worst = (T + 1) * ch;
        if (Lb > rs_rows) rs_rows = Lb;
        T *= r; ch /= 2;
        ++m->n_stages;
    }
    m->buf_floats = worst * max_batch;
    bool ok = hipMalloc((void**)&m->rs, rs_rows * max_batch * 4) == hipSuccess;
    for (int i = 0; i < 4; ++i) ok = ok && hipMalloc((void**)&m->buf[i], m->buf_floats * 4) == hipSuccess;
    if (!ok) { vox_snac_destroy(m); return vox_fail(VOX_ERR_NOMEM, "snac_create: hipMalloc failed"); }
    *out = m;
    return VOX_OK;
}

void vox_snac_destroy(vox_snac* m) {
    if (!m) return;
    for (int i = 0; i < 4; ++i) (void)hipFree(m->buf[i]);
    (void)hipFree(m->rs);
    delete m;
}

int vox_snac_decode(vox_snac* m, void* stream, const int32_t* codes, int n, int T, const float* noise, uint64_t seed,
                    const uint32_t* stream_base, float* out, int out_off, int out_len) {
    if (!m || !codes || !out) return vox_fail(VOX_ERR_INVALID, "snac_decode: NULL");
    const vox_snac_config& c = m->cfg;
    if (n < 1 || n > m->max_batch || T < 1 || T > m->max_T || T % c.vq_strides[0])
        return vox_fail(VOX_ERR_INVALID, "snac_decode: n %d / T %d out of range", n, T);
    hipStream_t st = (hipStream_t)stream;
    int code_row = 0;
    for (int i = 0; i < c.n_levels; ++i) code_row += T / c.vq_strides[i];
    float *x = m->buf[0], *y = m->buf[1], *u = m->buf[2], *pk = m->buf[3];
    const vox_snac_weights& w = m->w;
    // latent: from_codes -> depthwise k7 -> 1x1
    hipLaunchKernelGGL(k_snac_embed, dim3((c.latent_dim + 255) / 256, T, n), dim3(256), 0, st, codes, code_row, w.tab[0], w.tab[1], w.tab[2],
                       w.tab[3], c.n_levels, c.vq_strides[0], c.vq_strides[1] ? c.vq_strides[1] : 1, c.vq_strides[2] ? c.vq_strides[2] : 1,
                       c.vq_strides[3] ? c.vq_strides[3] : 1, c.codebook_size, T, c.latent_dim, x);
    SnacGeo g{n, T, 0, T, c.latent_dim};
    static const int off1[8] = {0, 0, 0, 0, 0, 0, 0, 0}, off2[8] = {0, 1, 0, 1, 0, 0, 0, 0};
    if (w.conv0.n_taps > 0) {      // non-depthwise: one dense k7 conv ("same" padding: tap j reads row t + j - 3), 2 weight planes
        static const int off7[14] = {3, 2, 1, 0, -1, -2, -3, 3, 2, 1, 0, -1, -2, -3};
        VOX_TRY(conv_gemm(st, w.conv0, x, nullptr, nullptr, n, T, 0, off7, y, nullptr, nullptr, 0));
        float* t = x; x = y; y = t;
    } else {
        hipLaunchKernelGGL(k_snac_dw, dim3(ew_grid((size_t)n * T * c.latent_dim)), dim3(256), 0, st, x, w.dw0_w, w.dw0_b, nullptr, nullptr,
                           nullptr, nullptr, y, g, 1);
        VOX_TRY(conv_gemm(st, w.pw0, y, nullptr, nullptr, n, T, 0, off1, x, nullptr, nullptr, 0));
    }
    g.C = c.decoder_dim;
    if (c.attn_window > 0) {       // LocalMHA: x += to_out(attention(rotary(to_qkv(LayerNorm(x)))))
        if (T % c.attn_window) return vox_fail(VOX_ERR_INVALID, "snac_decode: %d frames are not a multiple of the attention window %d", T, c.attn_window);
        hipLaunchKernelGGL(k_layernorm_f32, dim3(n * T), dim3(256), 0, st, x, w.attn_ln_w, w.attn_ln_b, y, g.C, 1e-5f);
        VOX_TRY(conv_gemm(st, w.attn_qkv, y, nullptr, nullptr, n, T, 0, off1, u, nullptr, nullptr, 0));          // u [nT][3C]
        hipLaunchKernelGGL(k_snac_local_attn, dim3(T / c.attn_window, g.C / 64, n), dim3(256), 0, st, u, y, T, g.C, c.attn_window);
        VOX_TRY(conv_gemm(st, w.attn_out, y, nullptr, nullptr, n, T, 0, off1, pk, x, nullptr, 0));                 // pk = x + out
        float* t = x; x = pk; pk = t;
    }
    size_t noise_off = 0;
    for (int bi = 0; bi < m->n_stages; ++bi) {
        const vox_snac_block_w& b = w.blocks[bi];
        const int r = c.rates[bi], cout = g.C / 2, Tin = g.Lv;
        // Snake -> compact rows + zero row; transposed conv as the 2-tap GEMM
        hipLaunchKernelGGL(k_snac_snake_pack, dim3(ew_grid((size_t)n * (Tin + 1) * g.C)), dim3(256), 0, st, x, b.snake0.alpha, b.snake0.inv_beta, pk, g);
        VOX_TRY(conv_gemm(st, b.tconv, pk, nullptr, nullptr, n, Tin + 1, 0, off2, x, nullptr, nullptr, 0));
        g = SnacGeo{n, (Tin + 1) * r, r / 2, Tin * r, cout};
        if (b.noise.n_taps > 0) {
            hipLaunchKernelGGL(k_snac_noise, dim3(ew_grid((size_t)n * g.Lb)), dim3(256), 0, st, noise ? noise + noise_off : nullptr, seed, stream_base, bi,
                               m->n_stages, m->rs, g);
            VOX_TRY(conv_gemm(st, b.noise, x, nullptr, nullptr, n, g.Lb, 0, off1, y, x, nullptr, 0, nullptr, nullptr, 0, m->rs));
            float* t = x; x = y; y = t;
            noise_off += (size_t)n * g.Lv;
        }
        static const int dils[3] = {1, 3, 9};
        for (int k = 0; k < 3; ++k) {
            const vox_snac_res_w& ru = b.res[k];
            if (ru.dense.n_taps > 0) {      // dense k7 conv: masked Snake -> 7-tap GEMM (taps read zeros outside the valid rows) with act2 fused
                const int d = dils[k];
                const int offd[14] = {3 * d, 2 * d, d, 0, -d, -2 * d, -3 * d, 3 * d, 2 * d, d, 0, -d, -2 * d, -3 * d};
                hipLaunchKernelGGL(k_snac_snake_mask, dim3(ew_grid((size_t)n * g.Lb * g.C)), dim3(256), 0, st, x, ru.act1.alpha, ru.act1.inv_beta, pk, g);
                VOX_TRY(conv_gemm(st, ru.dense, pk, nullptr, nullptr, n, g.Lb, 0, offd, nullptr, nullptr, nullptr, 0, u, &ru.act2, g.C));
            } else {
                hipLaunchKernelGGL(k_snac_dw, dim3(ew_grid((size_t)n * g.Lb * g.C)), dim3(256), 0, st, x, ru.dw_w, ru.dw_b, ru.act1.alpha, ru.act1.inv_beta,
                                   ru.act2.alpha, ru.act2.inv_beta, u, g, dils[k]);
            }
            VOX_TRY(conv_gemm(st, ru.pw, u, nullptr, nullptr, n, g.Lb, 0, off1, y, x, nullptr, 0));
            float* t = x; x = y; y = t;
        }
    }
    const int total_len = g.Lv;
    if (out_off < 0 || out_len < 1 || out_off + out_len > total_len) return vox_fail(VOX_ERR_INVALID, "snac_decode: output window out of range");
    hipLaunchKernelGGL(k_snac_final, dim3(((size_t)n * out_len + 3) / 4), dim3(256), 0, st, x, w.final_snake.alpha, w.final_snake.inv_beta, w.final_w,
                       w.final_b, out, g, out_off, out_len);
    return VOX_OK;
}

}  // extern "C"

// ====================================================================================================================
// HiFT vocoder (mel -> waveform; CosyVoice2 / GLM-4-Voice detokenizers).  See include/voxhip.h for the contract.
// Layout: fp32 time-major [request][t][C].  Every conv / transposed conv runs on conv_gemm (look-ahead taps, two weight planes);
// the harmonic source, the 16-point STFT / iSTFT and the strided source convs (Cin = 18) are direct kernels.
// ====================================================================================================================
// mel [n][Cm][T] -> x [n*T][Cp] (channels >= Cm zero)
__global__ __launch_bounds__(256) void k_hift_mel_in(const float* mel, float* x, int n, int Cm, int Cp, int T) {
    const size_t total = (size_t)n * T * Cp;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % Cp);
        const size_t row = i / Cp;
        const int b = (int)(row / T), t = (int)(row % T);
        x[i] = c < Cm ? mel[((size_t)b * Cm + c) * T + t] : 0.0f;
    }
}
// f0[row] = |w . x[row] + b|: one wave per row (hifigan.py:423-426)
__global__ __launch_bounds__(256) void k_hift_f0cls(const float* x, const float* w, float bias, float* f0, int rows, int C) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    float s = 0.0f;
    for (int c = lane; c < C; c += 64) s = fmaf(x[(size_t)row * C + c], w[c], s);
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) f0[row] = fabsf(s + bias);
}
// phase at the frame rate (hifigan.py:296-313): rad = (f0 h / sr) mod 1 (what the 1/scale linear resampling of the sample-rate
// track returns exactly), cumulative sum over the frames (accumulated in double like torch.cumsum on the CPU), * 2 * pi * scale
__global__ void k_hift_phase(const float* f0, float* ph, int n, int T, int H1, float sr, float scale) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * H1) return;
    const int b = i / H1, h = i % H1;
    double cum = 0.0;
    for (int t = 0; t < T; ++t) {
        const float fn = f0[(size_t)b * T + t] * (float)(h + 1);
        float r = fn / sr;
        r = r - floorf(r);
        cum += (double)r;
        ph[((size_t)b * T + t) * H1 + h] = (((float)cum * 2.0f) * 3.14159274101257324f) * scale;
    }
}
// merged harmonic source s[b][l] (hifigan.py:314-316, 334-343, 386-388): linear interpolation of the frame-rate phase back to the
// sample rate (torch upsample_linear1d, align_corners = False), sin, voiced / unvoiced noise, tanh(linear)
__global__ __launch_bounds__(256) void k_hift_source(const float* f0, const float* ph, const float* noise, uint64_t seed,
                                                      const uint32_t* stream_base, const float* lw, float lb, float* s, int n, int T,
                                                      int H1, int scale, float rscale, float alpha, float sigma, float vth) {
    const size_t L = (size_t)T * scale, total = (size_t)n * L;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int b = (int)(i / L);
        const size_t l = i % L;
        const float uv = f0[(size_t)b * T + l / scale] > vth ? 1.0f : 0.0f;
        const float amp = uv * sigma + (1.0f - uv) * alpha / 3.0f;
        float src = rscale * ((float)l + 0.5f) - 0.5f;
        src = src < 0.0f ? 0.0f : src;
        const int i0 = (int)src, i1 = i0 + (i0 < T - 1 ? 1 : 0);
        float l1 = src - (float)i0;
        l1 = l1 < 0.0f ? 0.0f : (l1 > 1.0f ? 1.0f : l1);
        const float l0 = 1.0f - l1;
        const uint32_t stream = stream_base ? stream_base[b] + 1u : (uint32_t)(2 * b + 1);
        float acc = 0.0f;
        for (int h = 0; h < H1; ++h) {
            const float p = l0 * ph[((size_t)b * T + i0) * H1 + h] + l1 * ph[((size_t)b * T + i1) * H1 + h];
            float nz;
            if (noise) nz = noise[i * H1 + h];
            else {
                uint32_t w0, w1;
                philox4((uint32_t)(l * H1 + h), stream, 0u, 0u, (uint32_t)seed, (uint32_t)(seed >> 32), &w0, &w1);
                const float u1 = ((float)(w0 >> 8) + 1.0f) * (1.0f / 16777216.0f), u2 = (float)(w1 >> 8) * (1.0f / 16777216.0f);
                nz = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
            }
            const float sw = (sinf(p) * alpha) * uv + amp * nz;
            acc = fmaf(sw, lw[h], acc);
        }
        s[i] = tanhf(acc + lb);
    }
}
// SineGen v1 (GLM-4-Voice's vocoder, tokenizer/glm.py:2298-2316): theta[b][l][h] = 2 pi ((cumulative sum over samples of f0 (h+1) / sr) mod 1),
// the sum accumulated in double like torch.cumsum on the CPU.  f0 is constant over the `scale` samples of a frame, so the running sum at
// sample q of frame t is start[t] + (q + 1) F_t with F_t = fl(fl(f0 (h+1)) / sr): the per-sample additions of the serial form are exact in
// double whenever F's last bit is above the sum's ulp (24-bit F >= 2^-18 against sums < 2^14: every voiced frame), so the closed form has
// the serial sum's bits; this kernel walks the T frames per (request, harmonic) — 172 dependent additions instead of 44 032 — and
// k_hift_source_v1 evaluates the phase of each sample from start[t].
__global__ void k_hift_theta_v1(const float* f0, double* start, int n, int T, int H1, int scale, float sr) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * H1) return;
    const int b = i / H1, h = i % H1;
    double cum = 0.0;
    for (int t = 0; t < T; ++t) {
        const float F = (f0[(size_t)b * T + t] * (float)(h + 1)) / sr;
        start[((size_t)b * H1 + h) * T + t] = cum;
        cum += (double)F * (double)scale;
    }
}
// merged source for SineGen v1: sin(theta + initial phase), voiced / unvoiced noise, tanh(linear).  Initial phases: -pi + 2 pi u with u
// given (rand_ini [n][H1], column 0 ignored) or word 0 of the seeded uniform stream stream_base[b] (element h); phase of the fundamental = 0
__global__ __launch_bounds__(256) void k_hift_source_v1(const float* f0, const double* start, float sr, const float* rand_ini, const float* noise, uint64_t seed,
                                                         const uint32_t* stream_base, const float* lw, float lb, float* s, int n, int T, int H1,
                                                         int scale, float alpha, float sigma, float vth) {
    const size_t L = (size_t)T * scale, total = (size_t)n * L;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int b = (int)(i / L);
        const size_t l = i % L;
        const int tf = (int)(l / scale), qf = (int)(l - (size_t)tf * scale);
        const float f0v = f0[(size_t)b * T + tf];
        const float uv = f0v > vth ? 1.0f : 0.0f;
        const float amp = uv * sigma + (1.0f - uv) * alpha / 3.0f;
        const uint32_t sb = stream_base ? stream_base[b] : (uint32_t)(2 * b);
        float acc = 0.0f;
        for (int h = 0; h < H1; ++h) {
            const float F = (f0v * (float)(h + 1)) / sr;
            const float cv = (float)(start[((size_t)b * H1 + h) * T + tf] + (double)F * (double)(qf + 1));
            const float theta = 6.28318548202514648f * (cv - floorf(cv));
            float ph = 0.0f;
            if (h > 0) {
                float u;
                if (rand_ini) u = rand_ini[(size_t)b * H1 + h];
                else {
                    uint32_t w0, w1;
                    philox4((uint32_t)h, sb, 0u, 0u, (uint32_t)seed, (uint32_t)(seed >> 32), &w0, &w1);
                    u = (float)(w0 >> 8) * (1.0f / 16777216.0f);
                }
                ph = -3.14159274101257324f + 6.28318548202514648f * u;
            }
            float nz;
            if (noise) nz = noise[i * H1 + h];
            else {
                uint32_t w0, w1;
                philox4((uint32_t)(l * H1 + h), sb + 1u, 0u, 0u, (uint32_t)seed, (uint32_t)(seed >> 32), &w0, &w1);
                const float u1 = ((float)(w0 >> 8) + 1.0f) * (1.0f / 16777216.0f), u2 = (float)(w1 >> 8) * (1.0f / 16777216.0f);
                nz = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
            }
            const float sw = (alpha * sinf(theta + ph)) * uv + amp * nz;
            acc = fmaf(sw, lw[h], acc);
        }
        s[i] = tanhf(acc + lb);
    }
}
// STFT of the source (torch.stft: n_fft 16, hop 4, periodic Hann, center = True with reflect padding): S[b][f][k] real rows
// 0..nb-1, imaginary rows nb..2nb-1; one thread per (b, frame, bin)
__global__ __launch_bounds__(256) void k_hift_stft(const float* s, float* S, int n, int L, int F, int nfft, int hop) {
    const int nb = nfft / 2 + 1;
    const size_t total = (size_t)n * F * nb;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int k = (int)(i % nb);
        const size_t bf = i / nb;
        const int b = (int)(bf / F), f = (int)(bf % F);
        float re = 0.0f, im = 0.0f;
        for (int j = 0; j < nfft; ++j) {
            int q = f * hop + j - nfft / 2;
            q = q < 0 ? -q : (q >= L ? 2 * (L - 1) - q : q);
            const float win = 0.5f - 0.5f * cospif(2.0f * (float)j / (float)nfft);
            const float v = s[(size_t)b * L + q] * win;
            const float ang = 2.0f * (float)((k * j) % nfft) / (float)nfft;      // in units of pi
            re = fmaf(v, cospif(ang), re);
            im = fmaf(-v, sinpif(ang), im);
        }
        S[bf * (2 * nb) + k] = re;
        S[bf * (2 * nb) + nb + k] = im;
    }
}
// source_downs[i]: strided conv over the STFT frames, Cin = 2 nb (hifigan.py:497-510): out[b][t][co]
__global__ __launch_bounds__(256) void k_hift_sd(const float* S, const float* wt, const float* bias, float* out, int n, int F, int Cin,
                                                  int Lo, int Cout, int k, int stride, int pad) {
    // wt = the weight transposed to [k][Cin][Cout] at creation: consecutive threads (output channels of one row) read consecutive
    // floats, the spectrum value is the same address for the whole row (the [Cout][Cin][k] original had every lane 4 k Cin bytes apart);
    // the accumulation order (tap, then input channel) is the original's
    const size_t total = (size_t)n * Lo * Cout;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int co = (int)(i % Cout);
        const size_t row = i / Cout;
        const int b = (int)(row / Lo), t = (int)(row % Lo);
        float acc = bias[co];
        for (int j = 0; j < k; ++j) {
            const int f = t * stride - pad + j;
            if (f < 0 || f >= F) continue;
            const float* sr = S + ((size_t)b * F + f) * Cin;
            const float* wr = wt + (size_t)j * Cin * Cout + co;
#pragma unroll 6
            for (int ci = 0; ci < Cin; ++ci) acc = fmaf(sr[ci], wr[(size_t)ci * Cout], acc);
        }
        out[i] = acc;
    }
}
// [Cout][Cin][k] -> [k][Cin][Cout]
__global__ __launch_bounds__(256) void k_hift_sd_transpose(const float* w, float* wt, int Cout, int Cin, int k) {
    const size_t total = (size_t)Cout * Cin * k;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int co = (int)(i % Cout), ci = (int)((i / Cout) % Cin), j = (int)(i / ((size_t)Cout * Cin));
        wt[i] = w[((size_t)co * Cin + ci) * k + j];
    }
}
// x = pad(y) + si (ReflectionPad1d((1, 0)) on the last stage: row 0 = row 1 of y) and the first Snake of the three resblocks
__global__ __launch_bounds__(256) void k_hift_add_snake3(const float* y, const float* si, float* x, float* a0, float* a1, float* a2,
                                                          const float* al0, const float* ib0, const float* al1, const float* ib1,
                                                          const float* al2, const float* ib2, int n, int Ly, int Lx, int C) {
    const size_t total = (size_t)n * Lx * C;
    const int padl = Lx - Ly;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % C);
        const size_t row = i / C;
        const int b = (int)(row / Lx), t = (int)(row % Lx);
        int ty = t - padl;
        ty = ty < 0 ? -ty : ty;
        const float v = y[((size_t)b * Ly + ty) * C + c] + si[i];
        x[i] = v;
        float s_;
        s_ = sinf(v * al0[c]); put_row(a0, row, C, c, v + ib0[c] * (s_ * s_), 3);
        if (a1) { s_ = sinf(v * al1[c]); put_row(a1, row, C, c, v + ib1[c] * (s_ * s_), 3); }
        if (a2) { s_ = sinf(v * al2[c]); put_row(a2, row, C, c, v + ib2[c] * (s_ * s_), 3); }
    }
}
// x = leaky_relu(((r0 + r1) + r2) / nk, slope)   (hifigan.py:613-621; r1 / r2 NULL when fewer kernels)
__global__ __launch_bounds__(256) void k_hift_avg_lrelu(const float* r0, const float* r1, const float* r2, float* x, size_t total, float nk,
                                                         float slope, int C, int terms) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        float v = r0[i];
        if (r1) v = v + r1[i];
        if (r2) v = v + r2[i];
        if (nk != 1.0f) v = v / nk;
        put_row(x, i / C, C, (int)(i % C), v > 0.0f ? v : v * slope, terms);
    }
}
// magnitude / phase heads -> irfft per frame -> window -> overlap-add / window^2 -> trim n_fft/2 -> clamp  (hifigan.py:554-594, 623-628)
// one thread per output sample; P[b][f][0..nb-1] = log-magnitude rows, [nb..2nb-1] = phase rows
__global__ __launch_bounds__(256) void k_hift_istft(const float* P, float* wav, int n, int F, int nfft, int hop, int Lout, float limit) {
    const int nb = nfft / 2 + 1;
    const size_t total = (size_t)n * Lout;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int b = (int)(i / Lout), l = (int)(i % Lout);
        const int q = l + nfft / 2;                        // position in the untrimmed signal
        float acc = 0.0f, den = 0.0f;
        int f_hi = q / hop;
        f_hi = f_hi > F - 1 ? F - 1 : f_hi;
        int f_lo = (q - nfft) / hop + 1;
        f_lo = (q - nfft) < 0 ? 0 : f_lo;
        for (int f = f_lo; f <= f_hi; ++f) {               // ascending frame order, like F.fold's accumulation
            const int j = q - f * hop;
            if (j < 0 || j >= nfft) continue;
            const float* pf = P + ((size_t)b * F + f) * (2 * nb);
            float v = 0.0f;
            for (int k = 0; k < nb; ++k) {
                float mag = expf(pf[k]);
                mag = mag > 1e2f ? 1e2f : mag;
                const float ph = sinf(pf[nb + k]);
                const float re = mag * cosf(ph), im = mag * sinf(ph);
                const float ang = 2.0f * (float)((k * j) % nfft) / (float)nfft;
                if (k == 0 || k == nb - 1) v += re * cospif(ang);                       // irfft ignores the imaginary part of DC / Nyquist
                else v += 2.0f * (re * cospif(ang) - im * sinpif(ang));
            }
            const float win = 0.5f - 0.5f * cospif(2.0f * (float)j / (float)nfft);
            acc += (v / (float)nfft) * win;
            den += win * win;
        }
        den = den > 1e-8f ? den : 1.0f;
        float o = acc / den;
        o = o < -limit ? -limit : (o > limit ? limit : o);
        wav[i] = o;
    }
}

struct vox_hift {
    vox_ctx* ctx;
    vox_hift_config cfg;
    vox_hift_weights w;
    int max_batch, max_T, scale;
    float* buf[9];
    size_t buf_floats;
    float *f0, *ph, *src, *stft, *post;
    double* theta = nullptr;               // SineGen v1: running phase sum at the start of every frame [n][H1][T]
    float* sd_wt[4] = {};                  // source_downs weights as [k][n_fft + 2][Cout] (k_hift_sd)
    int sine_v1 = 0;
};

static int hift_conv_offsets(int k, int dil, int* off, int planes = 2) {   // "same" conv: tap j reads row t + (j - (k-1)/2) dil
    const int pad = (k - 1) * dil / 2;
    for (int p = 0; p < planes; ++p)
        for (int j = 0; j < k; ++j) off[p * k + j] = pad - j * dil;
    return planes * k;
}
static int hift_tconv_offsets(int k, int u, int* off) {           // ConvTranspose1d(k, stride u, padding (k-u)/2): taps d = dmin..dmax, two planes
    const int p = (k - u) / 2;
    int dmin = -((p + (u - 1)) / u), dmax = (k - 1 - p) / u;
    while (dmin * u + (u - 1) + p < 0) ++dmin;
    const int nd = dmax - dmin + 1;
    for (int pl = 0; pl < 2; ++pl)
        for (int d = 0; d < nd; ++d) off[pl * nd + d] = dmin + d;
    return 2 * nd;
}

extern "C" {

void vox_hift_destroy(vox_hift* m) {
    if (!m) return;
    for (int i = 0; i < 9; ++i) (void)hipFree(m->buf[i]);
    (void)hipFree(m->f0); (void)hipFree(m->ph); (void)hipFree(m->src); (void)hipFree(m->stft); (void)hipFree(m->post); (void)hipFree(m->theta);
    for (int i = 0; i < 4; ++i) (void)hipFree(m->sd_wt[i]);
    delete m;
}

int vox_hift_create(vox_ctx* ctx, const vox_hift_config* cfg, const vox_hift_weights* w, int max_batch, int max_T, vox_hift** out) {
    if (!ctx || !cfg || !w || !out) return vox_fail(VOX_ERR_INVALID, "hift_create: NULL");
    if (cfg->n_stages < 1 || cfg->n_stages > 4 || cfg->n_kernels < 1 || cfg->n_kernels > 3 || max_batch < 1 || max_T < 1 ||
        cfg->in_channels_padded % 32 || cfg->in_channels > cfg->in_channels_padded || cfg->n_fft % 2 || cfg->nb_harmonics > 15)
        return vox_fail(VOX_ERR_INVALID, "hift_create: bad config");
    vox_hift* m = new vox_hift();
    m->ctx = ctx; m->cfg = *cfg; m->w = *w; m->max_batch = max_batch; m->max_T = max_T;
    m->scale = cfg->hop_len;
    size_t rows = max_T, worst = (size_t)max_T * cfg->base_channels;
    int ch = cfg->base_channels;
    if ((size_t)max_T * cfg->f0_channels > worst) worst = (size_t)max_T * cfg->f0_channels;
    if ((size_t)max_T * cfg->in_channels_padded > worst) worst = (size_t)max_T * cfg->in_channels_padded;
    for (int i = 0; i < cfg->n_stages; ++i) {
        if ((cfg->upsample_kernels[i] - cfg->upsample_rates[i]) < 0) { delete m; return vox_fail(VOX_ERR_INVALID, "hift_create: kernel < stride"); }
        rows *= cfg->upsample_rates[i]; ch /= 2; m->scale *= cfg->upsample_rates[i];
        if ((rows + 1) * ch > worst) worst = (rows + 1) * ch;
        if (ch % 32) { delete m; return vox_fail(VOX_ERR_INVALID, "hift_create: stage channels must be multiples of 32"); }
    }
    m->buf_floats = worst * max_batch;
    const size_t L = (size_t)max_T * m->scale, F = rows + 1;
    bool ok = true;
    for (int i = 0; i < 9; ++i) ok = ok && hipMalloc((void**)&m->buf[i], m->buf_floats * 6) == hipSuccess;      // (fp32 or S3 rows)
    ok = ok && hipMalloc((void**)&m->f0, (size_t)max_batch * max_T * 4) == hipSuccess &&
         hipMalloc((void**)&m->ph, (size_t)max_batch * max_T * (cfg->nb_harmonics + 1) * 4) == hipSuccess &&
         hipMalloc((void**)&m->src, (size_t)max_batch * L * 4) == hipSuccess &&
         hipMalloc((void**)&m->stft, (size_t)max_batch * F * (cfg->n_fft + 2) * 4) == hipSuccess &&
         hipMalloc((void**)&m->post, (size_t)max_batch * F * (cfg->n_fft + 2) * 4) == hipSuccess;
    m->sine_v1 = cfg->sine_gen_v1;
    if (m->sine_v1) ok = ok && hipMalloc((void**)&m->theta, (size_t)max_batch * max_T * (cfg->nb_harmonics + 1) * 8) == hipSuccess;
    ch = cfg->base_channels;
    for (int i = 0; i < cfg->n_stages && ok; ++i) {      // transposed source_downs weights
        int sstride = 1;
        for (int q = i + 1; q < cfg->n_stages; ++q) sstride *= cfg->upsample_rates[q];
        const int sk = sstride == 1 ? 1 : 2 * sstride, cin = cfg->n_fft + 2;
        ch /= 2;
        const size_t cnt = (size_t)ch * cin * sk;
        ok = hipMalloc((void**)&m->sd_wt[i], cnt * 4) == hipSuccess;
        if (ok) hipLaunchKernelGGL(k_hift_sd_transpose, dim3(ew_grid(cnt)), dim3(256), 0, 0, w->sd_w[i], m->sd_wt[i], ch, cin, sk);
    }
    ok = ok && hipStreamSynchronize(0) == hipSuccess;
    if (!ok) { vox_hift_destroy(m); return vox_fail(VOX_ERR_NOMEM, "hift_create: hipMalloc failed"); }
    *out = m;
    return VOX_OK;
}

// A conv with two weight planes over S3 rows.  A request's samples must not depend on how many others are decoded with it, so all tiles add
// in one order (64 channels at a time, two waves a half each): rows decide only which of them it is.  us, staged kernels before:
// 3584 rows x 256 channels, 7 taps 77 -> 22.5; 17 920 x 128 56 -> 36; 53 768 x 64 37 -> 27; one request: 448 x 256 36 -> 12, 6721 x 64 15 -> 9
static int hift_conv(hipStream_t st, ConvDmaArgs& a) {
    if (a.Cin % CG_BK || a.N % 16 || a.n_taps % 2 || a.n_taps > CG_MAXTAPS || a.bias_mod % 8)
        return vox_fail(VOX_ERR_INVALID, "hift conv: %d -> %d channels, %d taps", a.Cin, a.N, a.n_taps);
    a.n_taps /= 2;
    a.planes = 3;
    const auto tiles = [&](int bm, int bn) { return (long)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn); };
    if (a.Cin % 64) return conv_dma_launch<64, 64, 2, 2, 1, 32, 3, 3, 0, 2>(st, a);
    if (tiles(16, 32) <= 256) return conv_dma_launch<16, 32, 1, 1, 2, 64, 5, 3, 0, 2>(st, a);
    if (tiles(32, 64) <= 256) return conv_dma_launch<32, 64, 1, 2, 2, 64, 4, 3, 0, 2>(st, a);
    if (tiles(64, 64) <= 256) return conv_dma_launch<64, 64, 4, 2, 2, 64, 2, 3, 0, 2>(st, a);
    // many rows: rounds of a CU's tiles (17 920 x 128: 1120 of 32 x 64 in five small rounds; 53 768 x 64: 421 of 128 x 64 in two)
    if ((tiles(128, 64) + 255) / 256 * 4 <= (tiles(32, 64) + 255) / 256 * 1.3) return conv_dma_launch<128, 64, 4, 2, 2, 64, 2, 3, 0, 2>(st, a);
    return conv_dma_launch<32, 64, 1, 2, 2, 64, 2, 3, 0, 2>(st, a);
}

// one ResBlock (hifigan.py:134-141) on rows L per request: a = snake1_0(x) is given; result in `r` (x itself is left untouched);
// t1 scratch.  The next iteration's first Snake and this iteration's second Snake are fused into the producing conv's epilogue.
static int hift_resblock(hipStream_t st, const vox_hift_resblock_w& rb, const vox_hift_config& c, int k, const float* x, float* a, float* t1,
                         float* r, int n, int L) {
    int off1[CG_MAXTAPS], off2[CG_MAXTAPS];
    hift_conv_offsets(k, 1, off2);
    for (int j = 0; j < 3; ++j) {
        hift_conv_offsets(k, c.dilations[j], off1);
        ConvDmaArgs a1 = conv_s2_args(rb.c1[j], a, nullptr, nullptr, n, L, 0, off1), a2 = conv_s2_args(rb.c2[j], t1, nullptr, nullptr, n, L, 0, off2);
        a1.out2 = t1; a1.out2_s2 = 1; a1.sn_alpha = rb.a2[j].alpha; a1.sn_invb = rb.a2[j].inv_beta;
        a2.res = j == 0 ? x : r;
        a2.out = r;
        if (j < 2) { a2.out2 = a; a2.out2_s2 = 1; a2.sn_alpha = rb.a1[j + 1].alpha; a2.sn_invb = rb.a1[j + 1].inv_beta; }
        VOX_TRY(hift_conv(st, a1));
        VOX_TRY(hift_conv(st, a2));
    }
    return VOX_OK;
}

int vox_hift_decode(vox_hift* m, void* stream, const float* mel, int n, int T, const float* noise, uint64_t seed,
                    const uint32_t* stream_base, float* wav, float* source, const float* rand_ini) {
    if (!m || !mel || !wav) return vox_fail(VOX_ERR_INVALID, "hift_decode: NULL");
    if (n < 1 || n > m->max_batch || T < 1 || T > m->max_T) return vox_fail(VOX_ERR_INVALID, "hift_decode: n %d / T %d out of range", n, T);
    const vox_hift_config& c = m->cfg;
    const vox_hift_weights& w = m->w;
    hipStream_t st = (hipStream_t)stream;
    g_conv_planes = 3;
    g_conv_skinny_rows = 48; g_conv_rows_gemm = false;
    const int H1 = c.nb_harmonics + 1, nb2 = c.n_fft + 2;
    const size_t L = (size_t)T * m->scale;
    float** B = m->buf;
    int off[CG_MAXTAPS];
    // ---- f0 predictor: 5 x (conv k3 + ELU), linear, abs ----
    hipLaunchKernelGGL(k_hift_mel_in, dim3(ew_grid((size_t)n * T * c.in_channels_padded)), dim3(256), 0, st, mel, B[0], n, c.in_channels,
                       c.in_channels_padded, T);
    hift_conv_offsets(3, 1, off, 3);          // (three weight planes: the source's phase multiplies an f0 error by 2 pi scale T)
    {
        const float* in = B[0];
        for (int i = 0; i < 5; ++i) {
            float* o = (i & 1) ? B[2] : B[1];
            VOX_TRY(conv_gemm(st, w.f0_conv[i], in, nullptr, nullptr, n, T, 0, off, o, nullptr, nullptr, 0));
            elu(st, o, o, (size_t)n * T * c.f0_channels);
            in = o;
        }
        hipLaunchKernelGGL(k_hift_f0cls, dim3((n * T + 3) / 4), dim3(256), 0, st, in, w.f0_cls_w, w.f0_cls_b, m->f0, n * T, c.f0_channels);
    }
    // ---- harmonic source + its STFT ----
    if (m->sine_v1) {
        hipLaunchKernelGGL(k_hift_theta_v1, dim3((n * H1 + 63) / 64), dim3(64), 0, st, m->f0, m->theta, n, T, H1, m->scale, (float)c.sampling_rate);
        hipLaunchKernelGGL(k_hift_source_v1, dim3(ew_grid((size_t)n * L)), dim3(256), 0, st, m->f0, m->theta, (float)c.sampling_rate, rand_ini, noise, seed, stream_base,
                           w.src_lin_w, w.src_lin_b, m->src, n, T, H1, m->scale, c.nsf_alpha, c.nsf_sigma, c.voiced_threshold);
    } else {
        hipLaunchKernelGGL(k_hift_phase, dim3((n * H1 + 63) / 64), dim3(64), 0, st, m->f0, m->ph, n, T, H1, (float)c.sampling_rate, (float)m->scale);
        hipLaunchKernelGGL(k_hift_source, dim3(ew_grid((size_t)n * L)), dim3(256), 0, st, m->f0, m->ph, noise, seed, stream_base, w.src_lin_w,
                           w.src_lin_b, m->src, n, T, H1, m->scale, (float)(1.0 / (double)m->scale), c.nsf_alpha, c.nsf_sigma, c.voiced_threshold);
    }
    if (source) (void)hipMemcpyAsync(source, m->src, (size_t)n * L * 4, hipMemcpyDeviceToDevice, st);
    const int F = (int)(L / c.hop_len) + 1;
    hipLaunchKernelGGL(k_hift_stft, dim3(ew_grid((size_t)n * F * (c.n_fft / 2 + 1))), dim3(256), 0, st, m->src, m->stft, n, (int)L, F, c.n_fft,
                       c.hop_len);
    // ---- conv_pre ----
    hift_conv_offsets(7, 1, off);
    VOX_TRY(conv_gemm(st, w.conv_pre, B[0], nullptr, nullptr, n, T, 0, off, B[1], nullptr, nullptr, 0));
    hipLaunchKernelGGL(k_hift_avg_lrelu, dim3(ew_grid((size_t)n * T * c.base_channels)), dim3(256), 0, st, B[1], nullptr, nullptr, B[2],
                       (size_t)n * T * c.base_channels, 1.0f, c.lrelu_slope, c.base_channels, 3);
    float* cur = B[2];                     // leaky_relu'ed stage input (S3 rows; fp32 behind the last stage)
    int Lc = T, ch = c.base_channels;
    // strides of source_downs: cumulative products of the LATER stages' rates (hifigan.py:497-500)
    for (int i = 0; i < c.n_stages; ++i) {
        const int u = c.upsample_rates[i], k = c.upsample_kernels[i], cout = ch / 2;
        const bool last = i == c.n_stages - 1;
        const int Ly = Lc * u, Lx = last ? Ly + 1 : Ly;
        // pick working buffers distinct from `cur`
        float* pool[8];
        int np = 0;
        for (int q = 0; q < 9; ++q) if (B[q] != cur) pool[np++] = B[q];
        float *Y = pool[0], *S = pool[1], *A = pool[2], *T1 = pool[3], *X = pool[4], *A1 = pool[5], *A2 = pool[6], *R2 = pool[7];
        hift_tconv_offsets(k, u, off);
        { ConvDmaArgs a = conv_s2_args(w.ups[i], cur, nullptr, nullptr, n, Lc, 0, off); a.out = Y; VOX_TRY(hift_conv(st, a)); }
        int sstride = 1;
        for (int q = i + 1; q < c.n_stages; ++q) sstride *= c.upsample_rates[q];
        const int sk = sstride == 1 ? 1 : 2 * sstride, spad = sstride == 1 ? 0 : sstride / 2;
        if ((F + 2 * spad - sk) / sstride + 1 != Lx) return vox_fail(VOX_ERR_INVALID, "hift_decode: source / stage length mismatch at stage %d", i);
        hipLaunchKernelGGL(k_hift_sd, dim3(ew_grid((size_t)n * Lx * cout)), dim3(256), 0, st, m->stft, m->sd_wt[i], w.sd_b[i], S, n, F, nb2, Lx, cout,
                           sk, sstride, spad);
        // source resblock: S <- resblock(S)
        snake(st, S, w.src_rb[i].a1[0], A, (size_t)n * Lx, cout, 3);
        VOX_TRY(hift_resblock(st, w.src_rb[i], c, c.source_resblock_kernels[i], S, A, T1, X, n, Lx));       // result in X (scratch here)
        // x = pad(Y) + si, first Snakes of the stage's resblocks
        const vox_hift_resblock_w* rb = &w.rb[i * c.n_kernels];
        float* Si = X;                      // source branch output
        float* Xs = S;                      // stage tensor (S is free now)
        hipLaunchKernelGGL(k_hift_add_snake3, dim3(ew_grid((size_t)n * Lx * cout)), dim3(256), 0, st, Y, Si, Xs, A, c.n_kernels > 1 ? A1 : nullptr,
                           c.n_kernels > 2 ? A2 : nullptr, rb[0].a1[0].alpha, rb[0].a1[0].inv_beta, c.n_kernels > 1 ? rb[1].a1[0].alpha : nullptr,
                           c.n_kernels > 1 ? rb[1].a1[0].inv_beta : nullptr, c.n_kernels > 2 ? rb[2].a1[0].alpha : nullptr,
                           c.n_kernels > 2 ? rb[2].a1[0].inv_beta : nullptr, n, Ly, Lx, cout);
        float* Rs[3] = {Y, Si, R2};         // Y and the source output are free after the add
        float* As[3] = {A, A1, A2};
        for (int r = 0; r < c.n_kernels; ++r) VOX_TRY(hift_resblock(st, rb[r], c, c.resblock_kernels[r], Xs, As[r], T1, Rs[r], n, Lx));
        // average + the next stage's leaky_relu (slope 0.01 before conv_post: F.leaky_relu's default)
        hipLaunchKernelGGL(k_hift_avg_lrelu, dim3(ew_grid((size_t)n * Lx * cout)), dim3(256), 0, st, Rs[0], c.n_kernels > 1 ? Rs[1] : nullptr,
                           c.n_kernels > 2 ? Rs[2] : nullptr, Xs, (size_t)n * Lx * cout, (float)c.n_kernels, last ? 0.01f : c.lrelu_slope, cout, last ? 0 : 3);
        cur = Xs; Lc = Lx; ch = cout;
    }
    if (Lc != F) return vox_fail(VOX_ERR_INVALID, "hift_decode: frame count mismatch");
    hift_conv_offsets(7, 1, off);
    VOX_TRY(conv_gemm(st, w.conv_post, cur, nullptr, nullptr, n, Lc, 0, off, m->post, nullptr, nullptr, 0));
    hipLaunchKernelGGL(k_hift_istft, dim3(ew_grid((size_t)n * L)), dim3(256), 0, st, m->post, wav, n, F, c.n_fft, c.hop_len, (int)L, c.audio_limit);
    return VOX_OK;
}

}  // extern "C"

// ====================================================================================================================
// CosyVoice2 flow (speech tokens -> mel): conformer encoder + conditional flow matching.  See include/voxhip.h for the contract.
// ====================================================================================================================
// The exponential of the attention's scores: libm's, within one unit of the last place (0.82 at worst over -10 .. 0, 0.30 in the mean square), denormal results
// included.  exp2 of the unreduced product with a correction behind it was 1.24 and 0.41, and 0 below 2^-126 (k_flow_attn_mfma, 184 keys: 11.7 us for 12.0).
__device__ __forceinline__ float flow_exp(float d) { return expf(d); }
// (As v n / (n + 2) with n = e^v (e^v + 2) it saves 200 instructions and no time: k_flow_ln, 896 rows of 256, 4.69 us a launch and 4.71 so.  Its error
// over normal inputs is 3.63e-8, relative 2-norm; this one's 3.42e-8.)
__device__ __forceinline__ float mish_f(float v) { return v * tanhf(v > 20.0f ? v : log1pf(expf(v))); }

// x[row] = embedding[max(id, 0)]
__global__ __launch_bounds__(256) void k_flow_embed(const int* ids, const float* emb, float* x, size_t rows, int D) {
    const size_t total = rows * D;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int id = ids[i / D];
        x[i] = emb[(size_t)(id < 0 ? 0 : id) * D + i % D];
    }
}
// y = act(LayerNorm(x) * w + b) * post + add[row / rows_per_req]      (act 0 none, 1 Mish)
__global__ __launch_bounds__(256) void k_flow_ln(const float* x, const float* w, const float* b, float* y, int C, float eps, float post, int act,
                                                  const float* add, int rows_per_req, int rows, int ldx = 0, int ld_add = 0) {
    // ldx / ld_add: row strides of x and of add (0 = C): the ResNet blocks' first conv carries the residual conv as extra columns
    // one wave per row (4 rows per block): each of the wave's four 16-lane groups computes the row statistics (ln_row_stats: the bits the
    // fused-LayerNorm GEMMs get), then the 64 lanes apply them to one float4 chunk each per pass — a 112-row call is 28 blocks with 4 Mish
    // evaluations per lane instead of 7 blocks with 16
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float* xr = x + (size_t)row * (ldx ? ldx : C);
    const float* ad = add ? add + (size_t)(row / rows_per_req) * (ld_add ? ld_add : C) : nullptr;
    if (C == 256) {
        // 256-channel rows (every LayerNorm of the CosyVoice2 estimator): lane (l16 = lane % 16, k = lane / 16) of ln_row_stats' scheme
        // owns chunks l16, l16 + 16, l16 + 32, l16 + 48 — loaded once, both statistics passes run on the registers (same order: the
        // lane's chunks ascending, then the 16-lane butterfly), and the chunk this lane writes (index `lane` = l16 + 16 k) is its k-th
        const int l16 = lane & 15, kq = lane >> 4;
        const float4* x4 = reinterpret_cast<const float4*>(xr);
        const float4 c0 = x4[l16], c1 = x4[l16 + 16], c2 = x4[l16 + 32], c3 = x4[l16 + 48];
        const float4 wv = reinterpret_cast<const float4*>(w)[lane], bv = reinterpret_cast<const float4*>(b)[lane];
        float sm = 0.0f;
        sm += (c0.x + c0.y) + (c0.z + c0.w); sm += (c1.x + c1.y) + (c1.z + c1.w);
        sm += (c2.x + c2.y) + (c2.z + c2.w); sm += (c3.x + c3.y) + (c3.z + c3.w);
        sm = butterfly<16>(sm);
        const float mean = sm / 256.0f;
        float vs = 0.0f;
        {
            float d0 = c0.x - mean, d1 = c0.y - mean, d2 = c0.z - mean, d3 = c0.w - mean;
            vs += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
            d0 = c1.x - mean; d1 = c1.y - mean; d2 = c1.z - mean; d3 = c1.w - mean;
            vs += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
            d0 = c2.x - mean; d1 = c2.y - mean; d2 = c2.z - mean; d3 = c2.w - mean;
            vs += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
            d0 = c3.x - mean; d1 = c3.y - mean; d2 = c3.z - mean; d3 = c3.w - mean;
            vs += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
        }
        vs = butterfly<16>(vs);
        const float rstd = rsqrtf(vs / 256.0f + eps);
        const float4 xv = kq == 0 ? c0 : kq == 1 ? c1 : kq == 2 ? c2 : c3;
        float o[4] = {(xv.x - mean) * rstd * wv.x + bv.x, (xv.y - mean) * rstd * wv.y + bv.y, (xv.z - mean) * rstd * wv.z + bv.z, (xv.w - mean) * rstd * wv.w + bv.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (act == 1) o[e] = mish_f(o[e]);
            o[e] *= post;
        }
        if (ad) { const float4 av = reinterpret_cast<const float4*>(ad)[lane]; o[0] += av.x; o[1] += av.y; o[2] += av.z; o[3] += av.w; }
        reinterpret_cast<float4*>(y + (size_t)row * C)[lane] = make_float4(o[0], o[1], o[2], o[3]);
        return;
    }
    float mean, rstd;
    ln_row_stats(xr, C, lane & 15, eps, mean, rstd);
    for (int i = lane; i < C / 4; i += 64) {
        const float4 xv = reinterpret_cast<const float4*>(xr)[i], wv = reinterpret_cast<const float4*>(w)[i], bv = reinterpret_cast<const float4*>(b)[i];
        float o[4] = {(xv.x - mean) * rstd * wv.x + bv.x, (xv.y - mean) * rstd * wv.y + bv.y, (xv.z - mean) * rstd * wv.z + bv.z, (xv.w - mean) * rstd * wv.w + bv.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (act == 1) o[e] = mish_f(o[e]);
            o[e] *= post;
        }
        if (ad) { const float4 av = reinterpret_cast<const float4*>(ad)[i]; o[0] += av.x; o[1] += av.y; o[2] += av.z; o[3] += av.w; }
        reinterpret_cast<float4*>(y + (size_t)row * C)[i] = make_float4(o[0], o[1], o[2], o[3]);
    }
}
// in-place activation: 1 Mish, 2 SiLU, 3 leaky_relu(0.01)
__global__ __launch_bounds__(256) void k_flow_act(float* x, size_t total, int act) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const float v = x[i];
        x[i] = act == 1 ? mish_f(v) : act == 2 ? v / (1.0f + expf(-v)) : (v > 0.0f ? v : 0.01f * v);
    }
}
// nearest x2 along time: y[b][2t + j] = x[b][t]
__global__ __launch_bounds__(256) void k_flow_repeat2(const float* x, float* y, size_t rows, int C) {
    const size_t total = rows * 2 * C;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) y[i] = x[(i / C / 2) * C + i % C];
}
// EspnetRelPositionalEncoding.position_encoding(0, S): pe[j] = encoding of position S - 1 - j   (cosyvoice_flow.py:427-447, 483-486)
__global__ __launch_bounds__(256) void k_flow_relpos(float* pe, int S, int D) {
    const size_t total = (size_t)(2 * S - 1) * D;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int j = (int)(i / D), c = (int)(i % D);
        const float pos = (float)(S - 1 - j);
        const float div = expf((float)(c & ~1) * (float)(-(9.210340371976184 / (double)D)));
        pe[i] = (c & 1) ? cosf(pos * div) : sinf(pos * div);
    }
}
// Attention over [cached keys ; this chunk's keys], no mask.  One wave per (request n, head h, query i).
// qkv [N * T][3 HD] (q | k | v); cache [chalf][H][Tcap][2 dk] (K | V), Tc valid; output [N * T][HD].
// P != NULL: the relative-position term of RelPositionMultiHeadedAttention with its literal rel_shift (cosyvoice_flow.py:772-786, 830-857).
struct FlowAttn {
    const float *qkv, *cache, *P, *bu, *bv;
    float* out;
    int T, H, dk, Tc, Tcap, B;          // B: requests per classifier-free-guidance half (cache half = n / B); B <= 0: one shared cache
    size_t cache_half_stride;
    float scale;
    int mask_block;                     // > 0: key j is visible to query i iff j <= i or j / mask_block == i / mask_block (glm.py:452-470)
    // per-request evolving caches (CosyVoice2 use_detokenizer_cache): row n reads cache block cidx[n] (stride cache_half_stride); the
    // cached keys beyond the first `prefix` rows sit in a ring that starts at ring_head (logical row j -> physical row below)
    const int* cidx;
    int prefix, ring_head;
    // k_flow_attn_mfma<.., true>: the out projection's packed weights and the planes (one a head, ps floats apart, rows of 256) that take its sums over
    // that head's 64 columns, in the place of `out`
    const bf16_t* wo;
    float* parts;
    size_t ps;
    // and its items (request, head, query tile) as tb_item gives them: items of an XCD, XCDs with one more, the inverses (tb_inverse) of a request's items
    // and of its query tiles
    int per, rest;
    unsigned inv_n, inv_h;
};
__device__ __forceinline__ int flow_cache_row(int j, int prefix, int head, int cap) {
    return (head == 0 || j < prefix) ? j : prefix + (head + j - prefix) % (cap - prefix);
}
#define FLOW_MAXKEYS 1024
__global__ __launch_bounds__(256) void k_flow_attn(FlowAttn a) {
    touch_args(a);
    __shared__ float ps[4][FLOW_MAXKEYS];
    __shared__ __attribute__((aligned(16))) float qs[4][2][128];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i = blockIdx.x * 4 + wave, h = blockIdx.y, n = blockIdx.z;
    if (i >= a.T) return;
    const int HD = a.H * a.dk, ld = 3 * HD, S = a.Tc + a.T;
    const float* cache = a.cache ? a.cache + (a.cidx ? (size_t)a.cidx[n] * a.cache_half_stride : a.B > 0 ? (size_t)(n / a.B) * a.cache_half_stride : 0) +
                                       (size_t)h * a.Tcap * 2 * a.dk : nullptr;
    const float* qrow = a.qkv + ((size_t)n * a.T + i) * ld + h * a.dk;
    for (int d = lane; d < a.dk; d += 64) {
        qs[wave][0][d] = qrow[d] + (a.bu ? a.bu[h * a.dk + d] : 0.0f);
        qs[wave][1][d] = a.bv ? a.bv[h * a.dk + d] : 0.0f;
    }
    __builtin_amdgcn_wave_barrier();
    float mx = -INFINITY;
    const int dk4 = a.dk >> 2;
    const float4* q4 = reinterpret_cast<const float4*>(qs[wave][0]);
    const float4* v4 = reinterpret_cast<const float4*>(qs[wave][1]);
    for (int j = lane; j < S; j += 64) {
        const float4* kr = reinterpret_cast<const float4*>(j < a.Tc ? cache + (size_t)flow_cache_row(j, a.prefix, a.ring_head, a.Tcap) * 2 * a.dk
                                                                    : a.qkv + ((size_t)n * a.T + (j - a.Tc)) * ld + HD + h * a.dk);
        float ac = 0.0f;
#pragma unroll 4
        for (int d = 0; d < dk4; ++d) {
            const float4 k = kr[d], q = q4[d];
            ac = fmaf(q.x, k.x, ac); ac = fmaf(q.y, k.y, ac); ac = fmaf(q.z, k.z, ac); ac = fmaf(q.w, k.w, ac);
        }
        if (a.P) {
            const long f = (long)i * (2 * S - 1) + j + a.T;
            const int r = (int)(f / (2 * S)), ci = (int)(f % (2 * S));
            if (ci > 0) {
                const float4* qr = reinterpret_cast<const float4*>(a.qkv + ((size_t)n * a.T + r) * ld + h * a.dk);
                const float4* pr = reinterpret_cast<const float4*>(a.P + (size_t)(ci - 1) * HD + h * a.dk);
                float bd = 0.0f;
#pragma unroll 4
                for (int d = 0; d < dk4; ++d) {
                    const float4 q = qr[d], bv = v4[d], p = pr[d];
                    bd = fmaf(q.x + bv.x, p.x, bd); bd = fmaf(q.y + bv.y, p.y, bd); bd = fmaf(q.z + bv.z, p.z, bd); bd = fmaf(q.w + bv.w, p.w, bd);
                }
                ac += bd;
            }
        }
        ac *= a.scale;
        if (a.mask_block > 0 && j > i && j / a.mask_block != i / a.mask_block) ac = -INFINITY;
        ps[wave][j] = ac;
        mx = fmaxf(mx, ac);
    }
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    float sum = 0.0f;
    for (int j = lane; j < S; j += 64) {
        const float p = expf(ps[wave][j] - mx);
        ps[wave][j] = p;
        sum += p;
    }
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
    __builtin_amdgcn_wave_barrier();
    const float inv = 1.0f / sum;
    // PV: lane = (key group g = lane / 16, float4 chunk c = lane % 16 of the output dims); a pass reads four whole V rows (coalesced
    // 256-byte segments), four passes are in flight together; the four key groups are summed by two butterfly steps at the end.
    // (chunk c covers dims 4c .. 4c+3 of each 64-dim slab; lanes past dk idle)
    for (int c4 = (lane & 15) * 4, slab = 0; slab < a.dk; slab += 64, c4 += 64) {
        const int g = lane >> 4;
        const bool on = c4 < a.dk;
        float4 o[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) o[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        const float* vc = cache ? cache + a.dk + c4 : nullptr;
        const float* vn = a.qkv + (size_t)n * a.T * ld + 2 * HD + h * a.dk + c4;
        auto vrow = [&](int j) {
            return reinterpret_cast<const float4*>(j < a.Tc ? vc + (size_t)flow_cache_row(j, a.prefix, a.ring_head, a.Tcap) * 2 * a.dk : vn + (size_t)(j - a.Tc) * ld);
        };
        int j = g;
        if (on) {
            for (; j + 12 < S; j += 16) {
                float4 v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = *vrow(j + 4 * u);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float p = ps[wave][j + 4 * u];
                    o[u].x = fmaf(p, v[u].x, o[u].x); o[u].y = fmaf(p, v[u].y, o[u].y);
                    o[u].z = fmaf(p, v[u].z, o[u].z); o[u].w = fmaf(p, v[u].w, o[u].w);
                }
            }
            for (; j < S; j += 4) {
                const float4 v = *vrow(j);
                const float p = ps[wave][j];
                o[0].x = fmaf(p, v.x, o[0].x); o[0].y = fmaf(p, v.y, o[0].y); o[0].z = fmaf(p, v.z, o[0].z); o[0].w = fmaf(p, v.w, o[0].w);
            }
        }
        float4 r = make_float4((o[0].x + o[1].x) + (o[2].x + o[3].x), (o[0].y + o[1].y) + (o[2].y + o[3].y),
                               (o[0].z + o[1].z) + (o[2].z + o[3].z), (o[0].w + o[1].w) + (o[2].w + o[3].w));
#pragma unroll
        for (int off = 16; off <= 32; off <<= 1) {
            r.x += __shfl_xor(r.x, off, 64); r.y += __shfl_xor(r.y, off, 64); r.z += __shfl_xor(r.z, off, 64); r.w += __shfl_xor(r.w, off, 64);
        }
        if (on && g == 0)
            *reinterpret_cast<float4*>(a.out + ((size_t)n * a.T + i) * HD + h * a.dk + c4) = make_float4(r.x * inv, r.y * inv, r.z * inv, r.w * inv);
    }
}
// The same attention for the calls without a relative-position term (the CFM estimators' transformer blocks: thousands of launches per
// chunk), with the (request, head)'s keys and values staged ONCE per block in LDS: k_flow_attn has every wave stream all S key and value
// rows from L2 for its one query (94 KB per query at S = 184, dk = 64: 84 MB of L2 reads per call at one request).  A block owns QG
// consecutive queries, its four waves take them in turn; arithmetic and summation orders are k_flow_attn's, so the two kernels agree
// bit for bit (which one a call takes may depend on its batch size; a request's output may not).  K rows are padded to DK + 4 floats:
// lane = key reads of a float4 column then touch every bank once per 16 lanes.
template <int DK>
__global__ __launch_bounds__(256) void k_flow_attn_tile(FlowAttn a, int QG) {
    extern __shared__ __attribute__((aligned(16))) float fa_sm[];
    constexpr int KS = DK + 4, DK4 = DK / 4;
    const int S = a.Tc + a.T, S4 = (S + 3) & ~3;
    float* Ks = fa_sm;
    float* Vs = Ks + (size_t)S * KS;
    float* psm = Vs + (size_t)S * DK;
    float* qsm = psm + 4 * S4;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int h = blockIdx.y, n = blockIdx.z, i0 = blockIdx.x * QG;
    const int HD = a.H * DK, ld = 3 * HD;
    const float* cache = a.cache ? a.cache + (a.cidx ? (size_t)a.cidx[n] * a.cache_half_stride : a.B > 0 ? (size_t)(n / a.B) * a.cache_half_stride : 0) +
                                       (size_t)h * a.Tcap * 2 * DK : nullptr;
    for (int idx = tid; idx < S * DK4; idx += 256) {
        const int j = idx / DK4, c = idx - j * DK4;
        const float *kr, *vr;
        if (j < a.Tc) {
            kr = cache + (size_t)flow_cache_row(j, a.prefix, a.ring_head, a.Tcap) * 2 * DK;
            vr = kr + DK;
        } else {
            kr = a.qkv + ((size_t)n * a.T + (j - a.Tc)) * ld + HD + h * DK;
            vr = kr + HD;
        }
        *reinterpret_cast<float4*>(Ks + (size_t)j * KS + 4 * c) = reinterpret_cast<const float4*>(kr)[c];
        *reinterpret_cast<float4*>(Vs + (size_t)j * DK + 4 * c) = reinterpret_cast<const float4*>(vr)[c];
    }
    __syncthreads();
    float* ps = psm + wave * S4;
    float* qs = qsm + wave * DK;
    const int iend = (i0 + QG < a.T) ? i0 + QG : a.T;
    for (int i = i0 + wave; i < iend; i += 4) {
        const float* qrow = a.qkv + ((size_t)n * a.T + i) * ld + h * DK;
        for (int d = lane; d < DK; d += 64) qs[d] = qrow[d] + (a.bu ? a.bu[h * DK + d] : 0.0f);
        __builtin_amdgcn_wave_barrier();
        float mx = -INFINITY;
        const float4* q4 = reinterpret_cast<const float4*>(qs);
        for (int j = lane; j < S; j += 64) {
            const float4* kr = reinterpret_cast<const float4*>(Ks + (size_t)j * KS);
            float ac = 0.0f;
#pragma unroll
            for (int d = 0; d < DK4; ++d) {
                const float4 k = kr[d], q = q4[d];
                ac = fmaf(q.x, k.x, ac); ac = fmaf(q.y, k.y, ac); ac = fmaf(q.z, k.z, ac); ac = fmaf(q.w, k.w, ac);
            }
            ac *= a.scale;
            if (a.mask_block > 0 && j > i && j / a.mask_block != i / a.mask_block) ac = -INFINITY;
            ps[j] = ac;
            mx = fmaxf(mx, ac);
        }
        for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        float sum = 0.0f;
        for (int j = lane; j < S; j += 64) {
            const float p = expf(ps[j] - mx);
            ps[j] = p;
            sum += p;
        }
        for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
        __builtin_amdgcn_wave_barrier();
        const float inv = 1.0f / sum;
        // PV in k_flow_attn's order: lane = (key group g, float4 chunk c), keys g, g + 4, ... in four interleaved accumulators
        for (int c4 = (lane & 15) * 4, slab = 0; slab < DK; slab += 64, c4 += 64) {
            const int g = lane >> 4;
            const bool on = c4 < DK;
            float4 o[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) o[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            int j = g;
            if (on) {
                for (; j + 12 < S; j += 16) {
                    float4 v[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const float4*>(Vs + (size_t)(j + 4 * u) * DK + c4);
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const float p = ps[j + 4 * u];
                        o[u].x = fmaf(p, v[u].x, o[u].x); o[u].y = fmaf(p, v[u].y, o[u].y);
                        o[u].z = fmaf(p, v[u].z, o[u].z); o[u].w = fmaf(p, v[u].w, o[u].w);
                    }
                }
                for (; j < S; j += 4) {
                    const float4 v = *reinterpret_cast<const float4*>(Vs + (size_t)j * DK + c4);
                    const float p = ps[j];
                    o[0].x = fmaf(p, v.x, o[0].x); o[0].y = fmaf(p, v.y, o[0].y); o[0].z = fmaf(p, v.z, o[0].z); o[0].w = fmaf(p, v.w, o[0].w);
                }
            }
            float4 r = make_float4((o[0].x + o[1].x) + (o[2].x + o[3].x), (o[0].y + o[1].y) + (o[2].y + o[3].y),
                                   (o[0].z + o[1].z) + (o[2].z + o[3].z), (o[0].w + o[1].w) + (o[2].w + o[3].w));
#pragma unroll
            for (int off = 16; off <= 32; off <<= 1) {
                r.x += __shfl_xor(r.x, off, 64); r.y += __shfl_xor(r.y, off, 64); r.z += __shfl_xor(r.z, off, 64); r.w += __shfl_xor(r.w, off, 64);
            }
            if (on && g == 0)
                *reinterpret_cast<float4*>(a.out + ((size_t)n * a.T + i) * HD + h * DK + c4) = make_float4(r.x * inv, r.y * inv, r.z * inv, r.w * inv);
        }
        __builtin_amdgcn_wave_barrier();      // ps / qs are rewritten by the wave's next query
    }
}
// Parts of the estimator's fused transformer blocks (below) that their attention uses too.
//
// Which of a launch's items a block takes: the blocks of one XCD (block id modulo 8) take neighbouring ones, every XCD as many as the next, so that what
// blocks beside each other read, and what the launch before left for them, is in that XCD's L2.  All of a block's launches have their items in the
// order of the rows.  With the row tile or the query tile as the grid's fast index that was so only where eight divides it: a feed-forward of 42 row
// tiles 12.2 us, one of 48 11.3, now 10.6 and 10.6; q | k | v of later blocks of a level 8.8 (40 tiles 8.0), now 7.3.  (Padded to eight row tiles instead,
// 42 leave two XCDs more q | k | v blocks than CUs: 10.8.  Only q | k | v and feed-forward in this order: 8.1 and 10.6.)  The shares are counted on
// the host: counted in the kernels, a launch of few blocks took 0.1 longer.
struct tb_share {
    int per, rest;      // items of an XCD, of which the first `rest` have one more
};
static tb_share tb_shares(int items) { return tb_share{items >> 3, items & 7}; }
__device__ __forceinline__ int tb_item(tb_share s) {
    const int xcd = (int)blockIdx.x & 7;
    return xcd * s.per + (xcd < s.rest ? xcd : s.rest) + ((int)blockIdx.x >> 3);
}
// x / d as tb_quotient(x, tb_inverse(d)): exact while x * d < 2^24 and x / d < 256
static unsigned tb_inverse(int d) { return ((1u << 24) + (unsigned)d - 1) / (unsigned)d; }
__device__ __forceinline__ int tb_quotient(int x, unsigned inverse) { return (int)((unsigned)x * inverse >> 24); }
#define TB_C 256
#define TB_IN 512
#define TB_FF 1024
struct FlowPacked {
    const bf16_t *qkv = nullptr, *out = nullptr, *ff1 = nullptr, *ff2 = nullptr;
};
// w [N][K] bf16 -> tiles of 16 rows x 32 columns (row tile major), each as the 64 lanes of an MFMA operand hold it
__global__ __launch_bounds__(256) void k_pack_frag(const bf16_t* w, bf16_t* out, int K, size_t chunks) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= chunks) return;
    const int kb_n = K >> 5, lane = (int)(i & 63);
    const size_t tile = i >> 6, kb = tile % kb_n, rt = tile / kb_n;
    *reinterpret_cast<uint4*>(out + i * 8) = *reinterpret_cast<const uint4*>(w + (rt * 16 + (lane & 15)) * K + kb * 32 + (lane >> 4) * 8);
}
struct tb_split {
    uint2 t[3];      // four values' leading, second and third bf16 terms
};
__device__ __forceinline__ tb_split tb_split3(float4 v) {
    tb_split s;
    s.t[0] = make_uint2(pack_bf2(v.x, v.y), pack_bf2(v.z, v.w));
    const float4 r = make_float4(v.x - bflo(s.t[0].x), v.y - bfhi(s.t[0].x), v.z - bflo(s.t[0].y), v.w - bfhi(s.t[0].y));
    s.t[1] = make_uint2(pack_bf2(r.x, r.y), pack_bf2(r.z, r.w));
    s.t[2] = make_uint2(pack_bf2(r.x - bflo(s.t[1].x), r.y - bfhi(s.t[1].x)), pack_bf2(r.z - bflo(s.t[1].y), r.w - bfhi(s.t[1].y)));
    return s;
}
__device__ __forceinline__ float4 tb_add(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }
// Column tile 2 wave + t of 256 columns as an operand of the next product: k-block `wave`, k group 2 t + kq / 2
__device__ __forceinline__ void tb_put(uint4* pl, int kb_n, int wave, int t, int lane, float4 v) {
    const tb_split s = tb_split3(v);
    const int fr = lane & 15, kq = lane >> 4;
    uint2* d = reinterpret_cast<uint2*>(pl + wave * 64 + (2 * t + (kq >> 1)) * 16 + fr) + (kq & 1);
#pragma unroll
    for (int p = 0; p < 3; ++p) d[p * kb_n * 128] = s.t[p];
}
// A row's sum over its 256 columns from the sums s[t] of four neighbouring ones (two per lane): eight neighbouring columns, then the two
// 32-column blocks of a run of 64, then its four groups of eight, then the runs.  red: [8][16] x 4 floats, one for each call of a block
__device__ __forceinline__ float tb_row_sum(float s0, float s1, float4* red, int wave, int lane) {
    const int fr = lane & 15;
    s0 = xor_add<16>(s0);
    s1 = xor_add<16>(s1);
    if (!(lane & 16)) {
        float* d = reinterpret_cast<float*>(red + wave * 16 + fr) + (lane >> 5);
        d[0] = s0;
        d[2] = s1;
    }
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 a = red[2 * i * 16 + fr], b = red[(2 * i + 1) * 16 + fr];
        const float run = ((a.x + b.x) + (a.y + b.y)) + ((a.z + b.z) + (a.w + b.w));
        tot = i == 0 ? run : tot + run;
    }
    return tot;
}
// The same sum of a row that lies in one wave, four columns to a lane
__device__ __forceinline__ float tb_row_sum64(float s) {
    s = xor_add<1>(s);      // eight neighbouring columns
    s = xor_add<8>(s);      // the two 32-column blocks of a run of 64
    s = xor_add<2>(s);
    s = xor_add<4>(s);
    auto at = [&](int l) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s), l)); };
    return ((at(0) + at(16)) + at(32)) + at(48);
}
// LayerNorm of the rows whose columns lie 8 to a lane (two tiles of four) over the block's eight waves; red: [2][8][16] x 4 floats
__device__ __forceinline__ void tb_layernorm(float4 (&v)[2], const float4 (&w)[2], const float4 (&b)[2], float4* red, int wave, int lane) {
    const float mean = tb_row_sum((v[0].x + v[0].y) + (v[0].z + v[0].w), (v[1].x + v[1].y) + (v[1].z + v[1].w), red, wave, lane) / (float)TB_C;
    float q[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        v[t] = make_float4(v[t].x - mean, v[t].y - mean, v[t].z - mean, v[t].w - mean);
        q[t] = (v[t].x * v[t].x + v[t].y * v[t].y) + (v[t].z * v[t].z + v[t].w * v[t].w);
    }
    const float var = tb_row_sum(q[0], q[1], red + 128, wave, lane);
    const float rstd = rsqrtf(var / (float)TB_C + 1e-5f);
#pragma unroll
    for (int t = 0; t < 2; ++t)
        v[t] = make_float4(v[t].x * rstd * w[t].x + b[t].x, v[t].y * rstd * w[t].y + b[t].y, v[t].z * rstd * w[t].z + b[t].z, v[t].w * rstd * w[t].w + b[t].w);
}
// NT column tiles against the rows in pl (KB k-blocks, three terms, low terms first) as the sums of runs of RUN k-blocks
// (TURN: a row's place among the 16 of a k group is turned by the group, tb_turn)
__device__ __forceinline__ int tb_turn(int kb, int g, int row) { return row ^ ((g + 4 * kb) & 15); }
template <int KB, int RUN, int NT, bool TURN = false>
__device__ __forceinline__ void tb_runs(const uint4 (&wf)[NT][KB], const uint4* pl, int lane, f32x4 (&acc)[KB / RUN][NT]) {
#pragma unroll
    for (int i = 0; i < KB / RUN; ++i) {
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = i * RUN; kb < (i + 1) * RUN; ++kb)
#pragma unroll
            for (int p = 2; p >= 0; --p) {
                const uint4 x = pl[(p * KB + kb) * 64 + (TURN ? (lane & 48) + tb_turn(kb, lane >> 4, lane & 15) : lane)];
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_cbf8(wf[t][kb]), as_cbf8(x), acc[i][t], 0, 0, 0);
            }
    }
}
// the whole product: runs of two k-blocks, added in ascending order
template <int KB, int NT, bool TURN = false>
__device__ __forceinline__ void tb_product(const uint4 (&wf)[NT][KB], const uint4* pl, int lane, f32x4 (&acc)[NT]) {
    f32x4 r[KB / 2][NT];
    tb_runs<KB, 2, NT, TURN>(wf, pl, lane, r);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        acc[t] = r[0][t];
#pragma unroll
        for (int i = 1; i < KB / 2; ++i) acc[t] += r[i][t];
    }
}
template <int KB, int NT>
__device__ __forceinline__ void tb_weights(uint4 (&wf)[NT][KB], const bf16_t* w, int tile, int kb_all, int kb0, int lane) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) wf[t][kb] = *reinterpret_cast<const uint4*>(w + ((size_t)(tile + t) * kb_all + kb0 + kb) * 512 + lane * 8);
}
// floats of column tile 2 wave + t of row tile `rt` in lane order
__device__ __forceinline__ size_t tb_at(int rt, int wave, int t, int lane) { return ((((size_t)rt * 8 + wave) * 2 + t) * 64 + lane) * 4; }
// Planes of a block's scratch, ps floats apart: ff2's sums (the first two eighths, then an eighth each), the residual rows behind the out product,
// and those in front of it (the sum of the planes that the block before has left)
#define TB_PARTS 7
#define TB_PLANES 9
#define TB_HEADS 8      // planes of the heads' sums of the out product behind them, rows of 256
// rows [.][256] = residual + ((parts[0] + ... + parts[6]) + b2)
__device__ __forceinline__ float4 tb_sum(const float* p, size_t ps, float4 b2) {
    float4 v[TB_PARTS + 1];
#pragma unroll
    for (int i = 0; i <= TB_PARTS; ++i) v[i] = *reinterpret_cast<const float4*>(p + i * ps);
#pragma unroll
    for (int i = 1; i < TB_PARTS; ++i) v[0] = tb_add(v[0], v[i]);
    return tb_add(v[TB_PARTS], tb_add(v[0], b2));
}
// The largest value of a lane's row of 16 lanes (a maximum does not see the order it is taken in)
__device__ __forceinline__ float row16_max(float s) {
    s = fmaxf(s, vox_dpp<0x128, 0xF>(s, s));      // row_ror:8, 4, 2, 1
    s = fmaxf(s, vox_dpp<0x124, 0xF>(s, s));
    s = fmaxf(s, vox_dpp<0x122, 0xF>(s, s));
    return fmaxf(s, vox_dpp<0x121, 0xF>(s, s));
}
// The estimators' attention on the matrix cores (no relative-position term, dk = 64, at most 256 keys: every CosyVoice2 / GLM estimator
// call).  A block owns 16 consecutive queries of one (request, head); its WV (8) waves take the 16-key tiles w, w + WV for
// BOTH products, so nothing but the row maxima, the row sums and the 16 x 64 partial outputs crosses a wave:
//   scores  = Q K^T   v_mfma_f32_16x16x4_f32 (fp32 operands, fp32 accumulate), 16 per key tile; every operand is requested up front
//                     straight in operand layout (lane = (row l % 16, k group l / 16) holds four float4 chunks 16 c + 4 (l / 16) of its
//                     row: the contraction index is permuted the same way on both sides, which a dot product does not see)
//   softmax           row maximum by a 16-lane butterfly + one LDS exchange across the waves; p = exp(s - max)
//   out     = P V     p goes through a wave-private LDS tile to become an A operand; V rows are float4 loads whose four components
//                     are the four 16-dim output tiles (dim = 4 (l % 16) + tile), so a lane's four accumulators are one float4 of the row
// and the partial outputs of the WV waves are summed in the fixed order w0 + w1 + ... and scaled by 1 / sum.  A (request, head, query)'s
// result depends on that request's rows only.
// OUT (fused transformer blocks: 8 heads, 256 channels): the block multiplies its 16 x 64 outputs by the head's 64 columns of the out projection too (32 KB of
// weights), one of that product's eight runs of K: the feed-forward launch adds the heads' planes in order and has the product's bits without
// its 256 KB of weights a block.  896 rows: 11.4 -> 13.0 us here, 13.0 -> 10.8 there and 9.1 -> 8.3 in the next q | k | v.  (Two query
// tiles a block, which read each key once for both: 15.2.)
// Four waves share a SIMD, so what a wave issues counts: 184 keys, 13.6 us -> 12.0 with a tile's rows addressed together and clamped (each row had its own
// branches, a division among them, and a wait between the tiles) and DPP in the place of LDS permutes (2.6 are its fp32 MFMA).
template <int DK, int WV, bool OUT>
__global__ __launch_bounds__(64 * WV) void k_flow_attn_mfma(FlowAttn a) {
    static_assert(DK == 64, "operand layout below is written for 64-dim heads");
    constexpr int KT = 16 / WV, PS = KT * 16 + 4, OS = DK + 4;      // WV waves x KT key tiles of 16: at most 256 keys
    __shared__ __attribute__((aligned(16))) float red_mx[WV][16], red_sum[WV][16];
    __shared__ __attribute__((aligned(16))) float Ps[WV][16][PS];
    __shared__ __attribute__((aligned(16))) float Os[WV][16][OS];
    __shared__ uint4 pl[OUT ? 3 * 2 * 64 : 1];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, fr = lane & 15, kq = lane >> 4;
    int i0 = blockIdx.x * 16, h = blockIdx.y, n = blockIdx.z;
    if constexpr (OUT) {
        const int qt = (a.T + 15) >> 4, item = tb_item(tb_share{a.per, a.rest});
        n = tb_quotient(item, a.inv_n);
        const int nh = item - n * qt * a.H;
        h = tb_quotient(nh, a.inv_h);
        i0 = (nh - h * qt) * 16;
    }
    const int HD = a.H * DK, ld = 3 * HD, S = a.Tc + a.T, nt = (S + 15) >> 4;
    const float* const cache = a.cache ? a.cache + (a.cidx ? (size_t)a.cidx[n] * a.cache_half_stride : a.B > 0 ? (size_t)(n / a.B) * a.cache_half_stride : 0) +
                                       (size_t)h * a.Tcap * 2 * DK : nullptr;
    // Keys at or beyond S read key S - 1, whose products are dropped: no load stands behind a branch of its own
    const float* const fresh = a.qkv + ((ptrdiff_t)n * a.T - a.Tc) * ld + HD + h * DK;      // key j's K row: + j ld, its V row HD behind it
    const int iq = i0 + fr < a.T ? i0 + fr : a.T - 1;
    const float* qrow = a.qkv + (size_t)n * a.T * ld + h * DK;
    float4 q[4], k[KT][4], v[KT][4];
#pragma unroll
    for (int c = 0; c < 4; ++c) q[c] = *reinterpret_cast<const float4*>(qrow + (unsigned)(iq * ld + 4 * kq + 16 * c));
#pragma unroll
    for (int t = 0; t < KT; ++t) {
        const int j0 = (t * WV + wave) * 16, last = S - 1 - j0;
        if (last < 0) continue;
        const float *pk, *pv[4];      // B operand of P V: key j0 + 4 s4 + kq, dims 4 fr .. 4 fr + 3
        if (j0 >= a.Tc || (j0 + 16 <= a.Tc && a.ring_head == 0)) {      // the tile's keys lie one behind the other
            const bool old = j0 < a.Tc;
            const float* const base = old ? cache + j0 * 2 * DK : fresh + (ptrdiff_t)j0 * ld;
            const int step = old ? 2 * DK : ld, vo = old ? DK : HD;
            pk = base + (unsigned)((fr < last ? fr : last) * step + 4 * kq);
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4) pv[s4] = base + (unsigned)((4 * s4 + kq < last ? 4 * s4 + kq : last) * step + vo + 4 * fr);
        } else {
            auto row = [&](int j, int is_v) -> const float* {
                j = j < S ? j : S - 1;
                return j < a.Tc ? cache + (flow_cache_row(j, a.prefix, a.ring_head, a.Tcap) * 2 + is_v) * DK : fresh + (ptrdiff_t)j * ld + is_v * HD;
            };
            pk = row(j0 + fr, 0) + 4 * kq;
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4) pv[s4] = row(j0 + 4 * s4 + kq, 1) + 4 * fr;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) k[t][c] = ldg_f4(pk + 16 * c);
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) v[t][s4] = ldg_f4(pv[s4]);
    }
    f32x4 sc[KT];
    float mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
    for (int t = 0; t < KT; ++t) {
        const int kt = t * WV + wave;
        if (kt < nt) {
            sc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                sc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[c].x, k[t][c].x, sc[t], 0, 0, 0);
                sc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[c].y, k[t][c].y, sc[t], 0, 0, 0);
                sc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[c].z, k[t][c].z, sc[t], 0, 0, 0);
                sc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[c].w, k[t][c].w, sc[t], 0, 0, 0);
            }
            const int j = kt * 16 + fr;      // accumulator r: query i0 + 4 kq + r, key j
            const bool in = j < S;
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[t][r] = in ? sc[t][r] * a.scale : -INFINITY;
            if (a.mask_block > 0) {
                const int jb = j / a.mask_block;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = i0 + 4 * kq + r;
                    if (j > i && jb != i / a.mask_block) sc[t][r] = -INFINITY;
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], sc[t][r]);
        }
    }
    uint4 wf[OUT ? 2 : 1][2];      // (in flight while the outputs are formed)
    if constexpr (OUT) tb_weights<2, 2>(wf, a.wo, wave * 2, 16, h * 2, lane);
#pragma unroll
    for (int r = 0; r < 4; ++r) mx[r] = row16_max(mx[r]);
    if (fr == 0) *reinterpret_cast<float4*>(&red_mx[wave][4 * kq]) = make_float4(mx[0], mx[1], mx[2], mx[3]);
    __syncthreads();
    float4 gm = *reinterpret_cast<const float4*>(&red_mx[0][4 * kq]);
#pragma unroll
    for (int w = 1; w < WV; ++w) {
        const float4 m = *reinterpret_cast<const float4*>(&red_mx[w][4 * kq]);
        gm = make_float4(fmaxf(gm.x, m.x), fmaxf(gm.y, m.y), fmaxf(gm.z, m.z), fmaxf(gm.w, m.w));
    }
    const float top[4] = {gm.x, gm.y, gm.z, gm.w};
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < KT; ++t)
        if (t * WV + wave < nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = flow_exp(sc[t][r] - top[r]);
                Ps[wave][4 * kq + r][16 * t + fr] = p;
                sum[r] += p;
            }
#pragma unroll
    for (int r = 0; r < 4; ++r) sum[r] = butterfly<16>(sum[r]);
    if (fr == 0) *reinterpret_cast<float4*>(&red_sum[wave][4 * kq]) = make_float4(sum[0], sum[1], sum[2], sum[3]);
    __builtin_amdgcn_wave_barrier();      // the wave's own p tile: written in accumulator layout, read back as A operands
    f32x4 o[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < KT; ++t) {
        if (t * WV + wave < nt) {
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4) {
                const float pa = Ps[wave][fr][16 * t + 4 * s4 + kq];
                o[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa, v[t][s4].x, o[0], 0, 0, 0);
                o[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa, v[t][s4].y, o[1], 0, 0, 0);
                o[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa, v[t][s4].z, o[2], 0, 0, 0);
                o[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa, v[t][s4].w, o[3], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)      // o[d][r] = out[query 4 kq + r][dim 4 fr + d]
        *reinterpret_cast<float4*>(&Os[wave][4 * kq + r][4 * fr]) = make_float4(o[0][r], o[1][r], o[2][r], o[3][r]);
    __syncthreads();
    if constexpr (OUT) {      // two columns to a thread of the eight waves
        const int qi = tid >> 5, c2 = (tid & 31) * 2, g = c2 >> 3;
        float l = red_sum[0][qi];
        float2 o2 = *reinterpret_cast<const float2*>(&Os[0][qi][c2]);
#pragma unroll
        for (int w = 1; w < WV; ++w) {
            l += red_sum[w][qi];
            const float2 pw = *reinterpret_cast<const float2*>(&Os[w][qi][c2]);
            o2.x += pw.x; o2.y += pw.y;
        }
        const float inv = 1.0f / l;
        o2 = make_float2(o2.x * inv, o2.y * inv);
        u32* d = reinterpret_cast<u32*>(pl + (g >> 2) * 64 + (g & 3) * 16 + tb_turn(g >> 2, g & 3, qi)) + (tid & 3);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const u32 term = pack_bf2(o2.x, o2.y);
            d[p * 2 * 256] = term;
            o2 = make_float2(o2.x - bflo(term), o2.y - bfhi(term));
        }
    } else {
        const int qi = tid >> 4, c4 = (tid & 15) * 4;
        if (tid < 256 && i0 + qi < a.T) {
            float l = red_sum[0][qi];
            float4 o4 = *reinterpret_cast<const float4*>(&Os[0][qi][c4]);
#pragma unroll
            for (int w = 1; w < WV; ++w) {
                l += red_sum[w][qi];
                const float4 pw = *reinterpret_cast<const float4*>(&Os[w][qi][c4]);
                o4.x += pw.x; o4.y += pw.y; o4.z += pw.z; o4.w += pw.w;
            }
            const float inv = 1.0f / l;
            *reinterpret_cast<float4*>(a.out + ((size_t)n * a.T + i0 + qi) * HD + h * DK + c4) = make_float4(o4.x * inv, o4.y * inv, o4.z * inv, o4.w * inv);
        }
    }
    if constexpr (OUT) {
        __syncthreads();
        f32x4 y[1][2];
        tb_runs<2, 2, 2, true>(wf, pl, lane, y);
        if (i0 + fr < a.T)
#pragma unroll
            for (int t = 0; t < 2; ++t)
                *reinterpret_cast<f32x4*>(a.parts + h * a.ps + ((size_t)n * a.T + i0 + fr) * TB_C + (wave * 2 + t) * 16 + kq * 4) = y[0][t];
    }
}
// VOX_FLOW_ATTN_MFMA=0: the VALU attention kernels for every call (A/B timing)
static bool flow_attn_mfma_on() {
    static const bool on = [] { const char* e = getenv("VOX_FLOW_ATTN_MFMA"); return !(e && e[0] == '0'); }();
    return on;
}
// VOX_FLOW_ATTN_TILE=0: k_flow_attn for every call (A/B timing)
static bool flow_attn_tile_on() {
    static const bool on = [] { const char* e = getenv("VOX_FLOW_ATTN_TILE"); return !(e && e[0] == '0'); }();
    return on;
}
// the fused blocks' order of items; false: their numbers are beyond the divisions'
static bool flow_attn_near(FlowAttn& a, int T, int H, int N) {
    const long per_n = (long)((T + 15) / 16) * H;
    if (N >= 256 || H >= 256 || N * per_n * per_n >= 1l << 24) return false;
    const tb_share s = tb_shares((int)(N * per_n));
    a.per = s.per;
    a.rest = s.rest;
    a.inv_n = tb_inverse((int)per_n);
    a.inv_h = tb_inverse((T + 15) / 16);
    return true;
}
// VOX_FLOW_ATTN_WV=4: four waves x four key tiles, which leave their rows for the out product (A/B timing)
static bool flow_attn_wv4() {
    static const bool on = [] { const char* e = getenv("VOX_FLOW_ATTN_WV"); return e && atoi(e) == 4; }();
    return on;
}
static bool flow_attn_mfma_takes(const FlowAttn& a, int T) { return !a.P && !a.bu && a.dk == 64 && a.Tc + T <= 256 && flow_attn_mfma_on(); }
static void launch_flow_attn(hipStream_t st, const FlowAttn& a, int T, int H, int N) {
    const int S = a.Tc + T;
    const size_t lds = ((size_t)S * (2 * a.dk + 4) + 4 * ((S + 3) & ~3) + 4 * a.dk) * sizeof(float);
    if (flow_attn_mfma_takes(a, T)) {
        if (a.parts) hipLaunchKernelGGL((k_flow_attn_mfma<64, 8, true>), dim3((T + 15) / 16 * H * N), dim3(512), 0, st, a);
        else if (flow_attn_wv4()) hipLaunchKernelGGL((k_flow_attn_mfma<64, 4, false>), dim3((T + 15) / 16, H, N), dim3(256), 0, st, a);
        else hipLaunchKernelGGL((k_flow_attn_mfma<64, 8, false>), dim3((T + 15) / 16, H, N), dim3(512), 0, st, a);
        return;
    }
    if (!a.P && a.dk == 64 && lds <= 150 * 1024 && flow_attn_tile_on()) {
        static bool attr = false;
        if (!attr) {
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k_flow_attn_tile<64>), hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);
            attr = true;
        }
        int qg = 4;      // queries per block: one per wave while the grid stays within ~2 blocks per CU, more per wave beyond
        while ((T + qg - 1) / qg * H * N > 512 && qg < T) qg *= 2;
        hipLaunchKernelGGL(k_flow_attn_tile<64>, dim3((T + qg - 1) / qg, H, N), dim3(256), lds, st, a, qg);
        return;
    }
    hipLaunchKernelGGL(k_flow_attn, dim3((T + 3) / 4, H, N), dim3(256), 0, st, a);
}
// new K | V rows of request n -> cache [half = n][H][Tcap][2 dk], keeping the first `prefix` and the last Tcap - prefix of the T rows
__global__ __launch_bounds__(256) void k_flow_cache_store(const float* qkv, float* cache, int T, int H, int dk, int Tcap, int prefix,
                                                           size_t cache_half_stride, int N) {
    const int keep = T < Tcap ? T : Tcap;
    const size_t total = (size_t)N * H * keep * 2 * dk;
    const int HD = H * dk;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int e = (int)(i % (2 * dk));
        size_t r = i / (2 * dk);
        const int j = (int)(r % keep); r /= keep;
        const int h = (int)(r % H), n = (int)(r / H);
        const int src = (T <= Tcap || j < prefix) ? j : T - (Tcap - j);
        const float v = qkv[((size_t)n * T + src) * 3 * HD + (e < dk ? HD : 2 * HD) + h * dk + (e < dk ? e : e - dk)];
        cache[(size_t)n * cache_half_stride + ((size_t)h * Tcap + j) * 2 * dk + e] = v;
    }
}
// evolving caches: the T new K | V rows of request row n are appended to its cache block cidx[n] — logical position len + t; positions
// below `prefix` are stored in place, the others in the ring of Tcap - prefix rows that starts at `head` (a row past the capacity lands on
// the oldest ring row: the sliding-window truncation of cosyvoice2.py:1016-1046 without moving the rows that stay)
__global__ __launch_bounds__(256) void k_flow_cache_append(const float* qkv, float* cache, const int* cidx, size_t stride, int T, int H, int dk,
                                                            int Tcap, int prefix, int len, int head, int N) {
    const size_t total = (size_t)N * H * T * 2 * dk;
    const int HD = H * dk, R = Tcap - prefix;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int e = (int)(i % (2 * dk));
        size_t r = i / (2 * dk);
        const int t = (int)(r % T); r /= T;
        const int h = (int)(r % H), n = (int)(r / H);
        const int p = len + t;
        const int row = p < prefix ? p : prefix + (head + p - prefix) % R;
        const float v = qkv[((size_t)n * T + t) * 3 * HD + (e < dk ? HD : 2 * HD) + h * dk + (e < dk ? e : e - dk)];
        cache[(size_t)cidx[n] * stride + ((size_t)h * Tcap + row) * 2 * dk + e] = v;
    }
}
// last two rows of every request -> conv state [n][2][C] (slots != NULL: state row slots[n] instead of n)
__global__ __launch_bounds__(256) void k_flow_tail2(const float* x, float* st, int N, int T, int C, const int* slots = nullptr) {
    const size_t total = (size_t)N * 2 * C;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % C), p = (int)((i / C) % 2), n = (int)(i / (2 * C));
        const int t = T - 2 + p;
        const float v = t >= 0 ? x[((size_t)n * T + t) * C + c] : 0.0f;
        st[slots ? ((size_t)slots[n] * 2 + p) * C + c : i] = v;
    }
}
// estimator input [2B * T][4 mel] = x | mu | spk | cond, the second (unconditional) half with mu = spk = cond = 0   (cosyvoice_flow.py:2737-2745)
__global__ __launch_bounds__(256) void k_flow_pack(const float* x, const float* mu, const float* spk, const float* cond, float* y, int B, int T,
                                                    int M, int spk_stride = 0) {
    const size_t total = (size_t)2 * B * T * 4 * M;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % (4 * M));
        const size_t row = i / (4 * M);
        const int n = (int)(row / T), t = (int)(row % T), b = n % B;
        const bool un = n >= B;
        const int part = c / M, cc = c % M;
        float v;
        if (part == 0) v = x[((size_t)b * T + t) * M + cc];
        else if (un) v = 0.0f;
        else if (part == 1) v = mu[((size_t)b * T + t) * M + cc];
        else if (part == 2) v = spk[(size_t)b * spk_stride + cc];
        else v = cond ? cond[((size_t)b * T + t) * M + cc] : 0.0f;
        y[i] = v;
    }
}
// x <- x + dt * ((1 + r) d[b] - r d[B + b])   (classifier-free guidance + Euler step, cosyvoice_flow.py:2774-2778)
__global__ __launch_bounds__(256) void k_flow_euler(float* x, const float* d, int B, int T, int M, float dt, float rate) {
    const size_t total = (size_t)B * T * M;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const float g = (1.0f + rate) * d[i] - rate * d[total + i];
        x[i] = x[i] + dt * g;
    }
}
// start noise z [M][T] (given, or the seeded stream) -> x [B][T][M]
__global__ __launch_bounds__(256) void k_flow_noise(const float* z, uint64_t seed, uint32_t stream, float* x, int B, int T, int M) {
    const size_t total = (size_t)B * T * M;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % M), t = (int)((i / M) % T);
        float v;
        if (z) v = z[(size_t)c * T + t];
        else {
            uint32_t w0, w1;
            philox4((uint32_t)(c * T + t), stream, 0u, 0u, (uint32_t)seed, (uint32_t)(seed >> 32), &w0, &w1);
            const float u1 = ((float)(w0 >> 8) + 1.0f) * (1.0f / 16777216.0f), u2 = (float)(w1 >> 8) * (1.0f / 16777216.0f);
            v = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
        }
        x[i] = v;
    }
}
// [B][T][M] -> [B][M][T]
__global__ __launch_bounds__(256) void k_flow_to_bct(const float* x, float* y, int B, int T, int M) {
    const size_t total = (size_t)B * T * M;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int t = (int)(i % T), c = (int)((i / T) % M), b = (int)(i / ((size_t)T * M));
        y[i] = x[((size_t)b * T + t) * M + c];
    }
}
// L2-normalise the speaker embedding (F.normalize, eps 1e-12): one block
__global__ __launch_bounds__(256) void k_flow_l2norm(const float* x, float* y, int C) {
    __shared__ float red[4];
    float s = 0.0f;
    for (int i = threadIdx.x; i < C; i += 256) s += x[i] * x[i];
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float nrm = fmaxf(sqrtf(red[0] + red[1] + red[2] + red[3]), 1e-12f);
    for (int i = threadIdx.x; i < C; i += 256) y[i] = x[i] / nrm;
}
// cond [rows][M]: the first n_feat rows = prompt_feat, the rest 0
__global__ __launch_bounds__(256) void k_flow_cond(const float* feat, float* cond, int rows, int n_feat, int M) {
    const size_t total = (size_t)rows * M;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) cond[i] = (int)(i / M) < n_feat ? feat[i] : 0.0f;
}

// y[row] = a[row] | b[row]
__global__ __launch_bounds__(256) void k_flow_concat2(const float* a, const float* b, float* y, size_t rows, int C) {
    const size_t total = rows * 2 * C;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % (2 * C));
        const size_t r = i / (2 * C);
        y[i] = c < C ? a[r * C + c] : b[r * C + c - C];
    }
}
__global__ void k_flow_slots(int* slots, int N, int B) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) slots[i] = i / B;
}

// ---- estimator transformer block at 256 channels, 8 heads of 64, feed-forward 1024: two launches beside the attention ------------------
// Everything but the attention is row-local, so a block keeps 16 rows in LDS and walks its products there: the operands of a product are the
// rows' three bf16 terms in the order an MFMA operand is read (one 16-byte read per lane, no conflicts), the weights come from a
// fragment-major copy (1 KB per wave request, whole lines) straight into registers.  Products are taken transposed (weight rows x
// activation rows): a lane then holds four neighbouring columns of one row, which is what it stores, normalises and splits.
//   k_tb_qkv   rows = residual + feed-forward parts of the block before, LayerNorm, q | k | v: grid (row tiles, 256-column groups)
//   k_tb_ff    heads' sums of the out product + residual, LayerNorm, GELU feed-forward: grid (row tiles, 4); block y owns a quarter of the hidden
//              columns from ff1 to its two eighths of ff2's sums (they and the residual rows are added by whoever reads them).  Where the attention has
//              left its rows instead (tb_attn), the out product is done by all four
// Sums, LayerNorm statistics and the order of every addition are those of the general launches (k_rows_gemm: K in four runs of 64, or in eight
// from 512 on, added in ascending order), so the two forms give the same bits: the phase of the vocoder's source multiplies what a mel
// differs by some hundred times.
// What one of these leaves for another (parts, the residual rows) lies in the order of the lanes, [row tile][wave][tile][lane] x 4 floats:
// whole lines per request (as [row][256] every request touched 16 lines: k_tb_qkv 12.8 us against 8.3 with plain rows to read).
// Bound by the dependent chain of a block (row loads, three products, two LayerNorm exchanges) and the launch; 896 rows: 16.3 us (qkv) -> 7.4 /
// 8.3 (first / later blocks), 32 us (out, ff1, ff2 as three launches) -> 10.8, with 1.6 for the out product in
// the attention (13.1 with it here, in all four blocks of a row tile; with each product as one sum, four parts and other LayerNorm
// sums: 8.3 / 10.3 and 12.7).  A row's result depends on that row only.
// NT column tiles a wave, 128 NT columns a block.
// Grid: the blocks of a row tile beside each other, in tb_item's order, here and in the attention between them.
template <bool PARTS, int NT>
__global__ __launch_bounds__(512) void k_tb_qkv(const float* h, const float* parts, const float* b2, size_t ps, const bf16_t* w, const float* lnw, const float* lnb,
                                                float* qkv, float* h_out, int M, int N, tb_share share) {
    __shared__ uint4 pl[3 * 8 * 64];
    __shared__ float4 red[256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, fr = lane & 15, kq = lane >> 4;
    const int item = tb_item(share), rt = item / (12 / NT), part = item % (12 / NT);
    const int m = rt * 16 + fr, row = m < M ? m : M - 1, tile = (part * 8 + wave) * NT;
    float4 v[2], lw[2], lb[2];
    uint4 wf[NT][8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int c = (wave * 2 + t) * 16 + kq * 4;
        v[t] = PARTS ? tb_sum(parts + tb_at(rt, wave, t, lane), ps, *reinterpret_cast<const float4*>(b2 + c))
                     : *reinterpret_cast<const float4*>(h + (size_t)row * TB_C + c);
        lw[t] = *reinterpret_cast<const float4*>(lnw + c);
        lb[t] = *reinterpret_cast<const float4*>(lnb + c);
    }
    tb_weights<8, NT>(wf, w, tile, 8, 0, lane);
    if (PARTS && part == 0)
#pragma unroll
        for (int t = 0; t < 2; ++t) *reinterpret_cast<float4*>(h_out + (size_t)(rt * 16 + fr) * TB_C + (wave * 2 + t) * 16 + kq * 4) = v[t];
    tb_layernorm(v, lw, lb, red, wave, lane);
#pragma unroll
    for (int t = 0; t < 2; ++t) tb_put(pl, 8, wave, t, lane, v[t]);
    __syncthreads();
    f32x4 acc[NT];
    tb_product<8, NT>(wf, pl, lane, acc);
    if (m < M)
#pragma unroll
        for (int t = 0; t < NT; ++t)
            *reinterpret_cast<float4*>(qkv + (size_t)m * N + (tile + t) * 16 + kq * 4) = make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
}
// OUT: att = the heads' planes of the out product (os floats apart, rows of 256).  A wave takes two whole rows, which it adds up, normalises and splits by
// itself: a request is a row's 1 KB, and no LayerNorm sum waits for the other waves.  Else att = the attention rows, and the product is done here.
template <bool OUT>
__global__ __launch_bounds__(512) void k_tb_ff(const float* att, size_t os, const float* h, FlowPacked w, const float* b_out, const float* lnw, const float* lnb,
                                               const float* b1, float* parts, size_t ps, int M, tb_share share) {
    __shared__ uint4 pl[3 * 16 * 64];
    __shared__ float4 red[OUT ? 1 : 256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, fr = lane & 15, kq = lane >> 4;
    const int item = tb_item(share), rt = item >> 2, q = item & 3, m0 = rt * 16, m = m0 + fr, row = m < M ? m : M - 1;
    uint4 w1[2][8], w2[2][8];
    float4 bh[2];
    f32x4 acc[2];
    if constexpr (OUT) {
        float4 v[2][8], res[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const size_t r = m0 + 2 * wave + i < M ? m0 + 2 * wave + i : M - 1;
#pragma unroll
            for (int p = 0; p < 8; ++p) v[i][p] = *reinterpret_cast<const float4*>(att + p * os + r * TB_C + lane * 4);
            res[i] = *reinterpret_cast<const float4*>(h + r * TB_C + lane * 4);
        }
        const float4 bo = *reinterpret_cast<const float4*>(b_out + lane * 4), lw = *reinterpret_cast<const float4*>(lnw + lane * 4),
                     lb = *reinterpret_cast<const float4*>(lnb + lane * 4);
        tb_weights<8, 2>(w1, w.ff1, q * 16 + wave * 2, 8, 0, lane);
        const int kb = lane >> 3, g = (lane >> 1) & 3;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = 2 * wave + i;
#pragma unroll
            for (int p = 1; p < 8; ++p) v[i][0] = tb_add(v[i][0], v[i][p]);
            float4 x = tb_add(res[i], tb_add(v[i][0], bo));
            if (q == 0) *reinterpret_cast<float4*>(parts + TB_PARTS * ps + tb_at(rt, kb, (lane >> 2) & 1, (lane & 3) * 16 + r)) = x;
            const float mean = tb_row_sum64((x.x + x.y) + (x.z + x.w)) / (float)TB_C;
            x = make_float4(x.x - mean, x.y - mean, x.z - mean, x.w - mean);
            const float var = tb_row_sum64((x.x * x.x + x.y * x.y) + (x.z * x.z + x.w * x.w));
            const float rstd = rsqrtf(var / (float)TB_C + 1e-5f);
            const tb_split s = tb_split3(make_float4(x.x * rstd * lw.x + lb.x, x.y * rstd * lw.y + lb.y, x.z * rstd * lw.z + lb.z, x.w * rstd * lw.w + lb.w));
            uint2* d = reinterpret_cast<uint2*>(pl + kb * 64 + g * 16 + tb_turn(kb, g, r)) + (lane & 1);
#pragma unroll
            for (int p = 0; p < 3; ++p) d[p * 8 * 128] = s.t[p];
        }
    } else {
        float4 a[2][2], res[2], bo[2], lw[2], lb[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {      // the attention rows: thread = (row, 8 columns)
            const float* s = att + (size_t)(m0 + (tid & 15) < M ? m0 + (tid & 15) : M - 1) * TB_IN + ((tid >> 4) + 32 * i) * 8;
            a[i][0] = *reinterpret_cast<const float4*>(s);
            a[i][1] = *reinterpret_cast<const float4*>(s + 4);
        }
        uint4 wo[2][16];
        tb_weights<16, 2>(wo, w.out, wave * 2, 16, 0, lane);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int c = (wave * 2 + t) * 16 + kq * 4;
            res[t] = *reinterpret_cast<const float4*>(h + (size_t)row * TB_C + c);
            bo[t] = *reinterpret_cast<const float4*>(b_out + c);
            lw[t] = *reinterpret_cast<const float4*>(lnw + c);
            lb[t] = *reinterpret_cast<const float4*>(lnb + c);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const tb_split s0 = tb_split3(a[i][0]), s1 = tb_split3(a[i][1]);
            const int k8 = (tid >> 4) + 32 * i;
#pragma unroll
            for (int p = 0; p < 3; ++p) pl[(p * 16 + (k8 >> 2)) * 64 + (k8 & 3) * 16 + (tid & 15)] = make_uint4(s0.t[p].x, s0.t[p].y, s1.t[p].x, s1.t[p].y);
        }
        __syncthreads();
        tb_product<16, 2>(wo, pl, lane, acc);
        tb_weights<8, 2>(w1, w.ff1, q * 16 + wave * 2, 8, 0, lane);
        float4 n[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            n[t] = tb_add(res[t], tb_add(make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]), bo[t]));
            if (q == 0) *reinterpret_cast<float4*>(parts + TB_PARTS * ps + tb_at(rt, wave, t, lane)) = n[t];
        }
        tb_layernorm(n, lw, lb, red, wave, lane);      // (its barriers: every wave has read the attention rows)
#pragma unroll
        for (int t = 0; t < 2; ++t) tb_put(pl, 8, wave, t, lane, n[t]);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) bh[t] = *reinterpret_cast<const float4*>(b1 + q * 256 + (wave * 2 + t) * 16 + kq * 4);
    if (OUT) tb_weights<8, 2>(w2, w.ff2, wave * 2, 32, q * 8, lane);
    __syncthreads();
    tb_product<8, 2, OUT>(w1, pl, lane, acc);
    if (!OUT) tb_weights<8, 2>(w2, w.ff2, wave * 2, 32, q * 8, lane);
    uint4* const hid = pl + 3 * 8 * 64;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        tb_put(hid, 8, wave, t, lane, make_float4(gelu_f(acc[t][0] + bh[t].x), gelu_f(acc[t][1] + bh[t].y), gelu_f(acc[t][2] + bh[t].z), gelu_f(acc[t][3] + bh[t].w)));
    }
    __syncthreads();
    f32x4 y[2][2];
    tb_runs<8, 4, 2>(w2, hid, lane, y);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const size_t o = tb_at(rt, wave, t, lane);
        if (q == 0) {
            y[1][t] = y[0][t] + y[1][t];
        } else {
            *reinterpret_cast<f32x4*>(parts + (size_t)(2 * q - 1) * ps + o) = y[0][t];
        }
        *reinterpret_cast<f32x4*>(parts + (size_t)(2 * q) * ps + o) = y[1][t];
    }
}
__global__ __launch_bounds__(256) void k_tb_join(const float* parts, const float* b2, size_t ps, float* h, int M) {
    const int i = blockIdx.x * 256 + threadIdx.x, lane = i & 63, col = (i >> 6 & 15) * 16 + (lane >> 4) * 4, m = (i >> 10) * 16 + (lane & 15);
    if (m < M) *reinterpret_cast<float4*>(h + (size_t)m * TB_C + col) = tb_sum(parts + (size_t)i * 4, ps, *reinterpret_cast<const float4*>(b2 + col));
}
// fragment-major copies of every transformer block's weights, or an empty list where a block has other sizes (then the general launches run)
static bool tb_pack(const std::vector<vox_flow_tblock_w>& tb, int C, int inner, std::vector<FlowPacked>& out, void** mem) {
    if (C != TB_C || inner != TB_IN || tb.empty()) return true;
    const vox_conv_w vox_flow_tblock_w::*const which[4] = {&vox_flow_tblock_w::qkv, &vox_flow_tblock_w::out, &vox_flow_tblock_w::ff1, &vox_flow_tblock_w::ff2};
    const int n_of[4] = {3 * TB_IN, TB_C, TB_FF, TB_C}, k_of[4] = {TB_C, TB_IN, TB_C, TB_FF};
    size_t per = 0;
    for (int i = 0; i < 4; ++i) per += (size_t)n_of[i] * k_of[i];
    for (const vox_flow_tblock_w& t : tb)
        for (int i = 0; i < 4; ++i) {
            const vox_conv_w& w = t.*which[i];
            if (w.n_taps != 1 || w.n != n_of[i] || w.cin != k_of[i] || (i == 0) == (w.bias != nullptr) || ((size_t)w.w & 15) || ((size_t)w.bias & 15) ||
                ((size_t)t.ln1_w & 15) || ((size_t)t.ln1_b & 15) || ((size_t)t.ln3_w & 15) || ((size_t)t.ln3_b & 15)) return true;
        }
    if (hipMalloc(mem, per * tb.size() * 2) != hipSuccess) return false;
    bf16_t* p = (bf16_t*)*mem;
    for (const vox_flow_tblock_w& t : tb) {
        FlowPacked f;
        const bf16_t** const to[4] = {&f.qkv, &f.out, &f.ff1, &f.ff2};
        for (int i = 0; i < 4; ++i) {
            const size_t chunks = (size_t)n_of[i] * k_of[i] / 8;
            hipLaunchKernelGGL(k_pack_frag, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, (hipStream_t) nullptr, (const bf16_t*)(t.*which[i]).w, p, k_of[i], chunks);
            *to[i] = p;
            p += chunks * 8;
        }
        out.push_back(f);
    }
    return hipGetLastError() == hipSuccess;
}
static size_t tb_plane(size_t M) { return (M + 15) / 16 * 16 * TB_C; }      // floats of a plane of M rows
static float* tb_heads(float* ws, int M) { return ws + TB_PLANES * tb_plane(M); }
// the attention of a fused block: leaves the out product's planes where its matrix-core form runs (true), else the attention rows (ms, rows and planes:
// CosyVoice2 1 request of 10 tokens 19.9, 19.1; 8 of 28 28.2, 28.0; 16 48.6, 47.0; 32 83.4, 81.3; GLM-4-Voice 6 of 25 49.3, 48.4; 32 148.0, 144.7)
static bool tb_attn(hipStream_t st, FlowAttn a, const FlowPacked* pk, float* ws, int T, int H, int N) {
    const bool parts = pk && H == TB_HEADS && !flow_attn_wv4() && flow_attn_mfma_takes(a, T) && flow_attn_near(a, T, H, N);
    if (parts) { a.wo = pk->out; a.parts = tb_heads(ws, N * T); a.ps = tb_plane(N * T); }
    launch_flow_attn(st, a, T, H, N);
    return parts;
}
// q | k | v of the rows into qkv (before: the block before, which has left them in ws; NULL: of h itself)
static void tb_qkv(hipStream_t st, const FlowPacked& f, const vox_flow_tblock_w& w, const float* h, float* ws, const vox_flow_tblock_w* before, float* qkv, int M) {
    const int tiles = (M + 15) / 16;
    const size_t ps = tb_plane(M);
#define TB_QKV(NT_) \
    do { \
        const dim3 g(tiles * (12 / NT_)); \
        const tb_share share = tb_shares(tiles * (12 / NT_)); \
        if (!before) hipLaunchKernelGGL((k_tb_qkv<false, NT_>), g, dim3(512), 0, st, h, ws, nullptr, ps, f.qkv, w.ln1_w, w.ln1_b, qkv, ws, M, 3 * TB_IN, share); \
        else hipLaunchKernelGGL((k_tb_qkv<true, NT_>), g, dim3(512), 0, st, h, ws, before->ff2.bias, ps, f.qkv, w.ln1_w, w.ln1_b, qkv, ws + (TB_PLANES - 1) * ps, M, \
                                3 * TB_IN, share); \
    } while (0)
    // A block adds up its rows' planes (128 KB) whatever it multiplies them by (64 KB a tile of a wave): where two tiles a wave make more blocks than
    // CUs, three or four move less as long as theirs fit.  Detokenizers, ms, two, three and four tiles a wave: CosyVoice2 6 requests of 28 tokens
    // (672 rows) 26.3, 26.9, 27.5; 7 (784) 28.3, 27.4, 28.1; 8 (896) 28.8, 28.1, 28.7; GLM-4-Voice 5 (860) 37.6, 36.7, 37.5; 6 (1032) 49.6, 51.8, 49.4.
    if (tiles * 6 <= 256 || tiles * 3 > 256) TB_QKV(2);
    else if (tiles * 4 <= 256) TB_QKV(3);
    else TB_QKV(4);
#undef TB_QKV
}
// att: the attention rows, or (from_parts) the heads' planes of the out product, which the attention has left behind the block's own planes
static void tb_ff(hipStream_t st, const FlowPacked& f, const vox_flow_tblock_w& w, const float* att, float* h, float* ws, bool first, bool last, int M,
                  bool from_parts) {
    const size_t ps = tb_plane(M);
    const float* in = first ? h : ws + (TB_PLANES - 1) * ps;
    const dim3 g((M + 15) / 16 * 4);
    const tb_share share = tb_shares((M + 15) / 16 * 4);
    if (from_parts) hipLaunchKernelGGL(k_tb_ff<true>, g, dim3(512), 0, st, tb_heads(ws, M), ps, in, f, w.out.bias, w.ln3_w, w.ln3_b, w.ff1.bias, ws, ps, M, share);
    else hipLaunchKernelGGL(k_tb_ff<false>, g, dim3(512), 0, st, att, 0, in, f, w.out.bias, w.ln3_w, w.ln3_b, w.ff1.bias, ws, ps, M, share);
    if (last) hipLaunchKernelGGL(k_tb_join, dim3((unsigned)((M + 15) / 16 * 4)), dim3(256), 0, st, ws, w.ff2.bias, ps, h, M);
}

struct vox_flow {
    vox_ctx* ctx;
    vox_flow_config cfg;
    vox_flow_weights w;
    std::vector<vox_flow_conformer_w> enc;
    std::vector<vox_flow_resnet_w> resnets;
    std::vector<vox_flow_tblock_w> tblocks;
    std::vector<FlowPacked> packed;         // per transformer block, or empty
    void* packed_mem = nullptr;
    float* tb_ws = nullptr;                 // their scratch: TB_PLANES + TB_HEADS planes of the most rows
    int max_batch, max_T, max_prompt_T, n_res, n_att;
    std::vector<float> dt;                  // host: Euler step sizes
    float* tb = nullptr;                    // [n_steps][n_res][C]: mlp_r(Mish(time_mlp(emb_s)))
    float* buf[10] = {};
    size_t buf_floats = 0;
    float *spk = nullptr, *pe = nullptr, *pp = nullptr;
    int* slots = nullptr;                   // [2 * max_batch]: conv-state slot (= guidance half) of every estimator request row
    // ResNet blocks: block1's causal conv with the block's residual 1-tap conv stacked behind it as C more output columns (its weight in
    // the tap that reads the current row, zeros in the other taps): one launch less per ResNet block, 140 per chunk
    std::vector<vox_conv_w> conv1x;
    std::vector<void*> conv1x_mem;
    // static prompt caches
    float *enc_kv = nullptr, *up_kv = nullptr, *att_kv = nullptr, *cnn1 = nullptr, *cnn2 = nullptr;
    int enc_len = 0, up_len = 0, att_len = 0, cnn1_w = 0;
    bool have_prompt = false;
    // per-request evolving caches (use_detokenizer_cache=True, cosyvoice2.py:1010-1083): slot-major copies of the five caches, each
    // slot starting as a copy of the prompt's; the K/V caches keep their first `prefix` rows and run the rest as a ring
    struct SlotState { int enc_len = 0, enc_head = 0, up_len = 0, up_head = 0, att_len = 0, att_head = 0; bool live = false; };
    int n_slots = 0;
    std::vector<SlotState> slot;
    float *s_enc = nullptr, *s_up = nullptr, *s_att = nullptr, *s_cnn1 = nullptr, *s_cnn2 = nullptr;
    int *s_eidx = nullptr, *s_cidx = nullptr;      // device: slot of request b [max_batch]; cache block of estimator row n [2 max_batch]
};

static inline int flow_res_cin(const vox_flow_config& c, int r) { return r == 0 ? 4 * c.mel : (r == 1 + c.est_mid ? 2 * c.est_ch : c.est_ch); }

extern "C" {

void vox_flow_destroy(vox_flow* m) {
    if (!m) return;
    for (int i = 0; i < 10; ++i) (void)hipFree(m->buf[i]);
    (void)hipFree(m->tb); (void)hipFree(m->spk); (void)hipFree(m->pe); (void)hipFree(m->pp); (void)hipFree(m->slots);
    (void)hipFree(m->enc_kv); (void)hipFree(m->up_kv); (void)hipFree(m->att_kv); (void)hipFree(m->cnn1); (void)hipFree(m->cnn2);
    (void)hipFree(m->s_enc); (void)hipFree(m->s_up); (void)hipFree(m->s_att); (void)hipFree(m->s_cnn1); (void)hipFree(m->s_cnn2);
    (void)hipFree(m->s_eidx); (void)hipFree(m->s_cidx);
    for (void* p : m->conv1x_mem) (void)hipFree(p);
    (void)hipFree(m->packed_mem); (void)hipFree(m->tb_ws);
    delete m;
}

}  // extern "C"

// Rows up to which the flows' GEMMs take the few-row kernels (k_rows_gemm where the shape is eligible, the LDS-staged 16-row kernel
// otherwise) and normalise inside them.  Unbounded by default: the few-row kernels tile any row count, and ONE kernel per shape at
// every batch size is what keeps a request's mel independent of the batch it shares (k_rows_gemm sums its K quarters in a different
// order than the staged kernels).  VOX_FLOW_ROWS=<n> restores a row bound (A/B timing).
static int flow_skinny_rows() {
    static const int v = [] { const char* e = getenv("VOX_FLOW_ROWS"); return e ? atoi(e) : (1 << 30); }();
    return v;
}
#define FLOW_SKINNY_ROWS flow_skinny_rows()
static const int FLOW_OFF0[4] = {0, 0, 0, 0};
static const int FLOW_OFF_C3[3] = {2, 1, 0};            // causal k3
static const int FLOW_OFF_C5[5] = {4, 3, 2, 1, 0};      // causal k5 (Upsample1D after its left pad of 4)
static const int FLOW_OFF_LA[8] = {0, -1, -2, -3, -4, -5, -6, -7};   // look-ahead k (PreLookaheadLayer.conv1)

// one conformer layer (norm_mha -> rel-pos attention -> residual; norm_ff -> SiLU FFN -> residual) on x [n * T][D] in place
// LayerNorm(w, b, eps) followed by a one-tap GEMM of the normalised rows.  Calls that take the few-row GEMM normalise inside its operand
// staging (one launch less per attention / feed-forward half); larger batches normalise into `scratch` first.
static int ln_gemm(hipStream_t st, const vox_conv_w& w, const float* x, const float* lw, const float* lb, float eps, float* scratch, int n, int L,
                   float* out, int gelu) {
    if (n * L <= g_conv_skinny_rows && w.n_taps == 1)
        return conv_gemm(st, w, x, nullptr, nullptr, n, L, 0, FLOW_OFF0, out, nullptr, nullptr, gelu, nullptr, nullptr, 0, nullptr, lw, lb, eps);
    hipLaunchKernelGGL(k_flow_ln, dim3((n * L + 3) / 4), dim3(256), 0, st, x, lw, lb, scratch, w.cin, eps, 1.0f, 0, (const float*)nullptr, 1, n * L);
    return conv_gemm(st, w, scratch, nullptr, nullptr, n, L, 0, FLOW_OFF0, out, nullptr, nullptr, gelu);
}
// evolving mode (eidx != NULL): `cache` is layer l of the slot-major cache, request b reads and appends to block eidx[b] (stride
// slot_stride) whose rows past `prefix` form a ring starting at `head`
static int flow_conformer(vox_flow* m, hipStream_t st, const vox_flow_conformer_w& w, float* x, int n, int T, const float* cache, int Tc, int Tcap,
                          float* store_cache, int store_cap, int store_prefix, float** B, const int* eidx = nullptr, size_t slot_stride = 0,
                          int head = 0) {
    const vox_flow_config& c = m->cfg;
    const int D = c.dim, H = c.enc_heads, dk = D / H, S = Tc + T;
    if (S > FLOW_MAXKEYS) return vox_fail(VOX_ERR_INVALID, "flow: %d keys > %d", S, FLOW_MAXKEYS);
    float *nrm = B[0], *qkv = B[1], *att = B[2];
    VOX_TRY(ln_gemm(st, w.qkv, x, w.ln_mha_w, w.ln_mha_b, 1e-12f, nrm, n, T, qkv, 0));
    VOX_TRY(conv_gemm(st, w.pos, m->pe, nullptr, nullptr, 1, 2 * S - 1, 0, FLOW_OFF0, m->pp, nullptr, nullptr, 0));
    FlowAttn a{qkv, cache, m->pp, w.bias_u, w.bias_v, att, T, H, dk, Tc, Tcap, 0, eidx ? slot_stride : 0, 1.0f / sqrtf((float)dk)};
    a.cidx = eidx; a.prefix = store_prefix; a.ring_head = head;
    launch_flow_attn(st, a, T, H, n);
    if (eidx)
        hipLaunchKernelGGL(k_flow_cache_append, dim3(ew_grid((size_t)n * H * T * 2 * dk)), dim3(256), 0, st, qkv, const_cast<float*>(cache), eidx,
                           slot_stride, T, H, dk, Tcap, store_prefix, Tc, head, n);
    else if (store_cache)
        hipLaunchKernelGGL(k_flow_cache_store, dim3(ew_grid((size_t)H * store_cap * 2 * dk)), dim3(256), 0, st, qkv, store_cache, T, H, dk, store_cap,
                           store_prefix, (size_t)0, 1);
    VOX_TRY(conv_gemm(st, w.out, att, nullptr, nullptr, n, T, 0, FLOW_OFF0, x, x, nullptr, 0));
    VOX_TRY(ln_gemm(st, w.w1, x, w.ln_ff_w, w.ln_ff_b, 1e-12f, nrm, n, T, qkv, 0));
    hipLaunchKernelGGL(k_flow_act, dim3(ew_grid((size_t)n * T * c.enc_ffn)), dim3(256), 0, st, qkv, (size_t)n * T * c.enc_ffn, 2);
    VOX_TRY(conv_gemm(st, w.w2, qkv, nullptr, nullptr, n, T, 0, FLOW_OFF0, x, x, nullptr, 0));
    return VOX_OK;
}

// tokens [B][T] -> mel frames x [B][2T][mel] (time-major, in m->buf[9]); init: B == 1, caches are written instead of read
// evolve != NULL (decode only): the per-request caches of the given slot state (all requests of the call share one state: equal cache
// lengths, as the reference's batched caches require) are read through m->s_eidx / m->s_cidx and appended to
static int flow_run(vox_flow* m, hipStream_t st, const int32_t* tokens, int B, int T, bool init, const float* prompt_feat, int n_feat,
                    const float* noise, uint64_t seed, uint32_t nstream, float* mu_out, const vox_flow::SlotState* evolve = nullptr) {
    const vox_flow_config& c = m->cfg;
    const vox_flow_weights& w = m->w;
    const int D = c.dim, M = c.mel, C = c.est_ch, T2 = 2 * T, H = c.enc_heads, dk = D / H, inner = c.est_heads * c.est_head_dim;
    float** Bf = m->buf;
    g_conv_planes = 3;
    struct RowsGuard { ~RowsGuard() { g_conv_skinny_rows = 48; g_conv_rows_gemm = false; } } rows_guard;      // also on the error returns
    g_conv_skinny_rows = FLOW_SKINNY_ROWS; g_conv_rows_gemm = true;
    // ---- encoder ----
    float* x = Bf[3];
    hipLaunchKernelGGL(k_flow_embed, dim3(ew_grid((size_t)B * T * D)), dim3(256), 0, st, tokens, w.embedding, Bf[0], (size_t)B * T, D);
    VOX_TRY(conv_gemm(st, w.embed_lin, Bf[0], nullptr, nullptr, B, T, 0, FLOW_OFF0, Bf[1], nullptr, nullptr, 0));
    hipLaunchKernelGGL(k_flow_ln, dim3((B * T + 3) / 4), dim3(256), 0, st, Bf[1], w.embed_ln_w, w.embed_ln_b, x, D, 1e-5f, sqrtf((float)D), 0, nullptr, 1, B * T);
    // PreLookaheadLayer (empty context): conv k(pre+1) looking ahead, leaky_relu, causal conv k3, residual
    VOX_TRY(conv_gemm(st, w.pre1, x, nullptr, nullptr, B, T, 0, FLOW_OFF_LA, Bf[0], nullptr, nullptr, 0));
    hipLaunchKernelGGL(k_flow_act, dim3(ew_grid((size_t)B * T * D)), dim3(256), 0, st, Bf[0], (size_t)B * T * D, 3);
    VOX_TRY(conv_gemm(st, w.pre2, Bf[0], nullptr, nullptr, B, T, 0, FLOW_OFF_C3, x, x, nullptr, 0));
    {
        const int Tc = init ? 0 : (evolve ? evolve->enc_len : m->enc_len), S = Tc + T, cap = c.max_cache / 2;
        hipLaunchKernelGGL(k_flow_relpos, dim3(ew_grid((size_t)(2 * S - 1) * D)), dim3(256), 0, st, m->pe, S, D);
        const size_t lay = (size_t)H * cap * 2 * dk;
        for (int l = 0; l < c.enc_layers; ++l) {
            float* kv = (evolve ? m->s_enc : m->enc_kv) + (size_t)l * lay;
            VOX_TRY(flow_conformer(m, st, m->enc[l], x, B, T, init ? nullptr : kv, Tc, cap, init ? kv : nullptr, cap, c.prefix / 2, Bf,
                                   evolve ? m->s_eidx : nullptr, (size_t)c.enc_layers * lay, evolve ? evolve->enc_head : 0));
        }
        if (init) m->enc_len = T < cap ? T : cap;
    }
    // Upsample1D (nearest x2, causal conv k5), up_embed, the second conformer stack, after_norm, encoder_proj
    hipLaunchKernelGGL(k_flow_repeat2, dim3(ew_grid((size_t)B * T2 * D)), dim3(256), 0, st, x, Bf[0], (size_t)B * T, D);
    VOX_TRY(conv_gemm(st, w.up_conv, Bf[0], nullptr, nullptr, B, T2, 0, FLOW_OFF_C5, Bf[1], nullptr, nullptr, 0));
    VOX_TRY(conv_gemm(st, w.up_embed_lin, Bf[1], nullptr, nullptr, B, T2, 0, FLOW_OFF0, Bf[0], nullptr, nullptr, 0));
    hipLaunchKernelGGL(k_flow_ln, dim3((B * T2 + 3) / 4), dim3(256), 0, st, Bf[0], w.up_embed_ln_w, w.up_embed_ln_b, x, D, 1e-5f, sqrtf((float)D), 0, nullptr, 1, B * T2);
    {
        const int Tc = init ? 0 : (evolve ? evolve->up_len : m->up_len), S = Tc + T2, cap = c.max_cache;
        hipLaunchKernelGGL(k_flow_relpos, dim3(ew_grid((size_t)(2 * S - 1) * D)), dim3(256), 0, st, m->pe, S, D);
        const size_t lay = (size_t)H * cap * 2 * dk;
        for (int l = 0; l < c.up_layers; ++l) {
            float* kv = (evolve ? m->s_up : m->up_kv) + (size_t)l * lay;
            VOX_TRY(flow_conformer(m, st, m->enc[c.enc_layers + l], x, B, T2, init ? nullptr : kv, Tc, cap, init ? kv : nullptr, cap, c.prefix, Bf,
                                   evolve ? m->s_eidx : nullptr, (size_t)c.up_layers * lay, evolve ? evolve->up_head : 0));
        }
        if (init) m->up_len = T2 < cap ? T2 : cap;
    }
    hipLaunchKernelGGL(k_flow_ln, dim3((B * T2 + 3) / 4), dim3(256), 0, st, x, w.after_w, w.after_b, Bf[0], D, 1e-5f, 1.0f, 0, nullptr, 1, B * T2);
    float* mu = Bf[8];
    VOX_TRY(conv_gemm(st, w.enc_proj, Bf[0], nullptr, nullptr, B, T2, 0, FLOW_OFF0, mu, nullptr, nullptr, 0));
    if (mu_out) (void)hipMemcpyAsync(mu_out, mu, (size_t)B * T2 * M * 4, hipMemcpyDeviceToDevice, st);
    // ---- conditional flow matching: n_steps Euler steps of the estimator on the doubled (guidance) batch ----
    float *xs = Bf[9], *cond = Bf[7];
    if (init) hipLaunchKernelGGL(k_flow_cond, dim3(ew_grid((size_t)T2 * M)), dim3(256), 0, st, prompt_feat, cond, T2, n_feat, M);
    hipLaunchKernelGGL(k_flow_noise, dim3(ew_grid((size_t)B * T2 * M)), dim3(256), 0, st, noise, seed, nstream, xs, B, T2, M);
    const int N = 2 * B, capA = c.max_cache, hd = c.est_head_dim, HE = c.est_heads;
    const size_t att_layer = (size_t)HE * capA * 2 * hd, att_half = (size_t)c.n_steps * m->n_att * att_layer;
    const int Tc = init ? 0 : (evolve ? evolve->att_len : m->att_len);
    if (Tc + T2 > FLOW_MAXKEYS) return vox_fail(VOX_ERR_INVALID, "flow: chunk too long");
    hipLaunchKernelGGL(k_flow_slots, dim3((N + 63) / 64), dim3(64), 0, st, m->slots, N, B);
    // conv-state row / attention-cache block of estimator row n: the guidance half (shared prompt caches) or 2 slot + half (evolving)
    const int* crow = evolve ? m->s_cidx : m->slots;
    const int srows = evolve ? 2 * m->n_slots : 2;             // state rows per (step, resnet) block
    for (int s = 0; s < c.n_steps; ++s) {
        float *hA = Bf[0], *a1 = Bf[1], *a2 = Bf[2], *a3 = Bf[3], *skip = Bf[4], *cat = Bf[5], *hB = Bf[6];
        hipLaunchKernelGGL(k_flow_pack, dim3(ew_grid((size_t)N * T2 * 4 * M)), dim3(256), 0, st, xs, mu, m->spk, init ? cond : nullptr, cat, B, T2, M);
        const float* in = cat;
        float* h = hA;
        int li = 0;
        for (int r = 0; r < m->n_res; ++r) {
            const vox_flow_resnet_w& rw = m->resnets[r];
            const int cin = flow_res_cin(c, r);
            if (r == m->n_res - 1) {      // up block: pack([x, skip]) along channels
                hipLaunchKernelGGL(k_flow_concat2, dim3(ew_grid((size_t)N * T2 * 2 * C)), dim3(256), 0, st, in, skip, cat, (size_t)N * T2, C);
                in = cat;
            }
            h = (in == hA) ? hB : hA;
            float* st1 = (evolve ? m->s_cnn1 : m->cnn1) + ((size_t)s * m->n_res + r) * srows * 2 * m->cnn1_w;
            float* st2 = (evolve ? m->s_cnn2 : m->cnn2) + ((size_t)s * m->n_res + r) * srows * 2 * C;
            if (init) hipLaunchKernelGGL(k_flow_tail2, dim3(ew_grid((size_t)N * 2 * cin)), dim3(256), 0, st, in, st1, N, T2, cin, (const int*)nullptr);
            // block1: (cached) causal conv k3 -> LayerNorm -> Mish, + the time projection; block2 likewise; + res_conv(x)
            const bool fold = !m->conv1x.empty();      // a1 = [block1 conv | res_conv(in)], 2 C wide
            VOX_TRY(conv_gemm(st, fold ? m->conv1x[r] : rw.conv1, in, init ? nullptr : st1, crow, N, T2, 2, FLOW_OFF_C3, a1, nullptr, nullptr, 0));
            if (evolve) hipLaunchKernelGGL(k_flow_tail2, dim3(ew_grid((size_t)N * 2 * cin)), dim3(256), 0, st, in, st1, N, T2, cin, crow);
            hipLaunchKernelGGL(k_flow_ln, dim3((N * T2 + 3) / 4), dim3(256), 0, st, a1, rw.ln1_w, rw.ln1_b, a2, C, 1e-5f, 1.0f, 1,
                               m->tb + ((size_t)s * m->n_res + r) * C, N * T2, N * T2, fold ? 2 * C : 0, 0);
            if (init) hipLaunchKernelGGL(k_flow_tail2, dim3(ew_grid((size_t)N * 2 * C)), dim3(256), 0, st, a2, st2, N, T2, C, (const int*)nullptr);
            VOX_TRY(conv_gemm(st, rw.conv2, a2, init ? nullptr : st2, crow, N, T2, 2, FLOW_OFF_C3, fold ? a3 : a1, nullptr, nullptr, 0));
            if (evolve) hipLaunchKernelGGL(k_flow_tail2, dim3(ew_grid((size_t)N * 2 * C)), dim3(256), 0, st, a2, st2, N, T2, C, crow);
            if (fold) {      // h = Mish(LayerNorm(block2 conv)) + res_conv(in)
                hipLaunchKernelGGL(k_flow_ln, dim3((N * T2 + 3) / 4), dim3(256), 0, st, a3, rw.ln2_w, rw.ln2_b, h, C, 1e-5f, 1.0f, 1, a1 + C, 1, N * T2, 0,
                                   2 * C);
            } else {
                hipLaunchKernelGGL(k_flow_ln, dim3((N * T2 + 3) / 4), dim3(256), 0, st, a1, rw.ln2_w, rw.ln2_b, a2, C, 1e-5f, 1.0f, 1, nullptr, 1, N * T2);
                VOX_TRY(conv_gemm(st, rw.res, in, nullptr, nullptr, N, T2, 0, FLOW_OFF0, h, a2, nullptr, 0));       // h = block2 + res_conv(in)
            }
            for (int j = 0; j < c.est_blocks; ++j, ++li) {
                const vox_flow_tblock_w& tw = m->tblocks[li];
                float* kv = (evolve ? m->s_att : m->att_kv) + ((size_t)s * m->n_att + li) * att_layer;
                const FlowPacked* pk = m->packed.empty() ? nullptr : &m->packed[li];
                if (pk) tb_qkv(st, *pk, tw, h, m->tb_ws, j ? &m->tblocks[li - 1] : nullptr, a2, N * T2);
                else VOX_TRY(ln_gemm(st, tw.qkv, h, tw.ln1_w, tw.ln1_b, 1e-5f, a1, N, T2, a2, 0));
                FlowAttn a{a2, init ? nullptr : kv, nullptr, nullptr, nullptr, a3, T2, HE, hd, Tc, capA, B, att_half, 1.0f / sqrtf((float)hd)};
                if (evolve) { a.cidx = m->s_cidx; a.prefix = c.prefix; a.ring_head = evolve->att_head; }
                const bool parts = tb_attn(st, a, pk, m->tb_ws, T2, HE, N);
                if (evolve)
                    hipLaunchKernelGGL(k_flow_cache_append, dim3(ew_grid((size_t)N * HE * T2 * 2 * hd)), dim3(256), 0, st, a2, kv, m->s_cidx, att_half,
                                       T2, HE, hd, capA, c.prefix, Tc, evolve->att_head, N);
                if (init)
                    hipLaunchKernelGGL(k_flow_cache_store, dim3(ew_grid((size_t)N * HE * capA * 2 * hd)), dim3(256), 0, st, a2, kv, T2, HE, hd, capA,
                                       c.prefix, att_half, N);
                if (pk) { tb_ff(st, *pk, tw, a3, h, m->tb_ws, j == 0, j + 1 == c.est_blocks, N * T2, parts); continue; }
                VOX_TRY(conv_gemm(st, tw.out, a3, nullptr, nullptr, N, T2, 0, FLOW_OFF0, h, h, nullptr, 0));
                VOX_TRY(ln_gemm(st, tw.ff1, h, tw.ln3_w, tw.ln3_b, 1e-5f, a1, N, T2, a2, 1));
                VOX_TRY(conv_gemm(st, tw.ff2, a2, nullptr, nullptr, N, T2, 0, FLOW_OFF0, h, h, nullptr, 0));
            }
            in = h;
            if (r == 0) {                  // down block: keep the skip, then its (uncached) causal conv
                (void)hipMemcpyAsync(skip, h, (size_t)N * T2 * C * 4, hipMemcpyDeviceToDevice, st);
                float* o = (h == hA) ? hB : hA;
                VOX_TRY(conv_gemm(st, w.down_conv, skip, nullptr, nullptr, N, T2, 0, FLOW_OFF_C3, o, nullptr, nullptr, 0));
                in = o;
            }
        }
        VOX_TRY(conv_gemm(st, w.up_conv2, in, nullptr, nullptr, N, T2, 0, FLOW_OFF_C3, a1, nullptr, nullptr, 0));
        VOX_TRY(conv_gemm(st, w.final_conv, a1, nullptr, nullptr, N, T2, 0, FLOW_OFF_C3, a2, nullptr, nullptr, 0));
        hipLaunchKernelGGL(k_flow_ln, dim3((N * T2 + 3) / 4), dim3(256), 0, st, a2, w.final_ln_w, w.final_ln_b, a1, C, 1e-5f, 1.0f, 1, nullptr, 1, N * T2);
        VOX_TRY(conv_gemm(st, w.final_proj, a1, nullptr, nullptr, N, T2, 0, FLOW_OFF0, a2, nullptr, nullptr, 0));
        hipLaunchKernelGGL(k_flow_euler, dim3(ew_grid((size_t)B * T2 * M)), dim3(256), 0, st, xs, a2, B, T2, M, m->dt[s], c.cfg_rate);
    }
    if (init) m->att_len = T2 < capA ? T2 : capA;
    g_conv_skinny_rows = 48; g_conv_rows_gemm = false;
    return VOX_OK;
}

extern "C" {

int vox_flow_create(vox_ctx* ctx, const vox_flow_config* cfg, const vox_flow_weights* w, int max_batch, int max_T, int max_prompt_T,
                    const float* time_emb, const float* dt, vox_flow** out) {
    if (!ctx || !cfg || !w || !out || !time_emb || !dt) return vox_fail(VOX_ERR_INVALID, "flow_create: NULL");
    const vox_flow_config& c = *cfg;
    if (c.dim % c.enc_heads || c.dim / c.enc_heads > 128 || c.est_head_dim > 128 || c.dim % 32 || c.est_ch % 32 || (4 * c.mel) % 32 ||
        (c.est_heads * c.est_head_dim) % 32 || c.enc_ffn % 32 || c.spk_dim % 32 || c.pre_lookahead + 1 > 8 || max_batch < 1 || max_T < 1 ||
        max_prompt_T < 1 || c.n_steps < 1)
        return vox_fail(VOX_ERR_INVALID, "flow_create: bad config");
    vox_flow* m = new vox_flow();
    m->ctx = ctx; m->cfg = c; m->w = *w; m->max_batch = max_batch; m->max_T = max_T; m->max_prompt_T = max_prompt_T;
    m->n_res = 2 + c.est_mid; m->n_att = m->n_res * c.est_blocks;
    m->enc.assign(w->enc, w->enc + c.enc_layers + c.up_layers);
    m->resnets.assign(w->resnets, w->resnets + m->n_res);
    m->tblocks.assign(w->tblocks, w->tblocks + m->n_att);
    m->dt.assign(dt, dt + c.n_steps);
    const int D = c.dim, C = c.est_ch, TE = 4 * C, inner = c.est_heads * c.est_head_dim, dk = D / c.enc_heads;
    size_t rows = (size_t)2 * max_batch * 2 * max_T;
    if ((size_t)2 * 2 * (max_prompt_T + 3) > rows) rows = (size_t)2 * 2 * (max_prompt_T + 3);
    size_t wmax = 3 * (size_t)D;
    for (size_t v : {(size_t)c.enc_ffn, (size_t)4 * C, (size_t)3 * inner, (size_t)4 * c.mel, (size_t)TE}) wmax = v > wmax ? v : wmax;
    m->buf_floats = rows * wmax;
    m->cnn1_w = 4 * c.mel > 2 * C ? 4 * c.mel : 2 * C;
    const size_t capE = c.max_cache / 2, capU = c.max_cache;
    bool ok = true;
    auto alloc = [&](float** p, size_t n) { ok = ok && hipMalloc((void**)p, n * 4) == hipSuccess; };
    for (int i = 0; i < 10; ++i) alloc(&m->buf[i], m->buf_floats);
    alloc(&m->tb, (size_t)c.n_steps * m->n_res * C);
    alloc(&m->spk, c.mel);
    alloc(&m->pe, (size_t)2 * FLOW_MAXKEYS * D);
    alloc(&m->pp, (size_t)2 * FLOW_MAXKEYS * D);
    alloc(&m->enc_kv, (size_t)c.enc_layers * c.enc_heads * capE * 2 * dk);
    alloc(&m->up_kv, (size_t)c.up_layers * c.enc_heads * capU * 2 * dk);
    alloc(&m->att_kv, (size_t)2 * c.n_steps * m->n_att * c.est_heads * c.max_cache * 2 * c.est_head_dim);
    alloc(&m->cnn1, (size_t)c.n_steps * m->n_res * 4 * m->cnn1_w);
    alloc(&m->cnn2, (size_t)c.n_steps * m->n_res * 4 * C);
    ok = ok && hipMalloc((void**)&m->slots, (size_t)2 * (max_batch > 1 ? max_batch : 1) * 4) == hipSuccess;
    static const bool resfold = [] { const char* e = getenv("VOX_FLOW_RESFOLD"); return !(e && e[0] == '0'); }();
    for (int r = 0; r < m->n_res && ok && resfold; ++r) {
        const vox_flow_resnet_w& rw = m->resnets[r];
        if (rw.conv1.n_taps != 3 || rw.res.n_taps != 1 || rw.conv1.n != C || rw.res.n != C || rw.conv1.cin != rw.res.cin) { m->conv1x.clear(); break; }
        const size_t cin = rw.conv1.cin, blk = (size_t)C * cin * 2;      // bytes of one tap's [C][cin] bf16 block
        char* wx = nullptr; float* bx = nullptr;
        ok = hipMalloc((void**)&wx, 3 * 2 * blk) == hipSuccess && hipMalloc((void**)&bx, (size_t)2 * C * 4) == hipSuccess;
        if (wx) m->conv1x_mem.push_back(wx);
        if (bx) m->conv1x_mem.push_back(bx);
        if (!ok) break;
        (void)hipMemset(wx, 0, 3 * 2 * blk); (void)hipMemset(bx, 0, (size_t)2 * C * 4);
        for (int t = 0; t < 3; ++t) (void)hipMemcpy(wx + (size_t)t * 2 * blk, (const char*)rw.conv1.w + (size_t)t * blk, blk, hipMemcpyDeviceToDevice);
        (void)hipMemcpy(wx + (size_t)2 * 2 * blk + blk, rw.res.w, blk, hipMemcpyDeviceToDevice);      // FLOW_OFF_C3: tap 2 reads the current row
        if (rw.conv1.bias) (void)hipMemcpy(bx, rw.conv1.bias, (size_t)C * 4, hipMemcpyDeviceToDevice);
        if (rw.res.bias) (void)hipMemcpy(bx + C, rw.res.bias, (size_t)C * 4, hipMemcpyDeviceToDevice);
        vox_conv_w cx = rw.conv1;
        cx.w = wx; cx.bias = bx; cx.n = 2 * C; cx.bias_mod = 0;
        m->conv1x.push_back(cx);
    }
    ok = ok && tb_pack(m->tblocks, C, inner, m->packed, &m->packed_mem);
    if (!m->packed.empty()) alloc(&m->tb_ws, (TB_PLANES + TB_HEADS) * tb_plane(rows));
    if (!ok) { vox_flow_destroy(m); return vox_fail(VOX_ERR_NOMEM, "flow_create: hipMalloc failed"); }
    // time projections of every Euler step and resnet, once: tb[s][r] = mlp_r(Mish(linear_2(SiLU(linear_1(emb_s)))))
    hipStream_t st = nullptr;
    g_conv_planes = 3;
    int rc = VOX_OK;
    (void)hipMemcpy(m->buf[0], time_emb, (size_t)c.n_steps * 4 * c.mel * 4, hipMemcpyHostToDevice);
    rc = conv_gemm(st, w->time1, m->buf[0], nullptr, nullptr, 1, c.n_steps, 0, FLOW_OFF0, m->buf[1], nullptr, nullptr, 0);
    hipLaunchKernelGGL(k_flow_act, dim3(ew_grid((size_t)c.n_steps * TE)), dim3(256), 0, st, m->buf[1], (size_t)c.n_steps * TE, 2);
    if (rc == VOX_OK) rc = conv_gemm(st, w->time2, m->buf[1], nullptr, nullptr, 1, c.n_steps, 0, FLOW_OFF0, m->buf[2], nullptr, nullptr, 0);
    hipLaunchKernelGGL(k_flow_act, dim3(ew_grid((size_t)c.n_steps * TE)), dim3(256), 0, st, m->buf[2], (size_t)c.n_steps * TE, 1);
    for (int r = 0; r < m->n_res && rc == VOX_OK; ++r) {
        rc = conv_gemm(st, m->resnets[r].mlp, m->buf[2], nullptr, nullptr, 1, c.n_steps, 0, FLOW_OFF0, m->buf[3], nullptr, nullptr, 0);
        (void)hipMemcpy2DAsync(m->tb + (size_t)r * C, (size_t)m->n_res * C * 4, m->buf[3], (size_t)C * 4, (size_t)C * 4, c.n_steps,
                               hipMemcpyDeviceToDevice, st);
    }
    if (hipStreamSynchronize(st) != hipSuccess || rc != VOX_OK) { vox_flow_destroy(m); return rc != VOX_OK ? rc : vox_fail(VOX_ERR_HIP, "flow_create: time MLP failed"); }
    *out = m;
    return VOX_OK;
}

int vox_flow_set_prompt(vox_flow* m, void* stream, const int32_t* prompt_tokens, int n_prompt, const float* prompt_feat,
                        const float* embedding, const float* noise, uint64_t seed, uint32_t noise_stream, float* prompt_mel) {
    if (!m || !prompt_tokens || !prompt_feat || !embedding) return vox_fail(VOX_ERR_INVALID, "flow_set_prompt: NULL");
    if (n_prompt < 3 || n_prompt > m->max_prompt_T) return vox_fail(VOX_ERR_INVALID, "flow_set_prompt: %d prompt tokens out of range", n_prompt);
    hipStream_t st = (hipStream_t)stream;
    const vox_flow_config& c = m->cfg;
    const int T = n_prompt + 3;
    // speaker vector: spk_embed_affine_layer(normalize(embedding))
    hipLaunchKernelGGL(k_flow_l2norm, dim3(1), dim3(256), 0, st, embedding, m->buf[0], c.spk_dim);
    g_conv_planes = 3;
    VOX_TRY(conv_gemm(st, m->w.spk, m->buf[0], nullptr, nullptr, 1, 1, 0, FLOW_OFF0, m->spk, nullptr, nullptr, 0));
    // tokens = prompt + its first three again (cosyvoice2.py:864-867)
    int* tok = reinterpret_cast<int*>(m->buf[6]);
    (void)hipMemcpyAsync(tok, prompt_tokens, (size_t)n_prompt * 4, hipMemcpyDeviceToDevice, st);
    (void)hipMemcpyAsync(tok + n_prompt, prompt_tokens, (size_t)3 * 4, hipMemcpyDeviceToDevice, st);
    m->have_prompt = false;
    VOX_TRY(flow_run(m, st, tok, 1, T, true, prompt_feat, 2 * n_prompt, noise, seed, noise_stream, nullptr));
    if (prompt_mel) hipLaunchKernelGGL(k_flow_to_bct, dim3(ew_grid((size_t)2 * T * c.mel)), dim3(256), 0, st, m->buf[9], prompt_mel, 1, 2 * T, c.mel);
    m->have_prompt = true;
    return VOX_OK;
}

int vox_flow_decode_chunk(vox_flow* m, void* stream, const int32_t* tokens, int n, int T, const float* noise, uint64_t seed,
                          uint32_t noise_stream, float* mel, float* mu) {
    if (!m || !tokens || !mel) return vox_fail(VOX_ERR_INVALID, "flow_decode_chunk: NULL");
    if (!m->have_prompt) return vox_fail(VOX_ERR_INVALID, "flow_decode_chunk: no prompt set (vox_flow_set_prompt)");
    if (n < 1 || n > m->max_batch || T < 1 || T > m->max_T) return vox_fail(VOX_ERR_INVALID, "flow_decode_chunk: n %d / T %d out of range", n, T);
    hipStream_t st = (hipStream_t)stream;
    VOX_TRY(flow_run(m, st, tokens, n, T, false, nullptr, 0, noise, seed, noise_stream, mu));
    hipLaunchKernelGGL(k_flow_to_bct, dim3(ew_grid((size_t)n * 2 * T * m->cfg.mel)), dim3(256), 0, st, m->buf[9], mel, n, 2 * T, m->cfg.mel);
    return VOX_OK;
}

// ---- per-request evolving caches (CosyVoice2Decoder with shared_prompt_cache_mode=False; cosyvoice2.py:1010-1083) --------------------
int vox_flow_enable_slots(vox_flow* m, int n_slots) {
    if (!m || n_slots < 1) return vox_fail(VOX_ERR_INVALID, "flow_enable_slots: bad arguments");
    if (m->n_slots) return m->n_slots == n_slots ? VOX_OK : vox_fail(VOX_ERR_INVALID, "flow_enable_slots: already enabled with %d slots", m->n_slots);
    const vox_flow_config& c = m->cfg;
    const int D = c.dim, C = c.est_ch, dk = D / c.enc_heads;
    const size_t capE = c.max_cache / 2, capU = c.max_cache;
    const size_t e = (size_t)c.enc_layers * c.enc_heads * capE * 2 * dk, u = (size_t)c.up_layers * c.enc_heads * capU * 2 * dk;
    const size_t a = (size_t)2 * c.n_steps * m->n_att * c.est_heads * c.max_cache * 2 * c.est_head_dim;
    bool ok = true;
    auto alloc = [&](float** p, size_t n) { ok = ok && hipMalloc((void**)p, n * 4) == hipSuccess; };
    alloc(&m->s_enc, e * n_slots); alloc(&m->s_up, u * n_slots); alloc(&m->s_att, a * n_slots);
    alloc(&m->s_cnn1, (size_t)c.n_steps * m->n_res * 2 * n_slots * 2 * m->cnn1_w);
    alloc(&m->s_cnn2, (size_t)c.n_steps * m->n_res * 2 * n_slots * 2 * C);
    ok = ok && hipMalloc((void**)&m->s_eidx, (size_t)m->max_batch * 4) == hipSuccess && hipMalloc((void**)&m->s_cidx, (size_t)2 * m->max_batch * 4) == hipSuccess;
    if (!ok) return vox_fail(VOX_ERR_NOMEM, "flow_enable_slots: hipMalloc failed (%zu MB per slot)", (e + u + a) * 4 >> 20);
    m->n_slots = n_slots;
    m->slot.assign(n_slots, vox_flow::SlotState{});
    return VOX_OK;
}

// a request takes slot `slot`: its caches start as a copy of the prompt's (model/cosyvoice2.py:514-560: the per-request cache is the
// expanded initial cache of the default speaker)
int vox_flow_slot_reset(vox_flow* m, void* stream, int slot) {
    if (!m || slot < 0 || slot >= m->n_slots) return vox_fail(VOX_ERR_INVALID, "flow_slot_reset: slot %d out of range", slot);
    if (!m->have_prompt) return vox_fail(VOX_ERR_INVALID, "flow_slot_reset: no prompt set (vox_flow_set_prompt)");
    hipStream_t st = (hipStream_t)stream;
    const vox_flow_config& c = m->cfg;
    const int D = c.dim, C = c.est_ch, dk = D / c.enc_heads;
    const size_t e = (size_t)c.enc_layers * c.enc_heads * (c.max_cache / 2) * 2 * dk, u = (size_t)c.up_layers * c.enc_heads * c.max_cache * 2 * dk;
    const size_t a = (size_t)2 * c.n_steps * m->n_att * c.est_heads * c.max_cache * 2 * c.est_head_dim;
    VOX_HIP(hipMemcpyAsync(m->s_enc + e * slot, m->enc_kv, e * 4, hipMemcpyDeviceToDevice, st));
    VOX_HIP(hipMemcpyAsync(m->s_up + u * slot, m->up_kv, u * 4, hipMemcpyDeviceToDevice, st));
    VOX_HIP(hipMemcpyAsync(m->s_att + a * slot, m->att_kv, a * 4, hipMemcpyDeviceToDevice, st));
    // conv states: per (step, resnet) block [2 halves][2][cin] -> rows 2 slot, 2 slot + 1 of the slot-major block
    const size_t rows = (size_t)c.n_steps * m->n_res;
    for (int r = 0; r < m->n_res; ++r) {
        const int cin = flow_res_cin(c, r);
        VOX_HIP(hipMemcpy2DAsync(m->s_cnn1 + (size_t)r * 2 * m->n_slots * 2 * m->cnn1_w + (size_t)2 * slot * 2 * cin, (size_t)m->n_res * 2 * m->n_slots * 2 * m->cnn1_w * 4,
                                 m->cnn1 + (size_t)r * 4 * m->cnn1_w, (size_t)m->n_res * 4 * m->cnn1_w * 4, (size_t)4 * cin * 4, c.n_steps,
                                 hipMemcpyDeviceToDevice, st));
        VOX_HIP(hipMemcpy2DAsync(m->s_cnn2 + (size_t)r * 2 * m->n_slots * 2 * C + (size_t)2 * slot * 2 * C, (size_t)m->n_res * 2 * m->n_slots * 2 * C * 4,
                                 m->cnn2 + (size_t)r * 4 * C, (size_t)m->n_res * 4 * C * 4, (size_t)4 * C * 4, c.n_steps, hipMemcpyDeviceToDevice, st));
    }
    (void)rows;
    vox_flow::SlotState& ss = m->slot[slot];
    ss = vox_flow::SlotState{};
    ss.enc_len = m->enc_len; ss.up_len = m->up_len; ss.att_len = m->att_len; ss.live = true;
    return VOX_OK;
}

int vox_flow_slot_state(vox_flow* m, int slot, int32_t out[6]) {
    if (!m || !out || slot < 0 || slot >= m->n_slots) return vox_fail(VOX_ERR_INVALID, "flow_slot_state: bad arguments");
    const vox_flow::SlotState& x = m->slot[slot];
    out[0] = x.enc_len; out[1] = x.up_len; out[2] = x.att_len; out[3] = x.enc_head; out[4] = x.up_head; out[5] = x.att_head;
    return VOX_OK;
}

struct FlowSlotIdx {
    static constexpr int MAXN = 64;
    int e[MAXN], c[2 * MAXN];
};
__global__ void k_flow_slot_idx(FlowSlotIdx ix, int n, int* eidx, int* cidx) {
    const int t = threadIdx.x;
    if (t < n) eidx[t] = ix.e[t];
    else if (t >= FlowSlotIdx::MAXN && t - FlowSlotIdx::MAXN < 2 * n) cidx[t - FlowSlotIdx::MAXN] = ix.c[t - FlowSlotIdx::MAXN];
}

// one chunk of n requests that own slots[0..n): the flow runs against their caches, which then take this chunk's rows (sliding
// window: the first `prefix` rows + the most recent ones).  The requests of one call must share their cache lengths, as the reference's
// batched cache tensors do (DecoderCache.cat); the caller groups them.
int vox_flow_decode_chunk_slots(vox_flow* m, void* stream, const int32_t* tokens, int n, int T, const int32_t* slots, const float* noise,
                                uint64_t seed, uint32_t noise_stream, float* mel, float* mu) {
    if (!m || !tokens || !mel || !slots) return vox_fail(VOX_ERR_INVALID, "flow_decode_chunk_slots: NULL");
    if (!m->n_slots) return vox_fail(VOX_ERR_INVALID, "flow_decode_chunk_slots: vox_flow_enable_slots was not called");
    if (n < 1 || n > m->max_batch || T < 1 || T > m->max_T) return vox_fail(VOX_ERR_INVALID, "flow_decode_chunk_slots: n %d / T %d out of range", n, T);
    const vox_flow_config& c = m->cfg;
    std::vector<int> eidx(n), cidx(2 * n);
    for (int b = 0; b < n; ++b) {
        const int sl = slots[b];
        if (sl < 0 || sl >= m->n_slots || !m->slot[sl].live) return vox_fail(VOX_ERR_INVALID, "flow_decode_chunk_slots: slot %d not initialised", sl);
        for (int b2 = 0; b2 < b; ++b2)
            if (slots[b2] == sl) return vox_fail(VOX_ERR_INVALID, "flow_decode_chunk_slots: slot %d twice in one call", sl);
        const vox_flow::SlotState &x = m->slot[sl], &y = m->slot[slots[0]];
        if (x.enc_len != y.enc_len || x.enc_head != y.enc_head || x.up_len != y.up_len || x.up_head != y.up_head || x.att_len != y.att_len ||
            x.att_head != y.att_head)
            return vox_fail(VOX_ERR_INVALID, "flow_decode_chunk_slots: the requests of a call must have equal cache states (vox_flow_slot_state)");
        eidx[b] = sl; cidx[b] = 2 * sl; cidx[n + b] = 2 * sl + 1;
    }
    const int capE = c.max_cache / 2, capU = c.max_cache;
    if (T > capE - c.prefix / 2 || 2 * T > capU - c.prefix) return vox_fail(VOX_ERR_INVALID, "flow_decode_chunk_slots: chunk longer than the cache ring");
    hipStream_t st = (hipStream_t)stream;
    if (n <= FlowSlotIdx::MAXN) {
        // the slot index vectors travel as kernel arguments (copied at launch): no host buffer whose lifetime the stream depends on,
        // so the call returns without waiting for the chunks queued before it.  Host-side slot states advance at enqueue time: all
        // calls on one flow object must go through ONE stream (they are ordered against each other only there).
        FlowSlotIdx ix{};
        for (int b = 0; b < n; ++b) { ix.e[b] = eidx[b]; ix.c[b] = cidx[b]; ix.c[n + b] = cidx[n + b]; }
        hipLaunchKernelGGL(k_flow_slot_idx, dim3(1), dim3(3 * FlowSlotIdx::MAXN), 0, st, ix, n, m->s_eidx, m->s_cidx);
    } else {
        VOX_HIP(hipMemcpyAsync(m->s_eidx, eidx.data(), (size_t)n * 4, hipMemcpyHostToDevice, st));
        VOX_HIP(hipMemcpyAsync(m->s_cidx, cidx.data(), (size_t)2 * n * 4, hipMemcpyHostToDevice, st));
        VOX_HIP(hipStreamSynchronize(st));          // (the index vectors above are stack-owned host memory)
    }
    const vox_flow::SlotState cur = m->slot[slots[0]];
    VOX_TRY(flow_run(m, st, tokens, n, T, false, nullptr, 0, noise, seed, noise_stream, mu, &cur));
    hipLaunchKernelGGL(k_flow_to_bct, dim3(ew_grid((size_t)n * 2 * T * c.mel)), dim3(256), 0, st, m->buf[9], mel, n, 2 * T, c.mel);
    auto advance = [](int& len, int& head, int add, int cap, int prefix) {
        const int over = len + add - cap;
        if (over > 0) head = (head + over) % (cap - prefix);
        len = len + add < cap ? len + add : cap;
    };
    for (int b = 0; b < n; ++b) {
        vox_flow::SlotState& x = m->slot[slots[b]];
        advance(x.enc_len, x.enc_head, T, capE, c.prefix / 2);
        advance(x.up_len, x.up_head, 2 * T, capU, c.prefix);
        advance(x.att_len, x.att_head, 2 * T, capU, c.prefix);
    }
    return VOX_OK;
}

}  // extern "C"

// fade_in_out (tokenizer/cosyvoice2.py:46-54): the first `fade` samples of every row cross-fade with the tail of the previous chunk
// (prev NULL = silence), computed in double like the reference's float64 Hamming window
__global__ __launch_bounds__(256) void k_fade_in(float* wav, const float* prev, const double* win, int n, int L, int fade) {
    const size_t total = (size_t)n * fade;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int b = (int)(i / fade), t = (int)(i % fade);
        const double v = (double)wav[(size_t)b * L + t] * win[t] + (prev ? (double)prev[(size_t)b * fade + t] : 0.0) * win[fade + t];
        wav[(size_t)b * L + t] = (float)v;
    }
}
extern "C" int vox_fade_in_out(void* stream, float* wav, int n, int L, const float* prev_tail, const double* window, int fade) {
    if (!wav || !window || n < 1 || fade < 1 || fade > L) return vox_fail(VOX_ERR_INVALID, "fade_in_out: bad arguments");
    hipLaunchKernelGGL(k_fade_in, dim3(ew_grid((size_t)n * fade)), dim3(256), 0, (hipStream_t)stream, wav, prev_tail, window, n, L, fade);
    return VOX_OK;
}

// the seeded CFM start noise as a tensor [mel][frames] (what vox_flow_* draw when `noise` is NULL): lets a caller that replays a captured
// graph keep the draw outside it (a graph freezes scalar arguments such as the stream id)
__global__ __launch_bounds__(256) void k_flow_noise_z(uint64_t seed, uint32_t stream, float* z, size_t total) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        uint32_t w0, w1;
        philox4((uint32_t)i, stream, 0u, 0u, (uint32_t)seed, (uint32_t)(seed >> 32), &w0, &w1);
        const float u1 = ((float)(w0 >> 8) + 1.0f) * (1.0f / 16777216.0f), u2 = (float)(w1 >> 8) * (1.0f / 16777216.0f);
        z[i] = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
    }
}
extern "C" int vox_flow_fill_noise(void* stream, uint64_t seed, uint32_t noise_stream, int mel, int frames, float* z) {
    if (!z || mel < 1 || frames < 1) return vox_fail(VOX_ERR_INVALID, "flow_fill_noise: bad arguments");
    hipLaunchKernelGGL(k_flow_noise_z, dim3(ew_grid((size_t)mel * frames)), dim3(256), 0, (hipStream_t)stream, seed, noise_stream, z, (size_t)mel * frames);
    return VOX_OK;
}

// y = the function that the codecs' and flows' kernels use, one value a thread
__global__ __launch_bounds__(256) void k_flow_function(int which, const float* x, float* y, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = which == 0 ? gelu_f(x[i]) : which == 1 ? mish_f(x[i]) : flow_exp(x[i]);
}
extern "C" int vox_flow_function(void* stream, int which, const float* x, float* y, int n) {
    if (which < 0 || which > 2 || !x || !y || n < 1) return vox_fail(VOX_ERR_INVALID, "flow_function: bad arguments");
    hipLaunchKernelGGL(k_flow_function, dim3(((size_t)n + 255) / 256), dim3(256), 0, (hipStream_t)stream, which, x, y, (size_t)n);
    return VOX_OK;
}

// ====================================================================================================================
// GLM-4-Voice flow (speech tokens -> mel): block conformer encoder, length regulator, non-causal U-Net CFM.  include/voxhip.h has the contract.
// ====================================================================================================================
// GroupNorm over (channels of a group) x (all rows of a request) + Mish + optional per-channel addend; x [N][T][ld], C real channels
// (columns >= C are written 0); one block per (group, request)
__global__ __launch_bounds__(256) void k_flow_groupnorm(const float* x, const float* w, const float* b, float* y, int T, int C, int ld, int G,
                                                         float eps, const float* add) {
    __shared__ float red[8];
    const int g = blockIdx.x, n = blockIdx.y, cg = C / G;
    const float* xb = x + (size_t)n * T * ld;
    float* yb = y + (size_t)n * T * ld;
    const int cnt = T * cg;
    if (256 % cg == 0 && T <= 48 * (256 / cg)) {
        // the group fits the block's registers (GLM: 32 channels x <= 384 frames): element i = tid + 256 k is (frame tid / cg + k * 256 / cg,
        // channel tid % cg) — the general path's element -> thread assignment and accumulation order without its two integer divisions
        // per element and per pass, and with ONE read of x instead of three (the kernel is 16-128 blocks of pure latency)
        constexpr int KM = 48;
        const int c = g * cg + threadIdx.x % cg, r0 = threadIdx.x / cg, rs = 256 / cg;
        float xv[KM];
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < KM; ++k) {
            const int r = r0 + k * rs;
            xv[k] = r < T ? xb[(size_t)r * ld + c] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < KM; ++k)
            if (r0 + k * rs < T) s += xv[k];
        s = butterfly<64>(s);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
        __syncthreads();
        const float mean = (red[0] + red[1] + red[2] + red[3]) / (float)cnt;
        float v = 0.0f;
#pragma unroll
        for (int k = 0; k < KM; ++k)
            if (r0 + k * rs < T) { const float d = xv[k] - mean; v += d * d; }
        v = butterfly<64>(v);
        if ((threadIdx.x & 63) == 0) red[4 + (threadIdx.x >> 6)] = v;
        __syncthreads();
        const float rstd = rsqrtf((red[4] + red[5] + red[6] + red[7]) / (float)cnt + eps);
        const float wc = w[c], bc = b[c], ac = add ? add[c] : 0.0f;
#pragma unroll
        for (int k = 0; k < KM; ++k) {
            const int r = r0 + k * rs;
            if (r < T) {
                float o = mish_f((xv[k] - mean) * rstd * wc + bc);
                if (add) o += ac;
                yb[(size_t)r * ld + c] = o;
            }
        }
        if (g == G - 1 && ld > C)
            for (int i = threadIdx.x; i < T * (ld - C); i += 256) yb[(size_t)(i / (ld - C)) * ld + C + i % (ld - C)] = 0.0f;
        return;
    }
    float s = 0.0f;
    for (int i = threadIdx.x; i < cnt; i += 256) s += xb[(size_t)(i / cg) * ld + g * cg + i % cg];
    s = butterfly<64>(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float mean = (red[0] + red[1] + red[2] + red[3]) / (float)cnt;
    float v = 0.0f;
    for (int i = threadIdx.x; i < cnt; i += 256) { const float d = xb[(size_t)(i / cg) * ld + g * cg + i % cg] - mean; v += d * d; }
    v = butterfly<64>(v);
    if ((threadIdx.x & 63) == 0) red[4 + (threadIdx.x >> 6)] = v;
    __syncthreads();
    const float rstd = rsqrtf((red[4] + red[5] + red[6] + red[7]) / (float)cnt + eps);
    for (int i = threadIdx.x; i < cnt; i += 256) {
        const int c = g * cg + i % cg;
        const size_t o = (size_t)(i / cg) * ld + c;
        float r = mish_f((xb[o] - mean) * rstd * w[c] + b[c]);
        if (add) r += add[c];
        yb[o] = r;
    }
    if (g == G - 1 && ld > C)
        for (int i = threadIdx.x; i < T * (ld - C); i += 256) yb[(size_t)(i / (ld - C)) * ld + C + i % (ld - C)] = 0.0f;
}
// F.interpolate(mode="nearest") along time: y[b][t] = x[b][min(floor(t * T / To), T - 1)]
__global__ __launch_bounds__(256) void k_flow_interp(const float* x, float* y, int B, int T, int To, int ld) {
    const size_t total = (size_t)B * To * ld;
    const float sc = (float)T / (float)To;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % ld), t = (int)((i / ld) % To), b = (int)(i / ((size_t)ld * To));
        int src = (int)floorf((float)t * sc);
        src = src > T - 1 ? T - 1 : src;
        y[i] = x[((size_t)b * T + src) * ld + c];
    }
}
// Conv1d(k 3, stride 2, padding 1) as a 1-tap GEMM: y[n][t] = x[n][2t - 1] | x[n][2t] | x[n][2t + 1]  (zeros outside)
__global__ __launch_bounds__(256) void k_flow_stride2(const float* x, float* y, int N, int T, int To, int C) {
    const size_t total = (size_t)N * To * 3 * C;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % C), j = (int)((i / C) % 3), t = (int)((i / (3 * (size_t)C)) % To), n = (int)(i / (3 * (size_t)C * To));
        const int ts = 2 * t - 1 + j;
        y[i] = (ts >= 0 && ts < T) ? x[((size_t)n * T + ts) * C + c] : 0.0f;
    }
}
// per-request start noise z [B][M][T] (given, or stream first + b) -> x [B][T][M]
__global__ __launch_bounds__(256) void k_flow_noise_req(const float* z, uint64_t seed, uint32_t first, float* x, int B, int T, int M) {
    const size_t total = (size_t)B * T * M;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i % M), t = (int)((i / M) % T), b = (int)(i / ((size_t)M * T));
        float v;
        if (z) v = z[((size_t)b * M + c) * T + t];
        else {
            uint32_t w0, w1;
            philox4((uint32_t)(c * T + t), first + (uint32_t)b, 0u, 0u, (uint32_t)seed, (uint32_t)(seed >> 32), &w0, &w1);
            const float u1 = ((float)(w0 >> 8) + 1.0f) * (1.0f / 16777216.0f), u2 = (float)(w1 >> 8) * (1.0f / 16777216.0f);
            v = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
        }
        x[i] = v;
    }
}
// rows of x [n][C] L2-normalised (F.normalize, eps 1e-12): one block per row; x NULL = zeros
__global__ __launch_bounds__(256) void k_flow_l2norm_rows(const float* x, float* y, int C) {
    __shared__ float red[4];
    const float* xr = x ? x + (size_t)blockIdx.x * C : nullptr;
    float s = 0.0f;
    for (int i = threadIdx.x; i < C; i += 256) { const float v = xr ? xr[i] : 0.0f; s += v * v; }
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float nrm = fmaxf(sqrtf(red[0] + red[1] + red[2] + red[3]), 1e-12f);
    for (int i = threadIdx.x; i < C; i += 256) y[(size_t)blockIdx.x * C + i] = (xr ? xr[i] : 0.0f) / nrm;
}

struct vox_glmflow {
    vox_ctx* ctx;
    vox_glmflow_config cfg;
    vox_glmflow_weights w;
    std::vector<vox_flow_conformer_w> enc;
    std::vector<vox_flow_resnet_w> resnets;
    std::vector<vox_flow_tblock_w> tblocks;
    std::vector<FlowPacked> packed;         // per transformer block, or empty
    void* packed_mem = nullptr;
    float* tb_ws = nullptr;                 // their scratch: TB_PLANES + TB_HEADS planes of the most rows
    int max_batch, max_T, max_mel, n_res, n_att;
    std::vector<float> dt;
    float* tb = nullptr;
    float* buf[10] = {};
    size_t buf_floats = 0;
    float *spk = nullptr, *pe = nullptr, *pp = nullptr;
};
static const int FLOW_OFF_S3[3] = {1, 0, -1};           // "same" k3
static const int FLOW_OFF_T3[3] = {-1, 0, 1};           // ConvTranspose1d(4, 2, 1): taps d = -1, 0, 1 (tap d reads row t - d)

extern "C" {

void vox_glmflow_destroy(vox_glmflow* m) {
    if (!m) return;
    for (int i = 0; i < 10; ++i) (void)hipFree(m->buf[i]);
    (void)hipFree(m->tb); (void)hipFree(m->spk); (void)hipFree(m->pe); (void)hipFree(m->pp); (void)hipFree(m->packed_mem); (void)hipFree(m->tb_ws);
    delete m;
}

int vox_glmflow_create(vox_ctx* ctx, const vox_glmflow_config* cfg, const vox_glmflow_weights* w, int max_batch, int max_T, int max_mel,
                       const float* time_emb, const float* dt, vox_glmflow** out) {
    if (!ctx || !cfg || !w || !out || !time_emb || !dt) return vox_fail(VOX_ERR_INVALID, "glmflow_create: NULL");
    const vox_glmflow_config& c = *cfg;
    if (c.dim % c.enc_heads || c.dim / c.enc_heads > 128 || c.est_head_dim > 128 || c.dim % 32 || c.est_ch % 32 || (4 * c.mel) % 32 ||
        c.mel_padded % 32 || c.mel_padded < c.mel || (c.est_heads * c.est_head_dim) % 32 || c.enc_ffn % 32 || c.spk_dim % 32 ||
        c.est_ch % c.groups || max_batch < 1 || max_T < 1 || max_mel < 2 || c.n_steps < 1 || c.reg_layers > 4 || max_mel > FLOW_MAXKEYS ||
        max_T > FLOW_MAXKEYS)
        return vox_fail(VOX_ERR_INVALID, "glmflow_create: bad config");
    vox_glmflow* m = new vox_glmflow();
    m->ctx = ctx; m->cfg = c; m->w = *w; m->max_batch = max_batch; m->max_T = max_T; m->max_mel = max_mel;
    m->n_res = 4 + c.est_mid; m->n_att = m->n_res * c.est_blocks;
    m->enc.assign(w->enc, w->enc + c.enc_layers);
    m->resnets.assign(w->resnets, w->resnets + m->n_res);
    m->tblocks.assign(w->tblocks, w->tblocks + m->n_att);
    m->dt.assign(dt, dt + c.n_steps);
    const int D = c.dim, C = c.est_ch, TE = 4 * C, inner = c.est_heads * c.est_head_dim;
    size_t rows = (size_t)2 * max_batch * max_mel;
    if ((size_t)max_batch * max_T > rows) rows = (size_t)max_batch * max_T;
    size_t wmax = 3 * (size_t)D;
    for (size_t v : {(size_t)c.enc_ffn, (size_t)4 * C, (size_t)3 * inner, (size_t)4 * c.mel, (size_t)TE, (size_t)3 * C}) wmax = v > wmax ? v : wmax;
    m->buf_floats = rows * wmax;
    bool ok = true;
    auto alloc = [&](float** p, size_t n) { ok = ok && hipMalloc((void**)p, n * 4) == hipSuccess; };
    for (int i = 0; i < 10; ++i) alloc(&m->buf[i], m->buf_floats);
    alloc(&m->tb, (size_t)c.n_steps * m->n_res * C);
    alloc(&m->spk, (size_t)max_batch * c.mel);
    alloc(&m->pe, (size_t)2 * FLOW_MAXKEYS * D);
    alloc(&m->pp, (size_t)2 * FLOW_MAXKEYS * D);
    ok = ok && tb_pack(m->tblocks, C, inner, m->packed, &m->packed_mem);
    if (!m->packed.empty()) alloc(&m->tb_ws, (TB_PLANES + TB_HEADS) * tb_plane(rows));
    if (!ok) { vox_glmflow_destroy(m); return vox_fail(VOX_ERR_NOMEM, "glmflow_create: hipMalloc failed"); }
    hipStream_t st = nullptr;
    g_conv_planes = 3;
    g_conv_skinny_rows = 48; g_conv_rows_gemm = false;
    int rc = VOX_OK;
    (void)hipMemcpy(m->buf[0], time_emb, (size_t)c.n_steps * 4 * c.mel * 4, hipMemcpyHostToDevice);
    rc = conv_gemm(st, w->time1, m->buf[0], nullptr, nullptr, 1, c.n_steps, 0, FLOW_OFF0, m->buf[1], nullptr, nullptr, 0);
    hipLaunchKernelGGL(k_flow_act, dim3(ew_grid((size_t)c.n_steps * TE)), dim3(256), 0, st, m->buf[1], (size_t)c.n_steps * TE, 2);
    if (rc == VOX_OK) rc = conv_gemm(st, w->time2, m->buf[1], nullptr, nullptr, 1, c.n_steps, 0, FLOW_OFF0, m->buf[2], nullptr, nullptr, 0);
    hipLaunchKernelGGL(k_flow_act, dim3(ew_grid((size_t)c.n_steps * TE)), dim3(256), 0, st, m->buf[2], (size_t)c.n_steps * TE, 1);
    for (int r = 0; r < m->n_res && rc == VOX_OK; ++r) {
        rc = conv_gemm(st, m->resnets[r].mlp, m->buf[2], nullptr, nullptr, 1, c.n_steps, 0, FLOW_OFF0, m->buf[3], nullptr, nullptr, 0);
        (void)hipMemcpy2DAsync(m->tb + (size_t)r * C, (size_t)m->n_res * C * 4, m->buf[3], (size_t)C * 4, (size_t)C * 4, c.n_steps,
                               hipMemcpyDeviceToDevice, st);
    }
    if (hipStreamSynchronize(st) != hipSuccess || rc != VOX_OK) { vox_glmflow_destroy(m); return rc != VOX_OK ? rc : vox_fail(VOX_ERR_HIP, "glmflow_create: time MLP failed"); }
    *out = m;
    return VOX_OK;
}

int vox_glmflow_decode(vox_glmflow* m, void* stream, const int32_t* tokens, int n, int T, int Tm, const float* embedding, const float* noise,
                       uint64_t seed, uint32_t first_stream, float* mel) {
    if (!m || !tokens || !mel) return vox_fail(VOX_ERR_INVALID, "glmflow_decode: NULL");
    if (n < 1 || n > m->max_batch || T < 1 || T > m->max_T || Tm < 2 || Tm > m->max_mel)
        return vox_fail(VOX_ERR_INVALID, "glmflow_decode: n %d / T %d / mel frames %d out of range", n, T, Tm);
    hipStream_t st = (hipStream_t)stream;
    const vox_glmflow_config& c = m->cfg;
    const vox_glmflow_weights& w = m->w;
    const int D = c.dim, M = c.mel, MP = c.mel_padded, C = c.est_ch, H = c.enc_heads, dk = D / H, HE = c.est_heads, hd = c.est_head_dim;
    float** Bf = m->buf;
    g_conv_planes = 3;
    struct RowsGuard { ~RowsGuard() { g_conv_skinny_rows = 48; g_conv_rows_gemm = false; } } rows_guard;      // also on the error returns
    g_conv_skinny_rows = FLOW_SKINNY_ROWS; g_conv_rows_gemm = true;
    // speaker vector per request: spk_embed_affine_layer(normalize(embedding)); GLM-4-Voice passes zeros (glm.py:2647)
    hipLaunchKernelGGL(k_flow_l2norm_rows, dim3(n), dim3(256), 0, st, embedding, Bf[0], c.spk_dim);
    VOX_TRY(conv_gemm(st, w.spk, Bf[0], nullptr, nullptr, n, 1, 0, FLOW_OFF0, m->spk, nullptr, nullptr, 0));
    // ---- encoder: embed, LinearNoSubsampling, block-masked relative-position conformer layers, after_norm, encoder_proj ----
    float* x = Bf[3];
    hipLaunchKernelGGL(k_flow_embed, dim3(ew_grid((size_t)n * T * D)), dim3(256), 0, st, tokens, w.embedding, Bf[0], (size_t)n * T, D);
    VOX_TRY(conv_gemm(st, w.embed_lin, Bf[0], nullptr, nullptr, n, T, 0, FLOW_OFF0, Bf[1], nullptr, nullptr, 0));
    hipLaunchKernelGGL(k_flow_ln, dim3((n * T + 3) / 4), dim3(256), 0, st, Bf[1], w.embed_ln_w, w.embed_ln_b, x, D, 1e-5f, sqrtf((float)D), 0, nullptr, 1, n * T);
    hipLaunchKernelGGL(k_flow_relpos, dim3(ew_grid((size_t)(2 * T - 1) * D)), dim3(256), 0, st, m->pe, T, D);
    for (int l = 0; l < c.enc_layers; ++l) {
        const vox_flow_conformer_w& cw = m->enc[l];
        float *nrm = Bf[0], *qkv = Bf[1], *att = Bf[2];
        hipLaunchKernelGGL(k_flow_ln, dim3((n * T + 3) / 4), dim3(256), 0, st, x, cw.ln_mha_w, cw.ln_mha_b, nrm, D, 1e-12f, 1.0f, 0, nullptr, 1, n * T);
        VOX_TRY(conv_gemm(st, cw.qkv, nrm, nullptr, nullptr, n, T, 0, FLOW_OFF0, qkv, nullptr, nullptr, 0));
        VOX_TRY(conv_gemm(st, cw.pos, m->pe, nullptr, nullptr, 1, 2 * T - 1, 0, FLOW_OFF0, m->pp, nullptr, nullptr, 0));
        FlowAttn a{qkv, nullptr, m->pp, cw.bias_u, cw.bias_v, att, T, H, dk, 0, 0, 0, 0, 1.0f / sqrtf((float)dk), c.block_size};
        launch_flow_attn(st, a, T, H, n);
        VOX_TRY(conv_gemm(st, cw.out, att, nullptr, nullptr, n, T, 0, FLOW_OFF0, x, x, nullptr, 0));
        hipLaunchKernelGGL(k_flow_ln, dim3((n * T + 3) / 4), dim3(256), 0, st, x, cw.ln_ff_w, cw.ln_ff_b, nrm, D, 1e-12f, 1.0f, 0, nullptr, 1, n * T);
        VOX_TRY(conv_gemm(st, cw.w1, nrm, nullptr, nullptr, n, T, 0, FLOW_OFF0, qkv, nullptr, nullptr, 0));
        hipLaunchKernelGGL(k_flow_act, dim3(ew_grid((size_t)n * T * c.enc_ffn)), dim3(256), 0, st, qkv, (size_t)n * T * c.enc_ffn, 2);
        VOX_TRY(conv_gemm(st, cw.w2, qkv, nullptr, nullptr, n, T, 0, FLOW_OFF0, x, x, nullptr, 0));
    }
    hipLaunchKernelGGL(k_flow_ln, dim3((n * T + 3) / 4), dim3(256), 0, st, x, w.after_w, w.after_b, Bf[0], D, 1e-5f, 1.0f, 0, nullptr, 1, n * T);
    VOX_TRY(conv_gemm(st, w.enc_proj, Bf[0], nullptr, nullptr, n, T, 0, FLOW_OFF0, Bf[1], nullptr, nullptr, 0));       // [n*T][MP] (pad columns 0)
    // ---- length regulator: nearest resampling to Tm frames, (conv k3, GroupNorm(1), Mish) x reg_layers, conv k1 ----
    hipLaunchKernelGGL(k_flow_interp, dim3(ew_grid((size_t)n * Tm * MP)), dim3(256), 0, st, Bf[1], Bf[0], n, T, Tm, MP);
    for (int i = 0; i < c.reg_layers; ++i) {
        VOX_TRY(conv_gemm(st, w.reg_conv[i], Bf[0], nullptr, nullptr, n, Tm, 0, FLOW_OFF_S3, Bf[1], nullptr, nullptr, 0));
        hipLaunchKernelGGL(k_flow_groupnorm, dim3(1, n), dim3(256), 0, st, Bf[1], w.reg_gn_w[i], w.reg_gn_b[i], Bf[0], Tm, M, MP, 1, 1e-5f, nullptr);
    }
    float* mu = Bf[8];
    VOX_TRY(conv_gemm(st, w.reg_out, Bf[0], nullptr, nullptr, n, Tm, 0, FLOW_OFF0, mu, nullptr, nullptr, 0));           // [n*Tm][M]
    // ---- CFM: n_steps Euler steps of the U-Net on the doubled (classifier-free guidance) batch ----
    float* xs = Bf[9];
    hipLaunchKernelGGL(k_flow_noise_req, dim3(ew_grid((size_t)n * Tm * M)), dim3(256), 0, st, noise, seed, first_stream, xs, n, Tm, M);
    const int N = 2 * n, Th = (Tm - 1) / 2 + 1;
    auto tblocks = [&](float* h, int rows_T, int& li, float* a1, float* a2, float* a3) -> int {
        for (int j = 0; j < c.est_blocks; ++j, ++li) {
            const vox_flow_tblock_w& tw = m->tblocks[li];
            const FlowPacked* pk = m->packed.empty() ? nullptr : &m->packed[li];
            if (pk) tb_qkv(st, *pk, tw, h, m->tb_ws, j ? &m->tblocks[li - 1] : nullptr, a2, N * rows_T);
            else VOX_TRY(ln_gemm(st, tw.qkv, h, tw.ln1_w, tw.ln1_b, 1e-5f, a1, N, rows_T, a2, 0));
            FlowAttn a{a2, nullptr, nullptr, nullptr, nullptr, a3, rows_T, HE, hd, 0, 0, 0, 0, 1.0f / sqrtf((float)hd), 0};
            const bool parts = tb_attn(st, a, pk, m->tb_ws, rows_T, HE, N);
            if (pk) { tb_ff(st, *pk, tw, a3, h, m->tb_ws, j == 0, j + 1 == c.est_blocks, N * rows_T, parts); continue; }
            VOX_TRY(conv_gemm(st, tw.out, a3, nullptr, nullptr, N, rows_T, 0, FLOW_OFF0, h, h, nullptr, 0));
            VOX_TRY(ln_gemm(st, tw.ff1, h, tw.ln3_w, tw.ln3_b, 1e-5f, a1, N, rows_T, a2, 1));
            VOX_TRY(conv_gemm(st, tw.ff2, a2, nullptr, nullptr, N, rows_T, 0, FLOW_OFF0, h, h, nullptr, 0));
        }
        return VOX_OK;
    };
    for (int s = 0; s < c.n_steps; ++s) {
        float *hA = Bf[0], *a1 = Bf[1], *a2 = Bf[2], *a3 = Bf[3], *skip0 = Bf[4], *cat = Bf[5], *hB = Bf[6], *skip1 = Bf[7];
        hipLaunchKernelGGL(k_flow_pack, dim3(ew_grid((size_t)N * Tm * 4 * M)), dim3(256), 0, st, xs, mu, m->spk, nullptr, cat, n, Tm, M, M);
        int li = 0, r = 0;
        // ResnetBlock1D (conv k3, GroupNorm(groups), Mish; + time projection; again; + res_conv) then the transformer blocks, in -> out
        auto group = [&](const float* in, float* o, int rows_T) -> int {
            const vox_flow_resnet_w& rw = m->resnets[r];
            VOX_TRY(conv_gemm(st, rw.conv1, in, nullptr, nullptr, N, rows_T, 0, FLOW_OFF_S3, a1, nullptr, nullptr, 0));
            hipLaunchKernelGGL(k_flow_groupnorm, dim3(c.groups, N), dim3(256), 0, st, a1, rw.ln1_w, rw.ln1_b, a2, rows_T, C, C, c.groups, 1e-5f,
                               m->tb + ((size_t)s * m->n_res + r) * C);
            VOX_TRY(conv_gemm(st, rw.conv2, a2, nullptr, nullptr, N, rows_T, 0, FLOW_OFF_S3, a1, nullptr, nullptr, 0));
            hipLaunchKernelGGL(k_flow_groupnorm, dim3(c.groups, N), dim3(256), 0, st, a1, rw.ln2_w, rw.ln2_b, a2, rows_T, C, C, c.groups, 1e-5f, nullptr);
            VOX_TRY(conv_gemm(st, rw.res, in, nullptr, nullptr, N, rows_T, 0, FLOW_OFF0, o, a2, nullptr, 0));
            ++r;
            return tblocks(o, rows_T, li, a1, a2, a3);
        };
        VOX_TRY(group(cat, skip0, Tm));                                                       // down 0 (its output is the outer skip)
        hipLaunchKernelGGL(k_flow_stride2, dim3(ew_grid((size_t)N * Th * 3 * C)), dim3(256), 0, st, skip0, cat, N, Tm, Th, C);
        VOX_TRY(conv_gemm(st, w.down_s2, cat, nullptr, nullptr, N, Th, 0, FLOW_OFF0, hA, nullptr, nullptr, 0));
        VOX_TRY(group(hA, skip1, Th));                                                        // down 1
        VOX_TRY(conv_gemm(st, w.down_conv1, skip1, nullptr, nullptr, N, Th, 0, FLOW_OFF_S3, hA, nullptr, nullptr, 0));
        float *cur = hA, *nxt = hB;
        for (int i = 0; i < c.est_mid; ++i) {
            VOX_TRY(group(cur, nxt, Th));
            float* t = cur; cur = nxt; nxt = t;
        }
        hipLaunchKernelGGL(k_flow_concat2, dim3(ew_grid((size_t)N * Th * 2 * C)), dim3(256), 0, st, cur, skip1, cat, (size_t)N * Th, C);
        VOX_TRY(group(cat, nxt, Th));                                                         // up 0
        VOX_TRY(conv_gemm(st, w.up_tconv, nxt, nullptr, nullptr, N, Th, 0, FLOW_OFF_T3, cur, nullptr, nullptr, 0));      // [N][2 Th][C]
        // x[:, :, :skip.shape[-1]]: the transposed conv gives 2 Th rows per request, the skip has Tm (<= 2 Th)
        if (2 * Th != Tm) {
            for (int q = 0; q < N; ++q)
                (void)hipMemcpyAsync(nxt + (size_t)q * Tm * C, cur + (size_t)q * 2 * Th * C, (size_t)Tm * C * 4, hipMemcpyDeviceToDevice, st);
            float* t = cur; cur = nxt; nxt = t;
        }
        hipLaunchKernelGGL(k_flow_concat2, dim3(ew_grid((size_t)N * Tm * 2 * C)), dim3(256), 0, st, cur, skip0, cat, (size_t)N * Tm, C);
        VOX_TRY(group(cat, nxt, Tm));                                                         // up 1
        VOX_TRY(conv_gemm(st, w.up_conv1, nxt, nullptr, nullptr, N, Tm, 0, FLOW_OFF_S3, a1, nullptr, nullptr, 0));
        VOX_TRY(conv_gemm(st, w.final_conv, a1, nullptr, nullptr, N, Tm, 0, FLOW_OFF_S3, a2, nullptr, nullptr, 0));
        hipLaunchKernelGGL(k_flow_groupnorm, dim3(c.groups, N), dim3(256), 0, st, a2, w.final_gn_w, w.final_gn_b, a1, Tm, C, C, c.groups, 1e-5f, nullptr);
        VOX_TRY(conv_gemm(st, w.final_proj, a1, nullptr, nullptr, N, Tm, 0, FLOW_OFF0, a2, nullptr, nullptr, 0));
        hipLaunchKernelGGL(k_flow_euler, dim3(ew_grid((size_t)n * Tm * M)), dim3(256), 0, st, xs, a2, n, Tm, M, m->dt[s], c.cfg_rate);
    }
    g_conv_skinny_rows = 48; g_conv_rows_gemm = false;
    hipLaunchKernelGGL(k_flow_to_bct, dim3(ew_grid((size_t)n * Tm * M)), dim3(256), 0, st, xs, mel, n, Tm, M);
    return VOX_OK;
}

}  // extern "C"

// ================================================================================================
// Prompt-side encoders of a voice-clone request (run once per request, before prefill)
// ================================================================================================
// ---- speaker encoder: log-mel front end + ECAPA-TDNN  (model/qwen3_tts.py:21-88, 317-532, 835-891) ----
// Layout: fp32 time-major [t][C].  A reflect-padded "same" conv is a centred-tap conv_gemm over a reflect-padded copy of its input
// ([T + 2p][C]); rows p .. p+T-1 of the result are the conv's output (contiguous, so later stages just offset the pointer).
#define ENC_MAX_FFT 2048
__global__ __launch_bounds__(256) void k_enc_logmel(const float* audio, int N, const float* window, const float* basis, int n_fft, int hop,
                                                     int n_mels, int MP, float* mel) {
    __shared__ double xs[ENC_MAX_FFT], tw[ENC_MAX_FFT];
    __shared__ float mag[ENC_MAX_FFT / 2 + 1];
    const int t = blockIdx.x, pad = (n_fft - hop) / 2, mask = n_fft - 1, nb = n_fft / 2 + 1;
    for (int j = threadIdx.x; j < n_fft; j += 256) {
        int i = t * hop + j - pad;                       // F.pad(..., mode="reflect"): no edge repeat
        i = i < 0 ? -i : (i >= N ? 2 * (N - 1) - i : i);
        xs[j] = (double)(audio[i] * window[j]);
        tw[j] = cospi(2.0 * j / n_fft);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < nb; k += 256) {
        double re = 0.0, im = 0.0;
        const int q = 3 * n_fft / 4;                     // sin(a) = cos(a - pi/2)
        for (int n = 0; n < n_fft; ++n) {
            const int idx = (k * n) & mask;
            re += xs[n] * tw[idx];
            im += xs[n] * tw[(idx + q) & mask];
        }
        mag[k] = sqrtf((float)(re * re + im * im) + 1e-9f);
    }
    __syncthreads();
    for (int m = threadIdx.x; m < MP; m += 256) {
        float v = 0.f;
        if (m < n_mels) {
            const float* b = basis + (size_t)m * nb;
            float acc = 0.f;
            for (int k = 0; k < nb; ++k) acc += b[k] * mag[k];
            v = logf(fmaxf(acc, 1e-5f));
        }
        mel[(size_t)t * MP + m] = v;
    }
}
// dst [T + 2p][C]: dst[r][c] = s1[refl(r - p)][c] (+ s2[refl(r - p)][c]), reflect without edge repeat
__global__ __launch_bounds__(256) void k_enc_gather(float* dst, int T, int p, int C, const float* s1, int ld1, const float* s2, int ld2) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)(T + 2 * p) * C) return;
    const int r = (int)(i / C), c = (int)(i % C);
    int t = r - p;
    t = t < 0 ? -t : (t >= T ? 2 * (T - 1) - t : t);
    float v = s1[(size_t)t * ld1 + c];
    if (s2) v += s2[(size_t)t * ld2 + c];
    dst[i] = v;
}
__global__ __launch_bounds__(256) void k_enc_copy_cols(float* dst, int ldd, const float* src, int lds, int T, int C) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)T * C) return;
    const int t = (int)(i / C), c = (int)(i % C);
    dst[(size_t)t * ldd + c] = src[(size_t)t * lds + c];
}
// mode 2: ReLU; 3: tanh(ReLU); 4: sigmoid
__global__ __launch_bounds__(256) void k_enc_act(float* x, size_t n, int mode) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float v = x[i];
    if (mode == 2) v = fmaxf(v, 0.f);
    else if (mode == 3) v = tanhf(fmaxf(v, 0.f));
    else if (mode == 4) v = 1.0f / (1.0f + expf(-v));
    x[i] = v;
}
// Per-channel weighted statistics over time (AttentiveStatisticsPooling._compute_statistics): weights 1/T (att == NULL) or the softmax over
// time of att[:, c].  mean[c] = sum w x, std[c] = sqrt(max(sum w (x - mean)^2, 1e-12)).  Block = 64 channels x 4 time lanes.
__global__ __launch_bounds__(256) void k_enc_colstats(const float* x, int T, int C, const float* att, float* mean, float* stdv) {
    __shared__ float red[4][64];
    const int cl = threadIdx.x & 63, tl = threadIdx.x >> 6, c = blockIdx.x * 64 + cl;
    const bool ok = c < C;
    auto reduce = [&](float v, bool is_max) {
        red[tl][cl] = v;
        __syncthreads();
        float r = red[0][cl];
        for (int k = 1; k < 4; ++k) r = is_max ? fmaxf(r, red[k][cl]) : r + red[k][cl];
        __syncthreads();
        return r;
    };
    float amax = 0.f, inv = 1.0f / (float)T;
    if (att) {
        float mx = -INFINITY;
        if (ok) for (int t = tl; t < T; t += 4) mx = fmaxf(mx, att[(size_t)t * C + c]);
        amax = reduce(mx, true);
        float se = 0.f;
        if (ok) for (int t = tl; t < T; t += 4) se += expf(att[(size_t)t * C + c] - amax);
        inv = 1.0f / reduce(se, false);
    }
    float sm = 0.f;
    if (ok) for (int t = tl; t < T; t += 4) {
        const float w = att ? expf(att[(size_t)t * C + c] - amax) * inv : inv;
        sm += w * x[(size_t)t * C + c];
    }
    const float mu = reduce(sm, false);
    float sv = 0.f;
    if (ok) for (int t = tl; t < T; t += 4) {
        const float w = att ? expf(att[(size_t)t * C + c] - amax) * inv : inv;
        const float d = x[(size_t)t * C + c] - mu;
        sv += w * d * d;
    }
    const float var = reduce(sv, false);
    if (ok && tl == 0) {
        mean[c] = mu;
        if (stdv) stdv[c] = sqrtf(fmaxf(var, 1e-12f));
    }
}
// SE scale + residual (qwen3_tts.py:378, 532): out[t][c] = h[t][c] * s[c] + res[t][c]; a second copy goes into the aggregation buffer
__global__ __launch_bounds__(256) void k_enc_se_apply(const float* h, const float* s, const float* res, float* out, float* out2, int ld2, int T, int C) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)T * C) return;
    const int t = (int)(i / C), c = (int)(i % C);
    const float v = h[i] * s[c] + res[i];
    out[i] = v;
    out2[(size_t)t * ld2 + c] = v;
}
// [x, mean, std] along channels (qwen3_tts.py:452-454): out [T][3C]
__global__ __launch_bounds__(256) void k_enc_asp_cat(const float* x, const float* mean, const float* stdv, float* out, int T, int C) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)T * 3 * C) return;
    const int t = (int)(i / (3 * C)), c = (int)(i % (3 * C));
    out[i] = c < C ? x[(size_t)t * C + c] : (c < 2 * C ? mean[c - C] : stdv[c - 2 * C]);
}

struct vox_spkenc {
    vox_ctx* ctx;
    vox_spkenc_config cfg;
    vox_spkenc_weights w;
    int max_T, max_pad;
    float *mel = nullptr, *g = nullptr, *c0 = nullptr, *a = nullptr, *cat = nullptr, *h2 = nullptr, *hA = nullptr, *hB = nullptr,
          *co[8] = {}, *mfa_in = nullptr, *x = nullptr, *att_in = nullptr, *att_h = nullptr, *logits = nullptr, *vec = nullptr;
};
static inline unsigned enc_grid(size_t n) { return (unsigned)((n + 255) / 256); }
static inline void enc_act(hipStream_t st, float* x, size_t n, int mode) { hipLaunchKernelGGL(k_enc_act, dim3(enc_grid(n)), dim3(256), 0, st, x, n, mode); }

extern "C" {

void vox_spkenc_destroy(vox_spkenc* m) {
    if (!m) return;
    float* all[] = {m->mel, m->g, m->c0, m->a, m->cat, m->h2, m->hA, m->hB, m->mfa_in, m->x, m->att_in, m->att_h, m->logits, m->vec};
    for (float* p : all) if (p) (void)hipFree(p);
    for (float* p : m->co) if (p) (void)hipFree(p);
    delete m;
}

int vox_spkenc_create(vox_ctx* ctx, const vox_spkenc_config* cfg, const vox_spkenc_weights* w, int max_samples, vox_spkenc** out) {
    if (!ctx || !cfg || !w || !out) return vox_fail(VOX_ERR_INVALID, "spkenc_create: NULL");
    const vox_spkenc_config& c = *cfg;
    if (c.n_fft < 64 || c.n_fft > ENC_MAX_FFT || (c.n_fft & (c.n_fft - 1)) || c.hop < 1 || c.hop > c.n_fft || c.n_mels > c.n_mels_padded ||
        c.n_mels_padded % 32 || c.n_blocks < 1 || c.n_blocks > 4 || c.scale < 2 || c.scale > 8 || c.channels % (32 * c.scale) ||
        c.mfa_channels != c.n_blocks * c.channels || c.se_channels % 32 || c.att_channels % 32 || !(c.kernel0 & 1) || max_samples < c.n_fft)
        return vox_fail(VOX_ERR_INVALID, "spkenc_create: bad config");
    vox_spkenc* m = new vox_spkenc();
    m->ctx = ctx; m->cfg = c; m->w = *w;
    m->max_T = (max_samples + 2 * ((c.n_fft - c.hop) / 2) - c.n_fft) / c.hop + 1;
    int pad = c.dilation0 * (c.kernel0 - 1) / 2;
    for (int b = 0; b < c.n_blocks; ++b) {
        if (!(c.kernels[b] & 1)) { delete m; return vox_fail(VOX_ERR_INVALID, "spkenc_create: even kernel"); }
        pad = max(pad, c.dilations[b] * (c.kernels[b] - 1) / 2);
    }
    m->max_pad = pad;
    const size_t Tp = (size_t)m->max_T + 2 * pad, T = m->max_T, C = c.channels, M = c.mfa_channels, cw = C / c.scale;
    auto A = [&](float** p, size_t n) { return hipMalloc((void**)p, n * 4) == hipSuccess; };
    bool ok = A(&m->mel, T * c.n_mels_padded) && A(&m->g, Tp * (size_t)max(c.n_mels_padded, (int)cw)) && A(&m->c0, Tp * C) && A(&m->a, T * C) &&
              A(&m->cat, T * C) && A(&m->h2, T * C) && A(&m->hA, T * C) && A(&m->hB, T * C) && A(&m->mfa_in, T * M) && A(&m->x, T * M) &&
              A(&m->att_in, T * 3 * M) && A(&m->att_h, T * c.att_channels) && A(&m->logits, T * M) &&
              A(&m->vec, (size_t)(4 * M + 2 * C + c.se_channels + 64));
    for (int i = 1; i < c.scale && ok; ++i) ok = A(&m->co[i], Tp * cw);
    if (!ok) { vox_spkenc_destroy(m); return vox_fail(VOX_ERR_NOMEM, "spkenc_create: hipMalloc failed"); }
    *out = m;
    return VOX_OK;
}

int vox_spkenc_embed(vox_spkenc* m, void* stream, const float* audio, int n_samples, float* mel_out, int32_t* n_frames, float* emb_out) {
    if (!m || !audio || !emb_out) return vox_fail(VOX_ERR_INVALID, "spkenc_embed: NULL");
    const vox_spkenc_config& c = m->cfg;
    const vox_spkenc_weights& w = m->w;
    const int padw = (c.n_fft - c.hop) / 2;
    if (n_samples <= padw) return vox_fail(VOX_ERR_INVALID, "spkenc_embed: clip of %d samples is shorter than the STFT padding", n_samples);
    const int T = (n_samples + 2 * padw - c.n_fft) / c.hop + 1;
    if (T < 1 || T > m->max_T) return vox_fail(VOX_ERR_INVALID, "spkenc_embed: %d frames (capacity %d)", T, m->max_T);
    if (T <= m->max_pad) return vox_fail(VOX_ERR_INVALID, "spkenc_embed: %d frames, reflect padding needs more than %d", T, m->max_pad);
    if (n_frames) *n_frames = T;
    hipStream_t st = (hipStream_t)stream;
    const int saved_planes = g_conv_planes, saved_skinny = g_conv_skinny_rows;
    g_conv_planes = 3; g_conv_skinny_rows = 48; g_conv_rows_gemm = false;
    const int MP = c.n_mels_padded, C = c.channels, M = c.mfa_channels, cw = C / c.scale;
    int off[CG_MAXTAPS];
    static const int off0[1] = {0};
    hipLaunchKernelGGL(k_enc_logmel, dim3(T), dim3(256), 0, st, audio, n_samples, w.window, w.mel_basis, c.n_fft, c.hop, c.n_mels, MP, m->mel);
    if (mel_out) hipLaunchKernelGGL(k_enc_copy_cols, dim3(enc_grid((size_t)T * c.n_mels)), dim3(256), 0, st, mel_out, c.n_mels, m->mel, MP, T, c.n_mels);
    // blocks[0]: TDNN(mel -> C, k0, reflect)
    int p = c.dilation0 * (c.kernel0 - 1) / 2;
    hipLaunchKernelGGL(k_enc_gather, dim3(enc_grid((size_t)(T + 2 * p) * MP)), dim3(256), 0, st, m->g, T, p, MP, m->mel, MP, (const float*)nullptr, 0);
    hift_conv_offsets(c.kernel0, c.dilation0, off, 1);
    VOX_TRY(conv_gemm(st, w.conv0, m->g, nullptr, nullptr, 1, T + 2 * p, 0, off, m->c0, nullptr, nullptr, 0));
    enc_act(st, m->c0, (size_t)(T + 2 * p) * C, 2);
    const float* h = m->c0 + (size_t)p * C;
    float* hn = m->hA;
    float *vmean = m->vec, *vs1 = m->vec + C, *vs2 = vs1 + c.se_channels;       // SE vectors
    for (int b = 0; b < c.n_blocks; ++b) {
        const vox_spkenc_block_w& bw = w.blocks[b];
        VOX_TRY(conv_gemm(st, bw.tdnn1, h, nullptr, nullptr, 1, T, 0, off0, m->a, nullptr, nullptr, 0));
        enc_act(st, m->a, (size_t)T * C, 2);
        p = c.dilations[b] * (c.kernels[b] - 1) / 2;
        hift_conv_offsets(c.kernels[b], c.dilations[b], off, 1);
        for (int i = 1; i < c.scale; ++i) {                                       // Res2Net: chunk i sees chunk i + the previous output
            hipLaunchKernelGGL(k_enc_gather, dim3(enc_grid((size_t)(T + 2 * p) * cw)), dim3(256), 0, st, m->g, T, p, cw, m->a + i * cw, C,
                               i > 1 ? m->co[i - 1] + (size_t)p * cw : (const float*)nullptr, cw);
            VOX_TRY(conv_gemm(st, bw.res2[i - 1], m->g, nullptr, nullptr, 1, T + 2 * p, 0, off, m->co[i], nullptr, nullptr, 0));
            enc_act(st, m->co[i], (size_t)(T + 2 * p) * cw, 2);
        }
        hipLaunchKernelGGL(k_enc_copy_cols, dim3(enc_grid((size_t)T * cw)), dim3(256), 0, st, m->cat, C, m->a, C, T, cw);
        for (int i = 1; i < c.scale; ++i)
            hipLaunchKernelGGL(k_enc_copy_cols, dim3(enc_grid((size_t)T * cw)), dim3(256), 0, st, m->cat + i * cw, C, m->co[i] + (size_t)p * cw, cw, T, cw);
        VOX_TRY(conv_gemm(st, bw.tdnn2, m->cat, nullptr, nullptr, 1, T, 0, off0, m->h2, nullptr, nullptr, 0));
        enc_act(st, m->h2, (size_t)T * C, 2);
        hipLaunchKernelGGL(k_enc_colstats, dim3((C + 63) / 64), dim3(256), 0, st, m->h2, T, C, (const float*)nullptr, vmean, (float*)nullptr);
        VOX_TRY(conv_gemm(st, bw.se1, vmean, nullptr, nullptr, 1, 1, 0, off0, vs1, nullptr, nullptr, 0));
        enc_act(st, vs1, c.se_channels, 2);
        VOX_TRY(conv_gemm(st, bw.se2, vs1, nullptr, nullptr, 1, 1, 0, off0, vs2, nullptr, nullptr, 0));
        enc_act(st, vs2, C, 4);
        hipLaunchKernelGGL(k_enc_se_apply, dim3(enc_grid((size_t)T * C)), dim3(256), 0, st, m->h2, vs2, h, hn, m->mfa_in + (size_t)b * C, M, T, C);
        h = hn;
        hn = hn == m->hA ? m->hB : m->hA;
    }
    VOX_TRY(conv_gemm(st, w.mfa, m->mfa_in, nullptr, nullptr, 1, T, 0, off0, m->x, nullptr, nullptr, 0));
    enc_act(st, m->x, (size_t)T * M, 2);
    float *amean = m->vec + 2 * C + c.se_channels, *astd = amean + M, *pooled = astd + M;   // pooled = [mean | std], 2M
    hipLaunchKernelGGL(k_enc_colstats, dim3((M + 63) / 64), dim3(256), 0, st, m->x, T, M, (const float*)nullptr, amean, astd);
    hipLaunchKernelGGL(k_enc_asp_cat, dim3(enc_grid((size_t)T * 3 * M)), dim3(256), 0, st, m->x, amean, astd, m->att_in, T, M);
    VOX_TRY(conv_gemm(st, w.asp_tdnn, m->att_in, nullptr, nullptr, 1, T, 0, off0, m->att_h, nullptr, nullptr, 0));
    enc_act(st, m->att_h, (size_t)T * c.att_channels, 3);
    VOX_TRY(conv_gemm(st, w.asp_conv, m->att_h, nullptr, nullptr, 1, T, 0, off0, m->logits, nullptr, nullptr, 0));
    hipLaunchKernelGGL(k_enc_colstats, dim3((M + 63) / 64), dim3(256), 0, st, m->x, T, M, m->logits, pooled, pooled + M);
    VOX_TRY(conv_gemm(st, w.fc, pooled, nullptr, nullptr, 1, 1, 0, off0, emb_out, nullptr, nullptr, 0));
    g_conv_planes = saved_planes; g_conv_skinny_rows = saved_skinny;
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

}  // extern "C"

// ---- speech-tokenizer encoder: SEANet encoder + sliding-window transformer + downsample + split RVQ encode ----
// (tokenizer/qwen3_codec.py:1669-1773 over transformers' MimiModel; see include/voxhip.h).  Layout: fp32 time-major [t][C].
// A stride-r conv (kernel 2r, causal left pad r, zero right pad to a whole stride) is a two-tap conv_gemm over the same buffer
// viewed as [ceil(L/r)][r C]: output o reads view rows o-1 (kernel taps 0..r-1) and o (taps r..2r-1); row -1 reads as zero.
__global__ __launch_bounds__(256) void k_cenc_conv_in(const float* audio, int N, const float* w, const float* b, float* out, int nf, int k) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)N * nf) return;
    const int t = (int)(i / nf), co = (int)(i % nf);
    float acc = 0.f;
    for (int j = 0; j < k; ++j) {
        const int s = t - (k - 1) + j;
        if (s >= 0) acc += w[co * k + j] * audio[s];
    }
    out[i] = acc + b[co];
}
// rotate-half RoPE in place on the q and k thirds of qkv [T][3 A], A = H D
__global__ __launch_bounds__(256) void k_cenc_rope(float* qkv, int T, int H, int D, const float* inv_freq) {
    const int half = D / 2;
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)T * 2 * H * half) return;
    const int d = (int)(i % half), h = (int)((i / half) % H), which = (int)((i / ((size_t)half * H)) % 2), t = (int)(i / ((size_t)half * H * 2));
    const float ang = (float)t * inv_freq[d], cs = cosf(ang), sn = sinf(ang);
    float* p = qkv + (size_t)t * 3 * H * D + (size_t)which * H * D + (size_t)h * D;
    const float x1 = p[d], x2 = p[d + half];
    p[d] = x1 * cs - x2 * sn;
    p[d + half] = x2 * cs + x1 * sn;
}
// causal attention over the last `window` keys; one wave per query row, lane = head dim (D <= 64); online softmax
__global__ __launch_bounds__(256) void k_cenc_attn(const float* qkv, float* out, int T, int H, int D, int window, float scale) {
    const int h = blockIdx.x, i = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= T) return;
    const int A = H * D, ld = 3 * A;
    const bool on = lane < D;
    const float q = on ? qkv[(size_t)i * ld + h * D + lane] * scale : 0.f;
    float mx = -INFINITY, l = 0.f, acc = 0.f;
    const int j0 = i - window + 1 > 0 ? i - window + 1 : 0;
    for (int j = j0; j <= i; ++j) {
        float s = on ? q * qkv[(size_t)j * ld + A + h * D + lane] : 0.f;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        const float nm = fmaxf(mx, s), c = expf(mx - nm), p = expf(s - nm);
        l = l * c + p;
        acc = acc * c + (on ? p * qkv[(size_t)j * ld + 2 * A + h * D + lane] : 0.f);
        mx = nm;
    }
    if (on) out[(size_t)i * A + h * D + lane] = acc / l;
}
// frame pairs for the stride-2 downsample conv (kernel 4, replicate padding): dst [To][2 H] = [x[2o] | x[2o+1]] (the last frame
// repeated when T is odd); hist [2 H] = [x[0] | x[0]] (the replicate left padding, read as the conv's look-back row)
__global__ __launch_bounds__(256) void k_cenc_pairs(const float* x, int T, int Hd, float* dst, float* hist) {
    const int To = (T + 1) / 2;
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)(To + 1) * 2 * Hd) return;
    const int o = (int)(i / (2 * Hd)), c = (int)(i % (2 * Hd));
    if (o == To) { hist[c] = x[c % Hd]; return; }
    int t = 2 * o + c / Hd;
    t = t < T ? t : T - 1;
    dst[i] = x[(size_t)t * Hd + c % Hd];
}
// residual vector quantisation of one frame per block (MimiResidualVectorQuantizer.encode): per layer the nearest centroid by squared
// distance (lowest index on an exact tie), residual -= centroid.  One wave per centroid at a time, lanes over the dimension.
__global__ __launch_bounds__(256) void k_cenc_rvq(const float* x, const float* emb, int n_layers, int bins, int dim, int32_t* codes, int ld_codes) {
    __shared__ float r[512];
    __shared__ float bd[4];
    __shared__ int bi[4];
    const int t = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int d = threadIdx.x; d < dim; d += 256) r[d] = x[(size_t)t * dim + d];
    __syncthreads();
    for (int q = 0; q < n_layers; ++q) {
        const float* E = emb + (size_t)q * bins * dim;
        float best = INFINITY;
        int besti = 0x7fffffff;
        // eight centroids per pass: their rows' loads are independent and in flight together (the search is load-latency bound)
        for (int c0 = wave; c0 < bins; c0 += 32) {
            float s8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            for (int d = lane; d < dim; d += 64) {
                const float rd = r[d];
                float e8[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int c = c0 + 4 * u;
                    e8[u] = E[(size_t)(c < bins ? c : bins - 1) * dim + d];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) { const float df = rd - e8[u]; s8[u] += df * df; }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                float sv = s8[u];
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) sv += __shfl_xor(sv, o);
                const int c = c0 + 4 * u;
                if (c < bins && sv < best) { best = sv; besti = c; }
            }
        }
        if (lane == 0) { bd[wave] = best; bi[wave] = besti; }
        __syncthreads();
        float b = bd[0];
        int k = bi[0];
        for (int w = 1; w < 4; ++w)
            if (bd[w] < b || (bd[w] == b && bi[w] < k)) { b = bd[w]; k = bi[w]; }
        if (threadIdx.x == 0) codes[(size_t)t * ld_codes + q] = k;
        __syncthreads();
        for (int d = threadIdx.x; d < dim; d += 256) r[d] -= E[(size_t)k * dim + d];
        __syncthreads();
    }
}

struct vox_codecenc {
    vox_ctx* ctx;
    vox_codecenc_config cfg;
    vox_codecenc_weights w;
    int max_samples, hop25, max_T25;
    size_t big;
    float *A = nullptr, *B = nullptr, *C = nullptr, *tr[4] = {nullptr, nullptr, nullptr, nullptr}, *hist = nullptr, *proj = nullptr;
    int32_t* zero_slot = nullptr;
};

extern "C" {

void vox_codecenc_destroy(vox_codecenc* m) {
    if (!m) return;
    (void)hipFree(m->A); (void)hipFree(m->B); (void)hipFree(m->C); (void)hipFree(m->hist); (void)hipFree(m->proj); (void)hipFree(m->zero_slot);
    for (float* p : m->tr) (void)hipFree(p);
    delete m;
}

int vox_codecenc_create(vox_ctx* ctx, const vox_codecenc_config* cfg, const vox_codecenc_weights* w, int max_samples, vox_codecenc** out) {
    if (!ctx || !cfg || !w || !out) return vox_fail(VOX_ERR_INVALID, "codecenc_create: NULL");
    const vox_codecenc_config& c = *cfg;
    if (c.num_filters % (32 * c.compress) || c.compress < 1 || c.hidden % 32 || c.head_dim > 64 || c.head_dim % 2 || c.num_layers > 16 ||
        c.num_heads * c.head_dim % 32 || c.ffn % 32 || c.codebook_dim % 32 || c.codebook_dim > 512 || c.residual_kernel_size != 3 ||
        c.last_kernel_size != 3 || c.kernel_size > 16 || c.n_semantic < 1 || c.n_acoustic < 0 || max_samples < 1)
        return vox_fail(VOX_ERR_INVALID, "codecenc_create: bad config");
    vox_codecenc* m = new vox_codecenc();
    m->ctx = ctx; m->cfg = c; m->w = *w; m->max_samples = max_samples;
    // rows x channels shrinks by 2/r per stage, so the first stage bounds every SEANet buffer; + one padded stride of slack per stage
    size_t L = max_samples, ch = c.num_filters, big = (L + 64) * ch;
    m->hop25 = 1;
    for (int s = 0; s < 4; ++s) {
        if (c.ratios[s] < 1) { delete m; return vox_fail(VOX_ERR_INVALID, "codecenc_create: bad ratio"); }
        L = (L + c.ratios[s] - 1) / c.ratios[s];
        ch *= 2;
        m->hop25 *= c.ratios[s];
        big = big > (L + 64) * ch ? big : (L + 64) * ch;
    }
    m->max_T25 = (int)L;
    m->big = big;
    const size_t T = L + 2, A3 = (size_t)3 * c.num_heads * c.head_dim, wide = A3 > (size_t)c.ffn ? A3 : (size_t)c.ffn;
    bool ok = hipMalloc((void**)&m->A, big * 4) == hipSuccess && hipMalloc((void**)&m->B, big * 4) == hipSuccess &&
              hipMalloc((void**)&m->C, big * 4) == hipSuccess && hipMalloc((void**)&m->hist, (size_t)2 * c.hidden * 4) == hipSuccess &&
              hipMalloc((void**)&m->proj, T * c.codebook_dim * 4) == hipSuccess && hipMalloc((void**)&m->zero_slot, 4) == hipSuccess;
    for (int i = 0; i < 4 && ok; ++i) ok = hipMalloc((void**)&m->tr[i], T * (i < 2 ? (size_t)c.hidden * 2 : wide) * 4) == hipSuccess;
    if (!ok) { vox_codecenc_destroy(m); return vox_fail(VOX_ERR_NOMEM, "codecenc_create: hipMalloc failed"); }
    (void)hipMemset(m->zero_slot, 0, 4);
    *out = m;
    return VOX_OK;
}

int vox_codecenc_encode(vox_codecenc* m, void* stream, const float* audio, int n_samples, int32_t* codes, int32_t* n_frames, float* latents_out) {
    if (!m || !audio || !codes) return vox_fail(VOX_ERR_INVALID, "codecenc_encode: NULL");
    if (n_samples < 1 || n_samples > m->max_samples) return vox_fail(VOX_ERR_INVALID, "codecenc_encode: %d samples (capacity %d)", n_samples, m->max_samples);
    const vox_codecenc_config& c = m->cfg;
    const vox_codecenc_weights& w = m->w;
    hipStream_t st = (hipStream_t)stream;
    const int saved_planes = g_conv_planes, saved_skinny = g_conv_skinny_rows;
    g_conv_planes = 3; g_conv_skinny_rows = 48; g_conv_rows_gemm = false;
    static const int off0[1] = {0}, off3[3] = {2, 1, 0}, off2[2] = {1, 0};
    float *x = m->A, *t1 = m->B, *t2 = m->C;
    int L = n_samples, ch = c.num_filters;
    hipLaunchKernelGGL(k_cenc_conv_in, dim3(enc_grid((size_t)L * ch)), dim3(256), 0, st, audio, L, w.in_w, w.in_b, x, ch, c.kernel_size);
    for (int s = 0; s < 4; ++s) {
        const vox_codecenc_stage_w& sw = w.stage[s];
        const int r = c.ratios[s], Lo = (L + r - 1) / r;
        elu(st, x, t1, (size_t)L * ch);
        VOX_TRY(conv_gemm(st, sw.conv1, t1, nullptr, nullptr, 1, L, 0, off3, t2, nullptr, nullptr, 0));            // [L][ch / compress]
        elu(st, t2, t2, (size_t)L * (ch / c.compress));
        VOX_TRY(conv_gemm(st, sw.conv2, t2, nullptr, nullptr, 1, L, 0, off0, x, x, nullptr, 0));                   // x += conv2(...)
        elu(st, x, t1, (size_t)L * ch);
        if (Lo * r > L) VOX_HIP(hipMemsetAsync(t1 + (size_t)L * ch, 0, (size_t)(Lo * r - L) * ch * 4, st));      // zero right padding
        VOX_TRY(conv_gemm(st, sw.down, t1, nullptr, nullptr, 1, Lo, 0, off2, t2, nullptr, nullptr, 0));            // [Lo][2 ch]
        float* sw_ = x; x = t2; t2 = sw_;
        L = Lo; ch *= 2;
    }
    const int T = L, Hd = c.hidden, nh = c.num_heads, D = c.head_dim;
    float *h = m->tr[0], *nrm = m->tr[1], *qkv = m->tr[2], *att = m->tr[3];
    elu(st, x, t1, (size_t)T * ch);
    VOX_TRY(conv_gemm(st, w.last, t1, nullptr, nullptr, 1, T, 0, off3, h, nullptr, nullptr, 0));                   // h [T][hidden]
    for (int l = 0; l < c.num_layers; ++l) {
        const vox_mimi_layer_w& lw = w.layers[l];
        hipLaunchKernelGGL(k_layernorm_f32, dim3(T), dim3(256), 0, st, h, lw.ln1_w, lw.ln1_b, nrm, Hd, c.ln_eps);
        VOX_TRY(conv_gemm(st, lw.qkv, nrm, nullptr, nullptr, 1, T, 0, off0, qkv, nullptr, nullptr, 0));            // [T][3A]
        hipLaunchKernelGGL(k_cenc_rope, dim3(enc_grid((size_t)T * nh * D)), dim3(256), 0, st, qkv, T, nh, D, w.inv_freq);
        hipLaunchKernelGGL(k_cenc_attn, dim3(nh, (T + 3) / 4), dim3(256), 0, st, qkv, att, T, nh, D, c.window, 1.0f / sqrtf((float)D));
        VOX_TRY(conv_gemm(st, lw.o, att, nullptr, nullptr, 1, T, 0, off0, h, h, lw.scale1, 0));
        hipLaunchKernelGGL(k_layernorm_f32, dim3(T), dim3(256), 0, st, h, lw.ln2_w, lw.ln2_b, nrm, Hd, c.ln_eps);
        VOX_TRY(conv_gemm(st, lw.fc1, nrm, nullptr, nullptr, 1, T, 0, off0, qkv, nullptr, nullptr, 1));            // GELU
        VOX_TRY(conv_gemm(st, lw.fc2, qkv, nullptr, nullptr, 1, T, 0, off0, h, h, lw.scale2, 0));
    }
    const int To = (T + 1) / 2;
    hipLaunchKernelGGL(k_cenc_pairs, dim3(enc_grid((size_t)(To + 1) * 2 * Hd)), dim3(256), 0, st, h, T, Hd, nrm, m->hist);
    float* lat = latents_out ? latents_out : att;
    VOX_TRY(conv_gemm(st, w.downsample, nrm, m->hist, m->zero_slot, 1, To, 1, off2, lat, nullptr, nullptr, 0));    // [To][hidden]
    const int nq = c.n_semantic + c.n_acoustic;
    VOX_TRY(conv_gemm(st, w.sem_proj, lat, nullptr, nullptr, 1, To, 0, off0, m->proj, nullptr, nullptr, 0));
    hipLaunchKernelGGL(k_cenc_rvq, dim3(To), dim3(256), 0, st, m->proj, w.sem_emb, c.n_semantic, c.codebook_size, c.codebook_dim, codes, nq);
    if (c.n_acoustic > 0) {
        VOX_TRY(conv_gemm(st, w.ac_proj, lat, nullptr, nullptr, 1, To, 0, off0, m->proj, nullptr, nullptr, 0));
        hipLaunchKernelGGL(k_cenc_rvq, dim3(To), dim3(256), 0, st, m->proj, w.ac_emb, c.n_acoustic, c.codebook_size, c.codebook_dim,
                           codes + c.n_semantic, nq);
    }
    if (n_frames) *n_frames = To;
    g_conv_planes = saved_planes; g_conv_skinny_rows = saved_skinny;
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

}  // extern "C"
