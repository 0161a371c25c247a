// Fused 1D spectral layer: forward FFT along DY -> keep 64 modes -> complex GEMM over the channel
// dimension -> zero-pad -> backward FFT, in ONE kernel with no HBM round trip in between.
//
// Replaces fused_fft_cgemm_ifft_{7,8} of the reference
// (fusion_variants/1D_D_exp_fused_fft_cgemm_ifft/fused_fft_cgemm_ifft_7.cuh:9-222): same operands
//   x[K][S][DY]  (signal (k,s) at (k*S+s)*DY),  W[k + n*K],  y[N][S][DY],  M = 64*S,
// the same (S, N/64) blocks (as a 1D grid in an XCD-aware order), block 256, and the same "block traverses K" schedule, re-derived for wave64:
//   * an L = DY/16 lane group owns one signal; a 256-thread block transforms 256/L channels at once
//     (the reference does 8), so the K loop advances in chunks of 16 (DY=256) or 32 (DY=128) channels;
//   * the thread that accumulates C[m][n] is the thread that later needs it for the backward
//     transform, so the GEMM result never passes through LDS (the reference stages it in 8 rounds,
//     fused_fft_cgemm_ifft_7.cuh:203-218);
//   * exchange buffers are padded (row pitch 17 complex) for the 64-bank LDS of CDNA4.
#include "bf16_split.h"
#include "group_fft.h"
#include "kernels.h"

namespace tfno {

// FUSE_FWD: the A operand is produced by forward transforms of x; otherwise it is read from the column-major matrix A[m + k M]
//           (second half of the layer);
// FUSE_INV: the product goes straight into zero-padded backward transforms; otherwise it is stored as
//           C[m + n M] = alpha A W + beta C (first half).
template <int LOGDY, bool FUSE_FWD, bool FUSE_INV, bool KEEP>
__global__ __launch_bounds__(256) void fused_fft_cgemm_ifft_kernel(int S, int N, int K, const float2* __restrict__ x,
                                                                   const float2* __restrict__ W, float2* __restrict__ y,
                                                                   float2 alpha, float2 beta)
{
    using G = Geo1D<LOGDY>;
    constexpr int DY = G::DY, L = G::L, GROUPS = G::GROUPS, MM = G::MM, NN = G::NN;
    extern __shared__ float2 lds[];
    float2* sA = lds;                                  // [GROUPS][64]   truncated spectra of the K chunk
    float2* sW = sA + GROUPS * G::SA_PITCH;            // [GROUPS][64]   W chunk, sW[kk][n]
    float2* exch_all = sW + GROUPS * G::SW_PITCH;

    const int tid = threadIdx.x;
    const int g = tid / L, t = tid % L;
    long s;
    int ntile;
    decode_block_1d(S, N / 64, 1 << LOGDY, !KEEP, s, ntile);
    const int n0 = ntile * 64;
    const long M = 64L * S;
    // signals of 128 samples are transformed in pairs by 16-lane groups (128-byte accesses): lane t16 of pair g/2 holds
    // samples t16 + 16 i of both signals, and ends up with the modes an 8-lane group would give lane (g, t)
    constexpr bool PAIR = LOGDY == 7;
    const int t16 = tid % 16, gpair = (tid / 16) * 2;
    float2* exch = PAIR ? exch_all + (tid / 16) * (2 * G::EXCH) : exch_all + g * G::EXCH;

    cpx tw[16];
    load_lane_twiddles<LOGDY>(PAIR ? t16 : t, tw);

    cpx acc[MM][NN];
#pragma unroll
    for (int a = 0; a < MM; ++a)
#pragma unroll
        for (int b = 0; b < NN; ++b) acc[a][b] = make_float2(0.f, 0.f);

    for (int kc = 0; kc < K; kc += GROUPS) {
        if constexpr (FUSE_FWD) {
            const int k = kc + g;
            cpx out[MM];
            if (k < K) {
                cpx v[16];
                if constexpr (PAIR) {
                    const float2* src = x + ((long)(kc + gpair) * S + s) * DY + t16;
#pragma unroll
                    for (int i = 0; i < 8; ++i) { v[i] = src[16 * i]; v[8 + i] = src[(long)S * DY + 16 * i]; }
                    pair128_forward(v, tw, exch, t16, out);
                } else {
                    const float2* src = x + ((long)k * S + s) * DY + t;
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[i] = src[L * i];
                    group_forward<LOGDY, LOGDY == 10 && FUSE_INV>(v, tw, exch, t, out);    // SPREAD: not without the registers for it
                }
            } else {
#pragma unroll
                for (int a = 0; a < MM; ++a) out[a] = make_float2(0.f, 0.f);
            }
#pragma unroll
            for (int a = 0; a < MM; ++a) sA[g * G::SA_PITCH + (PAIR ? t + L * a : forward_mode_of_lane<LOGDY>(t, a))] = out[a];
        } else {
            // A tile of the chunk: 64 contiguous rows (this block's signal) of GROUPS columns
#pragma unroll
            for (int j = 0; j < (GROUPS * 64) / 256; ++j) {
                const int mloc = (tid + 256 * j) % 64, kk = (tid + 256 * j) / 64;
                sA[kk * G::SA_PITCH + mloc] = (kc + kk < K) ? x[s * 64 + mloc + (long)(kc + kk) * M] : make_float2(0.f, 0.f);
            }
        }
        // W chunk: GROUPS x 64 elements, consecutive threads read consecutive k (contiguous in memory)
#pragma unroll
        for (int j = 0; j < (GROUPS * 64) / 256; ++j) {
            int idx = tid + 256 * j;
            int kk = idx % GROUPS, n = idx / GROUPS;
            float2 w = make_float2(0.f, 0.f);
            if (kc + kk < K) w = W[(kc + kk) + (long)(n0 + n) * K];
            sW[kk * G::SW_PITCH + n] = w;
        }
        __syncthreads();
#pragma unroll 4
        for (int kk = 0; kk < GROUPS; ++kk) {
            cpx a[MM], b[NN];
#pragma unroll
            for (int i = 0; i < MM; ++i) a[i] = sA[kk * G::SA_PITCH + t + L * i];
#pragma unroll
            for (int j = 0; j < NN; ++j) b[j] = sW[kk * G::SW_PITCH + g + GROUPS * j];
#pragma unroll
            for (int i = 0; i < MM; ++i)
#pragma unroll
                for (int j = 0; j < NN; ++j) cfma(acc[i][j], a[i], b[j]);
        }
        __syncthreads();
    }

#pragma unroll
    for (int j = 0; j < NN; ++j) {
        const int n = n0 + g + GROUPS * j;
        if constexpr (FUSE_INV) {
            cpx c[MM], yv[16];
#pragma unroll
            for (int i = 0; i < MM; ++i) c[i] = cmul(acc[i][j], alpha);
            if constexpr (PAIR) {
                pair128_backward(c, tw, exch, t16, yv);
                float2* dst = y + ((long)(n0 + gpair + GROUPS * j) * S + s) * DY + t16;
                store_pair16<KEEP>(dst, (long)S * DY, yv);
            } else {
                group_backward<LOGDY>(c, tw, exch, t, yv);
                float2* dst = y + ((long)n * S + s) * DY + t;
                store_row16<L, KEEP>(dst, yv);
            }
        } else {
            float2* dst = y + s * 64 + t + (long)n * M;          // C[m + n M], m = 64 s + t + L i
#pragma unroll
            for (int i = 0; i < MM; ++i) {
                cpx r = cmul(acc[i][j], alpha);
                if (beta.x != 0.f || beta.y != 0.f) r = cadd(r, cmul(dst[L * i], beta));
                dst[L * i] = r;
            }
        }
    }
}

typedef float floatx4_1d __attribute__((ext_vector_type(4)));

// Fused 1D layer for DY = 128 and eight input channels: ONE WAVEFRONT per (signal set, 64 output channels), no block barrier
// and no staging of operands through LDS. The register layouts of the transforms and of v_mfma_f32_16x16x4_f32 coincide:
//   * the A operand row n' = 16 nt + t, k = g is one element of W (times alpha, as (re, -im) or (im, re)), read
//     straight from global memory (W is a few KiB and stays in the vector cache);
//   * a 16-lane group transforms two channels kc + 2 g + h at a time (lane t = r + 8 h finishes channel h with modes
//     r + 8 c, c < 8); one exchange between lanes t and t ^ 8 (a row rotation, no LDS) turns that into modes
//     t + 16 a of each of the two channels, i.e. two B operands;
//   * the accumulators D[row = 4 g + v][column = t] of tile (nt, a) hold, for j = 0, 1, the complex value
//     (v = 2 j, 2 j + 1) of output channel n = 8 nt + 2 g + j at mode t + 16 a; the same exchange leads to the paired
//     backward transform of output channels 8 nt + 2 g and 8 nt + 2 g + 1.
// 32 accumulator tiles (128 registers) per wave, two waves per SIMD; the only LDS traffic left is the exchange inside
// the transforms. With eight channels the split kernel (layer1d_split.hip) leaves three of four waves without a transform:
// S = 1000, N = 64: 16.4 here against 18.8 us, N = 128: 32.5 / 33.6, S = 16384, N = 64: 198 / 201; from 16 channels on that kernel is
// ahead (S = 1000, K = 16, N = 64: 20.5 / 18.7).
template <bool KEEP>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) void fused_fft_mfma_ifft_wave_kernel(
    int S, int N, int K, const float2* __restrict__ x, const float2* __restrict__ W, float2* __restrict__ y, float2 alpha)
{
    constexpr int DY = 128, EXCH = 16 * 17, CH = 8;               // CH = channels per round
    __shared__ float2 lds[4 * EXCH + kTwLdsSize];
    const int lane = threadIdx.x, g = lane >> 4, t = lane & 15;
    float2* exch = lds + g * EXCH;
    float2* twtab = lds + 4 * EXCH;
    fill_lds_twiddles<7>(twtab, lane, 64);
    const float2* twrow = twtab + t * kTwLdsPitch;
    __syncthreads();
    long s;
    int ntile;
    decode_block_1d(S, N / 64, DY, !KEEP, s, ntile);
    const int n0 = ntile * 64;
    const bool upper = t >> 3, odd = t & 1;

    floatx4_1d acc[8][4];
#pragma unroll
    for (int nt = 0; nt < 8; ++nt)
#pragma unroll
        for (int a = 0; a < 4; ++a) acc[nt][a] = floatx4_1d{ 0.f, 0.f, 0.f, 0.f };

    // lane (g, t): samples t + 16 i of channels kc + 2 g, kc + 2 g + 1
    const float2* src = x + ((long)(2 * g) * S + s) * DY + t;
    const float2* wsrc = W + (2 * g) + (long)(n0 + (t >> 1)) * K;   // W[k][n = n0 + 8 nt + t / 2]
    auto issue = [&](cpx (&dst)[16]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) { dst[i] = src[16 * i]; dst[8 + i] = src[(long)S * DY + 16 * i]; }
    };
    // one complex product row: acc += W'(row n', k) x B(k, column), W' = alpha W as (re, -im) / (im, re) by row parity
    auto contract = [&](floatx4_1d (&d)[4], float2 wk, const cpx (&b)[4]) {
        const float2 w = make_float2(wk.x * alpha.x - wk.y * alpha.y, wk.x * alpha.y + wk.y * alpha.x);
        const float ax = odd ? w.y : w.x, ay = odd ? w.x : -w.y;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            d[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(ax, b[a].x, d[a], 0, 0, 0);
            d[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(ay, b[a].y, d[a], 0, 0, 0);
        }
    };
    cpx v[16];
    issue(v);
    for (int kc = 0; kc < K; kc += CH) {                          // K is a multiple of 8 (caller contract)
        float2 wv[8], wv1[8];
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            wv[nt] = wsrc[kc + (long)(8 * nt) * K];
            wv1[nt] = wsrc[kc + 1 + (long)(8 * nt) * K];
        }
        cpx gg[16], out[8], b8[8];
        {
            cpx a8[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) { a8[i] = v[i]; b8[i] = v[8 + i]; }
            fft8<-1>(a8);
            fft8<-1>(b8);
#pragma unroll
            for (int r = 0; r < 8; ++r) gg[r] = a8[r];
        }
        if (kc + CH < K) { src += (long)CH * S * DY; issue(v); }
        gg[8] = b8[0];
#pragma unroll
        for (int r = 1; r < 8; ++r) {
            const cpx w = twrow[r];
            gg[r] = cmul(gg[r], w);
            gg[8 + r] = cmul(b8[r], w);
        }
        rows128_forward_finish(gg, exch, t, out);             // out[c] = mode (t & 7) + 8 c of channel t >> 3
        // lanes t < 8 keep the even c of their channel and take the even c of the other one; lanes t >= 8 the odd c
        cpx b0[4], b1[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const cpx got = rotate8(upper ? out[2 * a] : out[2 * a + 1]);
            b0[a] = upper ? got : out[2 * a];                 // channel kc + 2 g,     mode t + 16 a
            b1[a] = upper ? out[2 * a + 1] : got;             // channel kc + 2 g + 1, mode t + 16 a
        }
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            contract(acc[nt], wv[nt], b0);
            contract(acc[nt], wv1[nt], b1);
        }
    }
    // backward: the two output channels (j = 0, 1) a lane group owns per n tile are transformed together
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
        cpx c0[4], c1[4], y0[16];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            c0[a] = make_float2(acc[nt][a][0], acc[nt][a][1]);   // channel 8 nt + 2 g,     mode t + 16 a
            c1[a] = make_float2(acc[nt][a][2], acc[nt][a][3]);   // channel 8 nt + 2 g + 1, mode t + 16 a
        }
        float2* dst = y + ((long)(n0 + 8 * nt + 2 * g) * S + s) * DY + t;
        // lane t = r + 8 h finishes channel h: modes r + 8 c; even c come from lanes t < 8, odd c from lanes t >= 8
        cpx c8[8];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const cpx got = rotate8(upper ? c0[a] : c1[a]);
            c8[2 * a] = upper ? got : c0[a];
            c8[2 * a + 1] = upper ? c1[a] : got;
        }
        rows128_backward(c8, twrow, exch, t, y0);
        store_pair16<KEEP>(dst, (long)S * DY, y0);
    }
}

// Fused 1D layer for grids of more than half a block of 32 output channels per CU and at most one, DY = 256, more than 96 channels (fewer
// blocks or channels: layer1d_small.hip): the eight waves of a block share ONE
// item (signal set, 32 output channels) and split its K input channels: wave w transforms channels 32 r + 4 w + g in round r,
// g = 16-lane group. Four rounds give a lane four channels of its modes t + 16 a: with real and imaginary part the eight
// consecutive values of the contraction that a lane holds of the B operand of v_mfma_f32_16x16x32_bf16, so a wave multiplies its
// 16 channels straight out of its registers (exact three-way split, bf16_split.h) into its own partial accumulators (2 tiles of 16
// output channels x 4 m tiles). The K loop has no barrier and stages nothing through LDS. The eight partial products
// meet in LDS once (sP[w][n][m], pitch 72 complex: conflict-free b64 stores), every lane group sums the eight partials
// of one output channel and runs its backward transform. The chain of latencies of an item is K / 32 rounds + K / 128 products +
// one reduction + one backward pass. S = 64, K = N = 128: 17.6 us with fp32 matrix instructions in every round, 15.7 with the split, 16.0 with the search for operands that the split does not hold
// (for which the wave's share of the product is formed in fp32 instead); K = 64: 13.1 / 13.1 / 13.2.
constexpr int SPLIT_NT = 32, SPLIT_PP = 72;
constexpr size_t SPLIT_LDS = sizeof(float2) * 8 * SPLIT_NT * SPLIT_PP;       // 147,456 B; covers the 32 exchange regions

template <bool KEEP>
__global__ __launch_bounds__(512) void fused_fft_mfma_ifft_split_kernel(int S, int N, int K, const float2* __restrict__ x,
                                                                        const float2* __restrict__ W, float2* __restrict__ y,
                                                                        float2 alpha)
{
    constexpr int DY = 256, EXCH = 16 * 17, TILES = SPLIT_NT / 16;
    extern __shared__ float2 lds[];
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, t = lane & 15;
    float2* exch = lds + (4 * w + g) * EXCH;                      // the partials overlay these after the K loop
    long s;
    int ntile;
    decode_block_1d(S, N / SPLIT_NT, 256, !KEEP, s, ntile);
    const int n0 = ntile * SPLIT_NT;
    cpx tw[16];
    load_lane_twiddles<8>(t, tw);

    float4_v re[TILES][4], im[TILES][4];
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int a = 0; a < 4; ++a) re[i][a] = im[i][a] = float4_v{ 0.f, 0.f, 0.f, 0.f };

    // K is a multiple of 8 and a wave covers four consecutive channels: a wave is either fully inside K or idle
    const int k0 = 4 * w + g;
    const float2* src = x + ((long)k0 * S + s) * DY + t;
    const float2* wsrc = W + k0 + (long)(n0 + t) * K;             // W[k][n = n0 + 16 i + t]
    auto issue = [&](cpx (&dst)[16], int kc) {                    // samples t + 16 i of channel kc + k0
        const float2* p = src + (long)kc * S * DY;
#pragma unroll
        for (int i = 0; i < 16; ++i) dst[i] = p[16 * i];
    };
    // the buffer is refilled as soon as the first pass has consumed it (a second buffer, two rounds ahead, was
    // measured slower: a round is bound by its arithmetic, not by the latency of its loads)
    cpx v[16];
    bool low = false;                                             // values too small for the split among the wave's operands
    if (4 * w < K) issue(v, 0);
    for (int kc = 0; kc + 4 * w < K; kc += 128) {
        SplitOperand b[4];
        float2 wv[TILES][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int kr = kc + 32 * j;
            if (kr + 4 * w < K) {
#pragma unroll
                for (int i = 0; i < TILES; ++i) wv[i][j] = wsrc[kr + (long)(16 * i) * K];
                cpx gg[16], out[4];
                fwd_pass1(v, tw, gg);
                if (kr + 32 + 4 * w < K) issue(v, kr + 32);
                group_forward_finish<8>(gg, exch, t, out);
                low |= below_split_range(out);
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    unsigned h, m, l;
                    split_bf16_pair(out[a].x, out[a].y, h, m, l);
                    b[a].h[j] = h; b[a].m[j] = m; b[a].l[j] = l;
                }
            } else {                                              // beyond K: zeros
#pragma unroll
                for (int i = 0; i < TILES; ++i) wv[i][j] = make_float2(0.f, 0.f);
#pragma unroll
                for (int a = 0; a < 4; ++a) b[a].h[j] = b[a].m[j] = b[a].l[j] = 0u;
            }
        }
#pragma unroll
        for (int i = 0; i < TILES; ++i) {
            SplitOperand wre, wim;                                // rows (re, -im) and (im, re) of alpha W
#pragma unroll
            for (int j = 0; j < 4; ++j) wv[i][j] = cmul(wv[i][j], alpha);
            unsigned bits = ~0u;                                  // (zeros are common here: channels beyond K)
#pragma unroll
            for (int j = 0; j < 4; ++j) bits = lower(bits, wv[i][j]);
            low |= any_lane(bits < kSplitLow);
#pragma unroll
            for (int j = 0; j < 4; ++j) split_weight_rows(wv[i][j], wre, wim, j);
#pragma unroll
            for (int a = 0; a < 4; ++a) mac_split_pair(wre, wim, b[a], re[i][a], im[i][a]);
        }
    }
    float high[2] = { 0.f, 0.f };
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int a = 0; a < 4; ++a) { high[0] = larger(high[0], re[i][a]); high[1] = larger(high[1], im[i][a]); }
    if (__builtin_expect(low | any_lane(not_finite(high[0], high[1])), 0)) {
        // operands beyond the split: the wave's share of the product in fp32, one round of four channels at a time
#pragma unroll
        for (int i = 0; i < TILES; ++i)
#pragma unroll
            for (int a = 0; a < 4; ++a) re[i][a] = im[i][a] = float4_v{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll 1
        for (int kr = 0; kr + 4 * w < K; kr += 32) {
            cpx gg[16], out[4];
            issue(v, kr);
            fwd_pass1(v, tw, gg);
            group_forward_finish<8>(gg, exch, t, out);
#pragma unroll
            for (int i = 0; i < TILES; ++i) {
                const float2 wk = cmul(wsrc[kr + (long)(16 * i) * K], alpha);
#pragma unroll
                for (int a = 0; a < 4; ++a) mac_fp32(wk, out[a], re[i][a], im[i][a]);
            }
        }
    }
    __syncthreads();                                              // every wave is done with its exchange regions
    // D[row = 4 g + q][column = t] of tile (i, a): output channel 16 i + 4 g + q, mode t + 16 a
    float2* sP = lds + (long)w * SPLIT_NT * SPLIT_PP;
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int q = 0; q < 4; ++q) sP[(16 * i + 4 * g + q) * SPLIT_PP + t + 16 * a] = make_float2(re[i][a][q], im[i][a][q]);
    __syncthreads();
    // lane group (w, g) owns output channel n = 4 w + g: sum of the eight partials, modes t + 16 a
    const int n = 4 * w + g;
    cpx c[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        cpx sum = lds[n * SPLIT_PP + t + 16 * a];
#pragma unroll
        for (int ww = 1; ww < 8; ++ww) sum = cadd(sum, lds[(ww * SPLIT_NT + n) * SPLIT_PP + t + 16 * a]);
        c[a] = sum;
    }
    __syncthreads();                                              // the partials are consumed: exchange regions again
    cpx yv[16];
    group_backward<8>(c, tw, exch, t, yv);
    store_row16<16, KEEP>(y + ((long)(n0 + n) * S + s) * DY + t, yv);
}

// Stand-alone truncated forward / zero-padded backward transforms of contiguous signals (variants A, B, C):
//   fft_stride_DY : in[nsig][DY] -> out[nsig][64]      ifft_stride_DY : in[nsig][64] -> out[nsig][DY]
// Replace fft_N_stride_DY / ifft_N_stride_DY of the missing TurboFFT submodule (launched at
// fusion_variants/1D_A_exp_fft+cgemm+ifft/fused.cu:195,203). One L-lane group per signal, 256/L signals per block.
template <int LOGDY, bool INVERSE>
__global__ __launch_bounds__(256) void stride_DY_kernel(const float2* __restrict__ in, float2* __restrict__ out, long nsig)
{
    using G = Geo1D<LOGDY>;
    constexpr int DY = G::DY, L = G::L, GROUPS = G::GROUPS, MM = G::MM;
    extern __shared__ float2 lds[];
    const int tid = threadIdx.x, g = tid / L, t = tid % L;
    const long sig = (long)blockIdx.x * GROUPS + g;
    cpx tw[16];
    if constexpr (LOGDY == 7) {
        // signals of 128 samples go in pairs through 16-lane groups (128-byte accesses); lane (g, t) still ends up with /
        // starts from the modes t + 8 a of signal g. All 16 lanes take part for either signal, so a pair with one
        // signal beyond nsig loads zeros for it and skips its stores instead of leaving early.
        const int t16 = tid % 16;
        const long sigA = (long)blockIdx.x * GROUPS + (tid / 16) * 2;
        float2* exch = lds + (tid / 16) * (2 * G::EXCH);
        load_lane_twiddles<LOGDY>(t16, tw);
        if (sigA >= nsig) return;                    // whole pair out of range (uniform per 16-lane group)
        const bool hasB = sigA + 1 < nsig;
        if constexpr (!INVERSE) {
            const float2* src = in + sigA * DY + t16;
            cpx v[16], o[MM];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                v[i] = src[16 * i];
                v[8 + i] = hasB ? src[DY + 16 * i] : make_float2(0.f, 0.f);
            }
            pair128_forward(v, tw, exch, t16, o);
            if (sig < nsig) {
                float2* dst = out + sig * 64 + t;
#pragma unroll
                for (int a = 0; a < MM; ++a) dst[L * a] = o[a];
            }
        } else {
            cpx c[MM], yv[16];
#pragma unroll
            for (int a = 0; a < MM; ++a) c[a] = sig < nsig ? in[sig * 64 + t + L * a] : make_float2(0.f, 0.f);
            pair128_backward(c, tw, exch, t16, yv);
            float2* dst = out + sigA * DY + t16;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                store_streaming(dst + 16 * i, yv[i]);
                if (hasB) store_streaming(dst + DY + 16 * i, yv[8 + i]);
            }
        }
        return;
    } else {
    float2* exch = lds + g * G::EXCH;
    load_lane_twiddles<LOGDY>(t, tw);
    if (sig >= nsig) return;
    if constexpr (!INVERSE) {
        const float2* src = in + sig * DY + t;
        cpx v[16], o[MM];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = src[L * i];
        group_forward<LOGDY>(v, tw, exch, t, o);
        float2* dst = out + sig * 64;
#pragma unroll
        for (int a = 0; a < MM; ++a) dst[forward_mode_of_lane<LOGDY>(t, a)] = o[a];
    } else {
        const float2* src = in + sig * 64 + t;
        cpx c[MM], yv[16];
#pragma unroll
        for (int a = 0; a < MM; ++a) c[a] = src[L * a];
        group_backward<LOGDY>(c, tw, exch, t, yv);
        float2* dst = out + sig * DY + t;
#pragma unroll
        for (int i = 0; i < 16; ++i) store_streaming(dst + L * i, yv[i]);
    }
    }
}

// keep_y: the output is read again at once (Y stage of the three-kernel 2D pipeline): plain instead of streaming stores,
// as a template parameter of the kernels - a run-time branch around the stores cost the 1D layer up to 20 %
template <int LOGDY, bool FUSE_FWD, bool FUSE_INV, bool KEEP>
static hipError_t launch_fused_1d_k(long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, float2 beta,
                                    hipStream_t stream)
{
    using G = Geo1D<LOGDY>;
    if (S * (N / 64) > 0x7fffffffL) return hipErrorInvalidValue;
    if constexpr (G::LDS_BYTES > 64 * 1024) {          // DY = 128: 32 channels per chunk, 70 KiB
        static std::atomic<unsigned long long> served;
        if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(fused_fft_cgemm_ifft_kernel<LOGDY, FUSE_FWD, FUSE_INV, KEEP>),
                                             G::LDS_BYTES, served);
            e != hipSuccess)
            return e;
    }
    dim3 grid((unsigned)(S * (N / 64)), 1, 1), block(256, 1, 1);
    hipLaunchKernelGGL((fused_fft_cgemm_ifft_kernel<LOGDY, FUSE_FWD, FUSE_INV, KEEP>), grid, block, G::LDS_BYTES, stream, (int)S, N, K, x, W,
                       y, alpha, beta);
    return hipGetLastError();
}
template <int LOGDY>
static hipError_t launch_fused_1d(long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, hipStream_t stream, int keep_y)
{
    const float2 beta = make_float2(0.f, 0.f);
    return keep_y ? launch_fused_1d_k<LOGDY, true, true, true>(S, N, K, x, W, y, alpha, beta, stream)
                  : launch_fused_1d_k<LOGDY, true, true, false>(S, N, K, x, W, y, alpha, beta, stream);
}
static hipError_t dispatch_fused_1d(int logDY, long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha,
                                    hipStream_t stream, int keep_y)
{
    switch (logDY) {
    case 7: return launch_fused_1d<7>(S, N, K, x, W, y, alpha, stream, keep_y);
    case 8: return launch_fused_1d<8>(S, N, K, x, W, y, alpha, stream, keep_y);
    case 9: return launch_fused_1d<9>(S, N, K, x, W, y, alpha, stream, keep_y);
    case 10: return launch_fused_1d<10>(S, N, K, x, W, y, alpha, stream, keep_y);
    default: return hipErrorInvalidValue;
    }
}

// keep_y as for the other kernels: as the middle stage of one 256 x 256 image, K = 64, N = 128, the layer takes 37.1 us, 40.6 with streaming stores
template <bool KEEP>
static hipError_t launch_fused_split_channels(long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, hipStream_t stream)
{
    static std::atomic<unsigned long long> served;
    if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(fused_fft_mfma_ifft_split_kernel<KEEP>), SPLIT_LDS, served);
        e != hipSuccess)
        return e;
    if (S * (N / SPLIT_NT) > 0x7fffffffL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(fused_fft_mfma_ifft_split_kernel<KEEP>, dim3((unsigned)(S * (N / SPLIT_NT))), dim3(512), SPLIT_LDS, stream, (int)S, N,
                       K, x, W, y, alpha);
    return hipGetLastError();
}

static hipError_t launch_fused_wave(long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, hipStream_t stream,
                                    int keep_y)
{
    if (S * (N / 64) > 0x7fffffffL) return hipErrorInvalidValue;
    if (keep_y)
        hipLaunchKernelGGL((fused_fft_mfma_ifft_wave_kernel<true>), dim3((unsigned)(S * (N / 64))), dim3(64), 0, stream, (int)S, N, K, x, W,
                           y, alpha);
    else
        hipLaunchKernelGGL((fused_fft_mfma_ifft_wave_kernel<false>), dim3((unsigned)(S * (N / 64))), dim3(64), 0, stream, (int)S, N, K, x, W,
                           y, alpha);
    return hipGetLastError();
}

// Which fused 1D kernel runs for a problem: pure arithmetic on the sizes, the selector `algo`, the number of compute
// units and whether the stream has an exchange buffer attached (no device call), so that callers and tests can ask.
// algo: 0 = by size, 1 = SIMT kernel, 2 = matrix cores with 512-thread blocks of 64 output channels (layer1d_small.hip), 3 = matrix cores
// with 256-thread blocks of 64 output channels (layer1d_split.hip), 4 = as 2 with 32 output channels, 5 = as 3 for large grids: four
// blocks per CU, or with eight channels of length 128 one wavefront per (signal set, output tile), 6 = matrix cores, the eight waves of
// a block split the K channels of one item (DY = 256), 7 = matrix cores, a cluster of blocks splits the K channels of one signal set
// (DY = 256, N = 64 / 128, small grids), 8 = as 3 with 128 output channels per block where N allows
// The same rule holds where y is read again at once (middle stage of a 2D layer): the lines were drawn with x and y streamed, and of
// 3166 2D layers in three stages, lengths 128 to 1024, none lost against a rule that treated that case apart.
// The return value uses the same numbers (1 ... 8); chosen by size, 2 and 4 stand for blocks of 16, 32 or 64 output channels of
// the small-grid kernel, 8 for blocks of 64 or of 128 (tile_of_fused_1d_kernel). A selector value that a kernel is not built for
// falls back to the choice by size.
//
// By size (measured on MI355X, us; of two figures the second is the kernel named):
//  * Every block of 64 output channels has a CU to itself, any length: the small-grid kernel, with the fewest output channels per
//    block that leave it so (the best other kernel / this: N = 64: DY = 128, S = 256, K = 128 19.3 / 17.7; DY = 256, S = 128,
//    K = 64 16.9 / 11.3; DY = 512, S = 128, K = 64 28.9 / 18.7). With nearly a block per CU others take over where they are ahead:
//      DY = 256, up to 16 channels: split kernel (N = 256: S = 52, K = 16 9.8 / 9.4, S = 54, K = 8 9.7 / 9.5);
//      DY = 128, 49 to 64 channels, where a round of 48 leaves a short one: split kernel (N = 64, S = 256, K = 64 12.2 / 11.9);
//      DY = 128, 32 or 40 channels, N no multiple of 128: split kernel (S = 256, K = 32 9.0 / 8.8, S = 200 8.3 / 8.5); with 16 to
//      40 channels and exactly one block per CU in the layout for two per CU (S = 256, K = 16 8.2 / 8.1);
//      DY = 1024, eight channels, more than three quarters of the CUs: SIMT kernel (N = 64: S = 200 24.4 / 23.9, S = 245 28.5 /
//      27.3; with 192 blocks it is 4 us behind as the middle stage of three images).
//  * DY = 256, more than 96 channels (a fourth round), blocks of 32 output channels for more than half of the CUs and at most one
//    each: the K split, whose rounds have no barrier (S = 64, N = 128: K = 104 15.8 / 15.2, K = 128 17.6 / 17.1). Not with fewer
//    channels or blocks (S = 64, N = 128, K = 96: 14.6 / 15.3; S = 60, N = 64, K = 104: 13.0 / 13.5).
//  * More than one block of 64 output channels per CU, lengths 128 / 256: the split kernel.
//  * Lengths 512 / 1024, more than one block per CU: the SIMT kernel with few channels, the split kernel from where it is ahead
//    (SIMT / split: DY = 512: N = 64, S = 2048: K = 24 120 / 127, K = 40 185 / 170; N = 128, S = 1000: K = 32 144 / 123; DY = 1024:
//    N = 64, S = 2048, K = 32 325 / 318; N = 128, S = 1000: K = 32 246 / 257, K = 64 389 / 349). At DY = 1024 with N no multiple of
//    128 the split kernel fits two blocks on a CU, the SIMT kernel three: below 64 channels the latter stays where rounds of two
//    per CU would be at most three quarters full (N = 64, S = 600: K = 32 98 / 102, K = 64 159 / 143; S = 512, K = 40 88 / 80), and
//    on large grids with three blocks or more per signal set (N = 192, S = 600: K = 40 242 / 259, K = 64 341 / 319).
int pick_fused_1d_kernel(int logDY, long S, int N, int K, int algo, long cus, bool exchange_attached)
{
    const bool built = logDY >= 7 && logDY <= 10;
    const bool long_signal = logDY >= 9;            // 512 / 1024
    const long items = S * (N / 64);
    if (algo == 5 && !long_signal && built) return kFused1dDense;
    if (algo == 0 && !long_signal && built) {
        const long blocks = N % 128 == 0 ? S * (N / 128) : items;
        if (logDY == 7 && N % 128 != 0 && K >= 16 && (blocks > cus || (blocks == cus && K <= 40)) && blocks <= (K >= 128 ? 4 : 2) * cus)
            return kFused1dWide;
        if (blocks > cus) {
            if (N % 128 == 0 && K >= 16) return kFused1dWide;           // 128 or 64 output channels per block: wide_tiles()
            // blocks of 64 output channels, a few per CU
            if (logDY == 8 && N % 128 != 0 && K >= 128 && blocks <= 4 * cus) return kFused1dWide;
        }
        // DY = 128: several items per SIMD
        if (logDY == 7 && items >= (K <= 16 ? 2 : (K < 128 ? 4 : 8)) * cus) return kFused1dDense;
    }
    // small grids, 64 channels or more, N = 64 / 128: a cluster of blocks per signal set, no forward transform twice.
    // Only for streams that have an exchange buffer attached; without one the kernels below take over.
    // The line was drawn against the K split. The small-grid kernel has overtaken the cluster on part of this range (us, with / without
    // a buffer, S = 64: N = 128: K = 64 12.7 / 11.9, K = 96 15.7 / 14.8, K = 128 16.2 / 16.6; N = 64: K = 64 9.7 / 9.6, K = 128 11.4 / 13.9,
    // and 1.2 to 1.3 where K is no multiple of 32, which makes clusters of two): such streams are better off without one.
    if (algo == 7 || (algo == 0 && logDY == 8 && K >= 64)) {
        if (exchange_attached && cluster_size_1d(logDY, S, N, K, cus) > 0) return kFused1dCluster;
        if (algo == 7) algo = 0;                                // not applicable here: by size, as for every other value
    }
    if (algo == 8 && built) return kFused1dWide;
    if (algo == 8) algo = 0;
    if (algo == 0 && logDY == 7 && K >= 16 && N % 128 == 0 && items > cus && items <= 2 * cus) return kFused1dWide;
    // not quite one block per CU
    if (algo == 0 && items <= cus) {
        if (logDY == 7 && 4 * items >= 3 * cus && ((K > 48 && K <= 64) || (N % 128 != 0 && K >= 32 && K <= 40))) return kFused1dMfma256;
        if (logDY == 8 && K <= 16 && (K <= 8 ? 16 * items > 13 * cus : 4 * items > 3 * cus)) return kFused1dMfma256;
        if (logDY == 10 && 4 * items > 3 * cus && K <= 8) return kFused1dSimt;
    }
    // lengths 512 / 1024, more than one block per CU
    if (algo == 0 && long_signal && built && items > cus) {
        if (N % 128 == 0 && K >= (logDY == 9 ? 32 : 64)) return kFused1dWide;
        const long rounds = (items + 2 * cus - 1) / (2 * cus);
        const bool simt_fits_better = logDY == 10 && K < 64 && rounds > 1 && (2 * items <= 3 * rounds * cus || (N > 64 && items > 5 * cus));
        if (N % 128 != 0 && K >= (logDY == 9 ? 40 : 32) && !simt_fits_better) return kFused1dMfma256;
        const long blocks = N % 128 == 0 ? S * (N / 128) : 0;
        if (logDY == 10 && 4 * blocks >= 3 * cus && blocks <= cus) return kFused1dWide;
    }
    int pick = algo == 4 ? 2 : algo;
    if (pick == 0) pick = (built && items <= cus) ? 2 : (long_signal ? 1 : 3);
    const long split_blocks = S * (N / SPLIT_NT);
    if (logDY == 8 && (algo == 6 || (algo == 0 && K > 96 && 2 * split_blocks > cus && split_blocks <= cus))) return kFused1dSplitK;
    if (pick == 2 && (logDY == 7 || logDY == 8) && (algo == 4 || (algo == 0 && S * (N / 32) <= cus))) return kFused1dMfma512Tile32;
    if (pick == 2 && built) return kFused1dMfma512;
    if (pick == 3 && built) return kFused1dMfma256;
    return kFused1dSimt;
}

// Split kernel (layer1d_split.hip), N a multiple of 128: blocks of 128 output channels transform every input once per 128 outputs, blocks of 64 twice as
// often (the second time from L2), but they are finer and four fit a CU instead of three. 128 pays where the repeated transforms or reads
// are many (us, 64 / 128): DY = 256, S = 8192, K = 128: 1180 / 960; S = 4096, K = 40: 336 / 296, K = 32: 218 / 222; S = 1000, K = 96: 94 / 89,
// K = 64: 77 / 78; S = 333, K = 128: 46.6 / 50.9; just above three blocks of 64 per CU, which are two rounds of them (S = 400: K = 32: 31.8 / 28.4,
// K = 128: 58.5 / 50.7; S = 448: 30.2 / 29.9, 59.8 / 54.1). DY = 128, S = 8192, K = 128: 654 / 569; S = 3000, K = 64: 138 / 123, K = 32: 92 / 101; S = 1000,
// K = 96: 66 / 62, K = 40: 41.4 / 46.1; and where 128 fills one round of the CUs that 64 would need two for (S = 700, K = 64: 37.9 / 32.9).
// DY = 512, S = 2048, K = 128: 502 / 451; S = 1000, K = 64: 153 / 165. DY = 1024 (two blocks per CU either way): S = 512, K = 64: 173 / 163;
// S = 256, K = 32: 84 / 73, S = 512, K = 32: 134 / 140.
static bool wide_tiles(int logDY, long S, int N, int K, int algo, long cus)
{
    const long blocks = S * (N / 128), volume = (long)K * S / cus;       // forward transforms per CU
    if (N % 128 != 0) return false;
    if (algo == 8) return true;
    switch (logDY) {
    case 7: return (K >= 96 && blocks >= 2 * cus) || volume >= 625 || (K >= 40 && blocks > 2 * cus && blocks <= 3 * cus);
    case 8: return (volume >= 256 && (K >= 64 || volume >= 625)) || (K >= 16 && 2 * blocks > 3 * cus && 4 * blocks <= 7 * cus);
    case 9: return (K >= 96 && blocks >= 2 * cus) || (K >= 40 && volume >= 312);
    default: return K >= 64 ? blocks >= cus : blocks <= cus;
    }
}
// Output channels per block of the small-grid kernel: the fewest that leave every block a CU to itself. The blocks of a signal set
// repeat each other's forward transforms, but side by side, and each has fewer backward transforms to do one after the other (us,
// 16 / 32 / 64 channels, N = 64: S = 1, K = 32: DY = 128 5.3 / 5.9 / 7.0, DY = 1024 13.8 / 18.0 / 23.5; S = 64, K = 8: DY = 256 6.1 /
// 6.6 for 16 / 32, DY = 512 8.3 / 8.6 / 12.4; but with more blocks than CUs, S = 100, DY = 256, K = 24: 12.9 / 8.5 / 9.4).
static int small_tile(long S, int N, long cus)
{
    if (S * (N / 16) <= cus) return 16;
    return S * (N / 32) <= cus ? 32 : 64;
}
int tile_of_fused_1d_kernel(int kernel, int logDY, long S, int N, int K, int algo, long cus)
{
    switch (kernel) {
    case kFused1dMfma512: return algo == 2 ? 64 : small_tile(S, N, cus);
    case kFused1dMfma512Tile32: return algo == 4 ? 32 : small_tile(S, N, cus);
    case kFused1dSplitK: return SPLIT_NT;
    case kFused1dCluster: return N;
    case kFused1dWide: return wide_tiles(logDY, S, N, K, algo, cus) ? 128 : 64;
    default: return 64;
    }
}
// Blocks of 64 output channels at DY = 256: registers and LDS for four per CU once there are more than three (S = 1000, K = N = 64:
// 49.9 / 46.2 us); with two per CU the larger register budget is ahead (S = 512, K = 96: 37.4 / 39.3).
static bool dense_blocks(long S, int N, long cus) { return S * (N / 64) > 3 * cus; }

static bool overlap(const float2* a, long na, const float2* b, long nb) { return a < b + nb && b < a + na; }

hipError_t launch_fused_fft_cgemm_ifft(int logDY, long S, int N, int K, const float2* x, const float2* W, float2* y,
                                       float2 alpha, int algo, hipStream_t stream, bool y_is_reread)
{
    // y_is_reread (Y stage of the three-kernel 2D pipeline): the block kernels and the SIMT kernel then leave y in the
    // caches instead of streaming it past them; the clustered kernel ignores it
    const int keep_y = y_is_reread ? 1 : 0;
    const long cus = cu_count();
    // y in the place of x with 64 output channels: one block per signal set, which reads its rows of x before it writes them. (With more the
    // blocks of a signal set would race; the members of a cluster may read x again after others have written.)
    const bool in_place = N == 64 && overlap(x, (long)K * S << logDY, y, (long)N * S << logDY);
    int kernel = pick_fused_1d_kernel(logDY, S, N, K, algo, cus, !in_place && exchange_attached(stream));
    if (kernel == kFused1dCluster) {
        const hipError_t e = launch_fused_cluster(S, N, K, cluster_size_1d(logDY, S, N, K, cus), x, W, y, alpha, stream);
        if (e != hipErrorNotReady) return e;
        kernel = pick_fused_1d_kernel(logDY, S, N, K, algo, cus, false);    // detached in between
    }
    if (in_place && kernel == kFused1dSplitK) kernel = kFused1dMfma512;
    switch (kernel) {
    case kFused1dDense:
        if (logDY == 7 && K <= 8) return launch_fused_wave(S, N, K, x, W, y, alpha, stream, keep_y);
        return launch_fused_split(logDY, S, N, K, x, W, y, alpha, false, true, stream, keep_y);
    case kFused1dWide:
        return launch_fused_split(logDY, S, N, K, x, W, y, alpha, wide_tiles(logDY, S, N, K, algo, cus), dense_blocks(S, N, cus), stream, keep_y);
    case kFused1dSplitK:
        return keep_y ? launch_fused_split_channels<true>(S, N, K, x, W, y, alpha, stream) : launch_fused_split_channels<false>(S, N, K, x, W, y, alpha, stream);
    case kFused1dMfma512Tile32:
    case kFused1dMfma512: {
        const int tile = in_place ? 64 : tile_of_fused_1d_kernel(kernel, logDY, S, N, K, algo, cus);
        return launch_fused_small(logDY, S, N, K, x, W, y, alpha, tile, stream, keep_y);
    }
    case kFused1dMfma256:
        return launch_fused_split(logDY, S, N, K, x, W, y, alpha, false, logDY <= 8 && dense_blocks(S, N, cus), stream, keep_y);
    default: return dispatch_fused_1d(logDY, S, N, K, x, W, y, alpha, stream, keep_y);
    }
}

// The halves of the layer. While every block of 64 output channels has a CU to itself: the small-grid kernel (us, split kernel /
// small-grid kernel with 16, 32, 64 output channels per block).
//   First half: DY = 256, N = 64, K = 128: S = 1 20.3 / 11.3, 12.5, 15.1, S = 64 21.5 / 12.9, 13.5, 16.0; DY = 1024, K = 128, S = 64 65.8 /
//     39.4, 36.7, 37.8: blocks of 16 from 32 channels on and up to half of the CUs. Not with 49 to 64 channels of length 128 in
//     blocks of 64, whose rounds hold 48 (S = 200: K = 48 8.8 / 7.6, K = 56 9.5 / 9.8, K = 64 9.8 / 9.9, K = 72 11.8 / 10.5; with one
//     block on every CU only for multiples of 128: S = 128, N = 128, K = 56 9.8 / 10.1).
//   Second half (small_second_half): DY = 256, K = 32, S = 1 8.4 / 4.5, 5.3, 7.1; DY = 1024, K = 8: S = 1 19.4 / 6.2, 9.6, 15.8, S = 64
//     21.1 / 9.2, 11.1, 17.3. Length 128, and 256 with N a multiple of 128, up to one block per CU; else up to seven eighths (a block
//     of 64 on every CU: DY = 256, N = 64, K = 8 8.7 / 9.1; DY = 512 14.8 / 15.4; DY = 1024 26.8 / 28.1). Few channels: up to three
//     quarters with more than 64 outputs (DY = 256, K = 16, N = 256: S = 50 level, S = 54 8.8 / 9.1; DY = 512, K = 8, N = 192, against the
//     SIMT kernel: S = 62 0.98, S = 70 12.8 / 13.4), 13 of 16 at DY = 512 with 64; DY = 1024 with more than 128 outputs: 13 of 16 (N =
//     256, K = 48: S = 52 0.98, S = 56 27.3 / 28.8).
// Larger grids: the SIMT kernel with eight channels at lengths 512 / 1024, where a round of 16 would be half padding (split / SIMT:
// second half, DY = 512, S = 1000 58.5 / 54.8; first half with blocks of 64, DY = 1024, N = 64: S = 2048 49.4 / 46.4, S = 700 20.2 / 21.7);
// otherwise the split kernel (1232 shapes against the SIMT kernel: 0.66 of its time).
hipError_t launch_fused_fft_cgemm(int logDY, long S, int N, int K, const float2* x, const float2* W, float2* C,
                                  float2 alpha, float2 beta, hipStream_t stream)
{
    const long cus = cu_count(), items = S * (N / 64);
    const bool short_round = logDY == 7 && K > 48 && K <= 64 && 2 * items > cus && (items < cus || N % 128 == 0);
    if (items <= cus && !short_round) {
        // C over x (one signal, 64 output channels): one block, which reads before it writes
        const bool shared = overlap(x, (long)K * S << logDY, C, 64L * S * N);
        const int tile = shared ? 64 : K >= 32 && 2 * S * (N / 16) <= cus ? 16 : (S * (N / 32) <= cus ? 32 : 64);
        return launch_small_forward(logDY, S, N, K, x, W, C, alpha, beta, tile, stream);
    }
    // blocks of 128 output channels from one and a half per CU (N = 128, K = 64, DY = 256: S = 700 42.6 -> 34.4 us, S = 256 19.0 -> 19.9)
    const bool wide = N % 128 == 0 && 2 * S * (N / 128) >= 3 * cus;
    if (K <= 8 && !wide) {
        if (logDY == 9) return launch_fused_1d_k<9, true, false, false>(S, N, K, x, W, C, alpha, beta, stream);
        if (logDY == 10 && N % 128 != 0 && items > 3 * cus && items <= 8 * cus)
            return launch_fused_1d_k<10, true, false, false>(S, N, K, x, W, C, alpha, beta, stream);
    }
    return launch_split_forward(logDY, S, N, K, x, W, C, alpha, beta, wide, stream);
}

static bool small_second_half(int logDY, long items, int N, int K, long cus)
{
    if (items > cus || logDY == 7) return items <= cus;
    if (N > 64 && ((logDY == 8 && K <= 16) || (logDY == 9 && K <= 8))) return 4 * items <= 3 * cus;
    if (logDY == 8 && N % 128 == 0) return true;
    if ((logDY == 10 && N > 128) || (logDY == 9 && K <= 8)) return 16 * items <= 13 * cus;
    return 8 * items <= 7 * cus;
}
hipError_t launch_fused_cgemm_ifft(int logDY, long S, int N, int K, const float2* A, const float2* W, float2* y,
                                   float2 alpha, hipStream_t stream)
{
    const float2 beta = make_float2(0.f, 0.f);
    const long cus = cu_count(), items = S * (N / 64);
    if (small_second_half(logDY, items, N, K, cus)) {
        const bool shared = overlap(A, 64L * S * K, y, (long)N * S << logDY);   // y over A, likewise
        const int tile = shared ? 64 : S * (N / 16) <= cus ? 16 : (S * (N / 32) <= cus ? 32 : 64);
        return launch_small_backward(logDY, S, N, K, A, W, y, alpha, tile, stream);
    }
    if (K <= 8 && (logDY == 9 || (logDY == 10 && items > cus)))
        return logDY == 9 ? launch_fused_1d_k<9, false, true, false>(S, N, K, A, W, y, alpha, beta, stream)
                          : launch_fused_1d_k<10, false, true, false>(S, N, K, A, W, y, alpha, beta, stream);
    return launch_split_backward(logDY, S, N, K, A, W, y, alpha, stream);
}

template <int LOGDY, bool INVERSE>
static hipError_t launch_stride_DY_t(const float2* in, float2* out, long nsig, hipStream_t stream)
{
    using G = Geo1D<LOGDY>;
    const long blocks = (nsig + G::GROUPS - 1) / G::GROUPS;
    if (blocks <= 0 || blocks > 0x7fffffffL) return hipErrorInvalidValue;
    hipLaunchKernelGGL((stride_DY_kernel<LOGDY, INVERSE>), dim3((unsigned)blocks), dim3(256),
                       sizeof(float2) * G::GROUPS * G::EXCH, stream, in, out, nsig);
    return hipGetLastError();
}

hipError_t launch_fft_stride_DY(int logDY, const float2* in, float2* out, long nsig, hipStream_t stream)
{
    switch (logDY) {
    case 7: return launch_stride_DY_t<7, false>(in, out, nsig, stream);
    case 8: return launch_stride_DY_t<8, false>(in, out, nsig, stream);
    case 9: return launch_stride_DY_t<9, false>(in, out, nsig, stream);
    case 10: return launch_stride_DY_t<10, false>(in, out, nsig, stream);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_ifft_stride_DY(int logDY, const float2* in, float2* out, long nsig, hipStream_t stream)
{
    switch (logDY) {
    case 7: return launch_stride_DY_t<7, true>(in, out, nsig, stream);
    case 8: return launch_stride_DY_t<8, true>(in, out, nsig, stream);
    case 9: return launch_stride_DY_t<9, true>(in, out, nsig, stream);
    case 10: return launch_stride_DY_t<10, true>(in, out, nsig, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace tfno
