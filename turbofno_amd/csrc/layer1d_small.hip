// Fused 1D spectral layer for small grids (at most about one block per CU), and its halves: one 512-thread block per (signal set, NT
// output channels), NT = 16, 32 or 64, contraction on the bf16 matrix cores with exact three-way splits of both operands (bf16_split.h).
//
// Same operands and result as fused_fft_cgemm_ifft_{7,8} of the reference
// (fusion_variants/1D_D_exp_fused_fft_cgemm_ifft/fused_fft_cgemm_ifft_7.cuh:9-222: (S, N/64) blocks that each traverse K).
// What bounds it is the chain of latencies and instructions of one block, not memory: few blocks run, each with a CU to itself. So
//   * the output channels of a signal set are spread over as many blocks as there are CUs for (NT = 16, 32, 64), although each of
//     them repeats the forward transforms: 2 or 4 backward transforms in a row per lane group become one;
//   * the weights (32 to 128 channels at a time) are split and laid out in LDS once, while x is on its way: done per round they
//     cost every wave 76 vector instructions next to the 380 of a transform;
//   * a round (one transform per lane group) has one barrier: spectra go to one of two LDS tiles in operand order, every wave
//     multiplies its m tile with its tiles of output channels, and the accumulators of all rounds meet in LDS once before the
//     backward transforms. Two signals of 128 samples per group fill a tile of 48 or 64 channels, of which the LDS holds one: with
//     a forward transform at DY = 128 a round has two barriers.
// Rounds are bound by instruction issue, two waves per SIMD (vector ALUs 56 % busy; two rounds of x in flight: 3 - 10 % slower).
// Measured, N = 64 (us, a kernel with fp32 matrix instructions, three barriers per round, 32 or 64 output channels / this): S = 1,
// K = 8, DY = 128 5.6 / 5.0; S = 1, K = 64: DY = 128 8.8 / 6.4, DY = 256 10.9 / 8.6, DY = 512 23.0 / 13.2, DY = 1024 38.1 / 21.8; S = 256,
// K = 64, DY = 512 32.7 / 27.2. Halves: first, S = 1, DY = 256, K = 128 20.3 / 11.3; second, S = 1, DY = 1024, K = 8 19.4 / 6.2.
// Error against 64 bits as for the split kernel (layer1d_split.hip), over the whole range of floats: operands that the split does not hold are
// noticed as they are split or in the accumulators, and small_product_fp32() stands in.
#include "bf16_split.h"
#include "group_fft.h"
#include "kernels.h"

namespace tfno {

// FWD: the spectra are made by forward transforms of x; otherwise they are read from A[m + k M] (second half of the layer).
// INV: the product goes into zero-padded backward transforms; otherwise it is stored as C[m + n M] (+ beta C, first half).
template <int LOGDY, int NT, bool FWD> struct GeoSmall {
    static constexpr int THREADS = 512, WAVES = THREADS / 64;
    static constexpr int L = LOGDY <= 8 ? 16 : (1 << LOGDY) / 16;   // lanes per signal (DY = 128: per pair of signals)
    static constexpr bool PAIR = LOGDY == 7;                    // two signals of length 128 per 16-lane group
    // channels per pass: one per lane group (two of 128 samples; three quarters of the groups where 64 channels of both operands exceed the LDS)
    static constexpr int CP = !FWD ? 32 : (PAIR ? (NT == 64 ? 48 : 64) : THREADS / L);
    static constexpr int KC = CP > 16 ? CP : 16;                // channels per round
    static constexpr int STEPS = KC / 16;                       // matrix steps per round
    static constexpr int TILES = NT / 16;                       // tiles of 16 output channels
    // the waves: four m tiles x two groups, which share the tiles of output channels or (NT = 16) take every second step
    static constexpr int TPW = TILES >= 2 ? TILES / 2 : 1, SLICES = TILES >= 2 ? 1 : 2;
    static constexpr int EXCH = L * 17;
    static constexpr int STEP_BYTES = 12 * 1024, WSTEP_BYTES = TILES * 3 * 1024;    // spectra / weights of 16 channels
    static constexpr int BUFFERS = STEPS <= 2 ? 2 : 1;          // tiles of spectra: with two a round needs one barrier
    // steps that the tile of weights holds: one entry per thread (two where a round has more)
    static constexpr int WSTEPS = 8 / TILES > STEPS ? 8 / TILES : STEPS, WKC = 16 * WSTEPS;
    static constexpr int TILE_AT = THREADS * 17 * (int)sizeof(float2);
    static constexpr int WTILE_AT = TILE_AT + BUFFERS * STEPS * STEP_BYTES;
    static constexpr int PP = 68;                               // pitch (complex) of the product: rows 4 apart half the banks apart
    static constexpr int PRODUCT_BYTES = SLICES * NT * PP * (int)sizeof(float2);    // shares the operand tiles
    static constexpr int TW_AT = WTILE_AT + WSTEPS * WSTEP_BYTES;   // first-pass twiddles, then the powers w_L^e
    static_assert(PRODUCT_BYTES <= TW_AT - TILE_AT && WKC % KC == 0, "the product takes the place of the operand tiles");
    static constexpr int LOW_AT = TW_AT + (int)sizeof(float2) * (L * kTwLdsPitch + (L > 16 ? L : 0));   // a flag per wave
    static constexpr int LDS_BYTES = LOW_AT + WAVES * (int)sizeof(unsigned);
    static_assert(LDS_BYTES <= 160 * 1024, "LDS of a CU");
};

// The share of the product of one wave in fp32, for operands that the split does not hold: the wave transforms the channels by itself, as
// many at a time as it has lane groups for, and takes its m tile from them four channels at a time. `region`: the exchange regions of
// the wave, free of other use.
template <int LOGDY, int NT, bool FWD>
TFNO_DEV void small_product_fp32(long S, int K, long s, int n0, int mt, int tile0, int slice, const float2* __restrict__ x,
                                 const float2* __restrict__ W, float2 alpha, const cpx* twrow, const cpx* powers, cpx* region,
                                 float4_v (&re)[GeoSmall<LOGDY, NT, FWD>::TPW], float4_v (&im)[GeoSmall<LOGDY, NT, FWD>::TPW])
{
    using G = GeoSmall<LOGDY, NT, FWD>;
    constexpr int DY = 1 << LOGDY, L = G::L, CHANNELS = !FWD ? 4 : (G::PAIR ? 8 : 64 / L);
    const int lane = threadIdx.x & 63, group = lane / L, t = lane % L, kq = lane >> 4, col = lane & 15;
    cpx* exch = region + group * G::EXCH;
#pragma unroll
    for (int i = 0; i < G::TPW; ++i) re[i] = im[i] = float4_v{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll 1
    for (int k = 0; k < K; k += CHANNELS) {
        if (G::SLICES == 2 && ((k >> 4) & 1) != slice) continue;
        cpx own = make_float2(0.f, 0.f);
        if constexpr (!FWD) own = x[(k + kq) * (64 * S) + s * 64 + 16 * mt + col];
        else {
            const float2* p = x + ((long)(k + (G::PAIR ? 2 : 1) * group) * S + s) * DY + t;
            cpx v[16], gg[16];
            if constexpr (G::PAIR) {
                cpx out[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) { v[i] = p[16 * i]; v[8 + i] = p[S * DY + 16 * i]; }
                pair128_first_pass(v, twrow, gg);
                rows128_forward_finish(gg, exch, t, out);
                wave_lds_fence();
#pragma unroll
                for (int a = 0; a < 8; ++a) exch[(t >> 3) * 64 + (t & 7) + 8 * a] = out[a];
            } else {
                cpx out[64 / L];
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i] = p[L * i];
                fwd_pass1_lds(v, twrow, gg);
                if constexpr (L > 16) wide_forward_finish<L, true, true>(gg, exch, powers, t, out);
                else group_forward_finish<8>(gg, exch, t, out);
                wave_lds_fence();
#pragma unroll
                for (int a = 0; a < 64 / L; ++a) exch[t + L * a] = out[a];
            }
            wave_lds_fence();
        }
#pragma unroll
        for (int c0 = 0; c0 < CHANNELS; c0 += 4) {
            const int c = c0 + kq;                              // lanes without a channel multiply zeros
            const bool live = CHANNELS >= 4 || c < CHANNELS;
            if constexpr (FWD) {
                const cpx* modes = region + (G::PAIR ? (c >> 1) * G::EXCH + (c & 1) * 64 : (live ? c : 0) * G::EXCH) + 16 * mt + col;
                own = live ? *modes : make_float2(0.f, 0.f);
            }
#pragma unroll
            for (int i = 0; i < G::TPW; ++i) {
                const float2 wk = live ? cmul(W[k + c + (long)(n0 + 16 * (tile0 + i) + col) * K], alpha) : make_float2(0.f, 0.f);
                mac_fp32(wk, own, re[i], im[i]);
            }
        }
        wave_lds_fence();
    }
}

template <int LOGDY, int NT, bool KEEP, bool FWD, bool INV>
__global__ __launch_bounds__(512, 1) void fused_fft_small_ifft_kernel(int S, int N, int K, const float2* __restrict__ x,
                                                                      const float2* __restrict__ W, float2* __restrict__ y, float2 alpha,
                                                                      float2 beta)
{
    using G = GeoSmall<LOGDY, NT, FWD>;
    constexpr bool PAIR = G::PAIR, LONG = LOGDY >= 9;
    constexpr int DY = 1 << LOGDY, L = G::L, CP = G::CP, KC = G::KC, STEPS = G::STEPS, TPW = G::TPW, THREADS = G::THREADS;
    extern __shared__ char lds_small[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int grp = tid / L, t = tid % L;                       // transform role: lane t of L-lane group grp
    const int kq = lane >> 4, col = lane & 15;                  // matrix role
    const int mt = wave & 3, half = wave >> 2;
    const int tile0 = G::SLICES == 1 ? half * TPW : 0;          // first of the wave's TPW tiles of 16 output channels
    long s;
    int ntile;
    decode_block_1d(S, N / NT, DY, !KEEP, s, ntile);
    const int n0 = ntile * NT;
    const long M = 64L * S;
    float2* exch = reinterpret_cast<float2*>(lds_small) + grp * G::EXCH;
    char* tiles = lds_small + G::TILE_AT;
    float2* twtab = reinterpret_cast<float2*>(lds_small + G::TW_AT);
    float2* powers = twtab + L * kTwLdsPitch;
    unsigned* low_flags = reinterpret_cast<unsigned*>(lds_small + G::LOW_AT);
    fill_lds_twiddles<LOGDY, L>(twtab, tid, THREADS);
    if (LONG && tid < L) powers[tid] = kTwiddle1024[tid * (1024 / L)];
    const float2* twrow = twtab + t * kTwLdsPitch;

    // Weights of WKC channels, 16 bytes of each part per entry (step, tile, lane (kq, col) of the operand read): four channels of one
    // output channel, as (re, im) pairs. Requested before the x of the same round, because loads return in order; those of the first
    // channels are split while x is on its way.
    constexpr int ENTRIES = G::WSTEPS * G::TILES * 64, EPT = (ENTRIES + THREADS - 1) / THREADS;
    float2 wv[EPT][4];
    auto load_w = [&](int kc) {
#pragma unroll
        for (int u = 0; u < EPT; ++u) {
            const int e = tid + u * THREADS, l = e & 63, tile = (e >> 6) % G::TILES, st = (e >> 6) / G::TILES;
            const int k = kc + 16 * st + 4 * (l >> 4);
            const bool live = (ENTRIES % THREADS == 0 || e < ENTRIES) && k < K;
            const float2* p = live ? W + k + (long)(n0 + 16 * tile + (l & 15)) * K : W;
#pragma unroll
            for (int j = 0; j < 4; ++j) wv[u][j] = live ? p[j] : make_float2(0.f, 0.f);
        }
    };
    char* wtile = lds_small + G::WTILE_AT;
    bool low = false;                                           // values too small for the split among the wave's spectra and weights
    auto build_w = [&](int kc) {
#pragma unroll
        for (int u = 0; u < EPT; ++u) {
            const int e = tid + u * THREADS;
            if (kc + 16 * ((wave + u * G::WAVES) / G::TILES) >= K || (ENTRIES % THREADS != 0 && e >= ENTRIES)) break;    // uniform
            unsigned bits = ~0u;                                // (zeros are common here: channels beyond K)
            uint4_v h, m, lo;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float2 w = cmul(wv[u][j], alpha);
                bits = lower(bits, w);
                unsigned a, b, c;
                split_bf16_pair(w.x, w.y, a, b, c);
                h[j] = a; m[j] = b; lo[j] = c;
            }
            low |= any_lane(bits < kSplitLow);
            uint4_v* dst = reinterpret_cast<uint4_v*>(wtile + (e >> 6) * 3072) + (e & 63);
            dst[0] = h; dst[64] = m; dst[128] = lo;
        }
    };
    // x of the pass that starts at channel kc (second half of the layer: 16 lanes per channel, four modes each)
    const int first = !FWD ? tid >> 4 : (PAIR ? 2 * grp : grp); // channel of a pass that the group brings in (PAIR: the first of two)
    const float2* src = FWD ? x + ((long)first * S + s) * DY + t : x + (long)first * M + s * 64 + (tid & 15);
    constexpr int HELD = FWD ? 16 : 4;
    cpx v[HELD];
    auto issue = [&](int kc) {
        if (first >= CP || kc + first >= K) return;             // uniform over the wave
        const float2* p = src + (long)kc * (FWD ? (long)S * DY : M);
        if constexpr (PAIR && FWD) {
#pragma unroll
            for (int i = 0; i < 8; ++i) { v[i] = p[16 * i]; v[8 + i] = p[(long)S * DY + 16 * i]; }
        } else {
#pragma unroll
            for (int i = 0; i < HELD; ++i) v[i] = p[(FWD ? L : 16) * i];
        }
    };
    load_w(0);
    issue(0);

    float4_v re[TPW], im[TPW];
#pragma unroll
    for (int i = 0; i < TPW; ++i) re[i] = im[i] = float4_v{ 0.f, 0.f, 0.f, 0.f };
    // where the lane's modes go: channel c of the round, mode 16 a + column, in operand order
    auto place = [&](char* tile, int c, int a, int column) {
        return tile + (c >> 4) * G::STEP_BYTES + a * 3072 + ((c >> 2) & 3) * 256 + column * 16 + (c & 3) * 4;
    };
    __syncthreads();                                            // twiddles
    cpx tw[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) tw[r] = twrow[r];

    int buffer = 0;
    for (int kc = 0; kc < K; kc += KC) {
        char* tile = tiles + buffer * (STEPS * G::STEP_BYTES);
        const int kn = (K - kc) < KC ? (K - kc) : KC;           // a multiple of 8 (caller contract)
        const bool new_weights = kc % G::WKC == 0;
        if (kc > 0 && (G::BUFFERS == 1 || new_weights)) __syncthreads();    // the operands that are about to be replaced are read
        if (new_weights) {
            build_w(kc);
            if (kc + G::WKC < K) load_w(kc + G::WKC);
        }
#pragma unroll
        for (int pass = 0; pass < KC / CP; ++pass) {
            constexpr int MODES = !FWD ? 4 : (PAIR ? 8 : 64 / L);
            cpx out[MODES];
            const bool takes_part = first < CP;                 // uniform over the wave, as is the next
            if (takes_part && pass * CP + first < kn) {
                if constexpr (!FWD) {
#pragma unroll
                    for (int a = 0; a < 4; ++a) out[a] = v[a];
                    issue(kc + (pass + 1) * CP);
                } else if constexpr (PAIR) {
                    cpx gg[16];
                    pair128_first_pass(v, twrow, gg);
                    issue(kc + (pass + 1) * CP);
                    rows128_forward_finish(gg, exch, t, out);
                } else {
                    cpx gg[16];
                    fwd_pass1(v, tw, gg);
                    issue(kc + (pass + 1) * CP);
                    if constexpr (LONG) wide_forward_finish<L, true, true>(gg, exch, powers, t, out);
                    else group_forward_finish<8>(gg, exch, t, out);
                }
                low |= below_split_range(out);
            } else {                                            // channels beyond K
#pragma unroll
                for (int a = 0; a < MODES; ++a) out[a] = make_float2(0.f, 0.f);
            }
            if (!takes_part) continue;
#pragma unroll
            for (int a = 0; a < MODES; ++a) {
                unsigned h, m, l;
                split_bf16_pair(out[a].x, out[a].y, h, m, l);
                char* dst;
                if constexpr (!FWD) dst = place(tile, tid >> 4, a, tid & 15);
                else if constexpr (PAIR) dst = place(tile, 2 * grp + (t >> 3), a >> 1, (t & 7) + 8 * (a & 1));
                else dst = place(tile, pass * CP + grp, (t >> 4) + (L / 16) * a, t & 15);
                *reinterpret_cast<unsigned*>(dst) = h;
                *reinterpret_cast<unsigned*>(dst + 1024) = m;
                *reinterpret_cast<unsigned*>(dst + 2048) = l;
            }
        }
        if (kc + KC >= K && lane == 0) low_flags[wave] = low;
        __syncthreads();
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
            if (16 * st >= kn) break;                           // uniform
            if (G::SLICES == 2 && (((kc >> 4) + st) & 1) != half) continue;
            const uint4_v* frag = reinterpret_cast<const uint4_v*>(tile + st * G::STEP_BYTES + mt * 3072) + lane;
            const SplitOperand b{ frag[0], frag[64], frag[128] };
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
                const uint4_v* wf = reinterpret_cast<const uint4_v*>(wtile + (((kc % G::WKC) / 16 + st) * G::TILES + tile0 + i) * 3072) + lane;
                const SplitOperand w{ wf[0], wf[64], wf[128] };
                SplitOperand wre, wim;                          // rows (re, -im) and (im, re) of alpha W
                wre.h = w.h ^ 0x80000000u; wre.m = w.m ^ 0x80000000u; wre.l = w.l ^ 0x80000000u;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    wim.h[j] = __builtin_amdgcn_alignbit(w.h[j], w.h[j], 16);
                    wim.m[j] = __builtin_amdgcn_alignbit(w.m[j], w.m[j], 16);
                    wim.l[j] = __builtin_amdgcn_alignbit(w.l[j], w.l[j], 16);
                }
                mac_split_pair(wre, wim, b, re[i], im[i]);
            }
        }
        if (G::BUFFERS == 2) buffer ^= 1;
    }

    float high[2] = { 0.f, 0.f };
#pragma unroll
    for (int i = 0; i < TPW; ++i) { high[0] = larger(high[0], re[i]); high[1] = larger(high[1], im[i]); }
    if (__builtin_expect(any_lane((low_flags[lane & 7] != 0) | not_finite(high[0], high[1])), 0))
        small_product_fp32<LOGDY, NT, FWD>(S, K, s, n0, mt, tile0, half, x, W, alpha, twrow, powers,
                                           reinterpret_cast<float2*>(lds_small) + wave * (64 * 17), re, im);

    // D[row = 4 kq + q][col] of tile i: output channel n0 + 16 (tile0 + i) + 4 kq + q, mode 16 mt + col
    if constexpr (!INV && G::SLICES == 1) {
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            float2* dst = y + (long)(n0 + 16 * (tile0 + i) + 4 * kq) * M + s * 64 + 16 * mt + col;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                cpx r = make_float2(re[i][q], im[i][q]);
                if (beta.x != 0.f || beta.y != 0.f) r = cadd(r, cmul(dst[q * M], beta));
                dst[q * M] = r;
            }
        }
        return;
    }
    __syncthreads();                                            // every wave has read the operand tiles: the product takes their place
    float2* product = reinterpret_cast<float2*>(tiles);
#pragma unroll
    for (int i = 0; i < TPW; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            product[((G::SLICES == 2 ? half * NT : 16 * (tile0 + i)) + 4 * kq + q) * G::PP + 16 * mt + col] = make_float2(re[i][q], im[i][q]);
    __syncthreads();
    auto mode_of = [&](int n, int m) {
        const cpx a = product[n * G::PP + m];
        return G::SLICES == 2 ? cadd(a, product[(NT + n) * G::PP + m]) : a;
    };
    if constexpr (!INV) {
#pragma unroll
        for (int u = 0; u < NT * 64 / THREADS; ++u) {
            const int n = (tid >> 6) + u * G::WAVES;
            float2* dst = y + (long)(n0 + n) * M + s * 64 + lane;
            cpx r = mode_of(n, lane);
            if (beta.x != 0.f || beta.y != 0.f) r = cadd(r, cmul(*dst, beta));
            *dst = r;
        }
    } else if constexpr (PAIR) {
#pragma unroll 1
        for (int n = 2 * grp; n < NT; n += 2 * (THREADS / 16)) {
            cpx c8[8], yv[16];
#pragma unroll
            for (int a = 0; a < 8; ++a) c8[a] = mode_of(n + (t >> 3), (t & 7) + 8 * a);
            rows128_backward(c8, twrow, exch, t, yv);
            store_pair16<KEEP>(y + ((long)(n0 + n) * S + s) * DY + t, (long)S * DY, yv);
        }
    } else {
#pragma unroll 1
        for (int n = grp; n < NT; n += THREADS / L) {
            cpx c[64 / L], yv[16];
#pragma unroll
            for (int a = 0; a < 64 / L; ++a) c[a] = mode_of(n, t + L * a);
            if constexpr (LONG) {
                cpx e[16];
                wide_backward_inputs<L, true>(c, powers, exch, t, e);
                // twiddles from registers, for up to eight transforms in a row (DY = 1024, K = 8, N = 64, S = 129: 19.0 us with those
                // in LDS, 16.8; DY = 512, S = 144: 12.4 / 11.1; second half, K = 32, S = 130: DY = 1024 18.6 / 16.0, DY = 512 12.3 / 11.0)
                inv_pass2(e, tw, yv);
            } else {
                group_backward_lds<8>(c, twrow, exch, t, yv);
            }
            store_row16<L, KEEP>(y + ((long)(n0 + n) * S + s) * DY + t, yv);
        }
    }
}

template <int LOGDY, int NT, bool KEEP, bool FWD, bool INV>
static hipError_t launch_small_k(long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, float2 beta, hipStream_t stream)
{
    using G = GeoSmall<LOGDY, NT, FWD>;
    const long blocks = S * (N / NT);
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    static std::atomic<unsigned long long> served;
    if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(fused_fft_small_ifft_kernel<LOGDY, NT, KEEP, FWD, INV>), G::LDS_BYTES, served);
        e != hipSuccess)
        return e;
    hipLaunchKernelGGL((fused_fft_small_ifft_kernel<LOGDY, NT, KEEP, FWD, INV>), dim3((unsigned)blocks), dim3(G::THREADS), G::LDS_BYTES, stream,
                       (int)S, N, K, x, W, y, alpha, beta);
    return hipGetLastError();
}
template <int LOGDY, bool KEEP, bool FWD, bool INV>
static hipError_t launch_small_t(long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, float2 beta, int nt, hipStream_t stream)
{
    switch (nt) {
    case 16: return launch_small_k<LOGDY, 16, KEEP, FWD, INV>(S, N, K, x, W, y, alpha, beta, stream);
    case 32: return launch_small_k<LOGDY, 32, KEEP, FWD, INV>(S, N, K, x, W, y, alpha, beta, stream);
    case 64: return launch_small_k<LOGDY, 64, KEEP, FWD, INV>(S, N, K, x, W, y, alpha, beta, stream);
    default: return hipErrorInvalidValue;
    }
}
template <bool KEEP, bool FWD, bool INV>
static hipError_t launch_small(int logDY, long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, float2 beta, int nt, hipStream_t stream)
{
    switch (logDY) {
    case 7: return launch_small_t<7, KEEP, FWD, INV>(S, N, K, x, W, y, alpha, beta, nt, stream);
    case 8: return launch_small_t<8, KEEP, FWD, INV>(S, N, K, x, W, y, alpha, beta, nt, stream);
    case 9: return launch_small_t<9, KEEP, FWD, INV>(S, N, K, x, W, y, alpha, beta, nt, stream);
    case 10: return launch_small_t<10, KEEP, FWD, INV>(S, N, K, x, W, y, alpha, beta, nt, stream);
    default: return hipErrorInvalidValue;
    }
}

// nt: output channels per block (16, 32 or 64)
hipError_t launch_fused_small(int logDY, long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, int nt, hipStream_t stream, int keep_y)
{
    const float2 beta = make_float2(0.f, 0.f);
    return keep_y ? launch_small<true, true, true>(logDY, S, N, K, x, W, y, alpha, beta, nt, stream)
                  : launch_small<false, true, true>(logDY, S, N, K, x, W, y, alpha, beta, nt, stream);
}
hipError_t launch_small_forward(int logDY, long S, int N, int K, const float2* x, const float2* W, float2* C, float2 alpha, float2 beta, int nt, hipStream_t stream)
{
    return launch_small<true, true, false>(logDY, S, N, K, x, W, C, alpha, beta, nt, stream);
}
hipError_t launch_small_backward(int logDY, long S, int N, int K, const float2* A, const float2* W, float2* y, float2 alpha, int nt, hipStream_t stream)
{
    return launch_small<false, false, true>(logDY, S, N, K, A, W, y, alpha, make_float2(0.f, 0.f), nt, stream);
}

}  // namespace tfno
