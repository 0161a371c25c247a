// Fused 1D spectral layer for grids of about one block per CU and more, and its halves: one 256-thread block per
// (signal set, 64 NTW output channels), NTW = 1 or 2, contraction on the bf16 matrix cores with exact three-way splits of both
// operands (bf16_split.h).
//
// Same operands and result as fused_fft_cgemm_ifft_{7,8} of the reference
// (fusion_variants/1D_D_exp_fused_fft_cgemm_ifft/fused_fft_cgemm_ifft_7.cuh:9-222: (S, N/64) blocks that each traverse K).
// Per round of 16 channels (32 for DY = 128, two per group): forward transforms by the sixteen 16-lane groups (DY = 512 / 1024: in two / four
// passes by eight / four groups of 32 / 64 lanes); every lane splits
// its modes and writes them to LDS in operand order, a complex mode being one (re, im) pair of the contraction index, so that one
// matrix instruction covers 16 channels. Wave w owns 16 NTW output channels and all 64 modes:
//   * an element of W is used by one wave only and goes from global memory through its registers into the A operand, as the rows
//     (re, -im) and (im, re); nothing of W passes through LDS;
//   * the accumulators of a lane are, for each of four output channels, the modes t + 16 a: the input of the backward transform by
//     its own 16-lane group (DY = 128: after one row rotation; DY = 512 / 1024: through the exchange region of the group, inside
//     the wave). The product never passes a block barrier, nor does the backward phase.
// What bounds it: the chain of phases of a wave (x, transform, product, backward, stores), hidden by blocks in other phases, up to
// the rate of a mixed read and write stream (4.5 - 4.8 TB/s here; a copy of 2 GiB: 4.9). Hence, at lengths 128 / 256, the registers are
// held to three blocks per CU (NTW = 2: 158 - 166; NTW = 1: 135) or four (NTW = 1: 123 - 126, the operand tile sharing the exchange
// regions, x requested after the second pass), at 512 to two or three and at 1024 to two (the halves: up to four),
// without spills: with spills the kernel is up to 70 % slower, because a reload waits for the x in flight.
// Measured against the fp32 kernels it replaced (us, x and y from HBM): DY = 256, K = N = 128, S = 8192: 1135 -> 960;
// K = N = 64, S = 4096: 247 -> 213; DY = 128, K = N = 64, S = 16384: 533 -> 447; K = N = 128, S = 8192: 735 -> 569; K = 40, N = 128,
// S = 1000: 52 -> 41; DY = 512, K = N = 128, S = 2048: 652 -> 451; DY = 1024, K = N = 128, S = 1000: 601 -> 462. Halves against the SIMT kernel:
// forward DY = 256, K = N = 64, S = 2048: 103 -> 77, K = N = 128: 341 -> 171; backward 112 -> 65, 298 -> 149; S = 64, K = N = 64: 22 -> 13 both; which
// shapes stay with the SIMT kernel: launch_fused_fft_cgemm, launch_fused_cgemm_ifft.
// Error against 64 bits: 2.4e-7 -> 2.0e-7 (K = 64), 3.2e-7 -> 2.7e-7 (K = 128), the same from the smallest normal floats to the
// largest: operands that the split does not hold (bf16_split.h) are noticed - small spectra and weights as they are split, the rest in
// the accumulators - and product_fp32() stands in. Noticing costs 0 - 2 % (the most: DY = 128, S = 4096, K = N = 128: 295 -> 301), up to 4 % of the halves on small grids.
#include "bf16_split.h"
#include "group_fft.h"
#include "kernels.h"

namespace tfno {

// NTW = tiles of 16 output channels per wave (a block covers 64 NTW output channels).
// ALIAS: the operand tile of the spectra shares the exchange regions (one more barrier per round, LDS for four blocks per CU).
// BLOCKS: blocks per CU that the registers are held to.
// FWD: the spectra are made by forward transforms of x; otherwise they are read from A[m + k M] (second half of the layer).
// INV: the product goes into zero-padded backward transforms; otherwise it is stored as C[m + n M] (+ beta C, first half).
template <int LOGDY, bool ALIAS, bool FWD> struct GeoSplit {
    static constexpr int L = LOGDY <= 8 ? 16 : (1 << LOGDY) / 16;   // lanes per signal (DY = 128: per pair of signals)
    static constexpr bool PAIR = LOGDY == 7 && FWD;             // two channels of length 128 per 16-lane group
    static constexpr int CP = !FWD ? 16 : (PAIR ? 32 : 256 / L);    // channels per pass of the block
    static constexpr int KC = CP > 16 ? CP : 16;                // channels per round
    static constexpr int EXCH = L * 17;
    static constexpr int EXCH_BYTES = 256 * 17 * (int)sizeof(float2);
    static constexpr int STEP_BYTES = 12 * 1024;                // operand tile of 16 channels: 4 m tiles x 3 parts x 1 KiB
    static constexpr int TILE_BYTES = (KC / 16) * STEP_BYTES;
    static constexpr int TILE_AT = ALIAS ? 0 : EXCH_BYTES;
    static constexpr int TW_AT = ALIAS ? EXCH_BYTES : EXCH_BYTES + TILE_BYTES;      // first-pass twiddles, then the powers w_L^e
    static constexpr int LOW_AT = TW_AT + (int)sizeof(float2) * (L * kTwLdsPitch + (L > 16 ? L : 0));   // a flag per wave
    static constexpr size_t LDS_BYTES = LOW_AT + 4 * sizeof(unsigned);
    static_assert(!ALIAS || (TILE_BYTES <= EXCH_BYTES && CP == KC), "the operand tile must fit the exchange regions, one pass per round");
};

// Makes `offset` depend on g[]: loads that are addressed with it cannot be issued before g[] has been computed. The compiler
// otherwise moves loads from read-only arrays and the twiddle reads up to the start of the transform, where their
// registers (up to 78) come on top of those of the pass.
template <int COUNT> TFNO_DEV void after(int& offset, const cpx (&g)[COUNT])
{
#pragma unroll
    for (int i = 0; i < COUNT; ++i) asm volatile("" : "+v"(offset) : "v"(g[i].x));
}

// The product of one wave in fp32, for operands that the split does not hold: the wave transforms all K channels by itself, as many at
// a time as it has lane groups for, and takes its 16 NTW output channels from them four channels at a time. Several times as slow as
// the loop that it stands in for. `region`: the exchange regions of the wave, free of other use.
template <int LOGDY, int NTW, bool FWD>
TFNO_DEV void product_fp32(long S, int K, long s, int nw, int nstep, const float2* __restrict__ x, const float2* __restrict__ W, float2 alpha,
                           const cpx* twrow, const cpx* powers, cpx* region, float4_v (&re)[NTW][4], float4_v (&im)[NTW][4])
{
    using G = GeoSplit<LOGDY, false, FWD>;
    constexpr int DY = 1 << LOGDY, L = G::L, CHANNELS = !FWD ? 4 : (G::PAIR ? 8 : 64 / L);
    const int lane = threadIdx.x & 63, group = lane / L, t = lane % L, kq = lane >> 4, col = lane & 15;
    cpx* exch = region + group * G::EXCH;
    const float2* w = W + (long)(nw + nstep * col) * K;
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
        for (int a = 0; a < 4; ++a) re[i][a] = im[i][a] = float4_v{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll 1
    for (int k = 0; k < K; k += CHANNELS) {
        cpx b[4];
        if constexpr (!FWD) {
            const float2* p = x + (k + kq) * (64 * S) + s * 64 + col;
#pragma unroll
            for (int a = 0; a < 4; ++a) b[a] = p[16 * a];
        } else {
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
                if constexpr (L > 16) wide_forward_finish<L, true, L == 64>(gg, exch, powers, t, out);
                else group_forward_finish<8>(gg, exch, t, out);
                wave_lds_fence();
#pragma unroll
                for (int a = 0; a < 64 / L; ++a) exch[t + L * a] = out[a];
            }
            wave_lds_fence();
        }
#pragma unroll
        for (int c0 = 0; c0 < CHANNELS; c0 += 4) {
            // lane (kq, col): channel c of the round, modes col + 16 a; lanes without a channel multiply zeros
            const int c = c0 + kq;
            const bool live = CHANNELS >= 4 || c < CHANNELS;
            if constexpr (FWD) {
                const cpx* modes = region + (G::PAIR ? (c >> 1) * G::EXCH + (c & 1) * 64 : (live ? c : 0) * G::EXCH) + col;
#pragma unroll
                for (int a = 0; a < 4; ++a) b[a] = live ? modes[16 * a] : make_float2(0.f, 0.f);
            }
#pragma unroll
            for (int i = 0; i < NTW; ++i) {
                const float2 wk = live ? cmul(w[k + c + (long)(16 * i * nstep) * K], alpha) : make_float2(0.f, 0.f);
#pragma unroll
                for (int a = 0; a < 4; ++a) mac_fp32(wk, b[a], re[i][a], im[i][a]);
            }
        }
    }
}

template <int LOGDY, int NTW, bool ALIAS, int BLOCKS, bool KEEP, bool FWD = true, bool INV = true>
__global__ __launch_bounds__(256, BLOCKS) void fused_fft_split_ifft_kernel(int S, int N, int K, const float2* __restrict__ x,
                                                                             const float2* __restrict__ W, float2* __restrict__ y,
                                                                             float2 alpha, float2 beta, int wave_step)
{
    using G = GeoSplit<LOGDY, ALIAS, FWD>;
    constexpr bool PAIR = G::PAIR, LONG = LOGDY >= 9;
    constexpr int DY = 1 << LOGDY, KC = G::KC, CP = G::CP, L = G::L;
    // x of the next pass is requested after the second stage instead of before it: 32 registers fewer at the peak
    constexpr bool LATE = NTW > 1 || BLOCKS == 4;
    extern __shared__ char lds_split[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int grp = tid / L, t = tid % L;                       // transform role: lane t of L-lane group grp
    const int kq = lane >> 4, col = lane & 15;                  // matrix role
    long s;
    int ntile;
    decode_block_1d(S, N / (64 * NTW), DY, !KEEP, s, ntile);
    // output channels of the wave: nw, nw + nstep, ... (16 NTW of them)
    const int nstep = INV && LOGDY >= 8 ? wave_step : 1;
    const int nw = ntile * 64 * NTW + wave * (nstep == 1 ? 16 * NTW : 1);
    const long M = 64L * S;
    float2* exch = reinterpret_cast<float2*>(lds_split) + grp * G::EXCH;
    char* tile = lds_split + G::TILE_AT;
    float2* twtab = reinterpret_cast<float2*>(lds_split + G::TW_AT);
    float2* powers = twtab + L * kTwLdsPitch;
    unsigned* low_flags = reinterpret_cast<unsigned*>(lds_split + G::LOW_AT);
    fill_lds_twiddles<LOGDY, L>(twtab, tid, 256);
    if (LONG && tid < L) powers[tid] = kTwiddle1024[tid * (1024 / L)];
    const float2* twrow = twtab + t * kTwLdsPitch;

    // channel of a pass that the group brings in (PAIR: the first of two; without a forward transform 16 lanes per channel)
    const int first = !FWD ? tid >> 4 : (PAIR ? 2 * grp : grp);
    const float2* src = FWD ? x + ((long)first * S + s) * DY + t : x + (long)first * M + s * 64 + (tid & 15);
    // input of the pass that starts at channel kc. Branch free (a load under a condition would keep the old values alive and
    // cost 30 registers): channels beyond K read the first row(s) of the array, cache resident, and are masked later
    constexpr int HELD = FWD ? 16 : 4;
    cpx v[HELD];
    auto issue = [&](int kc, int offset) {
        const float2* p = (kc + first < K ? src + (long)kc * (FWD ? (long)S * DY : M) : x + (FWD ? t : tid & 15)) + offset;
        if constexpr (PAIR) {
#pragma unroll
            for (int i = 0; i < 8; ++i) { v[i] = p[16 * i]; v[8 + i] = p[(long)S * DY + 16 * i]; }
        } else {
#pragma unroll
            for (int i = 0; i < HELD; ++i) v[i] = p[(FWD ? L : 16) * i];
        }
    };
    issue(0, 0);
    float4_v re[NTW][4], im[NTW][4];
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
        for (int a = 0; a < 4; ++a) re[i][a] = im[i][a] = float4_v{ 0.f, 0.f, 0.f, 0.f };
    __syncthreads();                                            // twiddles

    // where the lane's modes go: channel c of the round, mode 16 a + column, in operand order (16 bytes per lane of the
    // operand read: four channels of one column)
    auto own_place = [&](int c, int a, int column) {
        return tile + (c >> 4) * G::STEP_BYTES + a * 3072 + ((c >> 2) & 3) * 256 + column * 16 + (c & 3) * 4;
    };

    bool low = false, low_weights = false;                      // spectra / weights of the wave that are too small for the split
    for (int kc = 0; kc < K; kc += KC) {
        const int kn = (K - kc) < KC ? (K - kc) : KC;           // a multiple of 8 (caller contract)
        constexpr int MODES = !FWD ? 4 : (PAIR ? 8 : 64 / L), WSTEPS = PAIR && NTW == 1 && BLOCKS < 4 ? 2 : 1;
        // W rows of the round: lane (kq, col) holds channels 4 kq ... 4 kq + 3 of 16, output channel col of the tile (a short
        // last round reads its first channels again: the spectra of the missing ones are zero). Requested before the next
        // pass's x: loads return in order, so a later request would wait for all of x first
        float2 wv[WSTEPS][NTW][4];
        auto load_w = [&](int step, float2 (&dst)[NTW][4], int offset) {
            const int k = 16 * step + 4 * kq;
            const float2* p = W + (kc + (k < kn ? k : 0)) + (long)(nw + nstep * col) * K + offset;
#pragma unroll
            for (int i = 0; i < NTW; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) dst[i][j] = p[(long)(16 * i * nstep) * K + j];
        };
#pragma unroll
        for (int pass = 0; pass < KC / CP; ++pass) {
            const bool busy = pass * CP + (CP / 4) * wave < kn; // uniform over the wave: CP / 4 channels each
            cpx out[MODES];
            if constexpr (!FWD) {
#pragma unroll
                for (int a = 0; a < 4; ++a) out[a] = busy ? v[a] : make_float2(0.f, 0.f);
#pragma unroll
                for (int u = 0; u < WSTEPS; ++u) load_w(u, wv[u], 0);
                issue(kc + CP, 0);
            } else if (busy) {
                cpx gg[16];
                if constexpr (PAIR) {
                    pair128_first_pass(v, twrow, gg);
                } else {
                    fft16<-1>(v);
                    int row = 0;
                    after(row, v);
                    const float2* tw = twrow + row;
                    gg[0] = v[0];
                    gg[1] = cmul(v[fft16_slot(1)], tw[1]);
#pragma unroll
                    for (int r = 2; r < 16; r += 2) {
                        const float4 w = *reinterpret_cast<const float4*>(tw + r);
                        gg[r] = cmul(v[fft16_slot(r)], make_float2(w.x, w.y));
                        gg[r + 1] = cmul(v[fft16_slot(r + 1)], make_float2(w.z, w.w));
                    }
                }
                int later = 0;
                after(later, gg);
                if (pass == 0) {
#pragma unroll
                    for (int u = 0; u < WSTEPS; ++u) load_w(u, wv[u], later);
                }
                if constexpr (!LATE) issue(kc + (pass + 1) * CP, later);
                if constexpr (PAIR) rows128_forward_finish(gg, exch, t, out);
                else if constexpr (LONG) wide_forward_finish<L, true, L == 64>(gg, exch, powers, t, out);
                else group_forward_finish<8>(gg, exch, t, out);
                if constexpr (LATE) {
                    later = 0;
                    after(later, out);
                    issue(kc + (pass + 1) * CP, later);
                }
            } else {                                            // the wave's channels are beyond K
                if (pass == 0) {
#pragma unroll
                    for (int u = 0; u < WSTEPS; ++u) load_w(u, wv[u], 0);
                }
                issue(kc + (pass + 1) * CP, 0);
#pragma unroll
                for (int a = 0; a < MODES; ++a) out[a] = make_float2(0.f, 0.f);
            }
            if (busy) low |= below_split_range(out);
            if (pass == 0) __syncthreads();                     // the operand tile of the last round is read / the exchanges are done
#pragma unroll
            for (int a = 0; a < MODES; ++a) {
                unsigned h, m, l;
                split_bf16_pair(out[a].x, out[a].y, h, m, l);
                char* dst;
                if constexpr (PAIR) dst = own_place(2 * grp + (t >> 3), a >> 1, (t & 7) + 8 * (a & 1));
                else if constexpr (!FWD) dst = own_place(tid >> 4, a, tid & 15);
                else dst = own_place(pass * CP + grp, (t >> 4) + (L / 16) * a, t & 15);
                *reinterpret_cast<unsigned*>(dst) = h;
                *reinterpret_cast<unsigned*>(dst + 1024) = m;
                *reinterpret_cast<unsigned*>(dst + 2048) = l;
            }
        }
        if (kc + KC >= K && lane == 0) low_flags[wave] = low;
        __syncthreads();
#pragma unroll
        for (int step = 0; step < KC / 16; ++step) {
            if (16 * step >= kn) break;                         // uniform
            const uint4_v* frag = reinterpret_cast<const uint4_v*>(tile + step * G::STEP_BYTES) + lane;
#pragma unroll
            for (int i = 0; i < NTW; ++i) {
                if constexpr (LATE) __builtin_amdgcn_sched_barrier(0);
                SplitOperand wre, wim;                          // rows (re, -im) and (im, re) of alpha W
                float2 (&w4)[4] = wv[WSTEPS == 2 ? step : 0][i];
#pragma unroll
                for (int j = 0; j < 4; ++j) w4[j] = cmul(w4[j], alpha);
                unsigned bits = ~0u;
#pragma unroll
                for (int j = 0; j < 4; ++j) bits = lower(bits, w4[j]);
                low_weights |= any_lane(bits < kSplitLow);
#pragma unroll
                for (int j = 0; j < 4; ++j) split_weight_rows(w4[j], wre, wim, j);
                if (WSTEPS == 1 && PAIR && step == 0 && 16 < kn && i == NTW - 1) load_w(1, wv[0], 0);
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    if constexpr (LATE) __builtin_amdgcn_sched_barrier(0);
                    const SplitOperand b{ frag[a * 192], frag[a * 192 + 64], frag[a * 192 + 128] };
                    mac_split_pair(wre, wim, b, re[i][a], im[i][a]);
                }
            }
        }
        if constexpr (ALIAS) __syncthreads();                   // the operand tile is read: exchange regions again
    }

    float high[2] = { 0.f, 0.f };
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
        for (int a = 0; a < 4; ++a) { high[0] = larger(high[0], re[i][a]); high[1] = larger(high[1], im[i][a]); }
    if (__builtin_expect(low_weights | any_lane((low_flags[lane & 3] != 0) | not_finite(high[0], high[1])), 0))
        product_fp32<LOGDY, NTW, FWD>(S, K, s, nw, nstep, x, W, alpha, twrow, powers, reinterpret_cast<float2*>(lds_split) + wave * (64 * 17), re, im);

    // D[row = 4 kq + q][col] of tile (i, a): output channel nw + nstep (16 i + 4 kq + q), mode col + 16 a
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
        if constexpr (!INV) {
            float2* dst = y + (long)(nw + 16 * i + 4 * kq) * M + s * 64 + col;
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    cpx r = make_float2(re[i][a][q], im[i][a][q]);
                    if (beta.x != 0.f || beta.y != 0.f) r = cadd(r, cmul(dst[q * M + 16 * a], beta));
                    dst[q * M + 16 * a] = r;
                }
        } else if constexpr (LONG) {
            // one output channel per L-lane group: the lanes that hold it store its 64 modes into the group's region
            constexpr int AT_ONCE = 64 / L;                     // channels per wave at a time
            float2* first_row = y + ((long)(nw + nstep * 4 * (lane / L)) * S + s) * DY + t;
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll 1
                for (int h = 0; h < 4 / AT_ONCE; ++h) {         // a loop: unrolled, the backward phase exceeds the instruction cache
                    wave_lds_fence();
                    if (kq / AT_ONCE == h) {
                        float2* dst = reinterpret_cast<float2*>(lds_split) + (wave * AT_ONCE + kq % AT_ONCE) * G::EXCH + col;
#pragma unroll
                        for (int a = 0; a < 4; ++a) dst[16 * a] = make_float2(re[i][a][q], im[i][a][q]);
                    }
                    cpx e[16], yv[16];
                    wide_backward_inputs_of_stored<L, true>(powers, exch, t, e);
                    inv_pass2_lds(e, twrow, yv);
                    store_row16<L, KEEP>(first_row + (long)(nstep * (16 * i + 4 * AT_ONCE * h + q)) * S * DY, yv);
                }
        } else if constexpr (LOGDY == 8) {
            float2* dst = y + ((long)(nw + nstep * (16 * i + 4 * kq)) * S + s) * DY + t;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                cpx c[4], yv[16];
#pragma unroll
                for (int a = 0; a < 4; ++a) c[a] = make_float2(re[i][a][q], im[i][a][q]);
                group_backward_lds<8>(c, twrow, exch, t, yv);
                store_row16<16, KEEP>(dst + (long)(q * nstep) * S * DY, yv);
            }
        } else {
            float2* dst = y + ((long)(nw + 16 * i + 4 * kq) * S + s) * DY + t;
            const bool upper = t >> 3;
#pragma unroll
            for (int q = 0; q < 4; q += 2) {
                // lane t = r + 8 h finishes channel h of the pair: modes r + 8 c; even c come from lanes t < 8, odd c from t >= 8
                cpx c8[8], yv[16];
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const cpx c0 = make_float2(re[i][a][q], im[i][a][q]), c1 = make_float2(re[i][a][q + 1], im[i][a][q + 1]);
                    const cpx got = rotate8(upper ? c0 : c1);
                    c8[2 * a] = upper ? got : c0;
                    c8[2 * a + 1] = upper ? c1 : got;
                }
                rows128_backward(c8, twrow, exch, t, yv);
                store_pair16<KEEP>(dst + (long)q * S * DY, (long)S * DY, yv);
            }
        }
    }
}

template <int LOGDY, int NTW, bool ALIAS, int BLOCKS, bool KEEP, bool FWD, bool INV>
static hipError_t launch_split_k(long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, float2 beta, hipStream_t stream)
{
    using G = GeoSplit<LOGDY, ALIAS, FWD>;
    const long blocks = S * (N / (64 * NTW));
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    // Channel strides of 1 or 2 MiB put all output channels of a signal set on the same memory channels: the four waves of a block then
    // take every fourth channel each, so that the rows that are stored at one time lie one stride apart and not 16 (DY = 512, S = 256,
    // N = 64, second half, K = 64: 23.5 -> 18.1 us, K = 8: 20.0 -> 15.2; whole layer DY = 256, S = 512, K = 64, N = 128: 44.9 -> 38.0).
    // At other strides neighbouring rows are better kept in one wave (S = 300: 3 % slower; 4 MiB, DY = 1024, S = 512: 5 - 13 %), and so
    // with 128 channels per block at DY = 512 (S = 512, K = N = 128: 101 / 112).
    const long stride = S * (8L << LOGDY);
    const bool step = (stride == (1L << 20) || stride == (2L << 20)) && !(LOGDY == 9 && NTW == 2);
    static_assert(G::LDS_BYTES <= 64 * 1024, "no attribute call needed below 64 KiB of dynamic LDS");
    hipLaunchKernelGGL((fused_fft_split_ifft_kernel<LOGDY, NTW, ALIAS, BLOCKS, KEEP, FWD, INV>), dim3((unsigned)blocks), dim3(256),
                       G::LDS_BYTES, stream, (int)S, N, K, x, W, y, alpha, beta, step ? 4 : 1);
    return hipGetLastError();
}
// keep_y: plain instead of streaming stores of y, for a consumer that reads it at once (a template parameter of the kernels)
template <int LOGDY, int NTW, bool ALIAS, int BLOCKS>
static hipError_t launch_split_t(long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, hipStream_t stream, int keep_y)
{
    const float2 beta = make_float2(0.f, 0.f);
    return keep_y ? launch_split_k<LOGDY, NTW, ALIAS, BLOCKS, true, true, true>(S, N, K, x, W, y, alpha, beta, stream)
                  : launch_split_k<LOGDY, NTW, ALIAS, BLOCKS, false, true, true>(S, N, K, x, W, y, alpha, beta, stream);
}

// wide: blocks of 128 output channels where N allows, else of 64; dense: the variant for four blocks per CU (64 output channels;
// DY = 256 only; always at DY = 128, where it is level or ahead from one block per CU on).
hipError_t launch_fused_split(int logDY, long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, bool wide,
                              bool dense, hipStream_t stream, int keep_y)
{
    wide = wide && N % 128 == 0;
    switch (logDY) {
    case 7:
        return wide ? launch_split_t<7, 2, true, 3>(S, N, K, x, W, y, alpha, stream, keep_y)
                    : launch_split_t<7, 1, true, 4>(S, N, K, x, W, y, alpha, stream, keep_y);
    case 8:
        if (wide) return launch_split_t<8, 2, false, 3>(S, N, K, x, W, y, alpha, stream, keep_y);
        return dense ? launch_split_t<8, 1, true, 4>(S, N, K, x, W, y, alpha, stream, keep_y)
                     : launch_split_t<8, 1, false, 3>(S, N, K, x, W, y, alpha, stream, keep_y);
    case 9:
        return wide ? launch_split_t<9, 2, false, 2>(S, N, K, x, W, y, alpha, stream, keep_y)
                    : launch_split_t<9, 1, false, 3>(S, N, K, x, W, y, alpha, stream, keep_y);
    case 10:
        return wide ? launch_split_t<10, 2, false, 2>(S, N, K, x, W, y, alpha, stream, keep_y)
                    : launch_split_t<10, 1, false, 2>(S, N, K, x, W, y, alpha, stream, keep_y);
    default: return hipErrorInvalidValue;
    }
}

// The halves of the layer (variants B and C): forward transforms and product, product and backward transforms.
hipError_t launch_split_forward(int logDY, long S, int N, int K, const float2* x, const float2* W, float2* C, float2 alpha, float2 beta,
                                bool wide, hipStream_t stream)
{
    wide = wide && N % 128 == 0;
    switch (logDY) {
    case 7:
        return wide ? launch_split_k<7, 2, true, 3, true, true, false>(S, N, K, x, W, C, alpha, beta, stream)
                    : launch_split_k<7, 1, true, 4, true, true, false>(S, N, K, x, W, C, alpha, beta, stream);
    case 8:
        return wide ? launch_split_k<8, 2, false, 3, true, true, false>(S, N, K, x, W, C, alpha, beta, stream)
                    : launch_split_k<8, 1, false, 3, true, true, false>(S, N, K, x, W, C, alpha, beta, stream);
    case 9:
        return wide ? launch_split_k<9, 2, false, 2, true, true, false>(S, N, K, x, W, C, alpha, beta, stream)
                    : launch_split_k<9, 1, false, 3, true, true, false>(S, N, K, x, W, C, alpha, beta, stream);
    case 10:
        return wide ? launch_split_k<10, 2, false, 2, true, true, false>(S, N, K, x, W, C, alpha, beta, stream)
                    : launch_split_k<10, 1, false, 2, true, true, false>(S, N, K, x, W, C, alpha, beta, stream);
    default: return hipErrorInvalidValue;
    }
}
hipError_t launch_split_backward(int logDY, long S, int N, int K, const float2* A, const float2* W, float2* y, float2 alpha, hipStream_t stream)
{
    const float2 beta = make_float2(0.f, 0.f);
    switch (logDY) {
    case 7: return launch_split_k<7, 1, true, 4, false, false, true>(S, N, K, A, W, y, alpha, beta, stream);
    case 8: return launch_split_k<8, 1, true, 4, false, false, true>(S, N, K, A, W, y, alpha, beta, stream);
    case 9: return launch_split_k<9, 1, true, 4, false, false, true>(S, N, K, A, W, y, alpha, beta, stream);
    case 10: return launch_split_k<10, 1, true, 3, false, false, true>(S, N, K, A, W, y, alpha, beta, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace tfno
