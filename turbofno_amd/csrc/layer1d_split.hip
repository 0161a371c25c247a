// Fused 1D spectral layer for grids of about one block per CU and more, DY = 128 and 256: one 256-thread block per
// (signal set, 64 NTW output channels), NTW = 1 or 2, contraction on the bf16 matrix cores with exact three-way splits of both
// operands (bf16_split.h).
//
// Same operands and result as fused_fft_cgemm_ifft_{7,8} of the reference
// (fusion_variants/1D_D_exp_fused_fft_cgemm_ifft/fused_fft_cgemm_ifft_7.cuh:9-222: (S, N/64) blocks that each traverse K).
// Per round of 16 channels (32 for DY = 128, two per group): forward transforms by the sixteen 16-lane groups; every lane splits
// its modes and writes them to LDS in operand order, a complex mode being one (re, im) pair of the contraction index, so that one
// matrix instruction covers 16 channels. Wave w owns 16 NTW output channels and all 64 modes:
//   * an element of W is used by one wave only and goes from global memory through its registers into the A operand, as the rows
//     (re, -im) and (im, re); nothing of W passes through LDS;
//   * the accumulators of a lane are, for each of four output channels, the modes t + 16 a: the input of the backward transform by
//     its own 16-lane group (DY = 128: after one row rotation). The product never leaves the registers and the backward phase
//     has no barrier.
// What bounds it: the chain of phases of a wave (x, transform, product, backward, stores), hidden by blocks in other phases, up to
// the rate of a mixed read and write stream (4.5 - 4.8 TB/s here; a copy of 2 GiB: 4.9). Hence the registers are held to three blocks per CU (NTW = 2: 158;
// NTW = 1: 144) or four (NTW = 1: 116 - 124, the operand tile sharing the exchange regions, x requested after the second pass)
// without spills: with spills the kernel is up to 70 % slower, because a reload waits for the x in flight.
// Measured against the fp32 kernels it replaced (us, x and y from HBM): DY = 256, K = N = 128, S = 8192: 1135 -> 960;
// K = N = 64, S = 4096: 247 -> 213; DY = 128, K = N = 64, S = 16384: 533 -> 447; K = N = 128, S = 8192: 735 -> 569; K = 40, N = 128,
// S = 1000: 52 -> 46. Error against 64 bits: 2.4e-7 -> 2.0e-7 (K = 64), 3.2e-7 -> 2.7e-7 (K = 128).
#include "bf16_split.h"
#include "group_fft.h"
#include "kernels.h"

namespace tfno {

// NTW = tiles of 16 output channels per wave (a block covers 64 NTW output channels).
// ALIAS: the operand tile of the spectra shares the exchange regions (one more barrier per round, LDS for four blocks per CU).
// BLOCKS: blocks per CU that the registers are held to.
template <int LOGDY, int NTW, bool ALIAS> struct GeoSplit {
    static constexpr bool PAIR = LOGDY == 7;
    static constexpr int KC = PAIR ? 32 : 16;                   // channels per round: a 16-lane group transforms one, or two of length 128
    static constexpr int EXCH = 16 * 17;
    static constexpr int EXCH_BYTES = 16 * EXCH * (int)sizeof(float2);
    static constexpr int STEP_BYTES = 12 * 1024;                // operand tile of 16 channels: 4 m tiles x 3 parts x 1 KiB
    static constexpr int TILE_BYTES = (KC / 16) * STEP_BYTES;
    static constexpr int TILE_AT = ALIAS ? 0 : EXCH_BYTES;
    static constexpr int TW_AT = ALIAS ? EXCH_BYTES : EXCH_BYTES + TILE_BYTES;
    static constexpr size_t LDS_BYTES = TW_AT + sizeof(float2) * kTwLdsSize;
    static_assert(!ALIAS || TILE_BYTES <= EXCH_BYTES, "the operand tile must fit the exchange regions");
};

// Makes `offset` depend on g[]: loads that are addressed with it cannot be issued before g[] has been computed. The compiler
// otherwise moves loads from read-only arrays and the twiddle reads up to the start of the transform, where their
// registers (up to 78) come on top of those of the pass.
template <int COUNT> TFNO_DEV void after(int& offset, const cpx (&g)[COUNT])
{
    static_assert(COUNT % 4 == 0, "in fours");
#pragma unroll
    for (int i = 0; i < COUNT; i += 4) asm volatile("" : "+v"(offset) : "v"(g[i].x), "v"(g[i + 1].x), "v"(g[i + 2].x), "v"(g[i + 3].x));
}

template <int LOGDY, int NTW, bool ALIAS, int BLOCKS, bool KEEP>
__global__ __launch_bounds__(256, BLOCKS) void fused_fft_split_ifft_kernel(int S, int N, int K, const float2* __restrict__ x,
                                                                             const float2* __restrict__ W, float2* __restrict__ y,
                                                                             float2 alpha)
{
    using G = GeoSplit<LOGDY, NTW, ALIAS>;
    constexpr bool PAIR = G::PAIR;
    constexpr int DY = 1 << LOGDY, KC = G::KC;
    // x of the next round is requested after the second pass instead of before it: 32 registers fewer at the peak
    constexpr bool LATE = NTW > 1 || BLOCKS == 4;
    extern __shared__ char lds_split[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int grp = tid >> 4, t = tid & 15;                     // transform role: lane t of 16-lane group grp
    const int kq = lane >> 4, col = lane & 15;                  // matrix role
    long s;
    int ntile;
    decode_block_1d(S, N / (64 * NTW), DY, !KEEP, s, ntile);
    const int nw = (ntile * 4 + wave) * (16 * NTW);             // first output channel of the wave
    float2* exch = reinterpret_cast<float2*>(lds_split) + grp * G::EXCH;
    char* tile = lds_split + G::TILE_AT;
    float2* twtab = reinterpret_cast<float2*>(lds_split + G::TW_AT);
    fill_lds_twiddles<LOGDY>(twtab, tid, 256);
    const float2* twrow = twtab + t * kTwLdsPitch;

    const int first = PAIR ? 2 * grp : grp;                     // channel of a round that the group transforms (first of two)
    const float2* src = x + ((long)first * S + s) * DY + t;
    // x of the round that starts at channel kc. Branch free (a load under a condition would keep the old values alive and
    // cost 30 registers): channels beyond K read the first row(s) of the array, cache resident, and are masked later
    cpx v[16];
    auto issue = [&](int kc, int offset) {
        const float2* p = (kc + first < K ? src + (long)kc * S * DY : x + t) + offset;
        if constexpr (PAIR) {
#pragma unroll
            for (int i = 0; i < 8; ++i) { v[i] = p[16 * i]; v[8 + i] = p[(long)S * DY + 16 * i]; }
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = p[16 * i];
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
    const int c_own = PAIR ? 2 * grp + (t >> 3) : grp, col_own = PAIR ? t & 7 : t;
    char* own = tile + (c_own >> 4) * G::STEP_BYTES + ((c_own >> 2) & 3) * 256 + col_own * 16 + (c_own & 3) * 4;

    for (int kc = 0; kc < K; kc += KC) {
        const int kn = (K - kc) < KC ? (K - kc) : KC;           // a multiple of 8 (caller contract)
        const bool busy = (PAIR ? 8 : 4) * wave < kn;           // uniform over the wave
        constexpr int MODES = PAIR ? 8 : 4, WSTEPS = PAIR && NTW == 1 && BLOCKS < 4 ? 2 : 1;
        // W rows of the round: lane (kq, col) holds channels 4 kq ... 4 kq + 3 of 16, output channel col of the tile (a short
        // last round reads its first channels again: the spectra of the missing ones are zero). Requested before the next
        // round's x: loads return in order, so a later request would wait for all of x first
        float2 wv[WSTEPS][NTW][4];
        auto load_w = [&](int step, float2 (&dst)[NTW][4], int offset) {
            const int k = 16 * step + 4 * kq;
            const float2* p = W + (kc + (k < kn ? k : 0)) + (long)(nw + col) * K + offset;
#pragma unroll
            for (int i = 0; i < NTW; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) dst[i][j] = p[(long)(16 * i) * K + j];
        };
        cpx out[MODES];
        if (busy) {
            cpx gg[16];
            if constexpr (PAIR) {
                cpx a8[8], b8[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) { a8[i] = v[i]; b8[i] = v[8 + i]; }
                fft8<-1>(a8);
                fft8<-1>(b8);
                gg[0] = a8[0];
                gg[8] = b8[0];
#pragma unroll
                for (int r = 1; r < 8; ++r) {
                    const cpx w = twrow[r];
                    gg[r] = cmul(a8[r], w);
                    gg[8 + r] = cmul(b8[r], w);
                }
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
#pragma unroll
            for (int u = 0; u < WSTEPS; ++u) load_w(u, wv[u], later);
            if constexpr (!LATE) issue(kc + KC, later);
            if constexpr (PAIR) rows128_forward_finish(gg, exch, t, out);
            else group_forward_finish<8>(gg, exch, t, out);
            if constexpr (LATE) {
                later = 0;
                after(later, out);
                issue(kc + KC, later);
            }
        } else {                                                // the wave's channels are beyond K
#pragma unroll
            for (int u = 0; u < WSTEPS; ++u) load_w(u, wv[u], 0);
            issue(kc + KC, 0);
#pragma unroll
            for (int a = 0; a < MODES; ++a) out[a] = make_float2(0.f, 0.f);
        }
        __syncthreads();                                        // the operand tile of the last round is read / the exchanges are done
#pragma unroll
        for (int a = 0; a < MODES; ++a) {
            unsigned h, m, l;
            split_bf16_pair(out[a].x, out[a].y, h, m, l);
            char* dst = own + (PAIR ? (a >> 1) * 3072 + (a & 1) * 128 : a * 3072);
            *reinterpret_cast<unsigned*>(dst) = h;
            *reinterpret_cast<unsigned*>(dst + 1024) = m;
            *reinterpret_cast<unsigned*>(dst + 2048) = l;
        }
        __syncthreads();
#pragma unroll
        for (int step = 0; step < KC / 16; ++step) {
            if (16 * step >= kn) break;                         // uniform
            const uint4_v* frag = reinterpret_cast<const uint4_v*>(tile + step * G::STEP_BYTES) + lane;
#pragma unroll
            for (int i = 0; i < NTW; ++i) {
                if constexpr (LATE) __builtin_amdgcn_sched_barrier(0);
                SplitOperand wre, wim;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float2 w = wv[WSTEPS == 2 ? step : 0][i][j];
                    unsigned h, m, l;
                    split_bf16_pair(w.x * alpha.x - w.y * alpha.y, w.x * alpha.y + w.y * alpha.x, h, m, l);
                    wre.h[j] = h ^ 0x80000000u; wre.m[j] = m ^ 0x80000000u; wre.l[j] = l ^ 0x80000000u;    // (re, -im)
                    wim.h[j] = __builtin_amdgcn_alignbit(h, h, 16);                                        // (im, re)
                    wim.m[j] = __builtin_amdgcn_alignbit(m, m, 16);
                    wim.l[j] = __builtin_amdgcn_alignbit(l, l, 16);
                }
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

    // D[row = 4 kq + q][col] of tile (i, a): output channel nw + 16 i + 4 kq + q, mode col + 16 a
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
        float2* dst = y + ((long)(nw + 16 * i + 4 * kq) * S + s) * DY + t;
        if constexpr (!PAIR) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                cpx c[4], yv[16];
#pragma unroll
                for (int a = 0; a < 4; ++a) c[a] = make_float2(re[i][a][q], im[i][a][q]);
                group_backward_lds<8>(c, twrow, exch, t, yv);
                store_row16<16, KEEP>(dst + (long)q * S * DY, yv);
            }
        } else {
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

template <int LOGDY, int NTW, bool ALIAS, int BLOCKS>
static hipError_t launch_split_t(long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, hipStream_t stream, int keep_y)
{
    using G = GeoSplit<LOGDY, NTW, ALIAS>;
    const long blocks = S * (N / (64 * NTW));
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    static_assert(G::LDS_BYTES <= 64 * 1024, "no attribute call needed below 64 KiB of dynamic LDS");
    // keep_y: plain instead of streaming stores of y, for a consumer that reads it at once (a template parameter of the kernels)
    if (keep_y)
        hipLaunchKernelGGL((fused_fft_split_ifft_kernel<LOGDY, NTW, ALIAS, BLOCKS, true>), dim3((unsigned)blocks), dim3(256), G::LDS_BYTES,
                           stream, (int)S, N, K, x, W, y, alpha);
    else
        hipLaunchKernelGGL((fused_fft_split_ifft_kernel<LOGDY, NTW, ALIAS, BLOCKS, false>), dim3((unsigned)blocks), dim3(256), G::LDS_BYTES,
                           stream, (int)S, N, K, x, W, y, alpha);
    return hipGetLastError();
}

// DY = 128 or 256. wide: blocks of 128 output channels where N allows, else of 64; dense: the variant for four blocks per CU
// (64 output channels; always at DY = 128, where it is level or ahead from one block per CU on).
hipError_t launch_fused_split(int logDY, long S, int N, int K, const float2* x, const float2* W, float2* y, float2 alpha, bool wide,
                              bool dense, hipStream_t stream, int keep_y)
{
    wide = wide && N % 128 == 0;
    if (logDY == 7)
        return wide ? launch_split_t<7, 2, true, 3>(S, N, K, x, W, y, alpha, stream, keep_y)
                    : launch_split_t<7, 1, true, 4>(S, N, K, x, W, y, alpha, stream, keep_y);
    if (logDY != 8) return hipErrorInvalidValue;
    if (wide) return launch_split_t<8, 2, false, 3>(S, N, K, x, W, y, alpha, stream, keep_y);
    return dense ? launch_split_t<8, 1, true, 4>(S, N, K, x, W, y, alpha, stream, keep_y)
                 : launch_split_t<8, 1, false, 3>(S, N, K, x, W, y, alpha, stream, keep_y);
}

}  // namespace tfno
