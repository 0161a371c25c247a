// How the mode GEMM (layer2d.hip) walks its contraction: channels per run over the tile of weights, whole or half steps, and
// its persistent blocks. Plain arithmetic on the sizes, so that it can be checked without a GPU.
#pragma once

namespace tfno {

constexpr int GEMM_KSTEP = 32;

struct GemmWalk {
    int run;          // channels covered by one run over the tile
    bool halves;      // steps in halves of 16 channels, an empty second half skipped
};

// K: all channels; Kw: period of the weights; nt: tiles of 16 output channels per block; threads per block; cap: steps that the tile
// can hold. One run covers one period of the weights where that wastes no part of a step, or else all K channels, if the tile can
// hold them. Half steps where the last step of a run holds at most 16 channels (us, whole steps / halves: M = 163,840, N = 128: K =
// 40 52.4 / 47.4, K = 104 102.2 / 98.3, K = 176 153.8 / 146.7; two parts of 24, M = 65,536, N = 128 25.1 / 22.7), and not where it is
// full or nearly so (M = 163,840, N = 128, K = 64 56.5 / 58.1; four parts of 40, M = 4,096, N = 64 8.0 / 8.7). Longest run that gains:
//   48 channels with tiles of 16 or 32 outputs, which have more per column to rearrange (M = 4,096, N = 64: two parts of 56 7.1 / 7.3);
//   128 with 64 outputs in blocks of 512 threads (M = 65,536, N = 64: K = 112 25.9 / 25.7, K = 136 29.8 / 30.6);
//   else whatever the tile holds (beyond that: M = 163,840, N = 128, K = 200 192.5 / 194.9).
inline GemmWalk gemm_walk(int K, int Kw, int nt, int threads, int cap)
{
    const bool periods = Kw % GEMM_KSTEP == 0 || (K + GEMM_KSTEP - 1) / GEMM_KSTEP > cap;
    const int run = periods ? Kw : K, last = run % GEMM_KSTEP;
    const int longest = nt < 4 ? 48 : (nt == 4 && threads == 512 ? 128 : GEMM_KSTEP * cap);
    return { run, last > 0 && last <= GEMM_KSTEP / 2 && run <= longest };
}

// Persistent blocks per tile of outputs, of `most` that the CUs hold: whole groups of eight, every XCD the same share. With up to 16
// channels not where the blocks left out make two rounds of one (us, whole groups / this: K = 16: N = 192, M = 21,120 11.6 / 9.4, N =
// 320, M = 12,800 11.8 / 9.6; 14 numbers of columns with N = 192 ... 576, beta or not: 0.83 of the time on average). With K = 24 and 32
// and beta the two rounds are ahead (N = 192, M = 20,608, K = 24 15.3 / 18.4).
inline long gemm_persistent_blocks(long nblocks, long most, int K)
{
    const long groups = most >= 8 ? most - most % 8 : (most > 0 ? most : 1);
    return nblocks <= (K <= 16 ? most : groups) ? nblocks : groups;
}

}  // namespace tfno
