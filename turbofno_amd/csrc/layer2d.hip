// Whole-image 2D spectral layer (the MI355X-first path of the 2D layer): images of DX x DY with DX in {128, 256} rows
// per block - 512 and 1024 rows as two and four interleaved parts of 256 ("decimated images" below) - and rows of DY in
// {128, 256, 512, 1024}.
//
// The reference's "fully fused" 2D variant is three kernels with two HBM round trips of
// half-truncated intermediates (fusion_variants/2D_D_exp_fused_fft_cgemm_ifft/fused_trunc_2D.cu:150-172:
// X transform -> t1[K*bs][64][DY], fused Y stage, t2[N*bs][64][DY] -> X inverse). Here one 1024-thread
// block owns a whole DX x DY image, so only fully truncated 64 x 64 spectra ever leave the CU:
//
//   fft2d_trunc    image (k,b): DX row FFTs along Y (coalesced rows, 64 modes kept, held in registers),
//                  redistribution through LDS, 64 column FFTs along X (64 modes kept)
//                  -> spec[k][b][4096]                          reads 8 DX DY bytes, writes 32 KiB
//   cgemm_modes    C[n][b][m] = alpha * sum_k W[k][n] spec[k][b][m] on the matrix cores
//   ifft2d_pad     exact mirror -> y[n][b][DX][DY]              reads 32 KiB, writes 8 DX DY bytes
//
// so x is read once and y written once; padded / discarded modes are never touched in memory.
// The 4096 modes of an image are stored in "lane order": element mm*(64 LX) + q*LX + t holds mode
// (p = t + LX mm, q), LX = DX/16. That order is private to the two image kernels (producer and consumer
// lanes coincide, every access is contiguous per wavefront) and the GEMM is oblivious to it.
#include "bf16_split.h"
#include "group_fft.h"
#include "gemm_steps.h"
#include "kernels.h"
#include <string>
#include <type_traits>

namespace tfno {

namespace {
constexpr int EXCH_ELEMS = 1024 * 17;            // exchange regions of all lane groups of a 1024-thread block

// Geometry of the whole-image kernels for a DX x DY image (DX rows of DY contiguous samples).
// Rows of 256: a 16-lane group owns one row (16 samples per lane). Rows of 128 ("paired"): a 16-lane group owns
// two rows, 8 samples per lane each, so that a group still covers 128 contiguous bytes per access. Rows of 512 / 1024
// ("wide"): a group of 32 / 64 lanes owns one row, 16 samples per lane, 256 / 512 contiguous bytes per access.
template <int LOGX, int LOGY> struct Geo2D {
    static constexpr int DX = 1 << LOGX, DY = 1 << LOGY;
    static constexpr bool PAIRED = LOGY == 7;
    static constexpr bool WIDE = LOGY >= 9;                   // rows of 512 / 1024: 32 / 64 lanes per row
    static constexpr int LX = DX / 16, LY = WIDE ? DY / 16 : 16;   // lanes per column / per row-pass group
    static constexpr int GY = 1024 / LY;                      // lane groups of the row pass
    static constexpr int RPP = PAIRED ? 2 * GY : GY;          // rows per pass
    static constexpr int ITY = DX / RPP;                      // row passes per image
    static constexpr int MMY = PAIRED ? 8 : 64 / LY;          // modes per lane after one row pass
    static constexpr int MMX = 64 / LX;                       // modes per lane after the column pass
    static constexpr int COLT = 64 * LX;                      // threads that take part in the column pass
    static constexpr int TILE = DX * 68;                      // the largest pitch of TileMap
    static constexpr int LDS_MAIN = EXCH_ELEMS > TILE ? EXCH_ELEMS : TILE;   // exchange regions alias the tile
    // after them: first-pass twiddles of the rows (one table row per lane of a group) and of the columns, and for rows
    // of 512 / 1024 the powers w_LY^e, e < LY, of the second pass
    static constexpr int TWY_ELEMS = LY * kTwLdsPitch, WSM_ELEMS = WIDE ? LY : 0;
    static constexpr size_t LDS_BYTES = sizeof(float2) * (size_t)(LDS_MAIN + TWY_ELEMS + kTwLdsSize + WSM_ELEMS);
    static_assert(LOGY >= 7 && LOGY <= 10, "rows of 128 to 1024");
    static_assert(ITY >= 1 && COLT <= 1024 && GY * LY * 17 <= EXCH_ELEMS, "unsupported image shape");
    // element offset of the lane's i-th sample from its first one; pair: rows between the two of a paired group
    // (logr: the rows of the image lie 2^logr rows of the array apart, see the decimated images below)
    static __device__ __forceinline__ constexpr int sample_off(int i, int pair, int logr = 0)
    {
        return PAIRED ? (i & 7) * 16 + (i >> 3) * ((pair * DY) << logr) : LY * i;
    }
    // column of the redistribution tile (mode along Y) that lane t of a row group holds in slot mm
    static __device__ __forceinline__ constexpr int tile_col(int t, int mm) { return PAIRED ? (t & 7) + 8 * mm : t + LY * mm; }
};

// The redistribution tile [DX][64] and which rows the lane groups take, laid out for the LDS banks: an 8-byte read serves 32 lanes per cycle
// over 64 banks (element numbers modulo 32 differ), an 8-byte write 16 lanes over 32 banks (modulo 16).
//   forward: rows are written (16 lanes: 16 modes of a row, or 8 modes of each row of a pair, which have to lie 8 elements apart modulo 16) and
//     columns are read (32 lanes: LX rows of 2 or 4 columns): a pitch of 2 modulo 32 for 16 rows, of 4 modulo 32 for 8 rows;
//   backward: columns are written (16 lanes: LX rows of 1 or 2 columns): an odd pitch for 16 rows, 2 modulo 16 for 8; rows are read (32 lanes: two
//     groups, whose rows have to lie 16 elements apart modulo 32, and 8 for the rows of a pair).
// With one pitch of 66 for all cases the writes of the backward kernel of 256 rows and the reads of the forward kernel of 128 rows
// met the same banks two by two (us per layer, before / now: 16 images of 256 x 256, K = N = 64: 211.6 / 204.8; 40 of 128 x 128, K = 72:
// 194.2 / 189.9; 16 of 512 x 128: 237.9 / 233.1). Backward kernels of decimated images other than 512 x 128 keep 66 and its order of
// the rows, which lie 2 or 4 rows apart in memory there (8 images of 1024 x 256: 312 / 331 with 65).
//   PAIR:    rows of 128: group g owns the rows a and a + PAIR (lanes 0-7 / 8-15 finish one each), a enumerating the rows in question;
//   PARTNER: rows between the first rows of the groups 2j and 2j + 1. Rows of 512 / 1024: a group is at least half a wavefront: any order.
template <int LOGX, int LOGY, int LOGR, bool FORWARD> struct TileMap {
    static constexpr bool ODD = !FORWARD && LOGX == 8 && (LOGR == 0 || (LOGR == 1 && LOGY == 7));
    static constexpr int PITCH = ODD ? 65 : FORWARD && LOGX == 7 ? 68 : 66;
    static constexpr int PAIR = ODD ? 8 : FORWARD && LOGX == 7 ? 2 : 4;
    static constexpr int PARTNER = ODD ? 16 : 8;
    // first row (within one pass) of lane group g
    template <bool PAIRED, bool WIDE> static __device__ __forceinline__ int first_row(int g)
    {
        const int jh = g & 1, rest = g >> 1;
        if constexpr (WIDE) return g;
        else if constexpr (!PAIRED) return jh * PARTNER + rest % PARTNER + (rest / PARTNER) * (2 * PARTNER);
        else {
            const int s = jh * PAIR + rest % PAIR + (rest / PAIR) * (2 * PAIR);    // pair index
            return s % PAIR + (s / PAIR) * (2 * PAIR);
        }
    }
};

// Decimated images (LOGR > 0): an image of R DX x DY, R = 2^LOGR, too long along X for one block, is handled as R parts
// of DX x DY: part r holds the rows R j + r. Its transform along X splits exactly (one radix-R decimation in time step):
//     X[p] = sum_{r<R} w_{R DX}^(r p) * DFT_DX(part r)[p],    p < 64
// so the forward kernel transforms every part like an image of its own and multiplies its 64 x 64 modes by w^(r p); the
// sum over r is a sum over "channels" and is done by the contraction that follows (channel r K + k, weight W[k]): the
// spectrum of part r of image i is stored at index r * nfull + i for that, nfull whole images. Backward, the R parts of
// an output image are transformed from the one spectrum of the image, multiplied by conj(w^(r p)). Nothing but x, y and
// the 64 x 64 modes ever leaves a CU, as for images of one block.
//
// Numbering of the block-images (one per block iteration). Side by side: image * R + part, the parts of an image run on
// neighbouring blocks at the same time and all rows of the array are in flight together, not every R-th one; part major:
// part * nfull + image. Measured: the forward kernels are 2-9 % faster side by side everywhere; the backward kernels as
// well for four parts and for rows up to 256, but 3 % slower for two parts of rows of 512 / 1024, which keep part major.
template <int LOGR, bool PART_MAJOR> struct PartNumbering {
    static constexpr int R = 1 << LOGR;
    static __device__ __forceinline__ unsigned part(long img, int nfull)
    {
        if constexpr (LOGR == 0) return 0;
        else if constexpr (PART_MAJOR) return (unsigned)img / (unsigned)nfull;
        else return (unsigned)img & (R - 1);
    }
    static __device__ __forceinline__ long image(long img, int nfull)
    {
        if constexpr (LOGR == 0) return img;
        else if constexpr (PART_MAJOR) return (unsigned)img % (unsigned)nfull;
        else return img >> LOGR;
    }
};
// first row in the array of block-image img: row `part` of image `image`, whose rows lie R rows apart
template <int LOGX, int LOGR, bool PART_MAJOR> __device__ __forceinline__ long first_array_row(long img, int nfull)
{
    using P = PartNumbering<LOGR, PART_MAJOR>;
    return (P::image(img, nfull) << (LOGX + LOGR)) + P::part(img, nfull);
}
constexpr int kDecimationTwiddles = 64 * 4;      // complex elements: R <= 4 parts
template <int LOGD> __device__ __forceinline__ void fill_decimation_twiddles(float2* tab, int tid, int nthreads)
{
    for (int e = tid; e < kDecimationTwiddles; e += nthreads)
        tab[e] = kTwiddle1024[(((e >> 6) * (e & 63)) << (10 - LOGD)) & 1023];
}
}  // namespace

// Forward image kernel: truncated 2D transform of one DX x DY image per block iteration.
// 1024 threads = 16 waves per CU (4 per SIMD: the arithmetic is issue bound, so full occupancy matters more
// than registers). A block is persistent over images (img = blockIdx.x, += gridDim.x). Pass 1 transforms the
// rows (along Y) with LY-lane groups and keeps the 64 retained modes of every row in registers; an
// LDS tile (TileMap) redistributes them; pass 2 transforms the 64 columns (along X) with LX-lane groups.
// Each group keeps ONE row in flight: the loads of its next row are issued as soon as the first radix-4
// stage has consumed the row registers, so they travel while the rest of the transform runs, across the
// column pass and across image boundaries. Inter-pass twiddles live in LDS to stay within 128 VGPRs.
// nimg counts block-images: the 2^LOGR parts of each of the nfull whole images (nimg = nfull when LOGR = 0).
template <int LOGX, int LOGY, int LOGR>
__global__ __launch_bounds__(1024) void fft2d_trunc_kernel(const float2* __restrict__ x, float2* __restrict__ spec,
                                                           int nimg, int nfull)
{
    using G = Geo2D<LOGX, LOGY>;
    using T2 = TileMap<LOGX, LOGY, LOGR, true>;
    constexpr int DY = G::DY, LX = G::LX, LY = G::LY, ITY = G::ITY, MMY = G::MMY, MMX = G::MMX;
    extern __shared__ float2 lds[];
    const int tid = threadIdx.x;
    const int gy = tid / LY, ty = tid % LY;            // row pass: group and lane
    const int gx = tid / LX, tx = tid % LX;            // column pass: group (= column q) and lane
    float2* exch_y = lds + gy * (LY * 17);
    float2* exch_x = lds + gx * (LX * 17);
    float2* twtab_y = lds + G::LDS_MAIN;               // after the exchange regions / tile
    float2* twtab_x = twtab_y + G::TWY_ELEMS;
    float2* wsm = twtab_x + kTwLdsSize;
    float2* twsub = wsm + G::WSM_ELEMS;                // decimated images: w^(r p) of the long axis, r < R, p < 64
    fill_lds_twiddles<LOGY, LY>(twtab_y, tid, 1024);
    fill_lds_twiddles<LOGX>(twtab_x, tid, 1024);
    if (G::WIDE && tid < LY) wsm[tid] = kTwiddle1024[tid * (1024 / LY)];
    const float2* twrow_y = twtab_y + ty * kTwLdsPitch;
    const float2* twrow_x = twtab_x + tx * kTwLdsPitch;
    if constexpr (LOGR > 0) fill_decimation_twiddles<LOGX + LOGR>(twsub, tid, 1024);
    __syncthreads();

    const int row0 = T2::template first_row<G::PAIRED, G::WIDE>(gy);
    // row the lane finishes after the exchange, and its first mode (paired rows: lanes 8-15 take the second row)
    const int trow = G::PAIRED ? row0 + T2::PAIR * (ty >> 3) : row0;
    // scalar base + 32-bit lane offset keeps the load addresses out of the vector registers
    const unsigned lane_off = (unsigned)(((row0 * DY) << LOGR) + ty);
    // x is streamed exactly once: non-temporal loads keep it from evicting the 64x64 spectra, which the
    // next kernel re-reads, out of L2 / Infinity Cache
    auto issue = [&](cpx (&dst)[16], long array_row, int it, unsigned off) {
        const float2* base = x + (array_row + ((G::RPP * it) << LOGR)) * (long)DY;
#pragma unroll
        for (int i = 0; i < 16; ++i) dst[i] = load_streaming(&base[off + (unsigned)G::sample_off(i, T2::PAIR, LOGR)]);
    };

    long img = blockIdx.x;
    long img_row = first_array_row<LOGX, LOGR, false>(img < nimg ? img : 0, nfull);
    cpx v[16];
    if (img < nimg) issue(v, img_row, 0, lane_off);
    for (; img < nimg; img += gridDim.x) {
        // look-ahead target: the next image's first rows; after the last image every lane group re-reads the
        // same row (row 0 of image 0, cache resident) so the loop stays branch free at no HBM cost
        const bool more = img + gridDim.x < nimg;
        const long pre_row = first_array_row<LOGX, LOGR, false>(more ? img + gridDim.x : 0, nfull);
        const unsigned pre_off = more ? lane_off : (unsigned)ty;
        // pass 1: rows (along Y). T[it][mm] = mode tq + 16 mm (paired rows: tq + 8 mm) of row trow + RPP it
        cpx T[ITY][MMY];
#pragma unroll
        for (int it = 0; it < ITY; ++it) {
            if constexpr (!G::PAIRED) {
                cpx bb[16], gg[16];
                fft16_stage1<-1>(v, bb);
                // v is dead after the first radix-4 stage: its registers become the landing zone of the next row;
                // the last pass already fetches the next image's first row
                if (it + 1 < ITY) issue(v, img_row, it + 1, lane_off);
                else issue(v, pre_row, 0, pre_off);
                fwd_pass1_lds_finish(bb, twrow_y, gg);
                if constexpr (G::WIDE) wide_rows_forward_finish<LY>(gg, exch_y, wsm, ty, T[it]);
                else group_forward_finish<8>(gg, exch_y, ty, T[it]);
            } else {
                cpx gg[16], b8[8];
                {
                    cpx a8[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) { a8[i] = v[i]; b8[i] = v[8 + i]; }
                    fft8<-1>(a8);
                    fft8<-1>(b8);
#pragma unroll
                    for (int r = 0; r < 8; ++r) gg[r] = a8[r];
                }
                if (it + 1 < ITY) issue(v, img_row, it + 1, lane_off);
                else issue(v, pre_row, 0, pre_off);
                gg[8] = b8[0];
#pragma unroll
                for (int r = 1; r < 8; ++r) {
                    const cpx w = twrow_y[r];
                    gg[r] = cmul(gg[r], w);
                    gg[8 + r] = cmul(b8[r], w);
                }
                rows128_forward_finish(gg, exch_y, ty, T[it]);
            }
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < ITY; ++it)
#pragma unroll
            for (int mm = 0; mm < MMY; ++mm)
                lds[(trow + G::RPP * it) * T2::PITCH + G::tile_col(ty, mm)] = T[it][mm];
        __syncthreads();
        // pass 2: columns (along X); group gx owns column q = gx, lane tx holds rows tx + LX i
        cpx c[16];
        if (tid < G::COLT) {
#pragma unroll
            for (int i = 0; i < 16; ++i) c[i] = lds[(tx + LX * i) * T2::PITCH + gx];
        }
        __syncthreads();
        if (tid < G::COLT) {
            cpx gg[16], z[MMX];
            fwd_pass1_lds(c, twrow_x, gg);
            group_forward_finish<LOGX>(gg, exch_x, tx, z);
            if constexpr (LOGR > 0) {
                // part r of a decimated image: its modes enter the sum over the parts with w^(r p) of the long axis
                const int r = (int)PartNumbering<LOGR, false>::part(img, nfull);
                if (r != 0) {
#pragma unroll
                    for (int mm = 0; mm < MMX; ++mm) z[mm] = cmul(z[mm], twsub[r * 64 + tx + LX * mm]);
                }
            }
            // lane order of the retained modes: element mm*COLT + q*LX + tx  <->  mode (p = tx + LX mm, q).
            // Written through as it is produced, so the end-of-kernel cache write-back has nothing left to flush
            // (decimated images: the spectrum of part r of image i is channel r of the contraction, index r * nfull + i)
            float2* dst = spec + (PartNumbering<LOGR, false>::part(img, nfull) * (long)nfull + PartNumbering<LOGR, false>::image(img, nfull)) * 4096;
#pragma unroll
            for (int mm = 0; mm < MMX; ++mm) store_streaming(dst + tid + G::COLT * mm, z[mm]);
        }
        img_row = pre_row;
    }
}

// Backward image kernel, mirror of the forward one: persistent blocks, 16 waves per CU, twiddles in LDS.
// The 32 KiB spectrum of the next image is fetched (a few registers per lane) while the current image's rows
// are being transformed and stored, so a CU never waits for its input between images.
//
// SHARE: the XCDs of this GPU do not store at the same rate. Workgroup b of a grid runs on XCD b mod 8, and the blocks on
// the odd XCDs need about a fifth longer per image than those on the even ones (21.3 against 17.5 us at 256 x 256, in
// every launch on every box measured; a store-only probe gives the same picture), so with the same number of images per
// block the even half of the chip idles for the last sixth of the kernel. Here blocks 2p and 2p + 1 share the images
// p, p + P, p + 2P, ... (P pairs) unevenly: of the J * ITY row passes of the pair's J images the even block takes a share
// of even_share / kEvenShareDen, in whole images plus the first row passes of one image that the two blocks split
// (each takes it last; both run its column pass). 1024 images of 256 x 256: the even block transforms 4 1/4 images, the odd one 3 3/4: 101.6 -> 96.5 us.
// Which row goes to which block does not change any value: the output is bit-identical to the equal split.
// (even_share / kEvenShareDen, see kernels.h; measured here: 17/32 and 18/32 level, -5.3 us per layer, 19/32 -3 us)

template <int LOGX, int LOGY, bool SHARE, int LOGR>
__global__ __launch_bounds__(1024) void ifft2d_pad_kernel(const float2* __restrict__ spec, float2* __restrict__ y,
                                                          int nimg, int even_share, int nfull)
{
    using G = Geo2D<LOGX, LOGY>;
    using T2 = TileMap<LOGX, LOGY, LOGR, false>;
    constexpr int DY = G::DY, LX = G::LX, LY = G::LY, ITY = G::ITY, MMY = G::MMY, MMX = G::MMX;
    extern __shared__ float2 lds[];
    const int tid = threadIdx.x;
    const int gy = tid / LY, ty = tid % LY;
    const int gx = tid / LX, tx = tid % LX;
    float2* exch_y = lds + gy * (LY * 17);
    float2* exch_x = lds + gx * (LX * 17);
    float2* twtab_y = lds + G::LDS_MAIN;
    float2* twtab_x = twtab_y + G::TWY_ELEMS;
    float2* wsm = twtab_x + kTwLdsSize;
    float2* twsub = wsm + G::WSM_ELEMS;
    fill_lds_twiddles<LOGY, LY>(twtab_y, tid, 1024);
    fill_lds_twiddles<LOGX>(twtab_x, tid, 1024);
    if (G::WIDE && tid < LY) wsm[tid] = kTwiddle1024[tid * (1024 / LY)];
    const float2* twrow_y = twtab_y + ty * kTwLdsPitch;
    const float2* twrow_x = twtab_x + tx * kTwLdsPitch;
    if constexpr (LOGR > 0) fill_decimation_twiddles<LOGX + LOGR>(twsub, tid, 1024);
    __syncthreads();

    const int row0 = T2::template first_row<G::PAIRED, G::WIDE>(gy);
    const int trow = G::PAIRED ? row0 + T2::PAIR * (ty >> 3) : row0;      // row whose modes the lane takes from the tile
    const unsigned lane_off = (unsigned)(((row0 * DY) << LOGR) + ty);
    const bool col_thread = tid < G::COLT;
    // part r of a decimated image is transformed from the spectrum of the whole image
    constexpr bool PART_MAJOR = LOGR == 1 && LOGY >= 9;
    using Parts = PartNumbering<LOGR, PART_MAJOR>;
    auto spectrum_of = [&](long img) { return spec + Parts::image(img, nfull) * 4096; };

    // The block transforms `count` images, image_at(k) for k < count; of its last one, if `split`, only the row passes
    // [pass0, pass1). Without SHARE: every block the images blockIdx.x, + gridDim.x, ... in full.
    long first = blockIdx.x, step = gridDim.x, last = 0;
    int count = (int)((nimg - first + step - 1) / step), pass0 = 0, pass1 = ITY;
    bool split = false;
    if constexpr (SHARE) {
        const int pairs = gridDim.x / 2, pr = blockIdx.x >> 1, odd = blockIdx.x & 1;     // the host launches an even grid
        const int J = (nimg - pr + pairs - 1) / pairs;                                    // images of this pair
        const int even_passes = (J * ITY * even_share + kEvenShareDen / 2) / kEvenShareDen;
        const int whole = even_passes / ITY, rest = even_passes % ITY;                    // of the even block
        step = pairs;
        split = rest != 0;
        last = pr + (long)pairs * whole;                    // the image the pair splits: the last one of either block
        if (!odd) {
            first = pr;                                     // images 0 .. whole - 1 of the pair, then the first `rest` passes
            count = whole + (split ? 1 : 0);
            pass1 = rest;
        } else {
            first = pr + (long)pairs * (whole + (split ? 1 : 0));   // the pair's remaining whole images, then the other passes
            count = J - whole;
            pass0 = rest;
        }
    }
    auto image_at = [&](int k) -> long { return (SHARE && split && k == count - 1) ? last : first + step * k; };

    cpx c[MMX];
    if (count > 0 && col_thread) {
        const float2* src = spectrum_of(image_at(0));
#pragma unroll
        for (int mm = 0; mm < MMX; ++mm) c[mm] = src[tid + G::COLT * mm];
    }
    for (int k = 0; k < count; ++k) {
        const long img = image_at(k);
        const long pre = k + 1 < count ? image_at(k + 1) : img;
        const bool partial = SHARE && split && k == count - 1;
        const int it0 = partial ? pass0 : 0, it1 = partial ? pass1 : ITY;
        // pass 1: columns (p -> x) of column q = gx
        cpx u[16];
        if constexpr (LOGR > 0) {
            const int r = (int)Parts::part(img, nfull);
            if (r != 0 && col_thread) {
#pragma unroll
                for (int mm = 0; mm < MMX; ++mm) c[mm] = cmulc(c[mm], twsub[r * 64 + tx + LX * mm]);
            }
        }
        if (col_thread) group_backward_lds<LOGX>(c, twrow_x, exch_x, tx, u);
        // the exchange regions alias the tile: every wave must be done with them before the tile is written
        __syncthreads();
        if (col_thread) {
#pragma unroll
            for (int i = 0; i < 16; ++i) lds[(tx + LX * i) * T2::PITCH + gx] = u[i];
            // next image's spectrum (for the last image: a harmless re-read of its own 32 KiB)
            const float2* src = spectrum_of(pre);
#pragma unroll
            for (int mm = 0; mm < MMX; ++mm) c[mm] = src[tid + G::COLT * mm];
        }
        __syncthreads();
        cpx cc[ITY][MMY];
#pragma unroll
        for (int it = 0; it < ITY; ++it)
#pragma unroll
            for (int mm = 0; mm < MMY; ++mm)
                cc[it][mm] = lds[(trow + G::RPP * it) * T2::PITCH + G::tile_col(ty, mm)];
        __syncthreads();
        // pass 2: rows (q -> y), coalesced row stores.
        // y is written once and not re-read by this layer: non-temporal stores stop half a gigabyte of
        // dirty lines from lingering in the Infinity Cache and being written back under the next kernel's reads
#pragma unroll
        for (int it = 0; it < ITY; ++it) {
            if (SHARE && (it < it0 || it >= it1)) continue;       // uniform: row passes of the split image left to the partner
            cpx yv[16];
            if constexpr (G::PAIRED) rows128_backward(cc[it], twrow_y, exch_y, ty, yv);
            else if constexpr (G::WIDE) wide_rows_backward<LY>(cc[it], twrow_y, wsm, exch_y, ty, yv);
            else group_backward_lds<8>(cc[it], twrow_y, exch_y, ty, yv);
            // uniform base + lane offset + immediates
            float2* dst = y + (first_array_row<LOGX, LOGR, PART_MAJOR>(img, nfull) + ((G::RPP * it) << LOGR)) * (long)DY;
#pragma unroll
            for (int i = 0; i < 16; ++i) store_streaming(dst + lane_off + G::sample_off(i, T2::PAIR, LOGR), yv[i]);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Mode-space complex GEMM on the matrix cores.
//   C[n][m] = alpha * sum_k W[k + n*K] * A[k][m] (+ beta C),   A: [K][Mtot], C: [N][Mtot]  (m contiguous)
// Same contraction as the reference's cgemm / the GEMM phase of its fused kernel
// (fusion_variants/1D_A_exp_fft+cgemm+ifft/cgemm.cuh:4-205, operand layout lda=M, ldb=K, ldc=M). Four real products per
// complex one, each from six bf16 matrix instructions per 32 channels (bf16_split.h).
// Rows of a tile are 16 output channels n, columns 16 consecutive m, contraction in steps of 32 channels (eight per lane
// of a quarter wavefront). A wave owns 16 m and all 16 NT output channels of its block: an element of A is loaded and split
// once per block, and its parts meet NT fragments of W read from LDS. The W tile holds the parts of alpha W as fragments
// in lane order, 6 x 1 KiB per (step, 16 channels): an operand is one conflict-free 16-byte read. With HALVES a step is two of 16
// channels whose (re, im) pairs share one instruction, so that a last step of at most 16 channels costs half (gemm_steps.h).
// Blocks are persistent over column blocks (XCD j takes the j-th eighth of them, so that an XCD keeps to one part of the
// memory system); the strip of the next step - of the next column block after the last - is requested before the matrix
// work of the current one, and nothing in the walk waits at a barrier, so loads, matrix work and stores of the waves overlap.
// With beta the values of C are read 16 at a time before any is stored (M = 262,144, N = 128, K = 24: 198 -> 124 us, K = 64: 221 -> 154;
// with a column block per block instead of the walk, so that nothing waits behind the strip of the next: 130, 175).
// Operands that the split does not hold (bf16_split.h) are found while they are split and in the accumulators, per wave and column
// block; the wave then forms its product again with fp32 matrix instructions (two to four times the time of the column block).
//   Kw    = period of W along the contraction: channel k is weighted with W[k mod Kw + n Kw] (Kw = K: the plain product;
//           Kw = K / R: the R parts of decimated images, see above, share the weights of their image's channel);
//   Kp    = channels covered by one run over the tile (K, or Kw: the contraction then runs over the tile K / Kw times);
//   cap   = steps that the tile can hold; with more steps in a run the tile is rebuilt as the contraction proceeds.
// ---------------------------------------------------------------------------------------------
constexpr size_t kSplitStepBytes = 6 * 1024;            // LDS of one step of 16 output channels

template <int NT, int THREADS, bool HALVES>
__global__ __launch_bounds__(THREADS, THREADS == 1024 ? 4 : 2) void cgemm_modes_split_kernel(
    const float2* __restrict__ A, const float2* __restrict__ W, float2* __restrict__ C, long Mtot, int K, float2 alpha,
    float2 beta, long nblocks, int Kw, int Kp, int cap)
{
    extern __shared__ uint4_v sW4[];
    __shared__ unsigned sLow[THREADS / 64];             // per wave: it has built fragments with weights below the split's range
    constexpr int MBLOCK = THREADS / 4;                 // columns per block: 16 per wave
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, col = lane & 15, kq = lane >> 4;
    const int n0 = blockIdx.y * (16 * NT);
    const int steps = (Kp + GEMM_KSTEP - 1) / GEMM_KSTEP, runs = K / Kp;
    const bool resident = steps <= cap;                 // the tile is built once
    const bool eighths = (gridDim.x & 7) == 0 && (nblocks & 7) == 0;
    auto block_of = [&](long v) { return eighths ? (v & 7) * (nblocks >> 3) + (v >> 3) : v; };

    // channels 8 kq ... 8 kq + 7 of step `step` of a run, of the lane's column. Branch free, so that the loads stay where
    // they are issued: lanes beyond the run (its last step may be short) read the first channels of the step again - the tile
    // holds zeros there - and waves beyond the last column read the first strip (nothing is stored from it). `live` is false
    // after the last step of the block: every lane then reads one line.
    // HALVES: channels 4 kq ... 4 kq + 3 of both halves of the step.
    constexpr int PER_LANE = HALVES ? 4 : 8;            // consecutive channels of a lane
    const unsigned lane_row = (unsigned)(PER_LANE * kq * Mtot), lane_col = wave * 16 + col;
    float2 bv[8];
    auto fetch = [&](long mb, int run, int step, bool live) {
        const bool column = mb * MBLOCK + wave * 16 < Mtot;       // Mtot is a multiple of 16; Kp of 8
        const float2* base = A + (column ? mb * MBLOCK : 0) + (long)(run * Kp + GEMM_KSTEP * step) * Mtot;    // uniform
        if constexpr (HALVES) {
            const int left = Kp - GEMM_KSTEP * step - PER_LANE * kq;      // channels of the step from the lane's first on
            const unsigned first = live ? (column ? lane_col : (unsigned)col) : 0u;
            const unsigned off = live && left > 0 ? first + lane_row : first, row = live && left > 0 ? (unsigned)Mtot : 0u;
            const bool second = live && left > 16;
            const float2* upper = base + (second ? 16 * Mtot + (long)(first + lane_row) : (long)first);
            const unsigned upper_row = second ? (unsigned)Mtot : 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) { bv[j] = base[off + j * row]; bv[4 + j] = upper[j * upper_row]; }
        } else {
            const unsigned off = live ? (column ? lane_col : (unsigned)col) + (GEMM_KSTEP * step + 8 * kq < Kp ? lane_row : 0u) : 0u;
#pragma unroll
            for (int j = 0; j < 8; ++j) bv[j] = (base + j * Mtot)[off];
        }
    };
    // fragments of the steps s0 ... s0 + count - 1: entry (step, tile, kq, n mod 16) = eight consecutive channels of one n, real and imaginary
    // parts apart. HALVES: entry (half step, tile, kq, n mod 16) = four consecutive channels as (re, im) pairs
    bool low_weights = false;                           // once seen it holds for all column blocks: they share the weights
    auto build = [&](int s0, int count) {
        for (int e = tid; e < (HALVES ? 2 : 1) * count * NT * 64; e += THREADS) {
            const int l = e & 63, t = (e >> 6) % NT, s = (e >> 6) / NT;
            const int k = GEMM_KSTEP * s0 + (HALVES ? 16 : GEMM_KSTEP) * s + PER_LANE * (l >> 4), n = n0 + 16 * t + (l & 15);
            float2 w[PER_LANE];
#pragma unroll
            for (int j = 0; j < PER_LANE; ++j) w[j] = make_float2(0.f, 0.f);
            if (k < Kp) {
                const float2* src = W + (k % Kw) + (long)n * Kw;    // Kw is a multiple of 8
#pragma unroll
                for (int j = 0; j < PER_LANE; ++j) w[j] = src[j];
            }
#pragma unroll
            for (int j = 0; j < PER_LANE; ++j) w[j] = make_float2(w[j].x * alpha.x - w[j].y * alpha.y, w[j].x * alpha.y + w[j].y * alpha.x);
            unsigned bits = ~0u;                        // (zeros are common here: channels beyond Kp)
#pragma unroll
            for (int j = 0; j < PER_LANE; ++j) bits = lower(bits, w[j]);
            low_weights |= any_lane(bits < kSplitLow);
            SplitOperand re, im;                        // HALVES: re holds the pairs
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                unsigned h, m, lo;
                if constexpr (HALVES) split_bf16_pair(w[j].x, w[j].y, h, m, lo);
                else split_bf16_pair(w[2 * j].x, w[2 * j + 1].x, h, m, lo);
                re.h[j] = h; re.m[j] = m; re.l[j] = lo;
                if constexpr (!HALVES) {
                    split_bf16_pair(w[2 * j].y, w[2 * j + 1].y, h, m, lo);
                    im.h[j] = h; im.m[j] = m; im.l[j] = lo;
                }
            }
            uint4_v* dst = sW4 + (e >> 6) * (HALVES ? 192 : 384) + l;
            dst[0] = re.h; dst[64] = re.m; dst[128] = re.l;
            if constexpr (!HALVES) { dst[192] = im.h; dst[256] = im.m; dst[320] = im.l; }
        }
        if (lane == 0) sLow[wave] = low_weights;
    };

    float4_v re[NT], im[NT];
    auto clear = [&]() {
#pragma unroll
        for (int t = 0; t < NT; ++t) re[t] = im[t] = float4_v{ 0.f, 0.f, 0.f, 0.f };
    };
    clear();
    // one loop over column blocks, runs and steps: nested ones cost a copy of the strip at every edge between them
    long v = blockIdx.x, mb = block_of(v);              // the grid is no larger than the number of column blocks
    int run = 0, step = 0, slot = 0;                    // slot: the step's place in the tile
    bool built = false, low_column = false;             // low_column: small values among the wave's columns
    unsigned low_tile = 0;
    fetch(mb, 0, 0, true);
    while (true) {
        if (slot == 0 && !(resident && built)) {        // uniform over the block
            if (built) __syncthreads();                 // not before the first build: the last waves of a block start microseconds late
            build(step, steps - step < cap ? steps - step : cap);
            __syncthreads();
            low_tile |= sLow[lane & (THREADS / 64 - 1)];
            built = true;
        }
        SplitOperand ar, ai;                            // HALVES: the (re, im) pairs of the two halves
        low_column |= below_split_range(bv);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            unsigned h, m, l;
            if constexpr (HALVES) split_bf16_pair(bv[j].x, bv[j].y, h, m, l);
            else split_bf16_pair(bv[2 * j].x, bv[2 * j + 1].x, h, m, l);
            ar.h[j] = h; ar.m[j] = m; ar.l[j] = l;
            if constexpr (HALVES) split_bf16_pair(bv[4 + j].x, bv[4 + j].y, h, m, l);
            else split_bf16_pair(bv[2 * j].y, bv[2 * j + 1].y, h, m, l);
            ai.h[j] = h; ai.m[j] = m; ai.l[j] = l;
        }
        const bool both = GEMM_KSTEP * step + 16 < Kp;  // HALVES: the second half has channels; uniform
        asm volatile("" ::: "memory");                  // operand reads of the tile stay inside the loop
        const bool run_ends = step + 1 == steps, last = run_ends && run + 1 == runs;
        const bool more = v + gridDim.x < nblocks;
        const int next_step = run_ends ? 0 : step + 1, next_run = last ? 0 : (run_ends ? run + 1 : run);
        const long next_mb = last && more ? block_of(v + gridDim.x) : mb;
        fetch(next_mb, next_run, next_step, !last || more);
        __builtin_amdgcn_sched_barrier(0);
        const uint4_v* frag = sW4 + slot * (NT * 384) + lane;
        if constexpr (HALVES) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                if (u == 1 && !both) break;
                const SplitOperand& a = u == 0 ? ar : ai;
                SplitOperand for_re, for_im;            // (re, -im) and (im, re): with (re, im) of a weight the real and the imaginary part
                for_re.h = a.h ^ 0x80000000u; for_re.m = a.m ^ 0x80000000u; for_re.l = a.l ^ 0x80000000u;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    for_im.h[j] = __builtin_amdgcn_alignbit(a.h[j], a.h[j], 16);
                    for_im.m[j] = __builtin_amdgcn_alignbit(a.m[j], a.m[j], 16);
                    for_im.l[j] = __builtin_amdgcn_alignbit(a.l[j], a.l[j], 16);
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const uint4_v* f = frag + (u * NT + t) * 192;
                    const SplitOperand w{ f[0], f[64], f[128] };
                    mac_split2(w, for_re, for_im, re[t], im[t]);
                }
            }
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                SplitOperand w{ frag[t * 384], frag[t * 384 + 64], frag[t * 384 + 128] };
                float4_v r = re[t], i = im[t];
                mac_split2(w, ar, ai, r, i);                            // Wr
                w = SplitOperand{ frag[t * 384 + 192], frag[t * 384 + 256], frag[t * 384 + 320] };
                i = mac_split(w, ar, i);                                // Wi
                w.h ^= 0x80008000u; w.m ^= 0x80008000u; w.l ^= 0x80008000u;
                r = mac_split(w, ai, r);                                // - Wi
                re[t] = r;
                im[t] = i;
            }
        }
        if (last) {
            if (mb * MBLOCK + wave * 16 < Mtot) {
                float high[2] = { 0.f, 0.f };
#pragma unroll
                for (int t = 0; t < NT; ++t) { high[0] = larger(high[0], re[t]); high[1] = larger(high[1], im[t]); }
                if (__builtin_expect(low_column | any_lane(low_tile != 0 | not_finite(high[0], high[1])), 0)) {
                    // operands beyond the split: the product in fp32
                    clear();
                    const float2* a = A + mb * MBLOCK + lane_col;
                    const float2* w = W + (long)(n0 + col) * Kw;
#pragma unroll 1
                    for (int k = kq; k < K; k += 4) {
                        const float2 ak = a[k * Mtot];
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            const float2 wk = w[k % Kw + (long)(16 * t) * Kw];
                            mac_fp32(make_float2(wk.x * alpha.x - wk.y * alpha.y, wk.x * alpha.y + wk.y * alpha.x), ak, re[t], im[t]);
                        }
                    }
                }
                // D[row = 4 kq + q][col] of tile t: output channel n0 + 16 t + 4 kq + q, the lane's column
                float2* dst = C + mb * MBLOCK + lane_col + (long)(n0 + 4 * kq) * Mtot;
                if (beta.x != 0.f || beta.y != 0.f) {               // variants A, B: C is read, up to 16 values at a time
                    constexpr int AT_ONCE = NT < 4 ? NT : 4;
#pragma unroll
                    for (int t0 = 0; t0 < NT; t0 += AT_ONCE) {
                        float2 c[AT_ONCE][4];
#pragma unroll
                        for (int t = 0; t < AT_ONCE; ++t)
#pragma unroll
                            for (int q = 0; q < 4; ++q) c[t][q] = dst[(long)(16 * (t0 + t) + q) * Mtot];
#pragma unroll
                        for (int t = 0; t < AT_ONCE; ++t)
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                c[t][q] = cmul(c[t][q], beta);
                                re[t0 + t][q] += c[t][q].x;
                                im[t0 + t][q] += c[t][q].y;
                            }
                    }
                }
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int q = 0; q < 4; ++q) dst[(long)(16 * t + q) * Mtot] = make_float2(re[t][q], im[t][q]);
            }
            if (!more) return;
            v += gridDim.x;
            low_column = false;
            clear();
        }
        mb = next_mb;
        run = next_run;
        step = next_step;
        slot = next_step == 0 || slot + 1 == cap ? 0 : slot + 1;
    }
}

// Few channels on some large products (K <= 16; K <= 32 in one range of sizes, see launch_cgemm_modes): fp32 matrix instructions
// over groups of four channels instead, three real products per complex one:
//   P1 = c (a + b),  P2 = (d - c) a,  P3 = (c + d) b   =>   re = P1 - P3,  im = P1 + P2      (alpha W = c + i d, A = a + i b)
// A block is 16 waves; wave w owns the 16-m strip w and 64 output channels; the strip sits in NG float2 registers per
// lane, all loads in flight while the W'' tile is built, and every n tile is stored as soon as it is complete.
// NG = channel groups of four that can hold data.
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int GEMM_THREADS = 1024;  // 16 waves x 16 m
constexpr int GEMM_MBLOCK = 256;    // m per block

// W'' tile in LDS: three planes (c, d - c, c + d) of floats at index (k / 4) * kW3Group + (k % 4) * kW3Row + n.
// An operand fetch (64 lanes: 4 k x 16 n) reads 16 consecutive floats of four rows 80 apart: one bank each. The
// build's lanes run along k, the contiguous direction of W: a group stride of 1 (mod 64 banks) spreads the lanes of a
// store over the banks as well.
constexpr int kW3Row = 80, kW3Group = 4 * kW3Row + 1;
template <int NG> constexpr int kW3Plane = NG * kW3Group;

template <int NG>
__device__ __forceinline__ void build_w3_tile(float* sW, const float2* __restrict__ W, int n0, int K, int Kw, float2 alpha, int tid)
{
    constexpr int KC = 4 * NG, WPT = KC * 64 / GEMM_THREADS;
    float2 wv[WPT];
#pragma unroll
    for (int u = 0; u < WPT; ++u) {
        const int idx = tid + u * GEMM_THREADS, k = idx % KC, n = idx / KC;
        wv[u] = (k < K) ? W[k % Kw + (long)(n0 + n) * Kw] : make_float2(0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < WPT; ++u) {
        const int idx = tid + u * GEMM_THREADS, k = idx % KC, n = idx / KC;
        const float c = wv[u].x * alpha.x - wv[u].y * alpha.y, d = wv[u].x * alpha.y + wv[u].y * alpha.x;
        float* dstw = &sW[(k >> 2) * kW3Group + (k & 3) * kW3Row + n];
        dstw[0] = c;
        dstw[kW3Plane<NG>] = d - c;
        dstw[2 * kW3Plane<NG>] = c + d;
    }
}

// one column block per block
template <int NG>
__global__ __launch_bounds__(GEMM_THREADS) void cgemm_modes3m_kernel(const float2* __restrict__ A,
                                                                     const float2* __restrict__ W, float2* __restrict__ C,
                                                                     long Mtot, int N, int K, float2 alpha, float2 beta,
                                                                     int Kw)
{
    __shared__ float sW[3 * kW3Plane<NG>];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, col = lane & 15, kq = lane >> 4;
    const int n0 = blockIdx.y * 64;
    const unsigned lane_off = (unsigned)(kq * Mtot) + (unsigned)(wave * 16 + col);
    // XCD j takes the j-th eighth of the column blocks, as above
    const unsigned mb = (unsigned)xcd_contiguous(blockIdx.x, gridDim.x);
    const float2* blk = A + (long)mb * GEMM_MBLOCK;
    const bool active = (long)mb * GEMM_MBLOCK + wave * 16 < Mtot;   // Mtot is a multiple of 16, not of 256
    float2* cblk = C + (long)mb * GEMM_MBLOCK;
    const bool has_beta = beta.x != 0.f || beta.y != 0.f;

    // the wave's whole A strip: lane (kq, col) holds channels 4 g + kq, g < NG; the loads overlap the tile build
    float2 bv[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) bv[g] = (active && 4 * g < K) ? (blk + (long)(4 * g) * Mtot)[lane_off] : make_float2(0.f, 0.f);
    build_w3_tile<NG>(sW, W, n0, K, Kw, alpha, tid);
    __syncthreads();
    if (!active) return;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        floatx4 p1 = floatx4{ 0.f, 0.f, 0.f, 0.f }, p2 = p1, p3 = p1;
        const float* wrow = &sW[kq * kW3Row + t * 16 + col];
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const float* w = wrow + g * kW3Group;
            p1 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[0], bv[g].x + bv[g].y, p1, 0, 0, 0);
            p2 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[kW3Plane<NG>], bv[g].x, p2, 0, 0, 0);
            p3 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[2 * kW3Plane<NG>], bv[g].y, p3, 0, 0, 0);
        }
        // D[row = 4 kq + v][col]: output channel n0 + 16 t + 4 kq + v, column m = wave * 16 + col
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            float2* p = cblk + (long)(n0 + 16 * t + 4 * kq + v) * Mtot + (wave * 16 + col);
            float2 r = make_float2(p1[v] - p3[v], p1[v] + p2[v]);
            if (has_beta) r = cadd(r, cmul(*p, beta));      // C = alpha A W + beta C (variants A, B)
            *p = r;
        }
    }
}

// Several column blocks per CU: persistent, beta = 0. A block builds the W'' tile once and walks column blocks; the strip of
// the next one is requested before the matrix work on the current one ends.
template <int NG>
__global__ __launch_bounds__(GEMM_THREADS) void cgemm_modes3m_persistent_kernel(const float2* __restrict__ A,
                                                                                const float2* __restrict__ W,
                                                                                float2* __restrict__ C, long Mtot, int N, int K,
                                                                                float2 alpha, long nblocks, int Kw)
{
    __shared__ float sW[3 * kW3Plane<NG>];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, col = lane & 15, kq = lane >> 4;
    const int n0 = blockIdx.y * 64;
    const unsigned lane_off = (unsigned)(kq * Mtot) + (unsigned)(wave * 16 + col);
    const bool eighths = (gridDim.x & 7) == 0 && (nblocks & 7) == 0;
    auto block_of = [&](long v) { return eighths ? (v & 7) * (nblocks >> 3) + (v >> 3) : v; };
    auto fetch = [&](float2 (&dst)[NG], long mb) {
        const bool active = mb * GEMM_MBLOCK + wave * 16 < Mtot;      // Mtot is a multiple of 16, not of 256
        const float2* blk = A + mb * GEMM_MBLOCK;
#pragma unroll
        for (int g = 0; g < NG; ++g) dst[g] = (active && 4 * g < K) ? (blk + (long)(4 * g) * Mtot)[lane_off] : make_float2(0.f, 0.f);
    };
    long v = blockIdx.x;                              // the grid is no larger than the number of column blocks
    float2 bv[NG];
    fetch(bv, block_of(v));
    build_w3_tile<NG>(sW, W, n0, K, Kw, alpha, tid);
    __syncthreads();
    for (; v < nblocks; v += gridDim.x) {
        asm volatile("" ::: "memory");                // keeps the operand fetches from the W'' tile inside the loop (192 registers otherwise)
        const long mb = block_of(v);
        const bool more = v + gridDim.x < nblocks;
        const long nb = more ? block_of(v + gridDim.x) : mb;
        const bool next_active = more && nb * GEMM_MBLOCK + wave * 16 < Mtot;
        const float2* nblk = A + nb * GEMM_MBLOCK;
        const bool active = mb * GEMM_MBLOCK + wave * 16 < Mtot;
        float2* cblk = C + mb * GEMM_MBLOCK;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            floatx4 p1 = floatx4{ 0.f, 0.f, 0.f, 0.f }, p2 = p1, p3 = p1;
            const float* wrow = &sW[kq * kW3Row + t * 16 + col];
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const float* w = wrow + g * kW3Group;
                p1 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[0], bv[g].x + bv[g].y, p1, 0, 0, 0);
                p2 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[kW3Plane<NG>], bv[g].x, p2, 0, 0, 0);
                p3 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[2 * kW3Plane<NG>], bv[g].y, p3, 0, 0, 0);
                // the last n tile has used this group of the strip: its registers take the next column block's
                if (t == 3 && more) bv[g] = (next_active && 4 * g < K) ? (nblk + (long)(4 * g) * Mtot)[lane_off] : make_float2(0.f, 0.f);
            }
            if (active) {
#pragma unroll
                for (int vv = 0; vv < 4; ++vv) {
                    float2* p = cblk + (long)(n0 + 16 * t + 4 * kq + vv) * Mtot + (wave * 16 + col);
                    *p = make_float2(p1[vv] - p3[vv], p1[vv] + p2[vv]);
                }
            }
        }
    }
}

int cu_count()
{
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    int v = cached[dev & 63].load(std::memory_order_relaxed);
    if (v > 0) return v;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    cached[dev & 63].store(v, std::memory_order_relaxed);
    return v;
}

int even_share_parts()
{
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return kEvenShareDen / 2;
    int v = cached[dev & 63].load(std::memory_order_relaxed);
    if (v > 0) return v;
    hipDeviceProp_t prop;
    v = kEvenShareDen / 2;
    if (hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount == 256 &&
        std::string(prop.gcnArchName).rfind("gfx950", 0) == 0)
        v = 17;
    cached[dev & 63].store(v, std::memory_order_relaxed);
    return v;
}

template <int LOGX, int LOGY, int LOGR>
static hipError_t launch_image_kernel(bool inverse, const float2* in, float2* out, int nfull, hipStream_t stream)
{
    using G = Geo2D<LOGX, LOGY>;
    if (nfull <= 0 || nfull > (0x7fffffff >> LOGR)) return hipErrorInvalidValue;
    const int nimg = nfull << LOGR;                    // images of one block each: the 2^LOGR parts of every image
    const size_t lds_bytes = G::LDS_BYTES + (LOGR > 0 ? sizeof(float2) * kDecimationTwiddles : 0);
    // persistent blocks: at most as many as fit at once (LDS allows one or two 1024-thread blocks per CU,
    // the thread count exactly one)
    const int blocks = nimg < cu_count() ? nimg : cu_count();
    // uneven shares between the blocks of a pair: a full grid (one block per CU, so that block parity is XCD parity), at
    // least two images per block (128 x 128 images are a single row pass each and are shared in whole images only)
    const bool share = inverse && blocks == cu_count() && blocks % 2 == 0 && nimg >= 2 * blocks && even_share_parts() != kEvenShareDen / 2;
    static std::atomic<unsigned long long> served[3];
    const void* fn = !inverse ? reinterpret_cast<const void*>(fft2d_trunc_kernel<LOGX, LOGY, LOGR>)
                     : share ? reinterpret_cast<const void*>(ifft2d_pad_kernel<LOGX, LOGY, true, LOGR>)
                             : reinterpret_cast<const void*>(ifft2d_pad_kernel<LOGX, LOGY, false, LOGR>);
    if (hipError_t e = allow_dynamic_lds(fn, lds_bytes, served[inverse ? (share ? 2 : 1) : 0]); e != hipSuccess) return e;
    if (share)
        hipLaunchKernelGGL((ifft2d_pad_kernel<LOGX, LOGY, true, LOGR>), dim3((unsigned)blocks), dim3(1024), lds_bytes, stream, in,
                           out, nimg, even_share_parts(), nfull);
    else if (inverse)
        hipLaunchKernelGGL((ifft2d_pad_kernel<LOGX, LOGY, false, LOGR>), dim3((unsigned)blocks), dim3(1024), lds_bytes, stream, in,
                           out, nimg, kEvenShareDen / 2, nfull);
    else
        hipLaunchKernelGGL((fft2d_trunc_kernel<LOGX, LOGY, LOGR>), dim3((unsigned)blocks), dim3(1024), lds_bytes, stream, in,
                           out, nimg, nfull);
    return hipGetLastError();
}

static hipError_t dispatch_image_kernel(bool inverse, int logDX, int logDY, const float2* in, float2* out, int nimg,
                                        hipStream_t stream)
{
    // columns: 128 or 256 rows per block, 512 / 1024 as 2 / 4 parts of 256; rows: any built length
    auto with_rows = [&](auto logy) -> hipError_t {
        constexpr int LOGY = decltype(logy)::value;
        switch (logDX) {
        case 7: return launch_image_kernel<7, LOGY, 0>(inverse, in, out, nimg, stream);
        case 8: return launch_image_kernel<8, LOGY, 0>(inverse, in, out, nimg, stream);
        case 9: return launch_image_kernel<8, LOGY, 1>(inverse, in, out, nimg, stream);
        case 10: return launch_image_kernel<8, LOGY, 2>(inverse, in, out, nimg, stream);
        default: return hipErrorInvalidValue;
        }
    };
    switch (logDY) {
    case 7: return with_rows(std::integral_constant<int, 7>{});
    case 8: return with_rows(std::integral_constant<int, 8>{});
    case 9: return with_rows(std::integral_constant<int, 9>{});
    case 10: return with_rows(std::integral_constant<int, 10>{});
    default: break;
    }
    return hipErrorInvalidValue;
}

hipError_t launch_fft2d_trunc(int logDX, int logDY, const float2* x, float2* spec, int nimg, hipStream_t stream)
{
    return dispatch_image_kernel(false, logDX, logDY, x, spec, nimg, stream);
}

hipError_t launch_ifft2d_pad(int logDX, int logDY, const float2* spec, float2* y, int nimg, hipStream_t stream)
{
    return dispatch_image_kernel(true, logDX, logDY, spec, y, nimg, stream);
}

// Which kernel (times of the stand-alone product on operands that come from HBM, us, the kernel before / this one):
//  * K <= 16: the split kernel (half a step) up to five blocks of 256 columns x 64 output channels per CU for N = 64 and multiples of
//    128, two for others, and for multiples of 128 from sixteen on (fp32 / split, K = 16: M = 4,096, N = 64, with beta, in tiles of
//    16 outputs 9.3 / 4.2; M = 98,304, N = 128 23.1 / 20.5; M = 163,840, N = 128 35.6 / 32.0; M = 524,288, N = 128 157 / 136).
//    Between, fp32 matrix instructions (M = 262,144, N = 128 55.3 / 64.7, N = 192 78.8 / 114; M = 524,288, N = 64 75.8 / 77.7), the
//    persistent kernel with several column blocks per CU. The split kernel is not the faster one everywhere on its side: N = 256 and
//    more from sixteen on with fewer than about six columns of blocks per CU (N = 256, K = 16: M = 262,144 102 / 123, M = 327,680
//    147 / 157, M = 508,416 334 / 240), inside 2D layers with N = 128 and 256 at three to five (1 to 3 % of the layer), M = 64 (3.5 /
//    3.6). It stays there for its error against 64 bits: 3.7e-8 (K = 16) and 3.2e-8 (K = 8), the three fp32 products 1.12e-7 and 8.7e-8.
//    K <= 32 goes to fp32 as well for N >= 128 and 8 to 16 such blocks per CU (M = 262,144, N = 128, K = 32: 77 against 88; from 16 on
//    the 128-channel tile below is ahead).
//  * otherwise the split kernel. Small products: blocks of 128 columns and the fewest output channels whose grid still fits one
//    block per CU (K = 64, N = 64, tiles of 64 / 32 / 16 output channels: M = 64: 7.5 / 5.5 / 4.7; M = 8,192: 8.5 / 6.3 / 5.5).
//    At most half a block of 256 columns x 64 output channels per CU: blocks of 128 columns (M = 16,384, N = 64, K = 64: fp32 18.6,
//    256 columns 14.0, 128 columns 11.1); also for N = 64 with one to two blocks per CU and more than 32 channels, where two blocks
//    of 128 columns on a CU overlap each other's phases (M = 65,536, K = 64: 22.7 / 21.5 / 19.6).
//    N a multiple of 128, up to 96 channels and 8 or more blocks per CU: tiles of 128 output channels, A is read once
//    (M = 524,288, K = 64: 271 / 214 / 197).
//    Else blocks of 256 columns, tiles of 64 (M = 163,840, N = 128, K = 72: 136 -> 90; M = 262,144, N = 128, K = 128: 259 -> 182).
hipError_t launch_cgemm_modes(const float2* A, const float2* W, float2* C, long Mtot, int N, int K, float2 alpha,
                              float2 beta, hipStream_t stream, int w_period)
{
    if (Mtot % 16 != 0 || Mtot <= 0 || Mtot >= (1L << 27) || N % 64 != 0 || K % 8 != 0) return hipErrorInvalidValue;
    const int Kw = w_period > 0 ? w_period : K;
    if (K % Kw != 0 || Kw % 8 != 0) return hipErrorInvalidValue;
    const long cus = cu_count(), columns = (Mtot + GEMM_MBLOCK - 1) / GEMM_MBLOCK, blocks = columns * (N / 64);
    const bool no_beta = beta.x == 0.f && beta.y == 0.f;

    auto launch_persistent = [&](auto ng_const) -> hipError_t {
        constexpr int NG = decltype(ng_const)::value;
        long g = cus;                                            // one block per CU and n tile
        if (g >= 8) g -= g % 8;                                  // whole groups of eight: every XCD the same share
        if (g > columns) g = columns;
        hipLaunchKernelGGL((cgemm_modes3m_persistent_kernel<NG>), dim3((unsigned)g, (unsigned)(N / 64), 1), dim3(GEMM_THREADS), 0,
                           stream, A, W, C, Mtot, N, K, alpha, columns, Kw);
        return hipGetLastError();
    };
    const bool split_ahead = N % 128 == 0 || N == 64 ? blocks <= 5 * cus || (no_beta && N % 128 == 0 && blocks >= 16 * cus) : blocks <= 2 * cus;
    const bool few = K <= 16 && !split_ahead;
    // Persistent not with beta: reading C back inside the walk waits for the strip requested just before it
    // (K = 32, M = 262,144: 79 against 74 us).
    if (few && no_beta && columns >= 2 * cus) return launch_persistent(std::integral_constant<int, 4>{});
    if (K > 16 && K <= 32 && no_beta && N >= 128 && blocks >= 8 * cus && blocks < 16 * cus)
        return launch_persistent(std::integral_constant<int, 8>{});
    if (few) {
        hipLaunchKernelGGL((cgemm_modes3m_kernel<4>), dim3((unsigned)columns, (unsigned)(N / 64), 1), dim3(GEMM_THREADS), 0, stream, A,
                           W, C, Mtot, N, K, alpha, beta, Kw);
        return hipGetLastError();
    }

    // cap: steps of 32 channels that the tile can hold; per_cu: blocks per CU
    auto launch_split_as = [&](auto nt_const, auto threads_const, auto halves_const, int Kp, int cap, int per_cu) -> hipError_t {
        constexpr int NT = decltype(nt_const)::value, THREADS = decltype(threads_const)::value;
        constexpr bool HALVES = decltype(halves_const)::value;
        const int steps = (Kp + GEMM_KSTEP - 1) / GEMM_KSTEP;
        const size_t lds_bytes = kSplitStepBytes * NT * (steps < cap ? steps : cap);
        static std::atomic<unsigned long long> served;
        if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(cgemm_modes_split_kernel<NT, THREADS, HALVES>), kSplitStepBytes * NT * cap, served);
            e != hipSuccess)
            return e;
        const long nblocks = (Mtot + THREADS / 4 - 1) / (THREADS / 4), tiles = N / (16 * NT);
        if (lds_bytes * per_cu > 160 * 1024) per_cu = 1;
        const long g = gemm_persistent_blocks(nblocks, per_cu * cus / tiles, K);
        hipLaunchKernelGGL((cgemm_modes_split_kernel<NT, THREADS, HALVES>), dim3((unsigned)g, (unsigned)tiles, 1), dim3(THREADS), lds_bytes, stream,
                           A, W, C, Mtot, K, alpha, beta, nblocks, Kw, Kp, cap);
        return hipGetLastError();
    };
    auto launch_split = [&](auto nt, auto threads, int cap, int per_cu) {
        const GemmWalk walk = gemm_walk(K, Kw, decltype(nt)::value, decltype(threads)::value, cap);
        return walk.halves ? launch_split_as(nt, threads, std::true_type{}, walk.run, cap, per_cu)
                           : launch_split_as(nt, threads, std::false_type{}, walk.run, cap, per_cu);
    };
    using Tiles4 = std::integral_constant<int, 4>;
    using Tiles8 = std::integral_constant<int, 8>;
    using Columns128 = std::integral_constant<int, 512>;
    using Columns256 = std::integral_constant<int, 1024>;
    using Tiles1 = std::integral_constant<int, 1>;
    using Tiles2 = std::integral_constant<int, 2>;
    // (64 output channels in place of the 64 input channels: one block has to hold all of a strip's outputs)
    const long strips = A == C ? cus : (Mtot + 127) / 128;
    if (strips * (N / 16) <= cus) return launch_split(Tiles1{}, Columns128{}, 6, 2);
    if (strips * (N / 32) <= cus) return launch_split(Tiles2{}, Columns128{}, 6, 2);
    if (2 * blocks <= cus || (N == 64 && K > 32 && blocks >= cus && blocks < 2 * cus)) return launch_split(Tiles4{}, Columns128{}, 6, 2);
    if (N % 128 == 0 && (Kw + GEMM_KSTEP - 1) / GEMM_KSTEP <= 3 && blocks >= 8 * cus) return launch_split(Tiles8{}, Columns128{}, 3, 1);
    return launch_split(Tiles4{}, Columns256{}, 6, 1);
}

}  // namespace tfno
