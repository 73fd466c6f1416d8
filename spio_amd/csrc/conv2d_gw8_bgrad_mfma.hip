// Fused backward kernel for conv2d_gw8 (gfx950): data gradient and weight gradient (and,
// optionally, the bias gradient) in one pass.
//
// Contract (reference kernels: spio/src/conv2d_gw8.cu:10-225 in its data-gradient mode and
// spio/src/conv2d_gw8_wgrad.cu:10-226; the reference launches them one after the other,
// spio/functional/conv2d_gw8_function.py:119-146):
//   dx[n,h,w,8g+c] = rn16(sum_{j,r,s} dy[n,h-r+py,w-s+px,8g+j] * w[8g+j,r,s,c])
//   dw[k,r,s,c]   += sum_{n,p,q} x[n,p+r-py,q+s-px,8g+c] * dy[n,p,q,k]            (fp32, atomics)
//   db[k]         += sum_{n,p,q} dy[n,p,q,k]                                      (with a bias)
//
// Why fuse: both gradients stream grad_output.  Run separately they move
// 2*|dy| + |x| + |dx| bytes through HBM; fused, dy is read once: 25 % less traffic for the
// backward step of an HBM-bound operator, and one launch instead of two.
//
// Scope: every filter size and padding the operator takes.  The kernel computes a "same"
// convolution (P = H and Q = W; padding PT rows above and PB below, PL columns left and PR right,
// PT + PB = R-1, PL + PR = S-1): then one copy of a dy row in LDS serves both gradients, and the dx
// row that completes at a step has the index of the x row of that step.  Any other padding is
// that convolution on a larger domain, DH x DW, in which x and dy sit at offsets that reproduce
// the problem's padding, with zeros around them: only the global addressing knows the tensors'
// real extents (domain rows and columns outside a tensor load zeros and store nothing), and below
// "row" and "column" are the domain's.
// A workgroup owns SPIO_BH rows (of dx, and of dy for the weight gradient) of SPIO_NB images
// side by side for SPIO_GB channel groups, repeated for SPIO_ITERS image blocks.  It streams the
// rows p0-PB .. p0+BH-1+PT of dy and p0-PT .. p0+BH-1+PB of x: step t stages dy row p0-PB+t and
// x row p0-(R-1)+t (an x row can only be multiplied once the dy rows up to PT below it are
// there).  The halo rows of dy above and below the block feed the
// data gradient only; the weight gradient masks them out of its dy fragments, so every dy row
// is counted by exactly one workgroup.  With SPIO_BH = DH a workgroup owns whole images and
// there is no halo.  Everything else is the separate kernels' design:
//   * rows of x and dy staged in LDS as [group][flattened pixel][8 ch], zero halo materialised
//     once, branch-free global loads SPIO_PF steps ahead;
//   * weight gradient: A = dy and dy one pixel on, B = x at two column taps, one accumulator per filter
//     row and four column taps, transposing LDS reads (see conv2d_gw8_wgrad_mfma.hip);
//   * data gradient: A = flipped, group-transposed filter for pairs of neighbouring pixels, B = every
//     second dy pixel (see conv2d_gw8_mfma.hip); dx rows take turns in R sets of accumulators;
//     a dy pixel (image i, column q) sits at flattened pixel i*WPI + q + PR, which is both its
//     place as a source pixel of the data gradient and, shifted by PR, its place opposite x
//     (column c at i*WPI + c + PL) in the weight gradient;
//   * a dy row is read from LDS for the weight gradient once, when it is the newest, and its fragments stay
//     in registers while the next R-1 x rows meet it: two ring rows of each tensor are enough;
//   * products of rows that do not exist (above, below, of neighbouring blocks) are left out at compile time;
//   * publishing of dw (and db) as in the weight-gradient kernel: sums staged in LDS in
//     grad_weight order, atomics of 64 consecutive floats;
//   * global memory through buffer instructions with the hardware bounds check as predicate
//     (lanes without data: out-of-range offset; rows the block does not need: empty descriptor;
//     such loads return zeros, such stores are dropped) and a fully unrolled step loop, so that
//     no memory instruction sits under a branch and the compiler's count of outstanding loads and
//     stores is exact (see conv2d_gw8_mfma.hip).
//
// With two rows instead of two neighbouring pixels side by side in both A operands a step had a third more
// products and twice the LDS reads, half of the lanes idled when a row was converted, and the sums took 32
// registers for a 3x3 filter and 128 for 7x7 (now 12 and 56).  What bounds the kernel is the chain of a step (barrier,
// LDS reads, products, conversion) on one or two waves a SIMD, then memory.  Before -> after: 128n 64c 56x56 35.2 ->
// 32.4 us (154 MB, 4.75 TB/s), 32n 15.4 -> 11.9, 512n 120.4 -> 112.2, 128n 96c 54.8 -> 52.9, 128n 768c 7x7 12.3 -> 9.9,
// 31n 1472c 27x17 38.2 -> 30.6, 54n 688c 18x18 5x5 44.2 -> 28.9, 128n 1392c 9x9 5x5 59 -> 42, 3n 224c 182x182 46 -> 38,
// 2n 1440c 161x87 1x1 68 -> 62.
#include "spio_conv_common.h"

using namespace spio;

#ifndef SPIO_NB
#define SPIO_NB 1
#endif
#ifndef SPIO_ITERS
#define SPIO_ITERS 1
#endif
#ifndef SPIO_PF
#define SPIO_PF 2
#endif
#ifndef SPIO_BQ
#define SPIO_BQ 0
#endif
#ifndef SPIO_PARTIALS
#define SPIO_PARTIALS 0
#endif
#ifndef SPIO_TS
#define SPIO_TS 1
#endif
#ifndef SPIO_HAS_BIAS
#define SPIO_HAS_BIAS 0
#endif
#ifndef SPIO_XCD_CHUNK
#define SPIO_XCD_CHUNK 0
#endif
#ifndef SPIO_HALO_CACHED
#define SPIO_HALO_CACHED 1
#endif
#ifndef SPIO_MAX_UNROLL
#define SPIO_MAX_UNROLL 40  // a step of this kernel is long: beyond this the unroller gives up
#endif

namespace {

// The kernel works on a size-preserving convolution of DH x DW images whose padding is PT rows
// above, PB below, PL columns left and PR right (PT + PB = R-1, PL + PR = S-1; equal halves for odd
// filter sizes, the larger half above and left for even ones).  x (and dx) and dy sit inside that
// domain at the offsets (XOY, XOX) and (DOY, DOX), one of each pair being 0, such that the
// problem's own padding comes out (DOY - XOY = PT - py), and count as zero around their real extent.
constexpr int PT = kR / 2, PB = kR - 1 - PT;
constexpr int PL = kS / 2, PR = kS - 1 - PL;
constexpr int DOY = PT > kPadY ? PT - kPadY : 0, XOY = PT > kPadY ? 0 : kPadY - PT;
constexpr int DOX = PL > kPadX ? PL - kPadX : 0, XOX = PL > kPadX ? 0 : kPadX - PL;
constexpr int DH = XOY + kH > DOY + kP ? XOY + kH : DOY + kP;
constexpr int DW = XOX + kW > DOX + kQ ? XOX + kW : DOX + kQ;

constexpr int GB = SPIO_GB;        // groups per workgroup
constexpr int BH = SPIO_BH;        // rows per workgroup
constexpr int NB = SPIO_NB;        // images side by side
constexpr int ITERS = SPIO_ITERS;  // image blocks per workgroup
constexpr int TS = SPIO_TS;        // waves per group: they split the 32-pixel chunks and the 16-pixel tiles
constexpr int PF = SPIO_PF;        // prefetch distance in rows (even)
constexpr int WAVES = GB * TS;
constexpr int THREADS = 64 * WAVES;
constexpr bool kDbias = SPIO_HAS_BIAS != 0;

// ---- weight gradient: column taps 4 nb .. 4 nb + 3 share one MFMA ----
constexpr int NB4 = (kS + 3) / 4;
// Column blocks (SPIO_BQ > 0): a workgroup owns BQ columns (of dx, and of dy for the weight
// gradient) and stages BQ + S - 1 columns of x and of dy: the extra columns hold the neighbouring
// blocks' pixels (the data gradient of the block's edge columns needs the neighbours' dy, the
// weight gradient the neighbours' x), or zeros at the image's edges.  The weight gradient's dy
// fragments are cleared where they reach into the extra columns, or the neighbour's dy would count twice.
// 0 = the whole width.
constexpr bool kColBlocks = SPIO_BQ > 0;
constexpr int BQ = kColBlocks ? SPIO_BQ : DW;
constexpr int QBLKS = (DW + BQ - 1) / BQ;
static_assert(!kColBlocks || NB == 1, "column blocks: one image per row");
constexpr int WPI = BQ + kS - 1;      // padded width of one image (block)
constexpr int F = NB * WPI;           // flattened pixels of a staged row
constexpr int KSPAN = (NB - 1) * WPI + BQ;
constexpr int KC = (KSPAN + 1 + 31) / 32;  // 32-pixel chunks; the first begins one pixel before the row
constexpr int CPW = (KC + TS - 1) / TS;   // chunks per wave
// ---- data gradient: a tile is 16 pairs of neighbouring pixels ----
constexpr int KB = (kS + 1 + 3) / 4;      // MFMA K-steps per dy row (4 of a pair's S + 1 columns each)
constexpr int WT = (F - kS + 1 + 31) / 32;   // 32-pixel tiles of a dx row
constexpr int TPW = (WT + TS - 1) / TS;      // tiles per wave
// ---- LDS geometry ----
// The pixels of a staged row lie in two planes, even ones first: lanes of the data gradient read every
// second pixel.  The planes are 8 cells (half the banks) apart modulo 16, the groups so that the cells a
// wave's threads write fall into different banks.  Chunks and tiles past the last one (waves share a
// row) read and write cells that exist; they hold zeros, and nobody looks at the results.
constexpr int plane_cells(int pixels) { return (pixels + 1) / 2 + ((8 - (pixels + 1) / 2 % 16) + 16) % 16; }
constexpr int GS_MOD = GB > 4 ? 9 : GB > 2 ? 2 : 4;
constexpr int group_cells(int plane, int pixels) { return plane + pixels / 2 + ((GS_MOD - (plane + pixels / 2) % 16) + 16) % 16; }
constexpr int FPX = 32 * CPW * TS + 4 * NB4 - 2;  // x pixels a weight-gradient read can touch
constexpr int HX = plane_cells(FPX);
constexpr int GSX = group_cells(HX, FPX);  // x group stride
constexpr int DL = PR > 0 ? PR : 1;  // pixel of the first dy column: at least one zero (or neighbour's) pixel before it
constexpr int DO = DL - PR;
constexpr int FPD_W = DL + 32 * CPW * TS;                    // dy pixels: weight-gradient reads
constexpr int FPD_D = DO + 32 * TPW * TS + 4 * KB - 2;       // dy pixels: data-gradient reads
constexpr int FPD = FPD_W > FPD_D ? FPD_W : FPD_D;
constexpr int HD = plane_cells(FPD);
constexpr int GSD = group_cells(HD, FPD);  // dy group stride
SPIO_DEVICE constexpr int pos(int pixel, int plane) { return (pixel >> 1) + (pixel & 1) * plane; }
// ring rows carry one spare unit behind the last group: the cell that threads without a source
// cell write their (zero) load result to
constexpr int XROW_UNITS = GB * GSX + 1;
constexpr int DROW_UNITS = GB * GSD + 1;
constexpr int XDUMP = GB * GSX;
constexpr int DDUMP = GB * GSD;
constexpr int OSTRIDE = stage_pitch(GB);     // bytes per pixel in the dx output stage, two planes as well
constexpr int OPLANE = 16 * TPW * TS * OSTRIDE + 128;
constexpr int OUT_ROW_BYTES = 2 * OPLANE;
constexpr int X_CELLS = F * GB;
constexpr int LPTX = (X_CELLS + THREADS - 1) / THREADS;
// dy cells a workgroup loads per row: the real columns of whole rows (the halo stays zero), all
// BQ + S - 1 columns of a column block
constexpr int D_CELLS = kColBlocks ? F * GB : NB * DW * GB;
constexpr int LPTD = (D_CELLS + THREADS - 1) / THREADS;  // dy loads per thread per row
constexpr int O_CELLS = NB * BQ * GB;
constexpr int LPTO = (O_CELLS + THREADS - 1) / THREADS;  // dx stores per thread per row
constexpr int GBLKS = (kGroups + GB - 1) / GB;
constexpr int NBLKS = (kN + NB * ITERS - 1) / (NB * ITERS);
constexpr int PBLKS = (DH + BH - 1) / BH;
constexpr int NUM_BLOCKS = GBLKS * PBLKS * QBLKS * NBLKS;
// steps: dy rows p0-PB .. p0+BH-1+PT, then PB more for the last x rows
constexpr int ROWS = BH + PB + kR - 1;

constexpr int gcd_(int a, int b) { return b == 0 ? a : gcd_(b, a % b); }
constexpr int lcm_(int a, int b) { return a / gcd_(a, b) * b; }
constexpr int LCM = lcm_(kR, PF);  // PF is even, so this is too
// up to SPIO_MAX_UNROLL steps the step loop is unrolled completely, longer ones run in chunks
constexpr bool kFullUnroll = ROWS <= SPIO_MAX_UNROLL;
constexpr int UNROLL = kFullUnroll ? (ROWS + LCM - 1) / LCM * LCM : LCM;
constexpr int pmod(int a, int m) { return ((a % m) + m) % m; }
// Where a workgroup has one block of whole rows, a finished dx row is converted and staged in the step after its last
// tap, while that step's fragment reads are on their way, instead of behind the products it would have to wait for.  Its
// sums are the ones that the step begins a new row in.  Before -> after in the same configuration: 1n 64c 56x56 5.8 ->
// 5.4 us, 8n 7.2 -> 6.8, 32n 11.9 -> 11.3, 128n in 28-row blocks 34.0 -> 31.5, 16n 64c 50x50 2x2 13.5 -> 10.5, 128n 128c 28x28
// 19.3 -> 18.8.  Elsewhere it gives nothing or takes registers that there are not: several blocks 16n 64c 128x512 79 -> 82,
// column blocks 1n 400c 211x211 37.7 -> 41.3, 5x5 4n 424c 84x84 61.6 -> 65.2, 1x1 8n 248c 42x42 10.3 -> 11.0.
constexpr bool kLateStage = ITERS == 1 && !kColBlocks && (kR == 2 || kR == 3);

constexpr int RING_UNITS = 2 * XROW_UNITS + 2 * DROW_UNITS;  // two rows each: a step's and the next one's
constexpr int STREAM_UNITS = RING_UNITS + 2 * OUT_ROW_BYTES / 16;
constexpr int FILTER_UNITS = GB * 8 * kR * kS;  // filters staged once at the start
constexpr int GROUP_FLOATS = kR * kS * 64;
// Two-stage publishing (SPIO_PARTIALS = 1): every workgroup stores its sums, in grad_weight order
// (and its GB * 8 bias sums behind them), into its own block of a workspace that takes the place
// of the grad_weight argument; the <name>_reduce kernel at the end of this file stores the sum of
// the blocks into grad_weight (and grad_bias).  No atomics: with one-round grids all workgroups
// reach the publish together and their atomic additions to the same lines retire one after the
// other (14 ns each: 3.6 us for 256 workgroups at N=128, C=64, 56x56); nothing to zero first.
constexpr int PART_FLOATS = GB * GROUP_FLOATS + (SPIO_HAS_BIAS ? GB * 8 : 0);  // one workgroup's block
constexpr int NPART = NBLKS * PBLKS * QBLKS;  // blocks per channel block
constexpr int PUBLISH_FLOATS = WAVES * GROUP_FLOATS + (SPIO_HAS_BIAS ? WAVES * 8 : 0);
constexpr int max3(int a, int b, int c) { return a > b ? (a > c ? a : c) : (b > c ? b : c); }
constexpr int LDS_UNITS = max3(STREAM_UNITS, FILTER_UNITS, (PUBLISH_FLOATS + 3) / 4);
static_assert(LDS_UNITS * 16 <= 160 * 1024, "LDS overflow");
static_assert(PF >= 2 && PF % 2 == 0 && WAVES <= 16, "bad configuration");

constexpr long long X_IMAGE_BYTES = (long long)kH * kW * kC * 2;  // of x
constexpr long long DX_IMAGE_BYTES = (long long)kH * kW * kC * kDstBytes;  // of dx
constexpr long long D_IMAGE_BYTES = (long long)kP * kQ * kC * kSrcBytes;  // of dy (SPIO_SRC_F32: fp32)
static_assert(NB * DX_IMAGE_BYTES < (1ll << 31) && NB * D_IMAGE_BYTES < (1ll << 31),
              "an image block must stay below 2 GiB (32-bit buffer offsets)");
constexpr int X_ROW_BYTES = kW * kC * 2;
constexpr int DX_ROW_BYTES = kW * kC * kDstBytes;
constexpr int D_ROW_BYTES = kQ * kC * kSrcBytes;
constexpr unsigned OOB = 0x80000000u;  // offset of a lane without data: beyond every descriptor
// Cache-policy operands of the buffer instructions: streamed (2) unless several channel blocks share the
// lines, then loaded with the default policy so that the second block finds them in L2.  Streamed -> default
// loads, best of four configurations: 94n 296c 43x47 129 -> 112 us, 50n 152c 21x41 17.1 -> 15.1, 64n 72c 56x56
// 41 -> 38, 32n 320c 28x28 17.8 -> 15.6, 16n 256c 56x56 38 -> 35, 128n 96c 56x56 equal.  Where a pixel is whole lines
// it can cost instead (64n 192c 28x28 18.6 -> 19.3, 8n 128c 112x112 35.6 -> 38.1); offering the sweep both
// there made a shape's first use 1 to 3 s longer and chose the same on the shapes tried.  SPIO_NT = 0 stores
// with the default policy: L2 then joins the parts of a line that different blocks store, see the
// configurations.
constexpr bool kSplitLines = splits_lines(GB, GBLKS);
constexpr int AUX_LD = kSplitLines ? 0 : 2;
constexpr int AUX_ST = SPIO_NT ? 2 : 0;

typedef __amdgpu_buffer_rsrc_t rsrc_t;
SPIO_DEVICE rsrc_t make_rsrc(const void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}

SPIO_DEVICE spio_half8 read_tr_pair(const unsigned char* lo, const unsigned char* hi) {
    typedef spio_short4 __attribute__((address_space(3))) * lds_ptr;
    union {
        spio_short4 s[2];
        spio_half8 h;
    } v;
    v.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)lo);
    v.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)hi);
    return v.h;
}

}  // namespace

extern "C" __global__ void SPIO_LAUNCH_BOUNDS(THREADS)
SPIO_KERNEL_NAME(spio_uint4* __restrict__ grad_input, float* __restrict__ grad_weight,
                 const spio_uint4* __restrict__ x, const spio_uint4* __restrict__ dy,
                 const spio_half* __restrict__ weights
#if SPIO_HAS_BIAS
                 , float* __restrict__ grad_bias  // [K] fp32, accumulated into; null = not wanted
#endif
) {
    // One LDS block: x ring, dy ring, two dx output-stage rows.  Before the first row it holds
    // the staged filters, after the last one the reduction scratch.
    __shared__ spio_uint4 lds[LDS_UNITS];
    spio_uint4* const xring = lds;
    spio_uint4* const dring = lds + 2 * XROW_UNITS;
    unsigned char* const ostage = reinterpret_cast<unsigned char*>(lds + RING_UNITS);

    const int tid = thread_id();
    const int lane = tid & 63;
    // scalar wave index: conditions on it become scalar branches, so no MFMA (which ignores the
    // lane mask) is issued under an empty mask
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wg = TS == 1 ? wave : wave % GB;
    const int ws = TS == 1 ? 0 : wave / GB;

    // Tile order: row blocks fastest, so that neighbours in a run of SPIO_XCD_CHUNK tiles share halo
    // rows through one XCD's L2.  Where channel blocks share lines they go fastest instead, a run
    // holding all of a pixel's: dealt to different XCDs, every one of them would fetch the whole lines
    // from memory (measured: twice the algorithmic reads).
    constexpr int RUN = kSplitLines ? line_run(SPIO_XCD_CHUNK, GBLKS) : SPIO_XCD_CHUNK;
    const int b = xcd_tile<RUN, NUM_BLOCKS>(block_id());
    // Column blocks go before the row blocks: neighbours share S - 1 columns of every row.
    constexpr int TILES = QBLKS * PBLKS;
    const int tile = kSplitLines ? (b / GBLKS) % TILES : b % TILES;
    const int cb = kSplitLines ? b % GBLKS : (b / TILES) % GBLKS;
    const int nbk = b / (TILES * GBLKS);
    const int pb = tile / QBLKS;
    const int q0 = (tile % QBLKS) * BQ;
    const int p0 = pb * BH;
    const int bh_eff = imin(BH, DH - p0);  // rows this block owns
    // first and last row (of the domain) the block needs: of x for the weight gradient of its dy
    // rows, of dy for its dx rows (which include the weight gradient's)
    const int xrow_lo = p0 - PT, xrow_hi = p0 + bh_eff - 1 + PB;
    const int drow_lo = p0 - PB, drow_hi = p0 + bh_eff - 1 + PT;
    const int gglob = cb * GB + wg;
    const bool wave_active = gglob < kGroups;

    // ---- data-gradient filter fragments: wfrag[r][u] ----
    // A[m = 8 j + ch][(kb, jj)] = w[8g+jj][R-1-r][S-1-s][ch], s = 4 u + kb - j: pixel j of a pair meets
    // column 4 u + kb of the pair's S + 1 source columns under tap s.  The workgroup copies its groups'
    // filters to LDS as they lie in memory and every wave reads its fragments with the
    // transposing LDS read (same scheme as the data-gradient mode of conv2d_gw8_mfma.hip).
    // The filter loads are issued here, the loads of the first rows right behind them, and only
    // then does anything wait: the fragments are built while the rows are on their way.
    constexpr int FLT = (FILTER_UNITS + THREADS - 1) / THREADS;
    spio_uint4 fpre[FLT];
    {
        const int valid_groups = imin(GB, kGroups - cb * GB);
        const rsrc_t rs_w = make_rsrc(reinterpret_cast<const unsigned char*>(weights) +
                                          (long long)cb * GB * (8 * kR * kS * 16),
                                      valid_groups * (8 * kR * kS * 16));
#pragma unroll
        for (int l = 0; l < FLT; ++l) {
            Pack16 v;  // units past the workgroup's groups lie beyond the descriptor: zeros
            v.i = __builtin_amdgcn_raw_buffer_load_b128(rs_w, (tid + THREADS * l) * 16, 0, 0);
            fpre[l] = v.u;
        }
    }
    __builtin_amdgcn_sched_barrier(0);  // keep the filter loads ahead of the row loads
    spio_half8 wfrag[kR][KB];

    // ---- lane roles ----
    // weight gradient (transposing reads): block kb = lane/16 covers pixels 8*kb..8*kb+7, source
    // lane 4*jr + t supplies pixel jr (+4 for the second read) of unit t/2 (dy: shift j, x: tap offset
    // 2 sj) and channel half t%2.
    const int kb = lane >> 4;
    const int jr = (lane & 15) >> 2;
    const int tt = lane & 3;
    const int sel = tt >> 1;
    const int xfrag_off = (wg * GSX + pos(8 * kb + jr + 2 * sel, HX)) * 16 + (tt & 1) * 8;
    const int dfrag_off = (wg * GSD + pos(DL - 1 + 8 * kb + jr + sel, HD)) * 16 + (tt & 1) * 8;
    // data gradient: D[m = 4*(lane/16)+i][n = lane%16]: pixel 2 n + out_j of the tile, channels
    // 4*((lane/16)&1) + i
    const int sfrag_unit = wg * GSD + (lane & 15) + pos(DO + kb, HD);
    const int out_off = (lane >> 5) * OPLANE + (lane & 15) * OSTRIDE + wg * 16 + ((lane >> 4) & 1) * 8;

    spio_float4 acc[kR][NB4];  // weight gradient
#pragma unroll
    for (int r = 0; r < kR; ++r)
#pragma unroll
        for (int nb = 0; nb < NB4; ++nb) acc[r][nb] = spio_float4{0.f, 0.f, 0.f, 0.f};
    spio_float4 accb = spio_float4{0.f, 0.f, 0.f, 0.f};  // bias gradient
    const spio_half8 ones8 = spio_half8{1, 1, 1, 1, 1, 1, 1, 1};
    (void)ones8;

    const spio_uint4 zero4 = spio_uint4{0u, 0u, 0u, 0u};
    const rsrc_t rs_none = make_rsrc(x, 0);  // nothing is in range: loads give zeros, stores vanish

    for (int it = 0; it < ITERS; ++it) {
        const int n0 = (nbk * ITERS + it) * NB;
        if (n0 >= kN) break;

        // ---- buffer descriptors of this image block; images past the end of the batch lie
        //      beyond their size ----
        const int images = imin(NB, kN - n0);
        const rsrc_t rs_x = make_rsrc(reinterpret_cast<const unsigned char*>(x) + n0 * X_IMAGE_BYTES,
                                      (int)(images * X_IMAGE_BYTES));
        const rsrc_t rs_dy = make_rsrc(reinterpret_cast<const unsigned char*>(dy) + n0 * D_IMAGE_BYTES,
                                       (int)(images * D_IMAGE_BYTES));
        const rsrc_t rs_dx = make_rsrc(reinterpret_cast<const unsigned char*>(grad_input) + n0 * DX_IMAGE_BYTES,
                                       (int)(images * DX_IMAGE_BYTES));

        // ---- loop-invariant addressing (cells without data carry the out-of-range offset: they
        //      load zeros, which is what halo and gap cells must hold) ----
        unsigned x_voff[LPTX];
        int x_lds[LPTX];
#pragma unroll
        for (int l = 0; l < LPTX; ++l) {
            const int cell = tid + THREADS * l;
            x_voff[l] = OOB;
            x_lds[l] = XDUMP;
            if (cell < X_CELLS) {
                const int g = cell % GB;
                const int f = cell / GB;
                const int img = f / WPI;
                const int col = q0 + f % WPI - PL - XOX;  // column of x
                x_lds[l] = g * GSX + pos(f, HX);
                if (col >= 0 && col < kW && cb * GB + g < kGroups)
                    x_voff[l] = (unsigned)(((img * kH * kW + col) * kGroups + cb * GB + g) * 16);
            }
        }
        // dy cells, and the dx cells of the same (image, domain column, group): where dy and x have
        // the same size, the same offset
        int d_voff[LPTD][kSrcLoads], d_lds[LPTD][kSrcLoads];  // (SPIO_SRC_F32: d_lds in bytes)
        unsigned o_voff[LPTO][kDstStores];
        int o_lds[LPTO][kDstStores];
#pragma unroll
        for (int l = 0; l < LPTD; ++l) {
#pragma unroll
            for (int j = 0; j < kSrcLoads; ++j) {
                const int cell = moved_unit(tid, j, kSrcLoads) + THREADS * l;
                unsigned voff = OOB;
                int unit = DDUMP;
                if (cell < D_CELLS) {
                    const int g = cell % GB;
                    // whole rows: the cells are the real columns; column blocks: every staged column
                    const int q = kColBlocks ? q0 + (cell / GB) % WPI - PR : (cell / GB) % DW;  // domain column
                    const int img = kColBlocks ? 0 : cell / (GB * DW);
                    unit = g * GSD + pos(kColBlocks ? cell / GB + DO : img * WPI + q + DL, HD);
                    const int qd = q - DOX;  // column of dy
                    if (qd >= 0 && qd < kQ && cb * GB + g < kGroups)
                        voff = (unsigned)(((img * kP * kQ + qd) * kGroups + cb * GB + g) * (8 * kSrcBytes));
                }
                d_voff[l][j] = (int)(voff + (unsigned)half_bytes(tid, kSrcLoads, 16));
                d_lds[l][j] = SPIO_SRC_F32 ? unit * 16 + half_bytes(tid, kSrcLoads, 8) : unit;
            }
        }
#pragma unroll
        for (int l = 0; l < LPTO; ++l) {
#pragma unroll
            for (int j = 0; j < kDstStores; ++j) {
                const int cell = moved_unit(tid, j, kDstStores) + THREADS * l;
                unsigned voff = OOB;
                int from = 0;
                if (cell < O_CELLS) {
                    const int g = cell % GB;
                    const int q = (cell / GB) % BQ;
                    const int img = cell / (GB * BQ);
                    const int o = img * WPI + q;
                    from = (o & 1) * OPLANE + (o >> 1) * OSTRIDE + g * 16;
                    const int wx = q0 + q - XOX;  // column of dx
                    if (q0 + q < DW && wx >= 0 && wx < kW && cb * GB + g < kGroups)
                        voff = (unsigned)(((img * kH * kW + wx) * kGroups + cb * GB + g) * (8 * kDstBytes));
                }
                o_voff[l][j] = voff + (unsigned)half_bytes(tid, kDstStores, 16);
                o_lds[l][j] = from + half_bytes(tid, kDstStores, 8);
            }
        }

        // Rows `t` of x (domain row p0-(R-1)+t) and of dy (p0-PB+t) for every cell of the thread.
        // Rows the block does not need, and domain rows outside the tensor, read through the empty
        // descriptor (zeros, no traffic).
        auto load_rows = [&](spio_uint4(&xr)[LPTX], spio_uint4(&dr)[LPTD][kSrcLoads], int t) {
            const int h = p0 - (kR - 1) + t;
            const rsrc_t rx = (h >= xrow_lo && h <= xrow_hi && h >= XOY && h < XOY + kH) ? rs_x : rs_none;
            const int sx = __builtin_amdgcn_readfirstlane(imin(imax(h - XOY, 0), kH - 1) * X_ROW_BYTES);
            const bool xhalo = h < p0 || h >= p0 + bh_eff;
#pragma unroll
            for (int l = 0; l < LPTX; ++l) {
                Pack16 v;
                v.i = (SPIO_HALO_CACHED && xhalo) ? __builtin_amdgcn_raw_buffer_load_b128(rx, (int)x_voff[l], sx, 0)
                                                  : __builtin_amdgcn_raw_buffer_load_b128(rx, (int)x_voff[l], sx, AUX_LD);
                xr[l] = v.u;
            }
            const int pr = p0 - PB + t;
            const rsrc_t rd = (pr >= drow_lo && pr <= drow_hi && pr >= DOY && pr < DOY + kP) ? rs_dy : rs_none;
            const int sd = __builtin_amdgcn_readfirstlane(imin(imax(pr - DOY, 0), kP - 1) * D_ROW_BYTES);
            const bool dhalo = pr < p0 || pr >= p0 + bh_eff;
#pragma unroll
            for (int l = 0; l < LPTD; ++l) {
#pragma unroll
                for (int j = 0; j < kSrcLoads; ++j) {
                    Pack16 v;
                    v.i = (SPIO_HALO_CACHED && dhalo) ? __builtin_amdgcn_raw_buffer_load_b128(rd, d_voff[l][j], sd, 0)
                                                      : __builtin_amdgcn_raw_buffer_load_b128(rd, d_voff[l][j], sd, AUX_LD);
                    dr[l][j] = v.u;
                }
            }
        };
        auto dy_to_ring = [&](const spio_uint4(&dr)[LPTD][kSrcLoads], int slot) {
            spio_uint4* const row = dring + slot * DROW_UNITS;
#pragma unroll
            for (int l = 0; l < LPTD; ++l) {
                if (!SPIO_SRC_F32) {
                    row[d_lds[l][0]] = dr[l][0];
                } else {
#pragma unroll
                    for (int j = 0; j < kSrcLoads; ++j)
                        *reinterpret_cast<spio_uint2*>(reinterpret_cast<unsigned char*>(row) + d_lds[l][j]) = narrow(dr[l][j]);
                }
            }
        };

        // ---- prologue: rows 0..PF-1 into registers ----
        spio_uint4 xpre[PF][LPTX], dpre[PF][LPTD][kSrcLoads];
#pragma unroll
        for (int t = 0; t < PF; ++t) load_rows(xpre[t], dpre[t], t);
        __builtin_amdgcn_sched_barrier(0);  // the first loads are on their way before anything waits
        if (it == 0) {
            // while the first loads are in flight: the filter fragments, through the LDS block
            // the rings will use ...
#pragma unroll
            for (int l = 0; l < FLT; ++l)
                if (tid + THREADS * l < FILTER_UNITS) lds[tid + THREADS * l] = fpre[l];
            block_sync();
            const int fkb = lane >> 4;
            const int fjr = (lane & 15) >> 2;
            const int ft4 = lane & 3;
            const int src_slot = ft4 >> 1;
            const int my_slot = (lane & 15) >> 3;
            typedef spio_short4 __attribute__((address_space(3))) * lds_ptr;
#pragma unroll
            for (int r = 0; r < kR; ++r) {
#pragma unroll
                for (int u = 0; u < KB; ++u) {
                    const int s_src = 4 * u + fkb - src_slot;
                    const int s_mine = 4 * u + fkb - my_slot;
                    const int rr = kR - 1 - r;
                    const int ss = s_src >= 0 && s_src < kS ? kS - 1 - s_src : 0;  // dead taps: any valid address
                    const unsigned char* base = reinterpret_cast<const unsigned char*>(lds) +
                                                ((((wg * 8 + fjr) * kR + rr) * kS + ss) * 16) + (ft4 & 1) * 8;
                    union {
                        spio_short4 q[2];
                        spio_half8 h;
                    } v;
                    v.q[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)base);
                    v.q[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(base + 4 * kR * kS * 16));
                    if (!(wave_active && s_mine >= 0 && s_mine < kS)) v.h = spio_half8{0, 0, 0, 0, 0, 0, 0, 0};
                    wfrag[r][u] = v.h;
                }
            }
            block_sync();  // everyone has its fragments before the rings are zero-filled
            // ... and both rings zeroed once: the slack cells behind each group's pixels are
            // never written
            for (int i = tid; i < RING_UNITS; i += THREADS) lds[i] = zero4;
        }
        block_sync();  // rings zeroed / previous image block finished
#pragma unroll
        for (int l = 0; l < LPTX; ++l) xring[x_lds[l]] = xpre[0][l];
        dy_to_ring(dpre[0], 0);
        block_sync();

        // Data gradient: dy row t reaches dx rows t - r (named by the step that completes them, less R-1);
        // each has one slot of sums, t - r modulo R, from its first dy row (r = 0) to its last.
        spio_float4 dacc[TPW][kR];
        // Weight gradient: fragments of the last R dy rows, row t in slot t modulo R.  They are read once, when
        // the row is the newest; rows the block does not own (halo, past the image) count as zero.
        spio_half8 afrag[kR][CPW];
#pragma unroll
        for (int r = 0; r < kR; ++r) {
#pragma unroll
            for (int i = 0; i < TPW; ++i) dacc[i][r] = spio_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ci = 0; ci < CPW; ++ci) afrag[r][ci] = spio_half8{0, 0, 0, 0, 0, 0, 0, 0};
        }

        // A finished dx row, from sums `slot` into the output stage.
        auto stage_dx_row = [&](int slot, int obuf) {
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
                Pack8 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o.h[e] = (spio_half)dacc[i][slot][e];
                *reinterpret_cast<spio_uint2*>(ostage + obuf * OUT_ROW_BYTES + 16 * (TPW * ws + i) * OSTRIDE + out_off) = o.u;
            }
        };
        // Coalesced store of the dx row that received its last tap at step `ts` (domain row p0 - (R-1) + ts), one step
        // after it was staged.  Steps that finish no row of the block, or a domain row outside dx, store through
        // the empty descriptor: the
        // instructions are issued all the same and the hardware drops them.
        auto store_dx_row = [&](int ts, int obuf) {
            const int h = p0 - (kR - 1) + ts;
            const bool real = ts >= kR - 1 && ts < kR - 1 + bh_eff && h >= XOY && h < XOY + kH;
            const rsrc_t rs = real ? rs_dx : rs_none;
            // The row offset is added to the per-lane offset; the scalar-offset operand stays the
            // constant 0.  A 16-byte buffer store reads its data registers for a few cycles after
            // it issues, and only for the constant form does the compiler keep the next
            // instructions from writing them: with the row offset in a scalar register a result
            // moved into the first data register right behind the store was stored in its place
            // (seen on gfx950 as stray values in the first two channels of some pixels).
            const unsigned row_off = (unsigned)(imin(imax(h - XOY, 0), kH - 1) * DX_ROW_BYTES);
#pragma unroll
            for (int l = 0; l < LPTO; ++l) {
                const unsigned char* row = ostage + obuf * OUT_ROW_BYTES;
#pragma unroll
                for (int j = 0; j < kDstStores; ++j) {
                    Pack16 v;
                    v.u = SPIO_DST_F32 ? widen(*reinterpret_cast<const spio_uint2*>(row + o_lds[l][j]))
                                       : *reinterpret_cast<const spio_uint4*>(row + o_lds[l][j]);
                    __builtin_amdgcn_raw_buffer_store_b128(v.i, rs, (int)(o_voff[l][j] + row_off), 0, AUX_ST);
                }
            }
            store_group_end();
        };

        for (int tb = 0; tb < ROWS; tb += UNROLL) {
#pragma unroll
            for (int uu = 0; uu < UNROLL; ++uu) {
                const int t = tb + uu;
                if (t >= ROWS) continue;  // (with a second way out of the loop the compiler leaves 12 steps rolled)
                const int sp = uu & 1;                   // parity of t: ring rows
                const int pbuf = uu % PF;                // register buffer that held row t
                const int ph = uu % kR;                  // t mod R
                // what the step has to do, known at compile time in an unrolled loop: dy rows are named by
                // the step that staged them (row p0-PB+tau at step tau; the block owns tau in [PB, PB+bh_eff)),
                // x row t (p0-(R-1)+t) meets dy rows t - r under filter row r, dy row t reaches the dx rows
                // that complete at steps t .. t+R-1
                const bool multiply_x = !kFullUnroll || t >= PB;
                const bool read_dy = !kFullUnroll || (t >= PB && t < PB + BH);
                const bool multiply_dy = !kFullUnroll || t < BH + kR - 1;

                // 1. fragment reads
                spio_half8 bfrag[CPW][NB4];
#pragma unroll
                for (int ci = 0; ci < CPW; ++ci) {
                    const int ch = CPW * ws + ci;
                    if (multiply_x) {
                        const unsigned char* xrow =
                            reinterpret_cast<const unsigned char*>(xring + sp * XROW_UNITS) + xfrag_off;
#pragma unroll
                        for (int nb = 0; nb < NB4; ++nb) {
                            const unsigned char* pb0 = xrow + (16 * ch + 2 * nb) * 16;
                            bfrag[ci][nb] = read_tr_pair(pb0, pb0 + 2 * 16);
                        }
                    }
                    if (read_dy) {
                        const unsigned char* pa0 = reinterpret_cast<const unsigned char*>(dring + sp * DROW_UNITS) +
                                                   dfrag_off + (16 * ch) * 16;
                        spio_half8 a = read_tr_pair(pa0, pa0 + 2 * 16);
                        if (kColBlocks) {  // the block's own columns only (the lane holds row m = lane % 16)
                            const int q = 32 * ch + 8 * kb + ((lane & 15) >> 3) - 1;
#pragma unroll
                            for (int e = 0; e < 8; ++e)
                                if (q + e < 0 || q + e >= BQ) a[e] = 0;
                        }
                        if ((!kFullUnroll && t < PB) || ((!kFullUnroll || DH % BH != 0) && t >= PB + bh_eff))
                            a = spio_half8{0, 0, 0, 0, 0, 0, 0, 0};
                        afrag[ph][ci] = a;
                    }
                }
                spio_half8 sfrag[TPW][KB];
                if (multiply_dy) {
                    const spio_uint4* rrow = dring + sp * DROW_UNITS + sfrag_unit;
#pragma unroll
                    for (int i = 0; i < TPW; ++i) {
#pragma unroll
                        for (int u = 0; u < KB; ++u) {
                            Pack16 v;
                            v.u = rrow[16 * (TPW * ws + i) + 2 * u];
                            if (in_no_window(u, kb)) v.u = zero4;
                            sfrag[i][u] = v.h;
                        }
                    }
                }

                // 2. prefetch rows t+PF.  Rows past the end read through the empty descriptor in the
                //    chunked loop (every step then issues the same loads); the unrolled loop leaves
                //    them out.
                if (!kFullUnroll || t + PF < ROWS) load_rows(xpre[pbuf], dpre[pbuf], t + PF);

                // 3. the dx row staged in the previous step goes out, one that was finished then is staged
                if (kLateStage) {
                    if (!kFullUnroll || t - 2 >= kR - 1) store_dx_row(t - 2, uu & 1);
                    if (!kFullUnroll || (t - 1 >= kR - 1 && t - 1 < kR - 1 + BH)) stage_dx_row(ph, (uu + 1) & 1);
                } else {
                    if (!kFullUnroll || t - 1 >= kR - 1) store_dx_row(t - 1, (uu + 1) & 1);
                }

                // 4. rows t+1 into LDS, where nothing of this step reads (dy rows past the last one become zero)
                if (t + 1 < ROWS) {
#pragma unroll
                    for (int l = 0; l < LPTX; ++l)
                        xring[(sp ^ 1) * XROW_UNITS + x_lds[l]] = xpre[(uu + 1) % PF][l];
                    dy_to_ring(dpre[(uu + 1) % PF], sp ^ 1);
                }

                // 5. multiply: data gradient, dy row t into the dx rows that exist ...
                if (multiply_dy) {
#pragma unroll
                    for (int i = 0; i < TPW; ++i) {
#pragma unroll
                        for (int u = 0; u < KB; ++u) {
#pragma unroll
                            for (int r = 0; r < kR; ++r) {
                                if (kFullUnroll && (t - r < 0 || t - r >= BH)) continue;
                                spio_float4& d = dacc[i][pmod(ph - r, kR)];
                                const spio_float4 before = r == 0 && u == 0 ? spio_float4{0.f, 0.f, 0.f, 0.f} : d;
                                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(wfrag[r][u], sfrag[i][u], before, 0, 0, 0);
                            }
                        }
                    }
                }
                //    ... and weight gradient
                if (multiply_x) {
#pragma unroll
                    for (int ci = 0; ci < CPW; ++ci) {
#pragma unroll
                        for (int nb = 0; nb < NB4; ++nb) {
#pragma unroll
                            for (int r = 0; r < kR; ++r) {
                                if (kFullUnroll && (t - r < PB || t - r >= PB + BH)) continue;
                                acc[r][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                    afrag[pmod(ph - r, kR)][ci], bfrag[ci][nb], acc[r][nb], 0, 0, 0);
                            }
                        }
                        if (kDbias && read_dy)
                            accb = __builtin_amdgcn_mfma_f32_16x16x32_f16(afrag[ph][ci], ones8, accb, 0, 0, 0);
                    }
                }

                // 6. the dx row that received its last tap (row p0-(R-1)+t): stage it
                if (!kLateStage && (!kFullUnroll || (t >= kR - 1 && t < kR - 1 + BH)))
                    stage_dx_row(pmod(ph - (kR - 1), kR), uu & 1);
                block_sync();
            }
        }
        // the row staged in the last step and one finished in it (if they are real ones)
        if (kLateStage) {
            store_dx_row(ROWS - 2, ROWS & 1);
            if (PB == 0) {
                stage_dx_row(ROWS % kR, (ROWS - 1) & 1);
                block_sync();
            }
        }
        if (!kLateStage || PB == 0) store_dx_row(ROWS - 1, (ROWS - 1) & 1);
    }

    // ---- publish grad_weight (and grad_bias) ----
    // Sum m = 8 j + k, n = 8 sj + c of acc[r][nb] belongs to filter row r and column 4 nb + 2 sj + 1 - j.  Every
    // wave stages its R*S*64 sums in grad_weight order; the waves of a group share the way out (64
    // consecutive floats at a time), where the sums of the group's waves meet.
    block_sync();  // every wave is done with the rings and the output stage
    {
        float* const sums = reinterpret_cast<float*>(lds);
        float* const gstage = sums + wg * GROUP_FLOATS;  // of the group's first wave
        {
            const int c = lane & 7;
            const int k4 = 4 * ((lane >> 4) & 1);
            float* const mine = sums + wave * GROUP_FLOATS;
#pragma unroll
            for (int nb = 0; nb < NB4; ++nb) {
                const int s = 4 * nb + 2 * ((lane & 15) >> 3) + 1 - (lane >> 5);
                if (s < kS) {
#pragma unroll
                    for (int r = 0; r < kR; ++r)
#pragma unroll
                        for (int e = 0; e < 4; ++e) mine[(((k4 + e) * kR + r) * kS + s) * 8 + c] = acc[r][nb][e];
                }
            }
        }
        if (TS > 1)
            block_sync();
        else
            wave_sync();  // all lanes read what all lanes staged
        auto total = [&](int i) {
            float v = gstage[64 * i + lane];
#pragma unroll
            for (int w2 = 1; w2 < TS; ++w2) v += gstage[w2 * GB * GROUP_FLOATS + 64 * i + lane];
            return v;
        };
#if SPIO_PARTIALS
        // this workgroup's block of the workspace: [group][k][r][s][c], then [group][k] bias sums
        float* const pblock = grad_weight + ((long long)cb * NPART + (nbk * PBLKS + pb) * QBLKS + q0 / BQ) * PART_FLOATS;
        float* const gout = pblock + wg * GROUP_FLOATS;  // groups past the last one store their zeros: the block is read whole
#pragma unroll
        for (int i = ws; i < kR * kS; i += TS) __builtin_nontemporal_store(wave_active ? total(i) : 0.f, gout + 64 * i + lane);
#else
        if (wave_active) {
            float* const gout = grad_weight + (long long)gglob * GROUP_FLOATS;
#pragma unroll
            for (int i = ws; i < kR * kS; i += TS) atomic_add_f32(gout + 64 * i + lane, total(i));
        }
#endif
#if SPIO_HAS_BIAS
        {
            float* bslots = sums + WAVES * GROUP_FLOATS;  // [wave][8]
            if ((lane & 47) == 0) {
#pragma unroll
                for (int e = 0; e < 4; ++e) bslots[wave * 8 + (lane >> 4) * 4 + e] = wave_active ? accb[e] : 0.f;
            }
            block_sync();
#if SPIO_PARTIALS
            if (wave == 0) {
                for (int i = lane; i < GB * 8; i += 64) {
                    float v = 0.f;
#pragma unroll
                    for (int w2 = 0; w2 < TS; ++w2) v += bslots[(w2 * GB + i / 8) * 8 + (i & 7)];
                    pblock[GB * GROUP_FLOATS + i] = v;
                }
            }
#else
            if (wave == 0 && grad_bias != nullptr) {
                for (int i = lane; i < GB * 8; i += 64) {
                    float v = 0.f;
#pragma unroll
                    for (int w2 = 0; w2 < TS; ++w2) v += bslots[(w2 * GB + i / 8) * 8 + (i & 7)];
                    if (cb * GB + i / 8 < kGroups) atomic_add_f32(grad_bias + 8 * cb * GB + i, v);
                }
            }
#endif
        }
#endif
    }
}

#if SPIO_PARTIALS
// Second stage: grad_weight (and grad_bias) = sum over the workgroups' blocks.  A workgroup of
// 256 threads owns 8 float4 columns of one channel block (128 contiguous bytes of every block);
// its 32 slices each add the blocks p = slice, slice + 32, ... with up to 16 loads in flight, the
// slices are added through LDS and slice 0 stores the totals.  A block is laid out like the
// channel block's part of grad_weight, so column `col` of channel block `cb` is the float4 at
// grad_weight[cb * GB * GROUP_FLOATS + 4 * col]; the columns behind it are the bias sums.
template <class T>
SPIO_DEVICE void reduce_partials(T* __restrict__ grad_weight, const spio_float4* __restrict__ partials,
                                 float* __restrict__ grad_bias) {
    constexpr int BLOCK_F4 = PART_FLOATS / 4;  // float4 columns of one block
    constexpr int COLS = 8;
    constexpr int SLICES = 256 / COLS;
    constexpr int UN = NPART <= 8 * SLICES ? 8 : 16;
    constexpr int WGS_PER_CB = (BLOCK_F4 + COLS - 1) / COLS;
    __shared__ spio_float4 red[SLICES][COLS];
    const int tid = thread_id();
    const int cl = tid % COLS;
    const int slice = tid / COLS;
    const int cb = block_id() / WGS_PER_CB;
    const int col = (block_id() % WGS_PER_CB) * COLS + cl;
    const bool live = col < BLOCK_F4;
    const spio_float4* base = partials + (long long)cb * NPART * BLOCK_F4 + (live ? col : 0);
    spio_float4 sum = spio_float4{0.f, 0.f, 0.f, 0.f};
    for (int p0 = slice; p0 < NPART; p0 += SLICES * UN) {
        spio_float4 v[UN];
#pragma unroll
        for (int i = 0; i < UN; ++i) {
            const int p = p0 + i * SLICES;
            v[i] = spio_float4{0.f, 0.f, 0.f, 0.f};
            if (p < NPART) v[i] = __builtin_nontemporal_load(base + (long long)p * BLOCK_F4);
        }
#pragma unroll
        for (int i = 0; i < UN; ++i) sum += v[i];
    }
    red[slice][cl] = sum;
    block_sync();
    if (slice == 0 && live) {
#pragma unroll 4
        for (int i = 1; i < SLICES; ++i) sum += red[i][cl];
        const int f = 4 * col;  // float index inside the block
        if (f < GB * GROUP_FLOATS) {
            if (cb * GB + f / GROUP_FLOATS < kGroups)
                store_sums(grad_weight + (long long)cb * GB * GROUP_FLOATS + f, sum);
        } else if (grad_bias != nullptr) {
            const int k = cb * GB * 8 + (f - GB * GROUP_FLOATS);
            if (k < kC) *reinterpret_cast<spio_float4*>(grad_bias + k) = sum;
        }
    }
}
extern "C" __global__ void SPIO_LAUNCH_BOUNDS(256)
SPIO_CONCAT(SPIO_KERNEL_NAME, _reduce)(float* __restrict__ grad_weight, const spio_float4* __restrict__ partials,
                                       float* __restrict__ grad_bias) {
    reduce_partials(grad_weight, partials, grad_bias);
}
extern "C" __global__ void SPIO_LAUNCH_BOUNDS(256)
SPIO_CONCAT(SPIO_KERNEL_NAME, _reduce_h)(spio_half* __restrict__ grad_weight, const spio_float4* __restrict__ partials,
                                         float* __restrict__ grad_bias) {
    reduce_partials(grad_weight, partials, grad_bias);
}
#endif
