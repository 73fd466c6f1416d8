// Row-streaming MFMA kernel for the conv2d_gw8 weight gradient (gfx950).
//
// Contract (reference kernel: spio/src/conv2d_gw8_wgrad.cu:10-226):
//   dw[k,r,s,c] += sum_{n,p,q} x[n,p+r-py,q+s-px,8g+c] * dy[n,p,q,k]      g = k / 8
// fp16 operands, fp32 accumulation, fp32 result added into `grad_weight`
// ([K][R][S][8] floats) with atomics, so the caller zeroes it first
// (spio/functional/conv2d_gw8_function.py:124-130).
//
// Design
//   * A workgroup owns SPIO_BH rows of dy (output rows) of SPIO_NB images side
//     by side, for SPIO_GB channel groups, and repeats that for SPIO_ITERS
//     image blocks before it publishes its sums.  Per step it stages SPIO_RB
//     (1 or 2) rows of x and of dy in LDS ([group][flattened pixel][8 ch],
//     zero halo materialised once, as in the forward kernel).
//   * One wave owns one group.  The contraction runs over pixels, so both MFMA
//     operands need "8 pixels of one channel" per lane while memory holds
//     "8 channels of one pixel"; the transposing LDS read of gfx950
//     (ds_read_b64_tr_b16) delivers exactly that from the pixel-major rows.
//   * v_mfma_f32_16x16x32_f16 per 32-pixel chunk:
//         A (16 x 32) = dy:  rows m = 8*j + k    (the chunk, j pixels on; 8 k)
//         B (32 x 16) = x:   cols n = 8*sj + c   (the chunk under two column taps, 2 sj; 8 c)
//     so one MFMA yields dw for one filter row and the four filter columns 4 nb + 2 sj + 1 - j.  Both
//     operands begin one pixel before the row: over all chunks each of the two copies of dy counts every
//     pixel once.  x row t meets dy row t - r under filter row r: R * ceil(S/4) MFMAs per chunk and x row,
//     as many accumulators, and nothing to combine between lanes.
//   * A dy row is read from LDS once, when it is the newest, and its fragments stay in registers for the R
//     x rows that meet it.
//   * With two dy rows side by side in A, as before, there were (R+1) * ceil(S/2) accumulators (32 of a 7x7
//     filter, now 14), 4, 9, 16 MFMAs per chunk and x row for 3x3, 5x5, 7x7 (now 3, 10, 14), R/2 + 1 reads
//     of dy a step, and an exchange of halves through LDS at the end.  Before -> after, best of 24
//     configurations: 128n 64c 56x56 21.0 -> 20.3 us (103 MB, 5.1 TB/s), 32n 10.0 -> 9.0, 32n 48c 224x224 55.4 -> 51.4, 256n 256c
//     14x14 7x7 24.7 -> 21.0, 54n 688c 18x18 5x5 24.9 -> 20.9, 7n 392c 68x64 7x7 33.9 -> 25.5, 2n 56c 102x102 7x7 23.2 -> 11.4.
//   * At the end the sums are staged in LDS in grad_weight order. Two ways to
//     publish: SPIO_PARTIALS=0 adds into grad_weight with fp32 atomics.  Atomics
//     of different workgroups to the same 128-byte line retire one after the
//     other, so the sums are first staged in LDS in grad_weight order and then
//     added with instructions that cover 64 consecutive floats (two full
//     lines): the fewest line operations possible.  SPIO_PARTIALS=1 stores each
//     workgroup's sums into its own part of a partial image of a workspace with plain
//     stores, and the small <name>_reduce kernel below stores the sum of the
//     partial images into grad_weight (which then needs no zero fill).  (Reducing inside the kernel by "the last workgroup of
//     a group to finish" was measured and rejected: the device-scope
//     release/acquire fences it needs write back and invalidate the L2 of an
//     XCD and cost more than the atomics they save.)
//   * The row loads do not stop at the end of an image block: they run on into the next one while the last
//     rows of this one are multiplied, so that only a workgroup's first block waits a memory latency for its
//     first row.  A step (barrier, fragment reads, ring writes, MFMAs) takes about 0.4 us on a compute unit
//     whatever is in it, so what bounds small images is the number of steps of the longest workgroup: the host
//     deals equal shares.  Rows in the padding or past the block go through an empty descriptor and cost no
//     traffic; the clamped loads that stood here before fetched a real row for each, PF of them per image
//     block.  20n 1024c 27x27 5x5 48.6 -> 43.8 us, with equal shares (3 images instead of 8 and 2 blocks of two) 23.4;
//     77n 168c 20x20 7x7 32.5 -> 22.1, 300n 88c 17x17 5x5 30.1 -> 20.4, 184n 288c 31x31 3x3 45.0 -> 39.7.
//   * With SPIO_HAS_BIAS the kernel takes a fourth pointer, grad_bias ([K]
//     fp32, accumulated into like grad_weight; null = not wanted), and sums dy
//     per channel in the same pass: one more MFMA per chunk and row with
//     an all-ones B operand (the reference runs a separate reduction,
//     spio/functional/conv2d_gw8_function.py:134-136).
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
#ifndef SPIO_PARTIALS
#define SPIO_PARTIALS 0
#endif
#ifndef SPIO_BQ
#define SPIO_BQ 0
#endif
#ifndef SPIO_TS
#define SPIO_TS 1
#endif
#ifndef SPIO_RB
#define SPIO_RB 1
#endif
#ifndef SPIO_HAS_BIAS
#define SPIO_HAS_BIAS 0
#endif
#ifndef SPIO_PIPE
#define SPIO_PIPE 0
#endif
#ifndef SPIO_MAX_UNROLL
#define SPIO_MAX_UNROLL 64
#endif

namespace {

constexpr int GB = SPIO_GB;        // groups (waves) per workgroup
constexpr int BH = SPIO_BH;        // dy rows per workgroup
constexpr int NB = SPIO_NB;        // images side by side
constexpr int ITERS = SPIO_ITERS;  // image blocks per workgroup
constexpr int TS = SPIO_TS;        // waves sharing the 32-pixel chunks of one group
constexpr int WAVES = GB * TS;
constexpr int THREADS = 64 * WAVES;
constexpr int PF = SPIO_PF;  // prefetch distance in steps (even)
constexpr int RB = SPIO_RB;  // x rows (and dy rows) per step: 1 or 2

constexpr int NB4 = (kS + 3) / 4;  // column taps 4 nb .. 4 nb + 3 share one MFMA
// Column blocks (SPIO_BQ > 0): a workgroup sums over BQ columns of dy and the BQ + S - 1 columns
// of x opposite them, so rows of any width fit the rings (the reference tiles the width with a
// fixed block of 8 columns, spio/kernels/conv2d_gw8_wgrad_kernel.py:40).  0 = the whole width.
constexpr int BQ = SPIO_BQ > 0 ? SPIO_BQ : kQ;
constexpr int QBLKS = (kQ + BQ - 1) / BQ;
constexpr int WPI = BQ + kS - 1;  // x cells staged per image (block): W + 2*px for whole rows
constexpr int F = NB * WPI;
// Where the images of a staged row sit.  dy pixel q of image i lies at flattened pixel
// off(i) + q and meets, for column tap s, the x pixel at off(i) + q + s; x column c of image i
// lies at off(i) + c + px.  Between the data of two images GAP = max(px, S-1-px) zero cells are
// enough: the right halo of one image is the left halo of the next.  The contraction runs over
// 32-pixel chunks of the dy row; where a chunk holds IPC >= 1 whole images and that takes fewer
// chunks than the images laid end to end, every chunk gets its own IPC images (14x14 images
// under a 7x7 filter: two per chunk, 28 of 32 pixels, instead of four in three chunks), and the
// x row, whose pixels q + s reach S-1 cells past a chunk, is staged as chunks XCP cells apart.
#ifndef SPIO_SHARED_HALO
#define SPIO_SHARED_HALO 1
#endif
constexpr int GAP = kPadX > kS - 1 - kPadX ? kPadX : kS - 1 - kPadX;
constexpr int IP = (SPIO_BQ > 0 || !SPIO_SHARED_HALO) ? WPI : BQ + GAP;  // pitch of the images in a run
// A chunk begins one pixel before its first image: 31 of its pixels are the images'.
constexpr int IPC_MAX = (31 + IP - BQ) / IP;                             // whole images per 32-pixel chunk
constexpr int KC_FLAT = ((NB - 1) * IP + BQ + 1 + 31) / 32;
constexpr int KC_PACKED = IPC_MAX > 0 ? (NB + IPC_MAX - 1) / IPC_MAX : KC_FLAT;
constexpr bool kPacked = SPIO_SHARED_HALO && KC_PACKED < KC_FLAT;
constexpr int IPC = kPacked ? IPC_MAX : NB;  // images per run: a chunk, or the whole row
constexpr int KC = kPacked ? KC_PACKED : KC_FLAT;  // 32-pixel chunks
constexpr int CPW = (KC + TS - 1) / TS;            // 32-pixel chunks per wave (past the last one: zeros)
constexpr int XCP = kPacked ? 16 * ((32 + 4 * NB4 - 2 + 15) / 16) : 32;  // x cells from chunk to chunk
constexpr int FPX = kPacked ? CPW * TS * XCP : 32 * CPW * TS + 4 * NB4 - 2;  // x pixels the reads can touch
constexpr int GSX = FPX + ((9 - FPX % 16) + 16) % 16;  // x group stride (pixels), = 9 mod 16
constexpr int FPD = 32 * CPW * TS + 1;                 // dy pixels, the first one a zero
constexpr int GSD = FPD + ((9 - FPD % 16) + 16) % 16;  // dy group stride
constexpr int d_image_offset(int img) { return (img / IPC) * 32 + (img % IPC) * IP; }
constexpr int x_image_offset(int img) { return (img / IPC) * XCP + (img % IPC) * IP; }
// ring rows carry spare units behind the last group, which lanes without a cell write to, each its own
constexpr int DUMPS = 16;
constexpr int XROW_UNITS = GB * GSX + DUMPS;
constexpr int DROW_UNITS = GB * GSD + DUMPS;
constexpr int XDUMP = GB * GSX, DDUMP = GB * GSD;
constexpr int X_CELLS = F * GB;
constexpr int LPTX = (X_CELLS + THREADS - 1) / THREADS;
constexpr int D_CELLS = NB * BQ * GB;
constexpr int LPTD = (D_CELLS + THREADS - 1) / THREADS;
constexpr int GBLKS = (kGroups + GB - 1) / GB;
constexpr int PBLKS = (kP + BH - 1) / BH;
constexpr int NBLKS = (kN + NB * ITERS - 1) / (NB * ITERS);
constexpr int NUM_BLOCKS = GBLKS * PBLKS * QBLKS * NBLKS;
constexpr bool kDbias = SPIO_HAS_BIAS != 0;  // also sum grad_output per channel (grad_bias)
constexpr int ROWS = BH + kR - 1;  // x rows a workgroup streams
constexpr int STEPS = (ROWS + RB - 1) / RB;  // barrier-separated steps of RB rows
// A workgroup that owns whole images (one row block) knows at compile time which of its x rows
// lie in the padding: the steps before the first real row would only stage dy rows, the steps
// after the last one nothing at all.  It starts at the first step with a real x row, with the dy
// rows up to that step staged in the prologue, and stops after the last.  (A padding of R or more has dy rows
// that meet no x row at all; the bias sum wants them.)
constexpr bool kSkipPadding = PBLKS == 1 && kPadY < kR && (ROWS + RB - 1) / RB <= SPIO_MAX_UNROLL;
constexpr int T_FIRST = kSkipPadding ? kPadY : 0;
constexpr int T_END = kSkipPadding && kH + kPadY < ROWS ? kH + kPadY : ROWS;
constexpr int S0 = T_FIRST / RB;               // first step
constexpr int S1 = (T_END + RB - 1) / RB;      // one past the last step
constexpr int LEAD = S0 * RB;                  // dy rows staged ahead of the first step's own
// The step loop is unrolled completely up to SPIO_MAX_UNROLL steps (which rows a step multiplies is then known at
// compile time, and products that do not exist are left out); longer loops run in chunks that are whole rounds of
// the row buffers and of the dy fragments.
constexpr bool kFullUnroll = S1 - S0 <= SPIO_MAX_UNROLL;
constexpr int gcd_(int a, int b) { return b == 0 ? a : gcd_(b, a % b); }
constexpr int lcm_(int a, int b) { return a / gcd_(a, b) * b; }
constexpr int NA = kR + RB - 1 + (SPIO_PIPE ? RB : 0);  // dy rows whose fragments are kept
constexpr int ROUND = kFullUnroll ? PF : lcm_(PF, NA / gcd_(NA, RB));
constexpr int SLOTS = (S1 - S0 + ROUND - 1) / ROUND * ROUND;  // steps of an image block, rounded up to whole rounds
constexpr int UNROLL = kFullUnroll ? SLOTS : ROUND;
// x ring rows: the step's rows and the next step's; dy ring rows: those, and the ones staged ahead of the first
// step (a dy row is read once, when it is the newest, and its fragments stay in registers while x rows meet it)
constexpr int NRX = 2 * RB;
constexpr int NRD = LEAD + 2 * RB;

// LDS: the two rings while streaming; at the end the same block holds the reduction scratch:
// every group's R*S*64 sums in grad_weight order and eight grad_bias sums per wave.
constexpr int RING_UNITS = NRX * XROW_UNITS + NRD * DROW_UNITS;
constexpr int GROUP_FLOATS = kR * kS * 64;  // grad_weight values of one group
constexpr int PUBLISH_FLOATS = GB * GROUP_FLOATS + (SPIO_HAS_BIAS ? WAVES * 8 : 0);
constexpr int LDS_UNITS = RING_UNITS > (PUBLISH_FLOATS + 3) / 4 ? RING_UNITS : (PUBLISH_FLOATS + 3) / 4;
static_assert(LDS_UNITS * 16 <= 160 * 1024, "LDS overflow");
static_assert(PF >= 2 && PF % 2 == 0, "prefetch distance must be even");
static_assert(RB == 1 || RB == 2, "one or two rows per step");
// Two stages: the partial block of a workgroup is its groups' sums in grad_weight order.
// Two stages with a bias: behind the partial blocks, every workgroup's bias sums, [block][channel], zeros
// for channels past the last one.
constexpr long long BIAS_PARTIALS = (long long)NBLKS * PBLKS * QBLKS * GBLKS * GB * GROUP_FLOATS;


constexpr long long X_ROW_BYTES = (long long)kW * kGroups * 16, X_IMAGE_BYTES = kH * X_ROW_BYTES;
constexpr long long D_ROW_BYTES = (long long)kQ * kGroups * 16, D_IMAGE_BYTES = kP * D_ROW_BYTES;
// Whether a row is read through a descriptor that begins at it, or through one of its image block with the row
// in the lanes' offsets.  Unrolled loops know the row at compile time and take the former (20n 1024c 27x27 5x5
// 23.6 us, 28.6 with one of the block); in others it is 64-bit arithmetic for every
// row (64n 64c 56x56 16.1 us, 14.2 with one of the block; 32n 48c 224x224 66.0 and 55.7).  It is also the one for
// images that side by side exceed 32-bit offsets.
constexpr bool kRowDescriptors = (kFullUnroll && PBLKS == 1) || NB * X_IMAGE_BYTES >= (1ll << 31) || NB * D_IMAGE_BYTES >= (1ll << 31);
// What a row adds to the offsets of its lanes.  Rows above the image and behind it (padding, slots without a step)
// have one too, which may wrap around; their loads go through an empty descriptor, which no offset is inside of.
// (It is not the scalar offset, which the range check may leave out, and it is not clamped to rows that exist.  A
// macro, since the compiler folds a row's offset into the lanes' only where the product stands in the expression:
// 32n 48c 224x224 55.7 us, 66.1 with a clamp or a function.)
#define ROW_OFFSET(row, row_bytes) ((unsigned)(row) * (unsigned)(row_bytes))
static_assert((NB - 1) * X_IMAGE_BYTES + X_ROW_BYTES < (1ll << 31) && (NB - 1) * D_IMAGE_BYTES + D_ROW_BYTES < (1ll << 31),
              "a row of all images side by side lies within 32-bit buffer offsets");
// Images side by side in an unrolled loop, one block of them a workgroup: plain loads.  There is no next block to
// run on into and the rows that do not exist are known at compile time, so nothing is left that a descriptor is good
// for, and they are faster: 128n 128c 28x28 14.8 -> 13.0 us, 128n 384c 14x14 12.8 -> 11.8, 128n 192c 28x28 19.5 ->
// 18.4, 300n 88c 17x17 5x5 22.3 -> 20.4, 256n 256c 14x14 7x7 eight images 30.9 -> 27.6.  With one image it is the
// other way round (128n 64c 56x56 21.8 and 22.2, 256n 39.0 and 41.1), as in loops that are not unrolled (32n 64c
// 56x56 two images 10.7 and 11.0).
constexpr bool kPlainLoads = kFullUnroll && PBLKS == 1 && ITERS == 1 && NB > 1;
constexpr int OUT_OF_RANGE = (int)0x80000000u;  // as an unsigned offset behind the end of every descriptor
constexpr bool kSplitLines = splits_lines(GB, GBLKS);
// Non-temporal, but for lines that channel blocks straddle (blocks that are halves of whole lines: 64n 64c
// 56x56 14.3 us with the default policy, 13.7 non-temporal, 20n 1024c 27x27 5x5 25.6 and 23.7).
constexpr int AUX_LD = kSplitLines && kC % 64 != 0 ? 0 : 2;
typedef __amdgpu_buffer_rsrc_t rsrc_t;
SPIO_DEVICE rsrc_t make_rsrc(const void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}

SPIO_DEVICE spio_uint4 load_plain(const unsigned char* base, int off) {
    return load_stream(reinterpret_cast<const spio_uint4*>(base + (unsigned)off));
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
SPIO_KERNEL_NAME(float* __restrict__ grad_weight, const spio_uint4* __restrict__ x,
                 const spio_uint4* __restrict__ dy
#if SPIO_HAS_BIAS
                 , float* __restrict__ grad_bias  // [K] fp32, accumulated into; null = not wanted
#endif
) {
    // One LDS block: the x ring, then the dy ring; reused as reduction scratch at the end.
    __shared__ spio_uint4 lds[LDS_UNITS];
    spio_uint4* const xring = lds;
    spio_uint4* const dring = lds + NRX * XROW_UNITS;

    const int tid = thread_id();
    const int lane = tid & 63;
    // the wave index as a scalar: conditions on it become scalar branches, so that no MFMA
    // (which ignores the lane mask) is ever issued under an empty mask
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wg = TS == 1 ? wave : wave % GB;  // group within the workgroup
    const int ws = TS == 1 ? 0 : wave / GB;  // which share of the 32-pixel chunks this wave multiplies

    // One contiguous range of tiles per XCD; column blocks fastest (neighbours share S - 1 columns of x),
    // then row blocks.  Where channel blocks share lines they go fastest, so that the lines are fetched
    // from memory once.
    const int b = xcd_tile<0, NUM_BLOCKS>(block_id());
    constexpr int TILES = QBLKS * PBLKS;
    const int tile = kSplitLines ? (b / GBLKS) % TILES : b % TILES;
    const int cb = kSplitLines ? b % GBLKS : (b / TILES) % GBLKS;
    const int nbk = b / (TILES * GBLKS);
    const int qb = tile % QBLKS;
    const int q0 = qb * BQ;
    const int pb = PBLKS == 1 ? 0 : tile / QBLKS;
    const int p0 = pb * BH;
    const int bh_eff = imin(BH, kP - p0);  // dy rows that exist in this block
    const int gglob = cb * GB + wg;
    const bool wave_active = gglob < kGroups;

    // lane roles inside the transposing reads: block kb = lane/16 covers pixels 8*kb..8*kb+7,
    // source lane sigma = lane%16 = 4*jr + t supplies pixel jr (+4 for the second read) of
    // unit t/2 (dy: shift j, x: tap offset 2 sj) and channel half t%2.
    const int kb = lane >> 4;
    const int jr = (lane & 15) >> 2;
    const int tt = lane & 3;
    const int sel = tt >> 1;
    const int xfrag_off = ((wg * GSX + 8 * kb + jr + 2 * sel) * 16) + (tt & 1) * 8;  // bytes in an x row
    const int dfrag_off = ((wg * GSD + 8 * kb + jr + sel) * 16) + (tt & 1) * 8;      // bytes in a dy row

    spio_float4 acc[kR][NB4];
#pragma unroll
    for (int r = 0; r < kR; ++r)
#pragma unroll
        for (int nb = 0; nb < NB4; ++nb) acc[r][nb] = spio_float4{0.f, 0.f, 0.f, 0.f};

    // grad_bias rides along as one more MFMA per dy row and chunk: dy (A) times an all-ones B
    // gives, in every column, the sum of the 32 pixels for the 16 (shift, channel) rows.
    spio_float4 accb = spio_float4{0.f, 0.f, 0.f, 0.f};
    const spio_half8 ones8 = spio_half8{1, 1, 1, 1, 1, 1, 1, 1};
    (void)ones8;
    // ---- addressing ----
    // Every thread issues the same loads in every slot, without branches, so that the compiler counts
    // outstanding loads exactly and a step waits only for the rows it needs (a load under a branch makes it
    // wait for all of them, which would serialise the prefetch).  The images are read
    // through a buffer descriptor that ends with the last image that exists; lanes without data (halo columns, missing groups) carry an offset no descriptor reaches,
    // and a row that nobody needs has an empty one: such loads give zeros and touch no memory.
    const int nfirst = nbk * ITERS * NB;  // the workgroup's first image
    // (Plain loads: lanes without data load the first pixel of a row and write it to a spare unit.)
    constexpr int NO_DATA = kPlainLoads ? 0 : OUT_OF_RANGE;
    int x_off[LPTX], x_lds[LPTX];
#pragma unroll
    for (int l = 0; l < LPTX; ++l) {
        const int cell = tid + THREADS * l;
        x_off[l] = NO_DATA;
        x_lds[l] = XDUMP + tid % DUMPS;
        if (cell < X_CELLS) {
            const int g = cell % GB;
            const int f = cell / GB;
            const int img = f / WPI;
            const int col = q0 + f % WPI - kPadX;
            x_lds[l] = g * GSX + x_image_offset(img) + f % WPI;
            if (col >= 0 && col < kW && cb * GB + g < kGroups && (!kPlainLoads || nfirst + img < kN))
                x_off[l] = (int)(img * X_IMAGE_BYTES) + (col * kGroups + cb * GB + g) * 16;
            else if (kPlainLoads)
                x_lds[l] = XDUMP + tid % DUMPS;
        }
    }
    int d_off[LPTD], d_lds[LPTD];
#pragma unroll
    for (int l = 0; l < LPTD; ++l) {
        const int cell = tid + THREADS * l;
        d_off[l] = NO_DATA;
        d_lds[l] = DDUMP + tid % DUMPS;
        if (cell < D_CELLS) {
            const int g = cell % GB;
            const int q = (cell / GB) % BQ;
            const int img = cell / (GB * BQ);
            d_lds[l] = g * GSD + 1 + d_image_offset(img) + q;
            if (q0 + q < kQ && cb * GB + g < kGroups && (!kPlainLoads || nfirst + img < kN))
                d_off[l] = (int)(img * D_IMAGE_BYTES) + ((q0 + q) * kGroups + cb * GB + g) * 16;
            else if (kPlainLoads)
                d_lds[l] = DDUMP + tid % DUMPS;
        }
    }
    const spio_uint4 zero4 = spio_uint4{0u, 0u, 0u, 0u};

    // Row t of the current image block (ahead = 0) or of the next one (1).
    const unsigned char* xbase[2] = {};
    const unsigned char* dbase[2] = {};
    int images[2] = {};
    auto enter_block = [&](int it) {
#pragma unroll
        for (int ahead = 0; ahead < (ITERS > 1 ? 2 : 1); ++ahead) {
            const int n0 = nfirst + (it + ahead) * NB;
            images[ahead] = it + ahead < ITERS ? imin(imax(kN - n0, 0), NB) : 0;
            xbase[ahead] = reinterpret_cast<const unsigned char*>(x) + (images[ahead] > 0 ? n0 : 0) * X_IMAGE_BYTES;
            dbase[ahead] = reinterpret_cast<const unsigned char*>(dy) + (images[ahead] > 0 ? n0 : 0) * D_IMAGE_BYTES;
        }
    };
    auto load_x = [&](int ahead, int t, spio_uint4(&v)[LPTX]) {
        const int h = p0 + t - kPadY;
        if (kPlainLoads) {  // (the loop is unrolled: h is known)
#pragma unroll
            for (int l = 0; l < LPTX; ++l)
                v[l] = t < ROWS && h >= 0 && h < kH ? load_plain(xbase[0] + h * X_ROW_BYTES, x_off[l]) : zero4;
            return;
        }
        const int n = t < ROWS && h >= 0 && h < kH ? images[ahead] : 0;
        const rsrc_t rs = kRowDescriptors ? make_rsrc(xbase[ahead] + (n > 0 ? h : 0) * X_ROW_BYTES,
                                                   n > 0 ? (int)((n - 1) * X_IMAGE_BYTES + X_ROW_BYTES) : 0)
                                       : make_rsrc(xbase[ahead], (int)(n * X_IMAGE_BYTES));
        const unsigned row = kRowDescriptors ? 0u : ROW_OFFSET(h, X_ROW_BYTES);
#pragma unroll
        for (int l = 0; l < LPTX; ++l)
            v[l] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)((unsigned)x_off[l] + row), 0, AUX_LD);
    };
    auto load_dy = [&](int ahead, int t, spio_uint4(&v)[LPTD]) {
        if (kPlainLoads) {
#pragma unroll
            for (int l = 0; l < LPTD; ++l) v[l] = t < bh_eff ? load_plain(dbase[0] + t * D_ROW_BYTES, d_off[l]) : zero4;
            return;
        }
        const int n = t < bh_eff ? images[ahead] : 0;
        const rsrc_t rs = kRowDescriptors ? make_rsrc(dbase[ahead] + (n > 0 ? p0 + t : 0) * D_ROW_BYTES,
                                                   n > 0 ? (int)((n - 1) * D_IMAGE_BYTES + D_ROW_BYTES) : 0)
                                       : make_rsrc(dbase[ahead], (int)(n * D_IMAGE_BYTES));
        const unsigned row = kRowDescriptors ? 0u : ROW_OFFSET(p0 + t, D_ROW_BYTES);
#pragma unroll
        for (int l = 0; l < LPTD; ++l)
            v[l] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)((unsigned)d_off[l] + row), 0, AUX_LD);
    };
    // The loads run PF slots ahead of the steps and straight on into the next image block: step S0 + i is slot
    // i, and SLOTS, a multiple of PF, holds an image block, so that the register buffer of a slot is known at
    // compile time.
    spio_uint4 xpre[PF][RB][LPTX], dpre[PF][RB][LPTD];
    spio_uint4 dlead[LEAD > 0 ? LEAD : 1][LPTD];
    auto load_slot = [&](int ahead, int slot, int buffer) {
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) {
            if (kFullUnroll && slot >= S1 - S0) continue;
            const int t = slot < S1 - S0 ? (S0 + slot) * RB + rr : ROWS + BH;  // a slot without a step: no rows
            load_x(ahead, t, xpre[buffer][rr]);
            load_dy(ahead, t, dpre[buffer][rr]);
        }
    };
    auto load_lead = [&](int ahead) {
#pragma unroll
        for (int i = 0; i < LEAD; ++i) load_dy(ahead, i, dlead[i]);
    };
    enter_block(0);
    load_lead(0);
#pragma unroll
    for (int slot = 0; slot < PF; ++slot) {
        load_slot(0, slot, slot);
        // in the order they are needed: loads return in order, and with the first slot's requested last the
        // first step waits for all of them (20n 1024c 27x27 5x5 25.3 us, 23.6 in order)
        __builtin_amdgcn_sched_barrier(0);
    }
    // zero both rings once, while the first loads are in flight: halo, gap and slack cells are never
    // written again
    for (int i = tid; i < NRX * XROW_UNITS; i += THREADS) xring[i] = zero4;
    for (int i = tid; i < NRD * DROW_UNITS; i += THREADS) dring[i] = zero4;
    block_sync();

    for (int it = 0; it < ITERS; ++it) {
        if (nfirst + it * NB >= kN) break;
        if (it > 0) enter_block(it);

        // ---- step S0 and the dy rows before it into LDS (every step ends with a barrier: the rings are free) ----
#pragma unroll
        for (int i = 0; i < LEAD; ++i) {
#pragma unroll
            for (int l = 0; l < LPTD; ++l)
                dring[(i % NRD) * DROW_UNITS + d_lds[l]] = dlead[i][l];
        }
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) {
            const int t = S0 * RB + rr;
#pragma unroll
            for (int l = 0; l < LPTX; ++l)
                xring[((S0 & 1) * RB + rr) * XROW_UNITS + x_lds[l]] = xpre[0][rr][l];
#pragma unroll
            for (int l = 0; l < LPTD; ++l)
                dring[(t % NRD) * DROW_UNITS + d_lds[l]] = dpre[0][rr][l];
        }
        block_sync();

        // Fragments: of the x rows of a step (and, with SPIO_PIPE, of the step before), and of the last NA dy
        // rows, row t in slot t modulo NA.  dy rows past the block are zeros, so are the ones before it.
        constexpr int FSETS = SPIO_PIPE ? 2 : 1;
        spio_half8 bfrag[FSETS][RB][CPW][NB4], afrag[NA][CPW];
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int ci = 0; ci < CPW; ++ci) afrag[a][ci] = spio_half8{0, 0, 0, 0, 0, 0, 0, 0};
        auto read_dy = [&](int t, int a, int ci) {
            const unsigned char* pa0 = reinterpret_cast<const unsigned char*>(dring + t % NRD * DROW_UNITS) + dfrag_off +
                                       (32 * (CPW * ws + ci)) * 16;
            afrag[a][ci] = read_tr_pair(pa0, pa0 + 4 * 16);
        };
        auto sum_bias = [&](int a, int ci) {
            if (kDbias) accb = __builtin_amdgcn_mfma_f32_16x16x32_f16(afrag[a][ci], ones8, accb, 0, 0, 0);
        };
        // x row t (row p0 + t - py) meets dy row t - r under filter row r
        auto x_exists = [&](int t) {
            return !kFullUnroll || (t < ROWS && (PBLKS > 1 || (t - kPadY >= 0 && t - kPadY < kH)));
        };
        // Share (rr, ci) of the fragment reads of step `st`, and of its products; `ta`: slot of dy row st * RB.
        auto read_share = [&](int st, int sp, int ta, int rr, int ci, int fs) {
            const int t = st * RB + rr;
            if (x_exists(t)) {
                const unsigned char* xrow =
                    reinterpret_cast<const unsigned char*>(xring + (sp * RB + rr) * XROW_UNITS) + xfrag_off;
#pragma unroll
                for (int nb = 0; nb < NB4; ++nb) {
                    const unsigned char* pb0 = xrow + (XCP * (CPW * ws + ci) + 4 * nb) * 16;
                    bfrag[fs][rr][ci][nb] = read_tr_pair(pb0, pb0 + 4 * 16);
                }
            }
            if (!kFullUnroll || t < BH) read_dy(t, (ta + rr) % NA, ci);
        };
        auto multiply_share = [&](int st, int ta, int rr, int ci, int fs) {
            const int t = st * RB + rr;
            if (!kFullUnroll || t < BH) sum_bias((ta + rr) % NA, ci);
            if (!x_exists(t)) return;
#pragma unroll
            for (int nb = 0; nb < NB4; ++nb) {
#pragma unroll
                for (int r = 0; r < kR; ++r) {
                    if (kFullUnroll && (t - r < 0 || t - r >= BH)) continue;
                    acc[r][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(afrag[(ta + rr - r + 2 * NA) % NA][ci],
                                                                        bfrag[fs][rr][ci][nb], acc[r][nb], 0, 0, 0);
                }
            }
        };
#pragma unroll
        for (int i = 0; i < (LEAD < BH ? LEAD : BH); ++i)
#pragma unroll
            for (int ci = 0; ci < CPW; ++ci) {
                read_dy(i, i % NA, ci);
                sum_bias(i % NA, ci);
            }
        // 2. the slot PF ahead: its register buffer held this slot's rows, now in LDS
        auto prefetch_rows = [&](int slot, int uf) {
            const bool next = slot + PF >= SLOTS;
            const int ahead = next ? slot + PF - SLOTS : slot + PF;
            if (LEAD > 0 && ITERS > 1 && next && ahead == 0) load_lead(1);  // (the loop is unrolled)
            if (ITERS > 1)
                load_slot(next, ahead, uf % PF);
            else if (!kFullUnroll || !next)
                load_slot(0, slot + PF, uf % PF);
        };
        // 3. the rows of step st+1 into LDS (rows that do not exist are zeros), where nothing of this step reads
        auto stage_x = [&](int st, int sp, int uf) {
            if (st + 1 >= S1) return;
#pragma unroll
            for (int rr = 0; rr < RB; ++rr) {
#pragma unroll
                for (int l = 0; l < LPTX; ++l)
                    xring[(((sp + 1) & 1) * RB + rr) * XROW_UNITS + x_lds[l]] = xpre[(uf + 1) % PF][rr][l];
            }
        };
        auto stage_dy = [&](int st, int uf) {
            if (st + 1 >= S1) return;
#pragma unroll
            for (int rr = 0; rr < RB; ++rr) {
                const int tn = (st + 1) * RB + rr;
                const int dslot = tn % NRD;
#pragma unroll
                for (int l = 0; l < LPTD; ++l)
                    dring[dslot * DROW_UNITS + d_lds[l]] = dpre[(uf + 1) % PF][rr][l];
            }
        };

        // With SPIO_PIPE the products of a step are issued one step later, from a second set of
        // fragment registers, and the step's own LDS reads, row loads and ring writes are dealt
        // out between the groups of MFMAs: the matrix pipe takes 16 cycles per MFMA and the wave
        // issues the other instructions in the slots that leaves.
        constexpr int SHARES = RB * CPW;
        for (int sb = 0; sb < SLOTS; sb += UNROLL) {
#pragma unroll
            for (int uf = 0; uf < UNROLL; ++uf) {
                const int slot = sb + uf;
                const int st = S0 + slot;
                // A slot without a step has the loads only; where the loop is not unrolled it runs through the
                // same code as the others (with nothing to read, stage or multiply), because loads on two paths
                // would cost the exact counts.
                if (kFullUnroll && st >= S1) {
                    prefetch_rows(slot, uf);
                    continue;
                }
                // PF is even, so the parity of the step is known at compile time: it fixes the
                // x ring rows.
                const int sp = (S0 + uf) & 1;
                const int ta = (S0 + uf) * RB % NA;
                const bool math = kFullUnroll || st < S1;
                if (SPIO_PIPE) {
                    const int fs = uf & 1;
#pragma unroll
                    for (int g = 0; g < SHARES; ++g) {
                        if (math) read_share(st, sp, ta, g / CPW, g % CPW, fs);
                        if (g == 0) prefetch_rows(slot, uf);
                        if (g == (SHARES > 1 ? 1 : 0)) stage_x(st, sp, uf);
                        if (g == (SHARES > 2 ? 2 : SHARES - 1)) stage_dy(st, uf);
                        if (st > S0 && math) multiply_share(st - 1, ta + NA - RB, g / CPW, g % CPW, fs ^ 1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
                    // all LDS reads first, so that their latency overlaps the loads and ring writes
                    if (math) {
#pragma unroll
                        for (int g = 0; g < SHARES; ++g) read_share(st, sp, ta, g / CPW, g % CPW, 0);
                    }
                    prefetch_rows(slot, uf);
                    stage_x(st, sp, uf);
                    stage_dy(st, uf);
                    if (math) {
#pragma unroll
                        for (int g = 0; g < SHARES; ++g) multiply_share(st, ta, g / CPW, g % CPW, 0);
                    }
                }
                block_sync();
            }
        }
        if (SPIO_PIPE) {
            constexpr int LAST = S1 - 1;
#pragma unroll
            for (int g = 0; g < SHARES; ++g) multiply_share(LAST, LAST * RB % NA, g / CPW, g % CPW, (LAST - S0) & 1);
        }
    }

    // ---- publish ----
    // Sum m = 8 j + k, n = 8 sj + c of acc[r][nb] belongs to filter row r and column 4 nb + 2 sj + 1 - j.  The sums
    // are staged in LDS in grad_weight order, where the waves of a group add theirs one after the other, and
    // leave 64 consecutive floats at a time: fp32 atomics into grad_weight (two full 128-byte lines an
    // instruction, which the memory system retires several times faster than the scattered half-lines of the
    // accumulator layout), or plain stores into this workgroup's partial block when a second kernel does the
    // reduction.
    block_sync();  // every wave is done with the rings; reuse them
    {
        float* const gstage = reinterpret_cast<float*>(lds) + wg * GROUP_FLOATS;
        const int k4 = 4 * ((lane >> 4) & 1);
        const int c = lane & 7;
#pragma unroll
        for (int w2 = 0; w2 < TS; ++w2) {
            if (TS == 1 || ws == w2) {
#pragma unroll
                for (int nb = 0; nb < NB4; ++nb) {
                    const int s = 4 * nb + 2 * ((lane & 15) >> 3) + 1 - (lane >> 5);
                    if (s < kS) {
#pragma unroll
                        for (int r = 0; r < kR; ++r)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                float* const sum = gstage + (((k4 + e) * kR + r) * kS + s) * 8 + c;
                                *sum = (w2 > 0 ? *sum : 0.f) + acc[r][nb][e];
                            }
                    }
                }
            }
            if (TS > 1)
                block_sync();
            else
                wave_sync();  // all lanes read what all lanes staged
        }
#if SPIO_PARTIALS
        if (wave_active && ws == 0) {  // (nobody reads the blocks of groups past the last one)
            spio_float4* const out = reinterpret_cast<spio_float4*>(grad_weight) +
                (((long long)((nbk * PBLKS + pb) * QBLKS + qb) * GBLKS + cb) * GB + wg) * (GROUP_FLOATS / 4);
            const spio_float4* const staged = reinterpret_cast<const spio_float4*>(gstage);
#pragma unroll
            for (int i = lane; i < GROUP_FLOATS / 4; i += 64) __builtin_nontemporal_store(staged[i], out + i);
        }
#else
        if (wave_active) {
            float* const out = grad_weight + (long long)gglob * GROUP_FLOATS;
#pragma unroll
            for (int i = ws; i < kR * kS; i += TS) atomic_add_f32(out + 64 * i + lane, gstage[64 * i + lane]);
        }
#endif
#if SPIO_HAS_BIAS
        // grad_bias[8g + k] = accb of shift 0 (every column holds the same sum): lanes 0 and 16 carry channels 0-3
        // and 4-7.  All waves leave their eight sums in LDS and one wave adds the workgroup's GB*8 consecutive
        // values with a single atomic instruction: atomics of different workgroups to the same
        // 128-byte line retire one after the other, so their number per line is what counts.
        {
            float* bslots = reinterpret_cast<float*>(lds) + GB * GROUP_FLOATS;  // [wave][8]
            if ((lane & 47) == 0) {
#pragma unroll
                for (int e = 0; e < 4; ++e) bslots[wave * 8 + k4 + e] = accb[e];
            }
            block_sync();
            if (wave == 0) {
                for (int i = lane; i < GB * 8; i += 64) {
                    float v = 0.f;
#pragma unroll
                    for (int w2 = 0; w2 < TS; ++w2) v += bslots[(w2 * GB + i / 8) * 8 + (i & 7)];
#if SPIO_PARTIALS
                    grad_weight[BIAS_PARTIALS + (((long long)nbk * PBLKS + pb) * QBLKS + qb) * GBLKS * GB * 8 + cb * GB * 8 + i] = v;
#endif
                    if (grad_bias != nullptr && cb * GB + i / 8 < kGroups) atomic_add_f32(grad_bias + 8 * cb * GB + i, v);
                }
            }
        }
#endif
    }
}

#if SPIO_PARTIALS
// Second stage: grad_weight = sum over the partial blocks (stored whole: a caller that runs the
// two-stage kernel need not zero grad_weight first).  A workgroup owns COLS float4 columns
// (COLS * 16 contiguous bytes of every partial image, which is grad_weight with the missing groups behind it); its slices each add the blocks
// p = slice, slice + SLICES, ... with UN loads in flight, the slices are added through LDS and slice 0
// stores the total.  With 32 columns (512 bytes: half a wave per load instruction) where that gives
// a workgroup per compute unit: with 8 columns, 3584 workgroups of 128-byte rows for a 7x7 filter on 256
// channels, the stage took 5.9 us for 14.7 MB, with 32 5.1 us, of which about 2.2 us are what any
// kernel costs in a stream.  With 8 where there are few columns: more workgroups, and more slices each.
// Every element of grad_weight has exactly one
// owner, so no atomics are needed and the sum does not depend on timing.
template <class T>
SPIO_DEVICE void reduce_partials(T* __restrict__ grad_weight, const spio_float4* __restrict__ partials) {
    constexpr int IMAGE_F4 = GBLKS * GB * GROUP_FLOATS / 4;  // float4 columns of one partial image
    constexpr int NPART = NBLKS * PBLKS * QBLKS;
    constexpr int COLS = SPIO_REDUCE_COLS;
    constexpr int SLICES = 256 / COLS;
    constexpr int UN = NPART <= 4 * SLICES ? 4 : NPART <= 8 * SLICES ? 8 : 16;
    __shared__ spio_float4 red[SLICES][COLS];
    const int tid = thread_id();
    const int cl = tid % COLS;
    const int slice = tid / COLS;
    const int col = block_id() * COLS + cl;
    const bool live = col < kGroups * GROUP_FLOATS / 4;
    spio_float4 sum = spio_float4{0.f, 0.f, 0.f, 0.f};
    for (int base = slice; base < NPART; base += SLICES * UN) {
        spio_float4 v[UN];
#pragma unroll
        for (int i = 0; i < UN; ++i) {
            const int p = base + i * SLICES;
            v[i] = spio_float4{0.f, 0.f, 0.f, 0.f};
            if (p < NPART && live) v[i] = partials[(long long)p * IMAGE_F4 + col];
        }
#pragma unroll
        for (int i = 0; i < UN; ++i) sum += v[i];
    }
    red[slice][cl] = sum;
    block_sync();
    if (slice == 0 && live) {
#pragma unroll 4
        for (int i = 1; i < SLICES; ++i) sum += red[i][cl];
        store_sums(grad_weight + 4 * (long long)col, sum);
    }
}
extern "C" __global__ void SPIO_LAUNCH_BOUNDS(256)
SPIO_CONCAT(SPIO_KERNEL_NAME, _reduce)(float* __restrict__ grad_weight, const spio_float4* __restrict__ partials) {
    reduce_partials(grad_weight, partials);
}
// The version for fp16 weights also sums the bias partials, in a workgroup of its own per channel block
// behind the others, and stores grad_bias (null = not wanted): nothing is left to clear before the main
// kernel, which gets a null grad_bias then.
#if SPIO_HAS_BIAS
SPIO_DEVICE void reduce_bias(float* __restrict__ grad_bias, const float* __restrict__ bias_partials, int cb) {
    constexpr int NPART = NBLKS * PBLKS * QBLKS;
    constexpr int CH = GB * 8;
    constexpr int SLICES = 256 / CH;
    constexpr int UN = 8;
    __shared__ float red[SLICES][CH];
    const int tid = thread_id();
    const int ch = tid % CH;
    const int slice = tid / CH;
    const int k = cb * CH + ch;
    float sum = 0.f;
    if (slice < SLICES) {
        for (int base = slice; base < NPART; base += SLICES * UN) {
            float v[UN];
#pragma unroll
            for (int i = 0; i < UN; ++i) {
                const int p = base + i * SLICES;
                v[i] = p < NPART ? bias_partials[(long long)p * GBLKS * CH + k] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < UN; ++i) sum += v[i];
        }
        red[slice][ch] = sum;
    }
    block_sync();
    if (slice == 0 && k < kC && grad_bias != nullptr) {
        for (int i = 1; i < SLICES; ++i) sum += red[i][ch];
        grad_bias[k] = sum;
    }
}
#endif
extern "C" __global__ void SPIO_LAUNCH_BOUNDS(256)
SPIO_CONCAT(SPIO_KERNEL_NAME, _reduce_h)(spio_half* __restrict__ grad_weight, const spio_float4* __restrict__ partials
#if SPIO_HAS_BIAS
                                         , float* __restrict__ grad_bias
#endif
) {
#if SPIO_HAS_BIAS
    constexpr int WEIGHT_BLOCKS = (GBLKS * GB * GROUP_FLOATS / 4 + SPIO_REDUCE_COLS - 1) / SPIO_REDUCE_COLS;
    if (block_id() >= WEIGHT_BLOCKS) {
        reduce_bias(grad_bias, reinterpret_cast<const float*>(partials) + BIAS_PARTIALS, block_id() - WEIGHT_BLOCKS);
        return;
    }
#endif
    reduce_partials(grad_weight, partials);
}
#endif
