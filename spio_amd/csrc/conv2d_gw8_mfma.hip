// Row-streaming MFMA kernel for conv2d_gw8 forward and data gradient (gfx950).
//
// Contract (reference kernel: spio/src/conv2d_gw8.cu:10-225, both modes):
//   fprop : y[n,p,q,k]     = rn16(bias[k] + sum_{c,r,s} x[n,p+r-py,q+s-px,8g+c] * w[k,r,s,c])
//   dgrad : dx[n,h,w,8g+c] = rn16(sum_{j,r,s} dy[n,h-r+py,w-s+px,8g+j] * w[8g+j,r,s,c])
// Both are "dst = conv(src, filter, effective padding)"; dgrad uses the flipped,
// group-transposed filter and padding (R-1-py, S-1-px), which may be negative.
//
// Design
//   * A workgroup owns SPIO_BP output rows of SPIO_NB images for SPIO_GB
//     channel groups.  It streams the BP+R-1 source rows it needs through a
//     two-row LDS ring, one row per step, so every source element is read
//     from HBM once per workgroup and every tap reuses it from LDS/registers.
//   * In LDS a row is stored group-major: [group][flattened pixel][8 ch], the
//     pixels of the NB images laid side by side, each image padded to
//     WPI = DW+S-1 columns so that the zero halo is materialised once and a
//     tap is a plain pixel offset.
//   * One wave owns one group.  Per tile of 16 pairs of neighbouring pixels and
//     source row it issues ceil((S+1)/4) 16-byte LDS reads per lane and R times
//     as many MFMAs v_mfma_f32_16x16x32_f16 with
//         A (16 x 32) = filter:  rows m = 8*j + k   (pixel j of a pair, 8 out channels k)
//                               cols  = 8*kb + c   (column kb of four of a pair's S+1 source
//                                                   columns, which meets tap kb - j; 8 in channels c)
//         B (32 x 16) = source:  col n = pair, rows = (column kb, channel c)
//     Lane (n, kb) of B is exactly the 16 bytes of pixel 2n+kb, so the fragment
//     needs no shuffling; even and odd pixels of a staged row lie in two planes,
//     so that its reads are free of bank conflicts.  A source row contributes to
//     R output rows, which live in R accumulators that take turns (accumulator =
//     output row mod R); products of rows that the tile does not own are left out
//     at compile time.
//   * A finished output row is converted to fp16, staged through LDS into
//     pixel-major order and stored with one coalesced 16-byte store per lane.
//   * One workgroup barrier per step; global loads run SPIO_PF rows ahead of
//     the row being computed.
//   * Global memory is reached through buffer instructions whose hardware
//     bounds check does the predication: lanes without data carry an
//     out-of-range offset, rows outside the image use a descriptor of size
//     zero.  Such loads return zeros (the zero padding of the convolution) and
//     such stores are dropped, so no memory instruction sits under a branch.
//     Together with the fully unrolled step loop this lets the compiler count
//     the outstanding loads and stores exactly: the wait before a row is used
//     is for that row only.  (A wait counter covers loads and stores alike; a
//     count merged over paths that issue different numbers of them degrades
//     to the smallest, i.e. to waiting for rows that are not needed yet.)
//
// What bounds it: 3x3 filters memory (128n 64c 56x56: 103 MB at 6.0 TB/s), larger ones the chain of a step (barrier,
// LDS reads, products) on two to four waves a SIMD.  The rows of A were two output rows, two slots of accumulators
// each; with two neighbouring pixels a 5x5 or 7x7 filter takes 5/6 and 7/8 of the products (3x3: 3/4), every filter
// half of the fragment reads and conversions, and all lanes convert.  Before -> after, best of the first 16
// configurations: 128n 64c 56x56 18.9 -> 17.1 us, 32n 48c 224x224 58.4 -> 55.6, 1n 64c 56x56 2.9 -> 2.7, 60n 200c 33x33
// 20.3 -> 17.2, 300n 1000c 9x12 34.7 -> 31.1, 13n 280c 63x93 5x5 32.1 -> 27.1, 4n 424c 84x84 5x5 23.1 -> 17.8, 2n 600c
// 147x147 7x7 55.7 -> 45.8; equal: 59n 456c 60x60 (lines shared by channel blocks), 128n 24c 144x144 47.2 -> 47.9, 4x4
// filters (twice the products of before, 16n 64c 50x50 5.6 -> 5.8 and 5.5 -> 5.4).
#include "spio_conv_common.h"

using namespace spio;

#ifndef SPIO_IGRAD
#define SPIO_IGRAD 0
#endif
#ifndef SPIO_HAS_BIAS
#define SPIO_HAS_BIAS 0
#endif
#ifndef SPIO_PF
#define SPIO_PF 2
#endif
#ifndef SPIO_PF0
#define SPIO_PF0 SPIO_PF
#endif
#ifndef SPIO_PF_RATE
#define SPIO_PF_RATE 1
#endif
#ifndef SPIO_BP2
#define SPIO_BP2 0
#endif
#ifndef SPIO_BQ
#define SPIO_BQ 0
#endif
#ifndef SPIO_TS
#define SPIO_TS 1
#endif
#ifndef SPIO_NB
#define SPIO_NB 1
#endif
#ifndef SPIO_XCD_CHUNK
#define SPIO_XCD_CHUNK 0
#endif

namespace {

constexpr bool kIgrad = SPIO_IGRAD != 0;
constexpr bool kHasBias = (SPIO_HAS_BIAS != 0) && !kIgrad;
constexpr int SH = kIgrad ? kP : kH;  // source rows / cols
constexpr int SW = kIgrad ? kQ : kW;
constexpr int DH = kIgrad ? kH : kP;  // destination rows / cols
constexpr int DW = kIgrad ? kW : kQ;
constexpr int EPY = kIgrad ? kR - 1 - kPadY : kPadY;
constexpr int EPX = kIgrad ? kS - 1 - kPadX : kPadX;

constexpr int GB = SPIO_GB;  // groups (waves along channels) per workgroup
constexpr int BP = SPIO_BP;  // output rows per workgroup
// Two tile heights (SPIO_BP2 > 0): the row blocks of an image alternate between BP and BP2 rows;
// the first half of the grid takes the BP-row tiles and the second half the BP2-row tiles.  A
// grid of two workgroups per compute unit is dispatched as two cohorts (ids below half the grid
// land one per CU first, the rest join them a moment later); memory serves requests in arrival
// order, so the first cohort's prefetch burst is served before the second cohort's first row,
// the second cohort trails by that burst for the whole kernel and then finishes alone at one
// workgroup per CU (measured at N=128, C=64, 56x56 with equal tiles: 13.3 us against 18.0 us).
// Taller tiles for the leading cohort and shorter ones for the trailing one let both end together.
constexpr int BP2 = SPIO_BP2;
constexpr int NB = SPIO_NB;  // images per workgroup
constexpr int TS = SPIO_TS;  // waves sharing the tiles of one group
constexpr int PF = SPIO_PF;  // prefetch distance in rows (register buffers for rows in flight)
// The distance is reached by a ramp: PF0 rows are requested before the first step and PF_RATE
// rows per step from then on until the requests run PF rows ahead.  All workgroups of a launch
// start within a fraction of a microsecond of each other and memory serves requests roughly in
// the order they arrive; a workgroup that asks for all PF rows at once gets them before a
// workgroup that started a moment later gets its first row, and the late ones then finish long
// after the others.  With a short first burst every workgroup has its first rows early.
constexpr int PF0 = SPIO_PF0 < SPIO_PF ? SPIO_PF0 : SPIO_PF;
constexpr int PF_RATE = SPIO_PF_RATE;
constexpr int WAVES = GB * TS;
constexpr int THREADS = 64 * WAVES;

constexpr int KB = (kS + 1 + 3) / 4;  // MFMA K-steps per source row (4 of a pair's S + 1 columns each)
// Column blocks (SPIO_BQ > 0): a workgroup owns BQ output columns of its rows and stages the
// BQ + S - 1 source columns they need; the S - 1 extra columns hold the neighbouring blocks'
// pixels, or zeros at the image's edges (reference: block_q / block_w = block_q + S - 1,
// spio/kernels/conv2d_gw8_kernel.py:92-108, and the column halo of spio/src/conv2d_gw8.cu:71-91).
// Rows of any width then fit the LDS ring.  0 = the whole width.
constexpr int BQ = SPIO_BQ > 0 ? SPIO_BQ : DW;
constexpr int QBLKS = (DW + BQ - 1) / BQ;
constexpr int WPI = BQ + kS - 1;        // padded width of one image (block) in LDS
constexpr int F = NB * WPI;             // flattened pixels of a staged row
constexpr int WT = (F - kS + 1 + 31) / 32;  // 32-pixel tiles per row
// Tiles per wave.  Those past the last one (waves share a row) read and write cells that exist; they hold
// zeros, and nobody looks at the results.
constexpr int TPW = (WT + TS - 1) / TS;
constexpr int FP = 32 * TPW * TS + 4 * KB - 2;  // pixels any fragment read can touch
// The planes of even and odd pixels are 8 cells (half the banks) apart modulo 16, the groups 9, so that the
// cells a wave's threads write fall into different banks.
constexpr int PLANE = (FP + 1) / 2 + ((8 - (FP + 1) / 2 % 16) + 16) % 16;
constexpr int GS = PLANE + FP / 2 + ((9 - (PLANE + FP / 2) % 16) + 16) % 16;  // group stride in cells
SPIO_DEVICE constexpr int pos(int pixel) { return (pixel >> 1) + (pixel & 1) * PLANE; }
constexpr int NR = 2;                               // ring rows
constexpr int RING_ROW_UNITS = GB * GS + 1;         // 16-byte units per ring row (+1: dump cell)
constexpr int DUMP_UNIT = GB * GS;                  // where lanes without a cell write
constexpr int OSTRIDE = stage_pitch(GB);            // bytes per pixel in the output stage
constexpr int OPLANE = 16 * TPW * TS * OSTRIDE + 128;  // even pixels, then odd ones, as in the ring
constexpr int OUT_ROW_BYTES = 2 * OPLANE;
constexpr int IN_CELLS = F * GB;
constexpr int LPT = (IN_CELLS + THREADS - 1) / THREADS;  // source cells per thread per row
constexpr int OUT_CELLS = NB * BQ * GB;
constexpr int SPT = (OUT_CELLS + THREADS - 1) / THREADS;  // stores per thread per row
constexpr int GBLKS = (kGroups + GB - 1) / GB;
constexpr int PAIRS = (DH + BP + BP2 - 1) / (BP + BP2);  // (BP, BP2) pairs of row blocks per image
constexpr int PBLKS = BP2 > 0 ? PAIRS : (DH + BP - 1) / BP;  // row blocks of one height per image
constexpr int NBLKS = (kN + NB - 1) / NB;
constexpr int HALF_BLOCKS = GBLKS * PBLKS * QBLKS * NBLKS;  // workgroups per tile height
constexpr int NUM_BLOCKS = (BP2 > 0 ? 2 : 1) * HALF_BLOCKS;

// The step loop is unrolled completely: every rotation index and every "is there a row to load
// / to store" is then a compile-time fact, and no memory instruction sits in a loop whose entry
// and back edge would disagree about the operations in flight.
#ifndef SPIO_MAX_UNROLL
#define SPIO_MAX_UNROLL 64
#endif
static_assert((BP > BP2 ? BP : BP2) + kR - 1 <= SPIO_MAX_UNROLL, "block_p + R - 1 exceeds the unrolled step limit");
static_assert(PF >= 2 && PF0 >= 2 && PF_RATE >= 1 && WAVES <= 16, "bad configuration");
constexpr int STREAM_UNITS = NR * RING_ROW_UNITS + 2 * OUT_ROW_BYTES / 16;
constexpr int FILTER_UNITS = kIgrad ? GB * 8 * kR * kS : 0;  // staged filters (data gradient only)
constexpr int LDS_UNITS = STREAM_UNITS > FILTER_UNITS ? STREAM_UNITS : FILTER_UNITS;
static_assert(LDS_UNITS * 16 <= 160 * 1024, "LDS overflow");

// Byte extents of the NB-image block a workgroup addresses through one buffer descriptor.
constexpr long long SRC_IMAGE_BYTES = (long long)SH * SW * kC * kSrcBytes;
constexpr long long DST_IMAGE_BYTES = (long long)DH * DW * kC * kDstBytes;
static_assert(NB * SRC_IMAGE_BYTES < (1ll << 31) && NB * DST_IMAGE_BYTES < (1ll << 31),
              "an image block must stay below 2 GiB (32-bit buffer offsets)");
static_assert(!SPIO_KEEP || !SPIO_SRC_F32 ||
                  (NB * SRC_IMAGE_BYTES < (1ll << 30) && EPY >= 0 && EPY < kR && EPX >= 0 && EPX < kS),
              "the fp16 copy: offsets are halved, and every source pixel has to be staged by the block that owns it");
static_assert(!(SPIO_W_F32 && SPIO_IGRAD), "the data gradient reads fp16 filters");
constexpr unsigned OOB = 0x80000000u;  // offset of a lane without data: beyond every descriptor

constexpr int cmin(int a, int b) { return a < b ? a : b; }
// Source rows requested once step t of `steps` has issued its loads (t = -1: before the first step).
constexpr int rows_requested(int t, int steps) { return cmin(cmin(steps, t + 1 + PF), PF0 + PF_RATE * (t + 1)); }

// Source rows shared with the neighbouring row blocks (the first and last R-1
// steps) can be served from L2 when the neighbour runs on the same XCD;
// SPIO_HALO_CACHED = 1 loads those with the default policy and only the
// interior rows with the non-temporal hint.
#ifndef SPIO_HALO_CACHED
#define SPIO_HALO_CACHED 0
#endif
// Cache-policy operands of the buffer instructions (gfx950: 1 = sc0, 2 = nt, 16 = sc1), one for
// the interior source rows, one for the rows shared with neighbouring row blocks, one for the
// stores.  SPIO_NT = 1 streams with the non-temporal hint unless a policy is given explicitly;
// source rows whose lines several channel blocks share are loaded with the default policy all the
// same: the block that comes second finds the line in L2.  Forward, non-temporal -> default loads:
// 64n 160c 40x40 22.5 -> 14.4 us, 46n 1072c 17x17 17.7 -> 15.0, 94n 296c 43x47 83.2 -> 76.7, 128n 96c
// 56x56 29.7 -> 29.1; where the blocks are whole lines the hint is worth 15 %.
constexpr bool kSplitLines = splits_lines(GB, GBLKS);
#ifndef SPIO_LD_POLICY
#define SPIO_LD_POLICY (SPIO_NT && !kSplitLines ? 2 : 0)
#endif
#ifndef SPIO_ST_POLICY
#define SPIO_ST_POLICY (SPIO_NT ? 2 : 0)
#endif
#ifndef SPIO_HALO_POLICY
#define SPIO_HALO_POLICY (SPIO_HALO_CACHED ? 0 : SPIO_LD_POLICY)
#endif
constexpr int AUX_LD = SPIO_LD_POLICY;
constexpr int AUX_HALO = SPIO_HALO_POLICY;
constexpr int AUX_ST = SPIO_ST_POLICY;

typedef __amdgpu_buffer_rsrc_t rsrc_t;
SPIO_DEVICE rsrc_t make_rsrc(const void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}

// pointers typed in the LDS address space: 32-bit address arithmetic, constant parts of an
// index end up in the instruction's offset field
typedef __attribute__((address_space(3))) spio_uint4* lds_u4p;
typedef __attribute__((address_space(3))) unsigned char* lds_bytep;

typedef __attribute__((address_space(3))) spio_uint2* lds_u2p;

// One tile: ROWS output rows starting at row p0 of the NB images from n0 on, channel block cb.
// kept_src, kept_weights: SPIO_KEEP.
template <int ROWS>
SPIO_DEVICE void conv_rows(spio_uint4* __restrict__ dst, const spio_uint4* __restrict__ src,
                           const spio_half* __restrict__ weights, const float* __restrict__ bias,
                           spio_uint4* __restrict__ kept_src, spio_uint4* __restrict__ kept_weights, const lds_u4p ring, const int p0, const int q0, const int n0, const int cb) {
    constexpr int STEPS = ROWS + kR - 1;
    const lds_bytep ostage = (lds_bytep)(ring + NR * RING_ROW_UNITS);

    const int tid = thread_id();
    const int lane = tid & 63;
    // the wave index as a scalar: whatever depends on it alone stays in scalar registers
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wg = wave % GB;  // group within the workgroup
    const int ws = wave / GB;  // tile split index
    const int gglob = cb * GB + wg;
    const bool wave_active = gglob < kGroups;  // idle waves compute on zeros and store nothing

    // ---- buffer descriptors: the workgroup's image block of src and of dst ----
    // Offsets are relative to the block's first image; images past the end of the batch lie
    // beyond the descriptor's size, so their loads give zeros and their stores are dropped.
    const int images = imin(NB, kN - n0);
    const rsrc_t rs_src = make_rsrc(reinterpret_cast<const unsigned char*>(src) + n0 * SRC_IMAGE_BYTES,
                                    (int)(images * SRC_IMAGE_BYTES));
    const rsrc_t rs_dst = make_rsrc(reinterpret_cast<const unsigned char*>(dst) + n0 * DST_IMAGE_BYTES,
                                    (int)(images * DST_IMAGE_BYTES));
    const rsrc_t rs_src_none = make_rsrc(reinterpret_cast<const unsigned char*>(src), 0);
    const rsrc_t rs_dst_none = make_rsrc(reinterpret_cast<const unsigned char*>(dst), 0);

    // ---- loop-invariant addressing of the cooperative row load ----
    // Every thread issues the same loads on every step.  Cells that hold no source data (halo
    // columns, missing groups) carry the out-of-range offset: the load returns zeros, which is
    // what the halo must hold.  Threads without a cell write to the row's dump cell.
    int in_voff[LPT][kSrcLoads];  // byte offset inside the image block; row term excluded
    int in_lds[LPT][kSrcLoads];   // 16-byte unit inside a ring row (SPIO_SRC_F32: byte)
#pragma unroll
    for (int l = 0; l < LPT; ++l) {
#pragma unroll
        for (int j = 0; j < kSrcLoads; ++j) {
            const int cell = moved_unit(tid, j, kSrcLoads) + THREADS * l;
            unsigned voff = OOB;
            int unit = DUMP_UNIT;
            if (cell < IN_CELLS) {
                const int g = cell % GB;
                const int f = cell / GB;
                const int img = f / WPI;
                const int col = q0 + f % WPI - EPX;
                unit = g * GS + pos(f);
                if (col >= 0 && col < SW && cb * GB + g < kGroups)
                    voff = (unsigned)(((img * SH * SW + col) * kGroups + cb * GB + g) * (8 * kSrcBytes));
            }
            in_voff[l][j] = (int)(voff + (unsigned)half_bytes(tid, kSrcLoads, 16));
            in_lds[l][j] = SPIO_SRC_F32 ? unit * 16 + half_bytes(tid, kSrcLoads, 8) : unit;
        }
    }
    constexpr int SRC_ROW_BYTES = SW * kC * kSrcBytes;
    constexpr int DST_ROW_BYTES = DW * kC * kDstBytes;

    // Source row `t` of this workgroup (image row p0 + t - EPY) for every cell of the thread.
    // Rows outside the image read through the empty descriptor: zeros, the vertical padding.
    auto load_row = [&](spio_uint4(&regs)[LPT][kSrcLoads], int t) {
        const int h = p0 + t - EPY;
        const bool inside = h >= 0 && h < SH;
        const rsrc_t rs = inside ? rs_src : rs_src_none;
        // (readfirstlane: the row offset must stay in a scalar register whatever the optimiser
        //  makes of the clamp)
        const int soff = __builtin_amdgcn_readfirstlane(imin(imax(h, 0), SH - 1) * SRC_ROW_BYTES);
        const bool halo = t < kR - 1 || t >= ROWS;
#pragma unroll
        for (int l = 0; l < LPT; ++l) {
#pragma unroll
            for (int j = 0; j < kSrcLoads; ++j) {
                Pack16 v;
                v.i = halo ? __builtin_amdgcn_raw_buffer_load_b128(rs, in_voff[l][j], soff, AUX_HALO)
                           : __builtin_amdgcn_raw_buffer_load_b128(rs, in_voff[l][j], soff, AUX_LD);
                regs[l][j] = v.u;
            }
        }
    };
    // A loaded row into a ring row; fp32 rows are rounded, and the ones this block owns stored as fp16:
    // rows p0 .. p0+ROWS-1, and what follows the last block of an image.
    const rsrc_t rs_kept = make_rsrc(reinterpret_cast<const unsigned char*>(kept_src) + (SPIO_KEEP ? n0 * SRC_IMAGE_BYTES / 2 : 0),
                                     (int)(SPIO_KEEP ? images * (SRC_IMAGE_BYTES / 2) : 0));
    auto row_to_ring = [&](const spio_uint4(&regs)[LPT][kSrcLoads], int t) {
        const lds_u4p row = ring + (t % NR) * RING_ROW_UNITS;
        if (!SPIO_SRC_F32) {
#pragma unroll
            for (int l = 0; l < LPT; ++l) row[in_lds[l][0]] = regs[l][0];
            return;
        }
        const int h = p0 + t - EPY;
        const bool owned = h < SH && (h < p0 + ROWS || p0 + ROWS >= DH);
        const rsrc_t rs = owned ? rs_kept : rs_src_none;
        const int row_off = imin(imax(h, 0), SH - 1) * (SRC_ROW_BYTES / 2);
#pragma unroll
        for (int l = 0; l < LPT; ++l) {
#pragma unroll
            for (int j = 0; j < kSrcLoads; ++j) {
                const spio_uint2 v = narrow(regs[l][j]);
                *(lds_u2p)((lds_bytep)row + in_lds[l][j]) = v;
                if (SPIO_KEEP && t >= EPY && (t < EPY + ROWS || SH > DH))
                    __builtin_amdgcn_raw_buffer_store_b64(v, rs, (int)(((unsigned)in_voff[l][j] >> 1) + (unsigned)row_off), 0, AUX_ST);
            }
        }
    };

    // ---- filter loads, first of all ----
    // Loads of one wave return in order, so what is requested first is what the first
    // multiplication waits for: the filters (a few loads per lane) go ahead of the PF source
    // rows, and the first step can start as soon as source row 0 has landed.  Branch-free: dead
    // taps and idle waves load a valid address and are zeroed when the fragments are built.
    constexpr int WLPT = kIgrad ? (GB * 8 * kR * kS + THREADS - 1) / THREADS : kR * KB;
    spio_uint4 wraw[WLPT][kFilterLoads];
    if (!kIgrad) {
        // A[m = out channel ch][c] = w[8g+ch][r][s][c]: 16 contiguous bytes per lane.
        // Lane (m = lane%16, kb = lane/16): pixel j = m/8 of a pair, channel m%8, column 4u+kb of the
        // pair's S+1, which this pixel meets under tap 4u+kb-j.
        const int m = lane & 15;
        const int kb = lane >> 4;
        const int j = m >> 3;
        const int ch = m & 7;
        const int gsafe = wave_active ? gglob : 0;
#pragma unroll
        for (int r = 0; r < kR; ++r) {
#pragma unroll
            for (int u = 0; u < KB; ++u) {
                const int s = 4 * u + kb - j;
                const int ss = s >= 0 && s < kS ? s : 0;
                load_filter_unit(wraw[r * KB + u], weights, ((long long)(8 * gsafe + ch) * kR + r) * kS + ss);
            }
        }
    } else {
        // the workgroup's filters as they lie in memory ([group][jj][r][s][8 ch]), WLPT units per thread
        constexpr int WUNITS = GB * 8 * kR * kS;
#pragma unroll
        for (int l = 0; l < WLPT; ++l) {
            const int i = imin(tid + THREADS * l, WUNITS - 1);
            const int g = i / (8 * kR * kS);
            const int rem = i % (8 * kR * kS);
            const int gs = cb * GB + g < kGroups ? cb * GB + g : 0;
            load_filter_unit(wraw[l], weights, (long long)gs * (8 * kR * kS) + rem);
        }
    }
    __builtin_amdgcn_sched_barrier(0);  // keep the filter loads ahead of the row loads

    // ---- rows 0..PF-1 into registers: their latency covers the rest of the set-up ----
    spio_uint4 pre[PF][LPT][kSrcLoads];
#pragma unroll
    for (int t = 0; t < PF0; ++t) load_row(pre[t], imin(t, STEPS - 1));
    __builtin_amdgcn_sched_barrier(0);  // ... and the row loads ahead of everything that waits

    // ---- loop-invariant addressing of the cooperative row store ----
    unsigned out_voff[SPT][kDstStores];  // byte offset inside the image block; row term excluded
    int out_lds[SPT][kDstStores];        // byte offset inside an output-stage row
#pragma unroll
    for (int s = 0; s < SPT; ++s) {
#pragma unroll
        for (int j = 0; j < kDstStores; ++j) {
            const int cell = moved_unit(tid, j, kDstStores) + THREADS * s;
            unsigned voff = OOB;
            int from = 0;
            if (cell < OUT_CELLS) {
                const int g = cell % GB;
                const int q = (cell / GB) % BQ;
                const int img = cell / (GB * BQ);
                const int o = img * WPI + q;
                from = (o & 1) * OPLANE + (o >> 1) * OSTRIDE + g * 16;
                if (cb * GB + g < kGroups && q0 + q < DW)
                    voff = (unsigned)(((img * DH * DW + q0 + q) * kGroups + cb * GB + g) * (8 * kDstBytes));
            }
            out_voff[s][j] = voff + (unsigned)half_bytes(tid, kDstStores, 16);
            out_lds[s][j] = from + half_bytes(tid, kDstStores, 8);
        }
    }

    // ---- filter fragments: wfrag[r][u] ----
    spio_half8 wfrag[kR][KB];
    if (!kIgrad) {
        const int m = lane & 15;
        const int kb = lane >> 4;
        const int j = m >> 3;
#pragma unroll
        for (int r = 0; r < kR; ++r) {
#pragma unroll
            for (int u = 0; u < KB; ++u) {
                const int s = 4 * u + kb - j;
                Pack16 v;
                v.u = (s >= 0 && s < kS) ? filter_unit(wraw[r * KB + u]) : spio_uint4{0u, 0u, 0u, 0u};
                wfrag[r][u] = v.h;
            }
        }
    } else {
        // A[m = dx channel ch][jj] = w[8g+jj][R-1-r][S-1-s][ch]: the filter transposed within
        // the group.  The workgroup copies its groups' filters to LDS as they lie in memory
        // ([jj][r][s][8 ch]) and every wave reads its fragments with the transposing LDS read:
        // in a 16-lane block source lane 4*jr+t supplies 4 channels (half t%2) of row jj = jr for
        // pixel t/2 of a pair, and result lane i receives rows jj = 0..3 of column i = 8*pixel + ch.
        constexpr int WUNITS = GB * 8 * kR * kS;
        const lds_u4p wlds = ring;  // ring and output stage are not in use yet
#pragma unroll
        for (int l = 0; l < WLPT; ++l) {
            const int i = tid + THREADS * l;
            if (i < WUNITS) wlds[i] = filter_unit(wraw[l]);
        }
        block_sync();
        const int kb = lane >> 4;
        const int jr = (lane & 15) >> 2;
        const int t4 = lane & 3;
        const int src_pixel = t4 >> 1;          // of a pair: whose data this lane fetches
        const int my_pixel = (lane & 15) >> 3;  // whose fragment row this lane receives
        typedef spio_short4 __attribute__((address_space(3))) * lds_ptr;
#pragma unroll
        for (int r = 0; r < kR; ++r) {
#pragma unroll
            for (int u = 0; u < KB; ++u) {
                const int s_src = 4 * u + kb - src_pixel;
                const int s_mine = 4 * u + kb - my_pixel;
                // clamp the address of dead taps; their result is discarded below
                const int rr = kR - 1 - r;
                const int ss = s_src >= 0 && s_src < kS ? kS - 1 - s_src : 0;
                const lds_bytep base = (lds_bytep)wlds + ((((wg * 8 + jr) * kR + rr) * kS + ss) * 16) + (t4 & 1) * 8;
                union {
                    spio_short4 q[2];
                    spio_half8 h;
                } v;
                v.q[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)base);
                v.q[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(base + 4 * kR * kS * 16));
                if (!(s_mine >= 0 && s_mine < kS)) v.h = spio_half8{0, 0, 0, 0, 0, 0, 0, 0};
                wfrag[r][u] = v.h;
            }
        }
        block_sync();  // everyone has its fragments before the ring is zero-filled
    }

    // Accumulator lane layout: D[m = 4*(lane/16)+i][n = lane%16]: pixel 2*(lane%16) + lane/32 of the
    // tile, channels 4*((lane/16)&1) + i.
    const int out_kh = (lane >> 4) & 1;
    // this lane's place in a staged output row (tile 0 of the wave) and in a ring row
    const lds_bytep ostage_lane =
        ostage + (lane >> 5) * OPLANE + (16 * TPW * ws + (lane & 15)) * OSTRIDE + wg * 16 + out_kh * 8;
    const int frag_unit = wg * GS + 16 * TPW * ws + (lane & 15) + pos(lane >> 4);
    // Columns in no window are read from the group's first slack cell, which is zero: clearing them in the fragments, four
    // instructions each between the reads and the products, took 4 % more than not clearing them (53n 144c 15x23 5x5 from the
    // cache 7.12 -> 7.43 us); this takes no more (0.97 to 1.01 times, 16 kernels of five shapes).
    static_assert((kS + 1) % 4 == 0 || FP > F, "no cell that stays zero");
    const int zero_unit = wg * GS + pos(F) - frag_unit;  // from frag_unit on
    spio_float4 bias_reg = spio_float4{0.f, 0.f, 0.f, 0.f};
    if (kHasBias && wave_active) {
#pragma unroll
        for (int i = 0; i < 4; ++i) bias_reg[i] = bias[8 * gglob + 4 * out_kh + i];
    }
    spio_float4 acc[TPW][kR];  // output row t of the tile in accumulator t mod R, from step t to step t + R - 1

    // ---- zero the slack cells behind each group's pixels once: fragment reads of the last
    //      tiles touch them (they meet zero filter taps, so they must be finite), nothing ever
    //      writes them ----
    {
        constexpr int SLACK = FP - F;
        constexpr int PER_GROUP = SLACK > 0 ? SLACK : 1;  // (none behind rows of whole tiles under 3- and 7-wide filters)
        for (int i = tid; i < NR * GB * SLACK; i += THREADS) {
            const int row = i / (GB * PER_GROUP);
            const int g = i / PER_GROUP % GB;
            ring[row * RING_ROW_UNITS + g * GS + pos(F + i % PER_GROUP)] = spio_uint4{0u, 0u, 0u, 0u};
        }
    }

    // ---- row 0 into the ring ----
    block_sync();  // slack zeroed
    row_to_ring(pre[0], 0);
    block_sync();

    // Coalesced store of the output row staged at step `ts` (in stage buffer `obuf`): the row
    // that received its last tap at that step.  Called one step later, after the barrier.  Rows
    // past the end of the image store through the empty descriptor: the instructions are issued
    // all the same and the hardware drops them.
    auto store_output_row = [&](int ts, int obuf) {
        const int p = p0 + ts - (kR - 1);
        const rsrc_t rs = p < DH ? rs_dst : rs_dst_none;
        // The row offset is added to the per-lane offset; the scalar-offset operand stays the
        // constant 0.  A 16-byte buffer store reads its data registers for a few cycles after it
        // issues, and only for the constant form does the compiler keep the next instructions
        // from writing them: with the row offset in a scalar register an accumulator moved into
        // the first data register right behind the store was stored in its place (seen on gfx950
        // as stray values in the first two channels of some pixels of one output row).
        const unsigned row_off = (unsigned)(imin(imax(p, 0), DH - 1) * DST_ROW_BYTES);
#pragma unroll
        for (int s = 0; s < SPT; ++s) {
            const lds_bytep row = ostage + obuf * OUT_ROW_BYTES;
#pragma unroll
            for (int j = 0; j < kDstStores; ++j) {
                Pack16 v;
                v.u = SPIO_DST_F32 ? widen(*(lds_u2p)(row + out_lds[s][j])) : *(lds_u4p)(row + out_lds[s][j]);
                __builtin_amdgcn_raw_buffer_store_b128(v.i, rs, (int)(out_voff[s][j] + row_off), 0, AUX_ST);
            }
        }
        store_group_end();
    };

    // Rows above and below the image are rows of zeros in the ring; their products are skipped (a
    // scalar branch around LDS reads and MFMAs only: with a 7-row filter on a 14-row image they
    // would be 6 of 20 steps).
    auto row_is_live = [&](int t) {
        const int h = p0 + t - EPY;
        return h >= 0 && h < SH;
    };
    spio_half8 bfrag[TPW][KB];
    auto read_fragments = [&](int ring_row) {
        const lds_u4p rrow = ring + ring_row * RING_ROW_UNITS + frag_unit;
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
#pragma unroll
            for (int u = 0; u < KB; ++u) {
                Pack16 v;
                v.u = rrow[in_no_window(u, lane >> 4) ? zero_unit : 16 * i + 2 * u];
                bfrag[i][u] = v.h;
            }
        }
    };
    // Stages the output row that received its last tap at step `te` (stage buffer te mod 2).
    auto emit_row = [&](int te) {
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            Pack8 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o.h[e] = (spio_half)acc[i][(te + 1) % kR][e];
            *(lds_u2p)(ostage_lane + (te & 1) * OUT_ROW_BYTES + 16 * i * OSTRIDE) = o.u;
        }
    };
#pragma unroll
    for (int t = 0; t < STEPS; ++t) {  // everything that depends on t is a compile-time constant after unrolling
        // 1. prefetch the next source rows, at most up to row t+PF (whose register buffer is
        //    free: row t is in LDS)
#pragma unroll
        for (int r = rows_requested(t - 1, STEPS); r < rows_requested(t, STEPS); ++r) load_row(pre[r % PF], r);

        // 2. fragment reads of this step's row.  While they are in flight the row staged in the previous step
        //    goes out, and the row that received its last tap in the previous step is converted and staged:
        //    its results are long complete, while behind this step's MFMAs it would have to wait.  Its accumulator is
        //    the one that this step's newest row begins in, below.
        const bool row_live = row_is_live(t);
        if (row_live) read_fragments(t % NR);
        if (t >= kR + 1) store_output_row(t - 2, t & 1);
        if (t >= kR) emit_row(t - 1);

        // 3. multiply source row t into the output rows t - r of the tile; row t starts from the bias
        if (row_live) {
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
#pragma unroll
                for (int u = 0; u < KB; ++u) {
#pragma unroll
                    for (int r = 0; r < kR; ++r) {
                        if (t - r < 0 || t - r >= ROWS) continue;
                        spio_float4& d = acc[i][(t - r) % kR];
                        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(wfrag[r][u], bfrag[i][u],
                                                                   r == 0 && u == 0 ? bias_reg : d, 0, 0, 0);
                    }
                }
            }
        } else if (t < ROWS) {
#pragma unroll
            for (int i = 0; i < TPW; ++i) acc[i][t % kR] = bias_reg;
        }

        // 4. the next source row not yet in the ring (loaded earlier) into its ring row
        if (t + 1 < STEPS) row_to_ring(pre[(t + 1) % PF], t + 1);

        block_sync();
    }
    // the row staged in the last step goes out, the last row is staged and follows
    if (STEPS >= kR + 1) store_output_row(STEPS - 2, STEPS & 1);
    emit_row(STEPS - 1);
    block_sync();
    store_output_row(STEPS - 1, (STEPS - 1) & 1);  // the last row

    if (SPIO_KEEP && SPIO_W_F32 && n0 == 0 && p0 == 0 && q0 == 0 && ws == 0 && wave_active) {
        // the rounded filters, by the first tile of the channel block: the first pixel's rows of the fragments
        const int m = lane & 15;
        const int kb = lane >> 4;
#pragma unroll
        for (int r = 0; r < kR; ++r)
#pragma unroll
            for (int u = 0; u < KB; ++u) {
                Pack16 v;
                v.h = wfrag[r][u];
                if (m < 8 && 4 * u + kb < kS) kept_weights[((long long)(8 * gglob + m) * kR + r) * kS + 4 * u + kb] = v.u;
            }
    }
}

}  // namespace

extern "C" __global__ void SPIO_LAUNCH_BOUNDS(THREADS)
SPIO_KERNEL_NAME(spio_uint4* __restrict__ dst, const spio_uint4* __restrict__ src,
                 const spio_half* __restrict__ weights, const float* __restrict__ bias
#if SPIO_KEEP
                 , spio_uint4* __restrict__ kept_src, spio_uint4* __restrict__ kept_weights
#endif
) {
#if !SPIO_KEEP
    spio_uint4 *const kept_src = nullptr, *const kept_weights = nullptr;
#endif
    // One LDS block: the source-row ring, then the two output-stage rows.  The data-gradient
    // mode first uses the same block to stage the filters of the workgroup's groups.
    __shared__ spio_uint4 lds[LDS_UNITS];
    const lds_u4p ring = (lds_u4p)lds;

    // Workgroup -> (image block, channel block, row block), row block fastest.
    // Consecutive workgroup ids are dealt round-robin to the 8 XCDs.  Remap so that runs of
    // SPIO_XCD_CHUNK consecutive tiles land on one XCD (neighbouring row blocks share halo rows
    // through that XCD's L2) while the tiles in flight on the whole device at any moment still
    // form one compact, advancing range of addresses (HBM streams best through such a front;
    // eight distant fronts, one per XCD, cost several per cent).  0 = one contiguous range of
    // tiles per XCD.
    // With two tile heights the two halves of the grid are two such sequences of tiles, one per
    // height, and a tile and the one below it (the other height) have the same index in both:
    // their workgroups run on the same XCD and share their halo rows.
    const int raw = block_id();
    const bool second = BP2 > 0 && raw >= HALF_BLOCKS;
    // Tile order: row blocks fastest, so that neighbours in a run share halo rows.  Where channel
    // blocks share lines they go fastest instead, a run holding all of a pixel's: dealt to different XCDs,
    // every one of them would fetch the whole lines from memory (measured: twice the algorithmic
    // reads).  Column blocks go before the row blocks: neighbours share S - 1 columns of every row.
    constexpr int RUN = kSplitLines ? line_run(SPIO_XCD_CHUNK, GBLKS) : SPIO_XCD_CHUNK;
    const int b = xcd_tile<RUN, HALF_BLOCKS>(second ? raw - HALF_BLOCKS : raw);
    constexpr int TILES = QBLKS * PBLKS;  // tiles of one image and channel block
    const int t = kSplitLines ? (b / GBLKS) % TILES : b % TILES;
    const int cb = kSplitLines ? b % GBLKS : (b / TILES) % GBLKS;
    const int nb = b / (TILES * GBLKS);
    const int pb = t / QBLKS;
    const int q0 = (t % QBLKS) * BQ;
    const int n0 = nb * NB;
    if (BP2 > 0) {
        const int p0 = pb * (BP + BP2);
        if (second)
            conv_rows<(BP2 > 0 ? BP2 : 1)>(dst, src, weights, bias, kept_src, kept_weights, ring, p0 + BP, q0, n0, cb);
        else
            conv_rows<BP>(dst, src, weights, bias, kept_src, kept_weights, ring, p0, q0, n0, cb);
    } else {
        conv_rows<BP>(dst, src, weights, bias, kept_src, kept_weights, ring, pb * BP, q0, n0, cb);
    }
}
