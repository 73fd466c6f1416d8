// Shared definitions for the grouped-width-8 convolution kernels (gfx950).
//
// Every kernel of this directory is specialised at compile time: the shape of
// one convolution and the tile configuration arrive as SPIO_* macros, either
// from hipRTC options at run time or from -D flags of an offline hipcc build.
// Kernels therefore take only pointers, as the reference's kernels do
// (spio/src/conv2d_gw8.cu:10-12, spio/src/conv2d_gw8_wgrad.cu:10-12).
//
// Memory layouts (physical):
//   activations  [N][H][W][C]      fp16   (NCHW tensors with channels_last strides)
//   weights      [K][R][S][8]      fp16   ([K,8,R,S] tensors with channels_last strides)
//   bias         [K]               fp32
//   grad_weight  [K][R][S][8]      fp32
// A group is 8 consecutive channels: 16 bytes of one pixel.
#ifndef SPIO_CONV_COMMON_H
#define SPIO_CONV_COMMON_H

#ifndef SPIO_N
#error "shape macros (SPIO_N, SPIO_C, SPIO_H, SPIO_W, SPIO_R, SPIO_S, SPIO_PY, SPIO_PX) are required"
#endif

typedef _Float16 spio_half;
typedef _Float16 spio_half2 __attribute__((ext_vector_type(2)));
typedef _Float16 spio_half4 __attribute__((ext_vector_type(4)));
typedef _Float16 spio_half8 __attribute__((ext_vector_type(8)));
typedef float spio_float4 __attribute__((ext_vector_type(4)));
typedef unsigned int spio_uint2 __attribute__((ext_vector_type(2)));
typedef unsigned int spio_uint4 __attribute__((ext_vector_type(4)));
typedef short spio_short4 __attribute__((ext_vector_type(4)));

namespace spio {

// The convolution as the user states it (forward orientation).
constexpr int kN = SPIO_N;
constexpr int kC = SPIO_C;
constexpr int kH = SPIO_H;
constexpr int kW = SPIO_W;
constexpr int kR = SPIO_R;
constexpr int kS = SPIO_S;
constexpr int kPadY = SPIO_PY;
constexpr int kPadX = SPIO_PX;
constexpr int kP = kH + 2 * kPadY - kR + 1;
constexpr int kQ = kW + 2 * kPadX - kS + 1;
constexpr int kGroups = kC / 8;

static_assert(kC % 8 == 0, "channels must be a multiple of the group width 8");
static_assert(kP > 0 && kQ > 0, "empty output");

// The kernels use compiler builtins only, so they compile identically under
// hipRTC and under an offline hipcc build without any runtime header.
#define SPIO_DEVICE __device__ inline __attribute__((always_inline))
#define SPIO_LAUNCH_BOUNDS(threads) __attribute__((amdgpu_flat_work_group_size(threads, threads)))

SPIO_DEVICE int imin(int a, int b) { return a < b ? a : b; }
SPIO_DEVICE int imax(int a, int b) { return a > b ? a : b; }
SPIO_DEVICE int thread_id() { return (int)__builtin_amdgcn_workitem_id_x(); }
SPIO_DEVICE int block_id() { return (int)__builtin_amdgcn_workgroup_id_x(); }

// Workgroup barrier with LDS/global visibility among the waves of the group.
SPIO_DEVICE void block_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Orders the LDS accesses of the lanes of one wave: what some lanes stored before it is what
// other lanes of the same wave load after it.  The hardware executes the LDS operations of a
// wave in order anyway; this keeps the compiler from moving them across (the store and the load
// sit under disjoint lane masks, so nothing else tells it they depend on each other).
SPIO_DEVICE void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Whether neighbouring channel blocks of `gb` groups share 128-byte lines of the activations: their
// boundary lies inside a line unless both the block (gb * 16 bytes) and the pixel (2 C bytes) are whole
// lines.  With C = 296 (592 bytes a pixel) every boundary does, whatever gb is.
constexpr bool splits_lines(int gb, int gblks) { return gblks > 1 && ((gb * 16) % 128 != 0 || (kC * 2) % 128 != 0); }

// Tile of workgroup `id` in a grid of TILES: workgroup ids are dealt round-robin to the 8 XCDs, here runs
// of RUN consecutive tiles go to one XCD (what neighbours share, halo rows and lines, they share in that
// XCD's L2) before the next run goes to the next XCD.  0 = one contiguous range of tiles per XCD.  The
// tiles behind the last whole turn of 8 runs are dealt as 8 contiguous ranges, so every tile count gets
// the order, not only multiples of 8 * RUN.
constexpr int kXcds = 8;
template <int RUN, int TILES>
SPIO_DEVICE int xcd_tile(int id) {
    constexpr int TURN = kXcds * RUN;
    constexpr int WHOLE = RUN > 0 ? TILES / TURN * TURN : 0;
    const int x = id % kXcds, k = id / kXcds;  // XCD, position in its sequence
    if (RUN == 1) return id;
    if (RUN > 0 && id < WHOLE) return k / (RUN > 0 ? RUN : 1) * TURN + x * RUN + k % (RUN > 0 ? RUN : 1);
    constexpr int REST = TILES - WHOLE;
    return WHOLE + x * (REST / kXcds) + imin(x, REST % kXcds) + k - WHOLE / kXcds;
}
// Run length where channel blocks share lines and go fastest in the tile order: whole pixels.
constexpr int line_run(int run, int gblks) { return run <= 1 ? run : (run + gblks - 1) / gblks * gblks; }

// Whether column 4 u + kb of a pair's source columns is in the filter window of neither pixel.  The pair meets S + 1
// columns and a product takes four, so the last one has up to three more; their taps are zeros, but zero times an
// infinity is not.  The lanes that hold them multiply zeros instead: an infinite or NaN source pixel then reaches, as NaN,
// no output beyond its window but the one next to it that is the other of a pair.
SPIO_DEVICE bool in_no_window(int u, int kb) { return (kS + 1) % 4 != 0 && 4 * u + kb > kS; }

// Streaming accesses: activations are touched once per kernel, so they are
// loaded and stored with the non-temporal hint (measured on MI355X: a plain
// 16-byte-per-lane copy gains about 10% from it).
#ifndef SPIO_NT
#define SPIO_NT 1
#endif
SPIO_DEVICE spio_uint4 load_stream(const spio_uint4* p) {
#if SPIO_NT
    return __builtin_nontemporal_load(p);
#else
    return *p;
#endif
}
SPIO_DEVICE void store_stream(spio_uint4 v, spio_uint4* p) {
#if SPIO_NT
    __builtin_nontemporal_store(v, p);
#else
    *p = v;
#endif
}

// Kernels that write activations can store them as fp32 (SPIO_DST_F32): the same values, rounded to fp16
// once and widened on the way out, for a caller whose tensors are fp32.  A pass of its own over the result
// reads 2 bytes and writes 4 per element behind the 2 written here; stored wide at once it is 4 written.
#ifndef SPIO_DST_F32
#define SPIO_DST_F32 0
#endif
constexpr int kDstBytes = SPIO_DST_F32 ? 4 : 2;
// Bytes from pixel to pixel where a finished row is staged in LDS, `groups` units of 16 bytes and a spare one, or two: an
// odd number, so that the 8 bytes that 16 lanes store for as many pixels lie in different banks.  An even one folds them
// onto those of 8, 4, 2 pixels or one, which all lanes of a wave run into since a tile is pairs of pixels and every lane converts.
// With one spare unit -> odd: forward 32n 56c 112x112 (7 groups, a pitch of 128) 21.8 -> 15.6 us, 128n 24c 144x144 (3, 64)
// 46.1 -> 45.0, in tiles of 24 whole rows 53.2 -> 48.1, 64n 40c 56x56 5x5 (5, 96) equal.
constexpr int stage_pitch(int groups) { return 16 * (groups + 1 + groups % 2); }

// A finished row leaves LDS as 16-byte units of 8 channels, one per lane, which widen to 32 bytes: two
// stores.  In store j lane i of a wave writes half i % 2 of the unit of lane 32 j + i / 2, so that every
// store covers whole lines (1024 consecutive bytes where the units are).  A lane that wrote its own two halves
// would leave every second 16 bytes of a line to the other store; with the units dealt to quads of lanes every
// access covered half of each line: 128n 384c 14x14, quads -> whole lines, fused backward that stores fp32
// 23.4 -> 20.6 us, that also reads it 28.7 -> 23.3, forward that reads and stores it 26.5 -> 22.3.
constexpr int kDstStores = SPIO_DST_F32 ? 2 : 1;
SPIO_DEVICE spio_uint4 widen(spio_uint2 v) {
    union {
        spio_float4 f;
        spio_uint4 u;
    } o;
    union {
        spio_uint2 u;
        spio_half4 h;
    } i;
    i.u = v;
#pragma unroll
    for (int e = 0; e < 4; ++e) o.f[e] = (float)i.h[e];
    return o.u;
}

// Kernels can read activations (SPIO_SRC_F32: x of the forward pass, grad_output of a backward one) and
// weights (SPIO_W_F32, forward pass) that are fp32 and round them to fp16 on their way into LDS, as a
// conversion beforehand would: that is a pass of 4 bytes read and 2 written per element and a launch.  With
// SPIO_KEEP they store what they rounded as fp16 tensors too, for the backward pass or the next kernel of it:
// the 2 written remain, the pass over the 4 and reading the 2 again do not.  128n 384c 14x14 forward and
// backward: 68 us with conversions, 46 without (of 33 that its bytes take).
// Loads are the float32 stores in reverse: in load j lane i reads half i % 2 of the 32-byte unit of lane
// 32 j + i / 2.  A row in flight takes twice the registers, so half as many are in flight: as many bytes as of
// fp16 rows.
#ifndef SPIO_SRC_F32
#define SPIO_SRC_F32 0
#endif
#ifndef SPIO_W_F32
#define SPIO_W_F32 0
#endif
#ifndef SPIO_KEEP
#define SPIO_KEEP 0
#endif
constexpr int kSrcBytes = SPIO_SRC_F32 ? 4 : 2;
constexpr int kSrcLoads = SPIO_SRC_F32 ? 2 : 1;  // loads (and LDS writes) per cell of 8 channels
constexpr int kFilterLoads = SPIO_W_F32 ? 2 : 1;
SPIO_DEVICE spio_uint2 narrow(spio_uint4 v) {
    union {
        spio_uint4 u;
        spio_float4 f;
    } i;
    union {
        spio_half4 h;
        spio_uint2 u;
    } o;
    i.u = v;
#pragma unroll
    for (int e = 0; e < 4; ++e) o.h[e] = (spio_half)i.f[e];
    return o.u;
}
// The unit that thread `tid` takes part in moving by access j, and the byte of its 8 (fp16) or 16 (fp32)
// that the thread moves where a unit is two accesses.
SPIO_DEVICE int moved_unit(int tid, int j, int accesses) {
    return accesses == 1 ? tid : (tid & ~63) + 32 * j + ((tid & 63) >> 1);
}
SPIO_DEVICE int half_bytes(int tid, int accesses, int bytes) { return accesses == 1 ? 0 : (tid & 1) * bytes; }

// Closes a group of 16-byte buffer stores.  Such a store reads its data registers for a few
// cycles after it issues; an instruction that writes one of them in the very next slot can have
// its value stored instead (seen on gfx950 as stray values in the first two channels of some
// pixels).  The compiler keeps that slot free only for some operand forms of the store, so the
// kernels do not rely on it: nothing is scheduled across this point, and the wait state between
// the last store and whatever follows is explicit.
#ifndef SPIO_STORE_GUARD
#define SPIO_STORE_GUARD 1
#endif
SPIO_DEVICE void store_group_end() {
#if SPIO_STORE_GUARD
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 0");
    __builtin_amdgcn_sched_barrier(0);
#endif
}

// Device-scope fp32 add without a return value.
SPIO_DEVICE void atomic_add_f32(float* address, float value) {
    __hip_atomic_fetch_add(address, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Stores four sums of a second stage: as they are, or rounded to fp16 for a caller whose weights are fp16.
SPIO_DEVICE void store_sums(float* p, spio_float4 v) { *reinterpret_cast<spio_float4*>(p) = v; }
SPIO_DEVICE void store_sums(spio_half* p, spio_float4 v) {
    spio_half4 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = (spio_half)v[e];
    *reinterpret_cast<spio_half4*>(p) = h;
}
// A second stage comes twice: <name>_reduce stores float sums, <name>_reduce_h the same rounded to fp16.
#define SPIO_CONCAT2(a, b) a##b
#define SPIO_CONCAT(a, b) SPIO_CONCAT2(a, b)

// Bit-cast helpers between the 16-byte vector views of one (pixel, group).
union Pack16 {
    spio_uint4 u;
    spio_uint4 i;  // the buffer builtins' 128-bit operand type
    spio_half8 h;
    spio_half4 h4[2];
};

union Pack8 {
    spio_uint2 u;
    spio_half4 h;
    spio_short4 s;
};

// Eight filter values as they were loaded, as fp16.
SPIO_DEVICE spio_uint4 filter_unit(const spio_uint4 (&raw)[kFilterLoads]) {
    if (!SPIO_W_F32) return raw[0];
    const spio_uint2 lo = narrow(raw[0]), hi = narrow(raw[kFilterLoads - 1]);
    return spio_uint4{lo[0], lo[1], hi[0], hi[1]};
}
// Unit `i` of a filter tensor.
SPIO_DEVICE void load_filter_unit(spio_uint4 (&raw)[kFilterLoads], const spio_half* weights, long long i) {
    const spio_uint4* p = reinterpret_cast<const spio_uint4*>(weights) + i * kFilterLoads;
#pragma unroll
    for (int j = 0; j < kFilterLoads; ++j) raw[j] = p[j];
}

}  // namespace spio

#endif  // SPIO_CONV_COMMON_H
