// Backward of the channel LayerNorm of layernorm_2d.hip (NHWC fp16 tensors, gfx950).
//
// The reference ships the forward device source only (spio/src/layernorm_2d.cu:81-222); this is
// the gradient of that contract, with the statistics recomputed from the input:
//   xhat[x][c] = (in[x][c] - mean[x]) * rstd[x]              mean, rstd as in the forward kernel
//   g[x][c]    = dout[x][c] * weight[c]                       (weight = 1 without one)
//   din[x][c]  = rn16(rstd[x] * (g - mean_c(g) - xhat * mean_c(g * xhat)))
//   dweight[c] = sum_x dout[x][c] * xhat[x][c]                fp32
//   dbias[c]   = sum_x dout[x][c]                             fp32
//
// Design: the lane mapping of the forward kernel (LPP lanes share a pixel, a lane keeps the same
// channels for all its pixels), so the per-channel sums stay in registers over the whole
// workgroup loop.  At the end the lanes of a wave that hold the same channels are added by an
// xor butterfly, the waves through LDS, and the workgroup writes one row of
// `partials[workgroup][2][C]` with plain stores: every row is written completely, so the
// workspace needs no zeroing and nothing is atomic (with atomics every workgroup would add to the
// same C addresses, one after the other).  The small <name>_reduce kernel below adds the rows
// into `sums[2][C]` (0 = grad_weight, 1 = grad_bias), which it overwrites.  HBM-bound: 4 bytes in,
// 2 bytes out per element.
//
// The channel sums keep workgroups few (one or two per CU), so a wave has its own loads to wait for: the next
// pass is requested before a pass is worked on.  With the instructions of a pass from 17.5 to 13.5 an element
// (mixed-precision multiply-adds instead of conversions), both stages: 128n 96c 56x56 (231 MB) 46.9 -> 41.3 us,
// 192c 28x28 26.2 -> 24.5, 384c 14x14 16.6 -> 15.2, 4n 96c 56x56 7.1 -> 6.4; 768c 7x7 10.9, as before: two
// launches and a pass.
#ifndef SPIO_LN_C
#error "SPIO_LN_C, SPIO_LN_PIXELS, SPIO_LN_LPP, SPIO_LN_THREADS, SPIO_LN_GRID are required"
#endif
#ifndef SPIO_LN_UNROLL
#define SPIO_LN_UNROLL 2
#endif
#ifndef SPIO_LN_HAS_WEIGHT
#define SPIO_LN_HAS_WEIGHT 1
#endif
#ifndef SPIO_LN_EPS
#define SPIO_LN_EPS 1e-6f
#endif

typedef _Float16 ln_half8 __attribute__((ext_vector_type(8)));
typedef unsigned int ln_uint4 __attribute__((ext_vector_type(4)));
typedef float ln_float4 __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t ln_rsrc;

namespace {

constexpr int C = SPIO_LN_C;
constexpr long long PIXELS = SPIO_LN_PIXELS;
constexpr int UNITS = C / 8;              // 16-byte units per pixel
constexpr int LPP = SPIO_LN_LPP;          // lanes per pixel (power of two, <= 64)
constexpr int UPL = (UNITS + LPP - 1) / LPP;  // units per lane
constexpr int THREADS = SPIO_LN_THREADS;
constexpr int WAVES = THREADS / 64;
constexpr int PPW = 64 / LPP;             // pixels per wave and pass
constexpr int PPB = PPW * WAVES;          // pixels per workgroup and pass
constexpr int UN = SPIO_LN_UNROLL;
constexpr unsigned OOB = 0x80000000u;
constexpr bool kAllLive = LPP * UPL == UNITS;  // no lane holds a unit past the pixel's last
static_assert(C % 8 == 0 && (LPP & (LPP - 1)) == 0 && LPP <= 64 && LPP * UPL >= UNITS, "bad geometry");

union Pack {
    ln_uint4 u;
    ln_half8 h;
};

template <int CTRL>
__device__ inline float dpp_add(float v) {
    const int other = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false);
    return v + __builtin_bit_cast(float, other);
}
__device__ inline float lane_xor_add(float v, int m) {
    const int lane = (int)__builtin_amdgcn_workitem_id_x() & 63;
    const int other = __builtin_amdgcn_ds_bpermute(((lane ^ m) << 2), __builtin_bit_cast(int, v));
    return v + __builtin_bit_cast(float, other);
}
template <int CTRL>
__device__ inline void dpp_add_all(float (&v)[UN]) {
#pragma unroll
    for (int u = 0; u < UN; ++u) v[u] = dpp_add<CTRL>(v[u]);
}
// Sums over the LPP lanes of each of UN pixels; every lane ends up with the totals (as in the forward kernel).
__device__ inline void pixel_sums(float (&v)[UN]) {
    if (LPP >= 2) dpp_add_all<0xB1>(v);    // quad_perm [1,0,3,2]
    if (LPP >= 4) dpp_add_all<0x4E>(v);    // quad_perm [2,3,0,1]
    if (LPP >= 8) dpp_add_all<0x141>(v);   // row_half_mirror
    if (LPP >= 16) dpp_add_all<0x140>(v);  // row_mirror
#pragma unroll
    for (int m = 16; m < LPP; m <<= 1)
#pragma unroll
        for (int u = 0; u < UN; ++u) v[u] = lane_xor_add(v[u], m);
}
// Sum over the PPW lanes of a wave that hold the same channels (lanes sub, sub + LPP, ...).
__device__ inline float channel_sum(float v) {
#pragma unroll
    for (int m = LPP; m < 64; m <<= 1) v = lane_xor_add(v, m);
    return v;
}

// Eight fp32 values of a [C] vector from byte offset `off` on; zeros where that is OOB.
__device__ inline void load_channels(float (&v)[8], const float* p, unsigned off) {
    const ln_rsrc rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, C * 4, 0x00020000);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const ln_float4 q =
            __builtin_bit_cast(ln_float4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off + 16 * h), 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * h + e] = q[e];
    }
}

}  // namespace

extern "C" __global__ void __attribute__((amdgpu_flat_work_group_size(THREADS, THREADS)))
SPIO_KERNEL_NAME(float* __restrict__ partials, ln_uint4* __restrict__ din, const ln_uint4* __restrict__ in,
                 const ln_uint4* __restrict__ dout, const float* __restrict__ weight) {
    constexpr long long num_workgroups = SPIO_LN_GRID;
    __shared__ float red[WAVES][2][LPP * UPL * 8];
    const int tid = (int)__builtin_amdgcn_workitem_id_x();
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int sub = lane % LPP;
    const int pix_in_pass = wave * PPW + lane / LPP;

    // SGPRs of 1 and -0 that the compiler does not know for constants: (float)h * one + c and (float)h * w + zero
    // are single mixed-precision instructions, where h + c and h * w are a conversion and another one (and the
    // same values).
    float one = 1.f, zero = -0.f;
    asm("" : "+s"(one), "+s"(zero));

    float w[UPL][8];
    bool live[UPL];
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
        const int unit = sub + k * LPP;
        live[k] = kAllLive || unit < UNITS;
#pragma unroll
        for (int e = 0; e < 8; ++e) w[k][e] = 1.f;
        if (SPIO_LN_HAS_WEIGHT) load_channels(w[k], weight, live[k] ? unit * 32 : OOB);
    }
    float dw[UPL][8], db[UPL][8];
#pragma unroll
    for (int k = 0; k < UPL; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) dw[k][e] = db[k][e] = 0.f;

    unsigned off[UN][UPL];
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
        for (int k = 0; k < UPL; ++k)
            off[u][k] = live[k] ? (unsigned)(((u * PPB + pix_in_pass) * UNITS + sub + k * LPP) * 16) : OOB;

    constexpr long long PASS_PIXELS = (long long)PPB * UN;
    constexpr long long PASSES = (PIXELS + PASS_PIXELS - 1) / PASS_PIXELS;
    static_assert(num_workgroups <= PASSES, "every workgroup has a pass");
    // 32-bit buffer offsets cover 2 GiB: the descriptors are rebased per pass.  Passes behind the last one
    // have descriptors of size zero: loads give zeros, stores are dropped.
    auto pass_rsrc = [&](const void* base, long long it) {
        const long long first = it < PASSES ? it * PASS_PIXELS : 0;
        const long long left = it < PASSES ? PIXELS - first : 0;
        const int npix = (int)(left < PASS_PIXELS ? left : PASS_PIXELS);
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<unsigned char*>(reinterpret_cast<const unsigned char*>(base)) + first * C * 2, 0, npix * C * 2,
            0x00020000);
    };
    auto load_pass = [&](Pack(&vx)[UN][UPL], Pack(&vd)[UN][UPL], long long it) {
        const ln_rsrc rs_in = pass_rsrc(in, it), rs_dout = pass_rsrc(dout, it);
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int k = 0; k < UPL; ++k) {
                vx[u][k].u = __builtin_amdgcn_raw_buffer_load_b128(rs_in, (int)off[u][k], 0, 2);
                vd[u][k].u = __builtin_amdgcn_raw_buffer_load_b128(rs_dout, (int)off[u][k], 0, 2);
            }
    };
    // Statistics as in the forward kernel (pixels past the end and dead units load zeros: rstd is finite, every
    // product below is zero, their stores are dropped).  The sums of all UN pixels take each step of their
    // butterflies together: one alone would wait for every step.
    auto work_pass = [&](const Pack(&vx)[UN][UPL], const Pack(&vd)[UN][UPL], long long it) {
        float mean[UN], rstd[UN], m1[UN], m2[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            float s[2] = {0.f, 0.f};  // two chains of additions: few pixels in flight wait for one
#pragma unroll
            for (int k = 0; k < UPL; ++k)
#pragma unroll
                for (int e = 0; e < 8; ++e) s[e & 1] = __builtin_fmaf((float)vx[u][k].h[e], one, s[e & 1]);
            mean[u] = s[0] + s[1];
        }
        pixel_sums(mean);
        float xhat[UN][UPL][8], g[UN][UPL][8];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            float s[2] = {0.f, 0.f};
#pragma unroll
            for (int k = 0; k < UPL; ++k) {
                const float nmean = live[k] ? mean[u] * (-1.0f / C) : 0.f;  // x - mean is zero in dead units
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    xhat[u][k][e] = __builtin_fmaf((float)vx[u][k].h[e], one, nmean);
                    s[e & 1] = __builtin_fmaf(xhat[u][k][e], xhat[u][k][e], s[e & 1]);
                }
            }
            rstd[u] = s[0] + s[1];
        }
        pixel_sums(rstd);
        // xhat, g = dy * w, the two means, the channel sums
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            rstd[u] = __builtin_amdgcn_rsqf(rstd[u] * (1.0f / C) + SPIO_LN_EPS);
            m1[u] = m2[u] = 0.f;
#pragma unroll
            for (int k = 0; k < UPL; ++k)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float dy = (float)vd[u][k].h[e];
                    xhat[u][k][e] *= rstd[u];
                    g[u][k][e] = SPIO_LN_HAS_WEIGHT ? __builtin_fmaf(dy, w[k][e], zero) : dy;
                    m1[u] += g[u][k][e];
                    m2[u] = __builtin_fmaf(g[u][k][e], xhat[u][k][e], m2[u]);
                    dw[k][e] = __builtin_fmaf(dy, xhat[u][k][e], dw[k][e]);
                    db[k][e] = __builtin_fmaf(dy, one, db[k][e]);
                }
        }
        pixel_sums(m1);
        pixel_sums(m2);
        const ln_rsrc rs_din = pass_rsrc(din, it);
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const float c1 = -rstd[u] * (m1[u] * (1.0f / C)), c2 = -rstd[u] * (m2[u] * (1.0f / C));
#pragma unroll
            for (int k = 0; k < UPL; ++k) {
                Pack o;
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    o.h[e] = (_Float16)__builtin_fmaf(xhat[u][k][e], c2, __builtin_fmaf(g[u][k][e], rstd[u], c1));
                __builtin_amdgcn_raw_buffer_store_b128(o.u, rs_din, (int)off[u][k], 0, 2);
            }
        }
    };

    // The next pass is requested before this one is worked on.  Stores and loads leave one queue in order, so a
    // wait for the loads of a pass counts what was issued behind them: the stores of the pass before and the
    // loads of the next one.  The first pass has no stores before it and gets dropped ones in their place;
    // without them the count that fits every pass would wait for the stores too.
    Pack vx0[UN][UPL], vd0[UN][UPL], vx1[UN][UPL], vd1[UN][UPL];
    // What a turn ends with in flight counts as used there: left unused on that way out the loads would be moved
    // behind the branch, next to their use.
    auto drop_pass = [&](const Pack(&vx)[UN][UPL], const Pack(&vd)[UN][UPL]) {
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int k = 0; k < UPL; ++k) asm volatile("" ::"v"(vx[u][k].u), "v"(vd[u][k].u));
    };
    long long it = (long long)__builtin_amdgcn_workgroup_id_x();
    load_pass(vx0, vd0, it);
    if (PASSES <= num_workgroups) {
        work_pass(vx0, vd0, it);
    } else {
        __builtin_amdgcn_sched_barrier(0);
        const ln_rsrc none = pass_rsrc(din, PASSES);
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int k = 0; k < UPL; ++k)
                __builtin_amdgcn_raw_buffer_store_b128(ln_uint4{0u, 0u, 0u, 0u}, none, (int)off[u][k], 0, 2);
        __builtin_amdgcn_sched_barrier(0);
        while (true) {  // (no workgroup is without a pass)
            load_pass(vx1, vd1, it + num_workgroups);
            __builtin_amdgcn_sched_barrier(0);
            work_pass(vx0, vd0, it);
            __builtin_amdgcn_sched_barrier(0);
            it += num_workgroups;
            if (it >= PASSES) {
                drop_pass(vx1, vd1);
                break;
            }
            load_pass(vx0, vd0, it + num_workgroups);
            __builtin_amdgcn_sched_barrier(0);
            work_pass(vx1, vd1, it);
            __builtin_amdgcn_sched_barrier(0);
            it += num_workgroups;
            if (it >= PASSES) {
                drop_pass(vx0, vd0);
                break;
            }
        }
    }

    // ---- the workgroup's row of partial sums: lanes with the same channels, then the waves ----
#pragma unroll
    for (int k = 0; k < UPL; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            dw[k][e] = channel_sum(dw[k][e]);
            db[k][e] = channel_sum(db[k][e]);
        }
    if (lane < LPP) {
#pragma unroll
        for (int k = 0; k < UPL; ++k)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                red[wave][0][(sub + k * LPP) * 8 + e] = dw[k][e];
                red[wave][1][(sub + k * LPP) * 8 + e] = db[k][e];
            }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    float* row = partials + (long long)__builtin_amdgcn_workgroup_id_x() * 2 * C;
    for (int i = tid; i < 2 * C; i += THREADS) {
        const int which = i / C;
        const int c = i % C;
        float v = 0.f;
#pragma unroll
        for (int wv = 0; wv < WAVES; ++wv) v += red[wv][which][c];
        row[i] = v;
    }
}

// Second stage: sums[i] = sum over the workgroups' rows of partials[row][i], i < 2*C.  A workgroup
// owns 32 columns; its 8 slices each add the rows r = slice, slice + 8, ... with up to 32 loads
// in flight, and meet in LDS.  Every element has one owner: no atomics, no dependence on timing.
#define SPIO_LN_CONCAT2(a, b) a##b
#define SPIO_LN_CONCAT(a, b) SPIO_LN_CONCAT2(a, b)
extern "C" __global__ void __attribute__((amdgpu_flat_work_group_size(256, 256)))
SPIO_LN_CONCAT(SPIO_KERNEL_NAME, _reduce)(float* __restrict__ sums, const float* __restrict__ partials) {
    constexpr int ROWS = SPIO_LN_GRID;
    constexpr int COLS = 32;
    constexpr int SLICES = 256 / COLS;
    // as many rows in flight per thread as a slice has, up to 32: one round trip to memory for up
    // to 256 rows (with 8 in flight the stage took 1.5-2 us longer on the 7x7 and 14x14 shapes)
    constexpr int UNR = (ROWS + SLICES - 1) / SLICES < 32 ? (ROWS + SLICES - 1) / SLICES : 32;
    __shared__ float red[SLICES][COLS];
    const int tid = (int)__builtin_amdgcn_workitem_id_x();
    const int cl = tid % COLS;
    const int slice = tid / COLS;
    const int col = (int)__builtin_amdgcn_workgroup_id_x() * COLS + cl;
    float sum = 0.f;
    if (col < 2 * C) {
        for (int base = slice; base < ROWS; base += SLICES * UNR) {
            float v[UNR];
#pragma unroll
            for (int i = 0; i < UNR; ++i) {
                const int r = base + i * SLICES;
                v[i] = r < ROWS ? partials[(long long)r * 2 * C + col] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < UNR; ++i) sum += v[i];
        }
    }
    red[slice][cl] = sum;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (slice == 0 && col < 2 * C) {
#pragma unroll
        for (int i = 1; i < SLICES; ++i) sum += red[i][cl];
        sums[col] = sum;
    }
}
