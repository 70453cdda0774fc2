// Dense int8 convolution with or without a window (also Gemm) for layers with few outputs: one image, the 20 x 20
// level of a detector, a classifier with a handful of classes.
//
// What it computes is conv2d_11cn / _33cn / _hwcn (esp-dl/dl/base/dl_base_conv2d.cpp:9-163) under
// conv_operation_shell's window clipping (esp-dl/dl/base/dl_base.hpp:940-1191) with the n_wise epilogue
// (esp-dl/dl/base/dl_base_activate_buffer.hpp:27-36, 61-72, 173-181, 201-210), any channel count.
//
// Such a launch is bound by latency, not by any throughput: a tile of 64 x 64 outputs per workgroup leaves most of
// the device without work and walks the reduction axis in dozens of steps with a barrier each (13 x 13 x 256 -> 128,
// 3 x 3, one image: six workgroups of 36 steps, 10 us).  Here a workgroup owns 16 pixels x 16 NT filters, its four
// wavefronts split the REDUCTION axis (SPLIT), and a wavefront reads both operands straight from memory in
// the layout the matrix instruction wants, G steps of 64 per batch of loads with the next batch in flight, so its
// life is a few memory round trips; the four partial sums meet in LDS, and wavefront t finishes filter tile t.
// For reductions of under four steps (not SPLIT) the wavefronts take neighbouring pixel tiles instead.
// Lane (col, quad) holds unit 4 step + quad of pixel col (operand B) and of filter row col (operand A); filter rows
// are permuted (row i of tile t is filter 4 NT (i / 4) + 4 t + i % 4) so that a lane's results are 4 NT neighbours.
// Measured against the kernels such layers took before, as nodes of a graph: 13 x 13 x 256 -> 64, 3 x 3 15.5 -> 5.0 us;
// 13 x 13 x 512 -> 256, 1 x 1 5.6 -> 3.3 us; 1 x 4096 -> 256 6.8 -> 4.7 us; 17 x 27 x 74 -> 11, 3 x 3 at stride 2 31.2 -> 3.8 us.
// In a chain of launches 1.2 us pass between a kernel's end and the next one's start; the rest is the instructions of ONE
// wavefront, four cycles each and more, in front of its loads and behind them.  So a lane finds its units by additions (a
// division takes six quarter-rate multiplications), layers of one tap have builds of their own, the epilogue's operands are
// requested before the loads and prepared while those are on their way (start values, the vote on the short form), and what is
// left behind the barrier is sums, a shift and a packed clamp.  14 x 14 x 64 -> 384 3.0 -> 2.4 us, 7 x 7 x 960 -> 160 3.1 -> 2.6,
// 26 x 26 x 64 -> 64, 3 x 3 3.2 -> 2.8 (launch to launch, kernel itself 2.0 -> 1.5).  What did not help: a reduction split eight
// ways (2 % at 36 steps, 9 % lost at 4: the loads of one compute unit's wavefronts take turns).
#include "conv_window.h"

namespace espdl {

namespace {

using namespace window;

constexpr int kThreads = 256;

struct NarrowArgs {
    WindowArgs win;
    const int32_t *bias, *shift;
    const int8_t *lut, *res;
    int8_t *out;
    int n_pix, out_c, out_pitch, res_pitch;
    int ksteps, relu, half_even, n_shift, res_shift;
    unsigned bound; // of a sum of products, see Short4
    int dense_pixels; // output pixel m of a pointwise layer reads input pixel m
    // From a lane's unit to its next one, where neither the channels nor the window's columns run out in between, and what
    // is added where they do.
    struct {
        int units, channels, column, row, in, filter;
        int tap_channels, in_tap, filter_tap;
        int window_columns, in_row;
    } step;
    int through; // whole dwords that go through the L2 caches as they are stored
};

// The units of one lane in steps of the launch's stride, without a division per unit: where a unit lies follows from where
// the one before it lay by additions, with one carry from channels to the tap's column and one from there to its row.
template <bool ALIGNED, bool POINT>
struct UnitWalk {
    int u, j16;       // unit, its first channel
    int ky, kx;       // row and column of its tap in the window, times the dilation
    int in_off, w_off;
    int base, iy, ix; // of the pixel's window
    bool alive;       // the pixel exists

    __device__ __forceinline__ void start(const NarrowArgs &a, int first, int m)
    {
        const WindowArgs &w = a.win;
        alive = m < a.n_pix;
        u = first;
        if constexpr (POINT) {
            // one tap: the window is the pixel
            j16 = 16 * first;
            base = (int)((unsigned)m * (unsigned)w.in_pitch);
            if (a.dense_pixels == 0) { // uniform: a stride
                const unsigned n = fastdiv((unsigned)m, w.fd_ohw), rem = (unsigned)m - n * w.fd_ohw.d;
                const unsigned oy = fastdiv(rem, w.fd_ow), ox = rem - oy * w.fd_ow.d;
                base = (((int)n * w.in_h + (int)oy * w.stride_h) * w.in_w + (int)ox * w.stride_w) * w.in_pitch;
            }
            w_off = 16 * first;
            in_off = base + 16 * first;
            ky = kx = iy = ix = 0;
        } else {
            const unsigned n = fastdiv((unsigned)m, w.fd_ohw), rem = (unsigned)m - n * w.fd_ohw.d;
            const unsigned oy = fastdiv(rem, w.fd_ow), ox = rem - oy * w.fd_ow.d;
            const unsigned tap = fastdiv((unsigned)first, w.fd_upt), row = fastdiv(tap, w.fd_kw);
            j16 = 16 * (first - (int)(tap * w.fd_upt.d));
            ky = (int)row * w.dil_h;
            kx = (int)(tap - row * w.fd_kw.d) * w.dil_w;
            iy = (int)oy * w.stride_h - w.pad_top;
            ix = (int)ox * w.stride_w - w.pad_left;
            base = (((int)n * w.in_h + iy) * w.in_w + ix) * w.in_pitch;
            in_off = base + (ky * w.in_w + kx) * w.in_pitch + j16;
            w_off = (int)tap * w.in_c + j16;
        }
    }
    __device__ __forceinline__ void advance(const NarrowArgs &a)
    {
        u += a.step.units;
        in_off += a.step.in;
        w_off += a.step.filter;
        if constexpr (POINT) {
            j16 += 16 * a.step.units;
        } else {
            j16 += a.step.channels;
            kx += a.step.column;
            ky += a.step.row;
            if (j16 >= a.step.tap_channels) {
                j16 -= a.step.tap_channels;
                kx += a.win.dil_w;
                in_off += a.step.in_tap;
                w_off += a.step.filter_tap;
            }
            if (kx >= a.step.window_columns) {
                kx -= a.step.window_columns;
                ky += a.win.dil_h;
                in_off += a.step.in_row;
            }
        }
    }
    // Channels the unit holds (<= 0: it does not exist).
    __device__ __forceinline__ int channels(const NarrowArgs &a) const
    {
        return u < a.win.n_units ? a.win.in_c - j16 : 0;
    }
    __device__ __forceinline__ v4i pixel(const NarrowArgs &a, __amdgpu_buffer_rsrc_t rsrc) const
    {
        bool ok = alive && u < a.win.n_units;
        if constexpr (!POINT)
            ok = ok && (unsigned)(iy + ky) < (unsigned)a.win.in_h && (unsigned)(ix + kx) < (unsigned)a.win.in_w;
        return load16<ALIGNED>(rsrc, ok ? in_off : kParked, a.win.in_bytes);
    }
    __device__ __forceinline__ v4i filter(const NarrowArgs &a, __amdgpu_buffer_rsrc_t rsrc, int row) const
    {
        return load16<ALIGNED>(rsrc, u < a.win.n_units ? row + w_off : kParked, a.win.w_bytes);
    }
};

template <int NT, bool SPLIT, bool ALIGNED, bool POINT>
__device__ __forceinline__ void narrow_tile(const NarrowArgs &a, int bx, int by)
{
    constexpr int G = NT >= 4 ? 2 : 4;
    constexpr int MINE = SPLIT ? 1 : NT; // filter tiles a wavefront finishes
    __shared__ v4i part[SPLIT ? 4 : 1][SPLIT ? NT : 1][64];
    __shared__ int8_t lut_l[256];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int m = (SPLIT ? bx : bx * 4 + wave) * 16 + col;
    const int n0 = by * 16 * NT;

    // What the epilogue needs is requested first, its addresses take no arithmetic: this wavefront's filter tiles.  Filters
    // past the last one lie past the descriptors' ends and read as zeros.
    const bool finisher = !SPLIT || wave < NT;
    v4i bias[MINE], shift[MINE];
    int res[MINE];
    int lut = 0;
    if (finisher) { // uniform
        const __amdgpu_buffer_rsrc_t b_rsrc =
            tensor_rsrc(reinterpret_cast<const int8_t *>(a.bias), a.bias != nullptr ? 4 * a.out_c : 0);
        const __amdgpu_buffer_rsrc_t s_rsrc = tensor_rsrc(reinterpret_cast<const int8_t *>(a.shift), 4 * a.n_shift);
#pragma unroll
        for (int t = 0; t < MINE; t++) {
            const int f = n0 + 4 * NT * quad + 4 * (SPLIT ? wave : t);
            if ((a.out_c & 3) == 0) { // uniform
                bias[t] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, 4 * f, 0, 0));
                shift[t] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(s_rsrc, 4 * f, 0, 0));
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    bias[t][r] = __builtin_amdgcn_raw_buffer_load_b32(b_rsrc, 4 * (f + r), 0, 0);
                    shift[t][r] = __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, 4 * (f + r), 0, 0);
                }
            }
            if (a.n_shift == 1) { // uniform
                const int s = __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, 0, 0, 0);
                shift[t] = v4i{s, s, s, s};
            }
        }
    }
    if (a.lut != nullptr)
        lut = a.lut[tid];

    const __amdgpu_buffer_rsrc_t in_rsrc = tensor_rsrc(a.win.in, a.win.in_bytes);
    const __amdgpu_buffer_rsrc_t w_rsrc = tensor_rsrc(a.win.w, a.win.w_bytes);
    int row[NT]; // a filter past the last one reads the last one again, its results are dropped
#pragma unroll
    for (int t = 0; t < NT; t++)
        row[t] = min(n0 + 4 * NT * (col >> 2) + 4 * t + (col & 3), a.out_c - 1) * a.win.w_len;

    struct Batch {
        v4i b[G], w[G][NT];
        int n[G];
    };
    UnitWalk<ALIGNED, POINT> walk;
    walk.start(a, 4 * (SPLIT ? wave : 0) + quad, m);
    const int steps = SPLIT ? (a.ksteps - wave + 3) >> 2 : a.ksteps; // of this wavefront
    auto request = [&](Batch &t) {
#pragma unroll
        for (int i = 0; i < G; i++) {
            if constexpr (!ALIGNED)
                t.n[i] = walk.channels(a);
            t.b[i] = walk.pixel(a, in_rsrc);
#pragma unroll
            for (int f = 0; f < NT; f++)
                t.w[i][f] = walk.filter(a, w_rsrc, row[f]);
            walk.advance(a);
        }
    };
    Batch cur, nxt;
    request(cur);
    // while the operands are on their way
    const bool half_even = a.half_even != 0;
    bool general = false;
    Short4 consts[MINE];
    int8_t *dst = nullptr;
    if (finisher) { // uniform
        dst = a.out + (long long)m * a.out_pitch;
        if (a.res != nullptr) // uniform
#pragma unroll
            for (int t = 0; t < MINE; t++) {
                const int f = n0 + 4 * NT * quad + 4 * (SPLIT ? wave : t);
                const int8_t *p = a.res + (long long)min(m, a.n_pix - 1) * a.res_pitch;
                res[t] = 0;
                if (f + 4 <= a.out_c) {
                    res[t] = *reinterpret_cast<const int_unaligned *>(p + f);
                } else {
#pragma unroll
                    for (int r = 0; r < 3; r++)
                        if (f + r < a.out_c)
                            res[t] |= (int)(unsigned char)p[f + r] << (8 * r);
                }
            }
        bool bad = false;
#pragma unroll
        for (int t = 0; t < MINE; t++) {
            const int f = n0 + 4 * NT * quad + 4 * (SPLIT ? wave : t);
            if (a.out_c & 3) // uniform
#pragma unroll
                for (int r = 0; r < 4; r++)
                    shift[t][r] = f + r < a.out_c ? shift[t][r] : 1;
            bad = bad || (f < a.out_c && !short4_ok(bias[t], shift[t], a.bound));
        }
        general = __any(bad);
#pragma unroll
        for (int t = 0; t < MINE; t++)
            consts[t] = make_short4(bias[t], shift[t], general, half_even);
    }

    v4i acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
        acc[t] = v4i{0, 0, 0, 0};
    // (steps past the last one have zeros on both sides)
    auto products = [&](const Batch &t) {
#pragma unroll
        for (int i = 0; i < G; i++)
#pragma unroll
            for (int f = 0; f < NT; f++)
                acc[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(mask_unit<ALIGNED>(t.w[i][f], ALIGNED ? 16 : t.n[i]), t.b[i], acc[f], 0, 0, 0);
    };
    for (int s = 0; s < steps; s += 2 * G) {
        if (s + G < steps)
            request(nxt);
        products(cur);
        if (s + G < steps) {
            if (s + 2 * G < steps)
                request(cur);
            products(nxt);
        }
    }
    if (a.lut != nullptr)
        lut_l[tid] = (int8_t)lut;
    if constexpr (SPLIT) {
#pragma unroll
        for (int t = 0; t < NT; t++)
            part[wave][t][lane] = acc[t];
    }
    if (SPLIT || a.lut != nullptr)
        __syncthreads();
    if (!finisher) // uniform
        return;
#pragma unroll
    for (int t = 0; t < MINE; t++) {
        v4i sum = acc[t] + consts[t].start;
        if constexpr (SPLIT) {
            sum = part[0][wave][lane] + part[1][wave][lane] + part[2][wave][lane] + part[3][wave][lane] + consts[t].start;
        }
        const int f = n0 + 4 * NT * quad + 4 * (SPLIT ? wave : t);
        int word;
        if (general) // uniform, as are the next ones
            word = finish_general4(sum, consts[t].shift, a.relu, a.half_even);
        else
            word = finish_short4(sum, consts[t].shift, a.relu != 0, half_even);
        if (a.lut != nullptr) {
            const int at = word ^ (int)0x80808080u;
            word = (int)(unsigned char)lut_l[at & 255] | (int)(unsigned char)lut_l[(at >> 8) & 255] << 8 |
                (int)(unsigned char)lut_l[(at >> 16) & 255] << 16 | (int)(unsigned char)lut_l[(unsigned)at >> 24] << 24;
        }
        if (a.res != nullptr)
            word = sat_add4_pairs(word, a.res_shift != 0 ? requant4_s8(res[t], make_requant4(a.res_shift)) : res[t]);
        if (m >= a.n_pix || f >= a.out_c)
            continue;
        if (f + 4 <= a.out_c) {
            if (a.through) // uniform
                __hip_atomic_store(reinterpret_cast<int *>(dst + f), word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else
                *reinterpret_cast<int_unaligned *>(dst + f) = word;
        } else {
#pragma unroll
            for (int r = 0; r < 3; r++)
                if (f + r < a.out_c)
                    dst[f + r] = (int8_t)(word >> (8 * r));
        }
    }
}

template <int NT, bool SPLIT, bool ALIGNED, bool POINT>
__global__ __launch_bounds__(kThreads) void conv2d_s8_narrow_kernel(const NarrowArgs a)
{
    narrow_tile<NT, SPLIT, ALIGNED, POINT>(a, (int)blockIdx.x, (int)blockIdx.y);
}

// Several layers that do not depend on one another in one launch (the same level of a detector's heads): each is too small for
// the device, and one after the other they pay a launch's 1.2 us and a wavefront's latency each (52, 26 and 13 pixels square, 64 ->
// 80 with a table, 1 x 1: 11 us one by one, 3.6 together; 3 x 3 of 64, 128, 256 -> 64: 15 and 6).  One filter tile per wavefront
// for all of them: what that costs a layer that took two by itself, workgroups of the others would have to wait for anyway.
struct NarrowGroup {
    NarrowArgs layer[kMostGrouped];
    int first[kMostGrouped]; // first workgroup of a layer; past the last one: no workgroup reaches it
    FastDiv columns[kMostGrouped]; // workgroups of a row of its grid
};
template <bool SPLIT, bool POINT>
__global__ __launch_bounds__(kThreads) void conv2d_s8_narrow_group_kernel(const NarrowGroup g)
{
    int i = 0;
#pragma unroll
    for (int k = 1; k < kMostGrouped; k++)
        i += (int)blockIdx.x >= g.first[k] ? 1 : 0;
    const unsigned at = blockIdx.x - g.first[i];
    const unsigned by = fastdiv(at, g.columns[i]);
    narrow_tile<1, SPLIT, true, POINT>(g.layer[i], (int)(at - by * g.columns[i].d), (int)by);
}

template <int NT, bool SPLIT>
void launch_split(const NarrowArgs &a, bool aligned, bool point, hipStream_t stream)
{
    const unsigned tiles = (unsigned)((a.n_pix + 15) / 16);
    const dim3 grid(SPLIT ? tiles : (tiles + 3) / 4, (unsigned)((a.out_c + 16 * NT - 1) / (16 * NT)));
    if (aligned && point)
        hipLaunchKernelGGL((conv2d_s8_narrow_kernel<NT, SPLIT, true, true>), grid, dim3(kThreads), 0, stream, a);
    else if (aligned)
        hipLaunchKernelGGL((conv2d_s8_narrow_kernel<NT, SPLIT, true, false>), grid, dim3(kThreads), 0, stream, a);
    else if (point)
        hipLaunchKernelGGL((conv2d_s8_narrow_kernel<NT, SPLIT, false, true>), grid, dim3(kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((conv2d_s8_narrow_kernel<NT, SPLIT, false, false>), grid, dim3(kThreads), 0, stream, a);
}

template <int NT>
void launch_narrow(const NarrowArgs &a, bool split, bool aligned, bool point, hipStream_t stream)
{
    if (split)
        launch_split<NT, true>(a, aligned, point, stream);
    else
        launch_split<NT, false>(a, aligned, point, stream);
}

void launch_one(const NarrowArgs &a, int nt, bool split, bool aligned, bool point, hipStream_t stream)
{
    if (nt == 4)
        launch_narrow<4>(a, split, aligned, point, stream);
    else if (nt == 2)
        launch_narrow<2>(a, split, aligned, point, stream);
    else
        launch_narrow<1>(a, split, aligned, point, stream);
}

// A launch held back in this thread's open group.
struct Held {
    NarrowArgs args;
    int nt;
    bool split, point;
    hipStream_t stream;
};
thread_local Held held[kMostGrouped];
thread_local int n_held = 0;

} // namespace

// Shape of the launch: the reduction split over the wavefronts where they have a step each, and the widest filter
// tile that leaves every compute unit two workgroups (pixels are read once per filter tile).
struct NarrowPlan {
    bool split;
    int nt;
    long long groups;
    int ksteps;
};

static NarrowPlan narrow_plan(const ConvGeom &g, int cu_count)
{
    NarrowPlan p;
    const long long cus = cu_count > 0 ? cu_count : 256;
    p.ksteps = (g.k_h * g.k_w * ((g.in_c + 15) / 16) + 3) / 4;
    p.split = p.ksteps >= 4;
    const long long tiles = ((long long)g.batch * g.out_h * g.out_w + 15) / 16;
    const long long rows = p.split ? tiles : (tiles + 3) / 4;
    for (p.nt = g.out_c > 32 ? 4 : (g.out_c > 16 ? 2 : 1); p.nt > 1; p.nt /= 2)
        if (rows * ((g.out_c + 16 * p.nt - 1) / (16 * p.nt)) >= 2 * cus)
            break;
    p.groups = rows * ((g.out_c + 16 * p.nt - 1) / (16 * p.nt));
    return p;
}

// Expected time (see dense_s8_route in espdl_hip_api.hip): launch, the steps of one wavefront, all steps in flight.  Fitted to 2840
// random layers on operands that change from launch to launch: 5 to 9 % off either way, 7 to 15 where channels are no whole units (over
// 5500 others, no multiple of 4: 6 to 9 % too small in the mean, 12 to 18 off around that, and up to 1.7 times too small where the
// launch takes several times the tiled GEMM's time; lines of their own for odd channels choose no better).
float conv2d_s8_narrow_us(const ConvGeom &g, const void *in, const void *filter, int cu_count)
{
    const NarrowPlan p = narrow_plan(g, cu_count);
    const long long tiles = ((long long)g.batch * g.out_h * g.out_w + 15) / 16;
    if ((p.split ? tiles : (tiles + 3) / 4) * kThreads >= 1ll << 32) // more threads than a launch may have
        return 1e30f;
    const float steps = (float)(p.split ? (p.ksteps + 3) / 4 : p.ksteps);
    const float waves = 4e-3f * (float)p.groups;
    const float nt = (float)p.nt;
    if (window_aligned(g, in, filter))
        return p.split ? 2.23f + 0.11f * steps + waves * (0.14f + steps * (0.02f + 0.077f * nt))
                       : 2.18f + 0.13f * steps + waves * nt * (g.k_h * g.k_w == 1 ? 0.36f + 0.075f * steps : 0.08f + 0.13f * steps);
    if (((g.in_c | g.in_pitch) & 3) == 0) // units of whole dwords
        return p.split ? 2.7f + 0.18f * steps + waves * (0.25f + nt * (0.06f + 0.082f * steps))
                       : 2.95f + 0.05f * steps + waves * (0.55f * nt + 0.1f * steps);
    if (p.split)
        return 2.42f + 0.34f * steps + waves * (0.18f + steps * (0.085f + 0.206f * nt));
    // (under 16 channels neighbouring pixels' units are bytes of the same lines: 0.65 to 0.85 of what more channels take, 450 layers)
    return 2.78f + 0.23f * steps + (g.in_c < 16 ? 0.65f : 1.f) * waves * (0.39f * nt + steps * (0.123f + 0.165f * nt));
}

hipError_t launch_conv2d_s8_narrow(const ConvGeom &g, const int8_t *in, const int8_t *filter, const int32_t *bias,
                                   const int32_t *shift, const int8_t *lut, const int8_t *residual, int8_t *out,
                                   int cu_count, hipStream_t stream)
{
    NarrowArgs a;
    a.through = ((reinterpret_cast<uintptr_t>(out) | (unsigned)g.out_pitch) & 3) == 0 &&
        writes_through((long long)g.batch * g.out_h * g.out_w * g.out_c);
    a.win = window_args(g, in, filter);
    a.bias = bias;
    a.shift = shift;
    a.lut = lut;
    a.res = residual;
    a.out = out;
    a.n_pix = g.batch * g.out_h * g.out_w;
    a.out_c = g.out_c;
    a.out_pitch = g.out_pitch;
    a.res_pitch = g.res_pitch;
    a.ksteps = (a.win.n_units + 3) / 4;
    a.relu = g.relu;
    a.half_even = g.half_even;
    a.n_shift = g.n_shift;
    a.res_shift = g.res_shift;
    if (a.n_pix == 0)
        return hipSuccess;
    const NarrowPlan p = narrow_plan(g, cu_count);
    const bool aligned = window_aligned(g, in, filter);
    const bool point = g.k_h == 1 && g.k_w == 1 && g.pad_top == 0 && g.pad_left == 0 && (g.out_h - 1) * g.stride_h < g.in_h &&
        (g.out_w - 1) * g.stride_w < g.in_w;
    const long long products = 16384ll * a.win.w_len;
    a.bound = products < 1ll << 30 ? (unsigned)products : 0x80000000u;
    a.dense_pixels = g.out_h == g.in_h && g.out_w == g.in_w && g.stride_h == 1 && g.stride_w == 1;
    a.step.units = p.split ? 16 : 4;
    const int taps = a.step.units / a.win.upt, rows = taps / g.k_w, columns = taps % g.k_w;
    a.step.channels = 16 * (a.step.units % a.win.upt);
    a.step.column = columns * g.dil_w;
    a.step.row = rows * g.dil_h;
    a.step.in = (a.step.row * g.in_w + a.step.column) * g.in_pitch + a.step.channels;
    a.step.filter = taps * g.in_c + a.step.channels;
    a.step.tap_channels = 16 * a.win.upt;
    a.step.in_tap = g.dil_w * g.in_pitch - a.step.tap_channels;
    a.step.filter_tap = g.in_c - a.step.tap_channels;
    a.step.window_columns = g.k_w * g.dil_w;
    a.step.in_row = (g.dil_h * g.in_w - a.step.window_columns) * g.in_pitch;
    if (point) { // channels past the tap's last one are no next tap
        a.step.in = a.step.filter = 16 * a.step.units;
    }
    if (group_open && aligned && p.nt <= 2 && n_held < kMostGrouped) {
        held[n_held++] = Held{a, p.nt, p.split, point, stream};
        return hipSuccess;
    }
    launch_one(a, p.nt, p.split, aligned, point, stream);
    return hipGetLastError();
}

// Which of a group's launches a layer takes (0: none), for tensors at aligned addresses.
int conv2d_s8_narrow_group_kind(const ConvGeom &g, int cu_count)
{
    const NarrowPlan p = narrow_plan(g, cu_count);
    if ((g.in_c & 15) != 0 || (g.in_pitch & 15) != 0 || p.nt > 2)
        return 0;
    return 1 + (p.split ? 2 : 0) + (g.k_h == 1 && g.k_w == 1 ? 1 : 0);
}

// The launches held back since the group was opened: those of one build together, in the order of the first of each.
hipError_t flush_conv2d_s8_narrow()
{
    const int n = n_held;
    n_held = 0;
    bool done[kMostGrouped] = {};
    for (int i = 0; i < n; i++) {
        if (done[i])
            continue;
        const Held &h = held[i];
        NarrowGroup group;
        long long blocks = 0;
        int members = 0;
        for (int j = i; j < n; j++) {
            const Held &o = held[j];
            if (o.split != h.split || o.point != h.point || o.stream != h.stream)
                continue;
            const unsigned tiles = (unsigned)((o.args.n_pix + 15) / 16);
            const unsigned columns = o.split ? tiles : (tiles + 3) / 4;
            done[j] = true;
            group.layer[members] = o.args;
            group.first[members] = (int)blocks;
            group.columns[members] = make_fastdiv(columns);
            blocks += (long long)columns * ((o.args.out_c + 15) / 16);
            members++;
        }
        if (members == 1 || blocks > 1 << 20) { // (a group's layers are small)
            for (int j = i; j < n; j++)
                if (held[j].split == h.split && held[j].point == h.point && held[j].stream == h.stream)
                    launch_one(held[j].args, held[j].nt, h.split, true, h.point, h.stream);
        } else {
            for (int k = members; k < kMostGrouped; k++) {
                group.layer[k] = group.layer[0];
                group.first[k] = (int)blocks;
                group.columns[k] = group.columns[0];
            }
            const auto kernel = h.split ? (h.point ? conv2d_s8_narrow_group_kernel<true, true> : conv2d_s8_narrow_group_kernel<true, false>)
                                        : (h.point ? conv2d_s8_narrow_group_kernel<false, true> : conv2d_s8_narrow_group_kernel<false, false>);
            hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kThreads), 0, h.stream, group);
        }
    }
    return n > 0 ? hipGetLastError() : hipSuccess;
}

} // namespace espdl
