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
// Measured against the kernels such layers took before, as nodes of a graph: 56 x 56 x 64 -> 64, 3 x 3, one image 6.0 ->
// 4.1 us; 13 x 13 x 256 -> 64, 3 x 3 15.5 -> 5.0 us; 13 x 13 x 512 -> 256, 1 x 1 5.6 -> 3.3 us; 1 x 4096 -> 256 6.8 -> 4.7 us;
// 17 x 27 x 74 -> 11, 3 x 3 at stride 2 31.2 -> 3.8 us.
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
    int through; // whole dwords that go through the L2 caches as they are stored
};

template <int NT, bool SPLIT, bool ALIGNED>
__global__ __launch_bounds__(kThreads) void conv2d_s8_narrow_kernel(const NarrowArgs a)
{
    constexpr int G = NT >= 4 ? 2 : 4;
    constexpr int MINE = SPLIT ? 1 : NT; // filter tiles a wavefront finishes
    __shared__ v4i part[SPLIT ? 4 : 1][SPLIT ? NT : 1][64];
    __shared__ int8_t lut_l[256];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int m = (SPLIT ? (int)blockIdx.x : (int)blockIdx.x * 4 + wave) * 16 + col;
    const int n0 = blockIdx.y * 16 * NT;

    const __amdgpu_buffer_rsrc_t in_rsrc = tensor_rsrc(a.win.in, a.win.in_bytes);
    const __amdgpu_buffer_rsrc_t w_rsrc = tensor_rsrc(a.win.w, a.win.w_bytes);
    const PixelWindow px = pixel_window(a.win, m, a.n_pix);
    int row[NT]; // a filter past the last one reads the last one again, its results are dropped
#pragma unroll
    for (int t = 0; t < NT; t++)
        row[t] = min(n0 + 4 * NT * (col >> 2) + 4 * t + (col & 3), a.out_c - 1) * a.win.w_len;

    struct Batch {
        v4i b[G], w[G][NT];
        int n[G];
    };
    const int first = SPLIT ? wave : 0, stride = SPLIT ? 4 : 1;
    auto request = [&](int s0, Batch &t) {
#pragma unroll
        for (int i = 0; i < G; i++) {
            const Unit u = locate_unit(a.win, 4 * (first + (s0 + i) * stride) + quad);
            t.n[i] = u.n;
            t.b[i] = load_pixel_unit<ALIGNED>(a.win, in_rsrc, px, u);
#pragma unroll
            for (int f = 0; f < NT; f++)
                t.w[i][f] = load_filter_unit<ALIGNED>(a.win, w_rsrc, row[f], u);
        }
    };
    const int steps = SPLIT ? (a.ksteps - wave + 3) >> 2 : a.ksteps; // of this wavefront
    Batch cur, nxt;
    request(0, cur);

    // what the epilogue needs is requested before the products: this wavefront's filter tiles
    const bool finisher = !SPLIT || wave < NT;
    int bias[MINE][4], shift[MINE][4];
    int res[MINE];
    const int8_t *res_p = a.res != nullptr ? a.res + (long long)min(m, a.n_pix - 1) * a.res_pitch : nullptr;
#pragma unroll
    for (int t = 0; t < MINE; t++) {
        const int f = n0 + 4 * NT * quad + 4 * (SPLIT ? wave : t);
        res[t] = 0;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int n = min(f + r, a.out_c - 1);
            bias[t][r] = (finisher && a.bias != nullptr) ? a.bias[n] : 0;
            shift[t][r] = finisher ? a.shift[a.n_shift == 1 ? 0 : n] : 0;
            if (finisher && res_p != nullptr)
                res[t] |= (int)(unsigned char)res_p[n] << (8 * r);
        }
    }
    if (a.lut != nullptr)
        lut_l[tid] = a.lut[tid];

    v4i acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
        acc[t] = v4i{0, 0, 0, 0};
    auto products = [&](const Batch &t, int left) {
#pragma unroll
        for (int i = 0; i < G; i++)
            if (i < left) // uniform
#pragma unroll
                for (int f = 0; f < NT; f++)
                    acc[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(mask_unit<ALIGNED>(t.w[i][f], t.n[i]), t.b[i], acc[f], 0, 0, 0);
    };
    for (int s = 0; s < steps; s += 2 * G) {
        if (s + G < steps)
            request(s + G, nxt);
        products(cur, steps - s);
        if (s + G < steps) {
            if (s + 2 * G < steps)
                request(s + 2 * G, cur);
            products(nxt, steps - s - G);
        }
    }
    if constexpr (SPLIT) {
#pragma unroll
        for (int t = 0; t < NT; t++)
            part[wave][t][lane] = acc[t];
    }
    if (SPLIT || a.lut != nullptr)
        __syncthreads();
    if (!finisher) // uniform
        return;
    const bool relu = a.relu != 0, half_even = a.half_even != 0;
#pragma unroll
    for (int t = 0; t < MINE; t++) {
        v4i sum = acc[t];
        if constexpr (SPLIT)
            sum = part[0][wave][lane] + part[1][wave][lane] + part[2][wave][lane] + part[3][wave][lane];
        const int f = n0 + 4 * NT * quad + 4 * (SPLIT ? wave : t);
        int q[4];
        const int word = a.res_shift != 0 ? requant4_s8(res[t], make_requant4(a.res_shift)) : res[t];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            q[r] = requant_s8(sum[r] + bias[t][r], shift[t][r], relu, half_even);
            if (a.lut != nullptr)
                q[r] = lut_l[q[r] + 128];
            if (a.res != nullptr)
                q[r] = clamp_s8(q[r] + (int)(int8_t)(word >> (8 * r)));
        }
        if (m >= a.n_pix || f >= a.out_c)
            continue;
        int8_t *dst = a.out + (long long)m * a.out_pitch + f;
        if (f + 4 <= a.out_c) {
            const int word = pack4_s8(q[0], q[1], q[2], q[3]);
            if (a.through) // uniform
                __hip_atomic_store(reinterpret_cast<int *>(dst), word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else
                *reinterpret_cast<int_unaligned *>(dst) = word;
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (f + r < a.out_c)
                    dst[r] = (int8_t)q[r];
        }
    }
}

template <int NT>
void launch_narrow(const NarrowArgs &a, bool split, bool aligned, hipStream_t stream)
{
    const unsigned tiles = (unsigned)((a.n_pix + 15) / 16);
    const dim3 grid(split ? tiles : (tiles + 3) / 4, (unsigned)((a.out_c + 16 * NT - 1) / (16 * NT)));
    if (split && aligned)
        hipLaunchKernelGGL((conv2d_s8_narrow_kernel<NT, true, true>), grid, dim3(kThreads), 0, stream, a);
    else if (split)
        hipLaunchKernelGGL((conv2d_s8_narrow_kernel<NT, true, false>), grid, dim3(kThreads), 0, stream, a);
    else if (aligned)
        hipLaunchKernelGGL((conv2d_s8_narrow_kernel<NT, false, true>), grid, dim3(kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((conv2d_s8_narrow_kernel<NT, false, false>), grid, dim3(kThreads), 0, stream, a);
}

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

// Expected time (see dense_s8_route in espdl_hip_api.hip): launch, the steps of one wavefront, all steps in flight.
float conv2d_s8_narrow_us(const ConvGeom &g, const void *in, const void *filter, int cu_count)
{
    const NarrowPlan p = narrow_plan(g, cu_count);
    const long long tiles = ((long long)g.batch * g.out_h * g.out_w + 15) / 16;
    if ((p.split ? tiles : (tiles + 3) / 4) * kThreads >= 1ll << 32) // more threads than a launch may have
        return 1e30f;
    const float steps = (float)(p.split ? (p.ksteps + 3) / 4 : p.ksteps);
    const float waves = 4e-3f * (float)p.groups;
    if (window_aligned(g, in, filter))
        return 2.7f + 0.12f * steps + waves * (0.25f + 0.077f * steps * (float)p.nt);
    return 3.3f + waves * (0.12f + 0.264f * steps * (float)p.nt);
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
    if (p.nt == 4)
        launch_narrow<4>(a, p.split, aligned, stream);
    else if (p.nt == 2)
        launch_narrow<2>(a, p.split, aligned, stream);
    else
        launch_narrow<1>(a, p.split, aligned, stream);
    return hipGetLastError();
}

} // namespace espdl
