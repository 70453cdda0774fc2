// Dense int8 convolution of images with a handful of channels (the first layer of a network) as a walk down the image.
//
// A wavefront owns 32 output columns of an image, as a tile of 16 even and a tile of 16 odd ones, and goes down them RS rows
// per step.
//   input   The image rows under a step come into LDS by direct-to-LDS copies, a lane per 16 consecutive bytes, one step ahead.
//           Image rows are whole 16-byte pieces, so a piece lies inside its row or is zeros: that is all the padding needs.
//   tiles   A lane group reads one filter row, the at most 12 bytes from the dword that its first byte lies in, as three
//           aligned dwords.  How far into that dword the row starts is the same for every second column, so it goes into the
//           filters as zeros in front of the row, and nothing is shifted.  Filters, start values and shifts stay in registers.
//   output  Results pass through LDS and leave as 16-byte pieces in memory order.
// Copies or stores of 16 bytes a lane at other distances (a lane's own window, a lane's own pixel) are taken apart lane by lane
// by the memory pipeline: the same walk with them took 77 us on the first layer below.
//
// Bound by memory and the start of the launch: 64 images of 640 x 640 x 3, 3 x 3 at stride 2 under 16 filters with a table
// (184 MB) 50 us, 78 before; 512 of 48 x 320 17 us (30); 64 of 224 x 224 under 32 filters 16 us (24), 32 under 64 22.5 us
// (37); one image of 416 x 416 the same 5.1 us.  Two and three steps ahead instead of one: 52 and 53 us.
//
// The kernel in conv2d_s8_stem.hip, which takes the layers that this one does not, copies rows through registers and cuts
// every window row out of LDS with an unaligned 16-byte read, which is what bounds it (LDS active 64 % of the time, 71 cycles
// per 16 pixels).
//
// What it computes: conv2d_33cn / _hwcn for int8 (esp-dl/dl/base/dl_base_conv2d.cpp:9-163) under conv_operation_shell's
// window clipping (esp-dl/dl/base/dl_base.hpp:382-1196), with the n_wise epilogue (dl_base_activate_buffer.hpp:10-74) and an
// optional 256-entry table on the stored value (dl_base_lut.cpp:10-15).
#include "mbconv_s8_walk_kernel.h"

namespace espdl {
namespace {
using namespace mbwalk;

struct StemWalkArgs {
    const int8_t *in, *w, *lut;
    const int32_t *bias, *shift;
    int8_t *out;
    int img_h, c, out_h, out_w, n, k_h, k_w, s_h, s_w, pad_top, pad_left, n_shift, relu, out_pitch;
    int in_row, in_img, out_row;
    long long out_img;
    int strips, steps;          // of 32 columns per image; per strip
    int total, per_wave;        // steps
    int n_groups;
    int pieces, pitch;          // 16-byte pieces of a copied row, its bytes
    int skew0, skew1; // bytes between the dword's first and the filter row's first byte: even tile, odd tile
    int bound;        // largest sum of products
    FastDiv fd_steps, fd_strips, fd_pieces;
};

constexpr int kWaves = 4, kThreads = 64 * kWaves;
constexpr int kCols = 32;
constexpr int kCopies = 2; // instructions per step: 128 pieces
constexpr int kAhead = 1, kSlots = kAhead + 2, kSlot = kCopies * 1024;

template <int RT, int RS, bool HE, bool LUT>
__global__ __launch_bounds__(kThreads) void conv2d_s8_walk_stem_kernel(const StemWalkArgs a)
{
    constexpr int kPx = 16 * RT, kStores = RS * kCols * RT / 64;
    __shared__ __align__(16) unsigned char ring[kWaves][kSlots][kSlot];
    __shared__ __align__(16) unsigned char slab[kWaves][RS * kCols * kPx];
    __shared__ unsigned char lut_l[LUT ? 256 : 1];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int group = (int)(blockIdx.x & 7u) * (a.n_groups >> 3) + (int)(blockIdx.x >> 3);
    const int begin = (group * kWaves + wave) * a.per_wave, end = min(a.total, begin + a.per_wave);

    // step -> image, strip, first output row
    const auto place = [&](int step, int &n, int &x0, int &y0) __attribute__((always_inline)) {
        const int q = (int)fastdiv((unsigned)step, a.fd_steps);
        n = (int)fastdiv((unsigned)q, a.fd_strips);
        x0 = (q - n * a.strips) * kCols;
        y0 = (step - q * a.steps) * RS;
    };

    // ---- copies: piece p of row r of the step, from 16 bytes in front of the strip's first column on
    const unsigned ring0 = (unsigned)reinterpret_cast<uintptr_t>(&ring[wave][0][0]);
    int pr[kCopies], pp[kCopies];
#pragma unroll
    for (int j = 0; j < kCopies; j++) {
        const int i = lane + 64 * j, r = (int)fastdiv((unsigned)i, a.fd_pieces);
        pr[j] = r;
        pp[j] = 16 * (i - r * a.pieces) - 16;
    }
    int f_step = begin;
    unsigned f_slot = 0;
    const auto feed = [&]() __attribute__((always_inline)) { // one step; past the last one nothing is read (the counts stay the same)
        const bool live = f_step < end;
        int n, x0, y0;
        place(live ? f_step : 0, n, x0, y0);
        const int row = y0 * a.s_h - a.pad_top, xb = x0 * a.s_w * a.c;
        const __amdgpu_buffer_rsrc_t rs = rsrc_of(a.in + (long long)n * a.in_img, __builtin_amdgcn_readfirstlane(live ? a.in_img : 0));
        const unsigned base = __builtin_amdgcn_readfirstlane(ring0 + f_slot);
#pragma unroll
        for (int j = 0; j < kCopies; j++) {
            const int y = row + pr[j], x = xb + pp[j];
            const bool ok = (unsigned)y < (unsigned)a.img_h && (unsigned)x < (unsigned)a.in_row;
            copy16(base + 1024 * j, ok ? y * a.in_row + x : kParked, rs);
        }
        f_step++;
        f_slot = f_slot + kSlot == kSlots * kSlot ? 0 : f_slot + kSlot;
    };
    const auto no_stores = [&]() __attribute__((always_inline)) { // dropped: the number of instructions behind a copy is known in every step
#pragma unroll
        for (int i = 0; i < kStores; i++)
            asm volatile("s_nop 4\n\tbuffer_store_byte %0, %0, %1, 0 offen" ::"v"(kParked), "s"(rsrc_of(a.out, 0)) : "memory");
    };

    // ---- set-up: the first copies, filters and constants
#pragma unroll
    for (int i = 0; i <= kAhead; i++) {
        feed();
        no_stores();
    }
    // Row i of filter tile t is filter 4 RT (i / 4) + 4 t + i % 4: a lane ends up with 4 RT neighbouring channels.
    const int taps = a.k_w * a.c;
    v4i wa[RT][2], start[RT], shift[RT];
    int ok = 1, low = 0;
#pragma unroll
    for (int t = 0; t < RT; t++) {
        const int f = 4 * RT * (col >> 2) + 4 * t + (col & 3);
        const int8_t *src = a.w + (f * a.k_h + min(quad, a.k_h - 1)) * taps;
        unsigned b[12];
#pragma unroll
        for (int i = 0; i < 12; i++)
            b[i] = (unsigned char)src[min(i, taps - 1)];
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int skew = e != 0 ? a.skew1 : a.skew0;
            unsigned long long lo = 0, hi = 0; // the filter row, then moved up by the distance
#pragma unroll
            for (int i = 0; i < 12; i++)
                if (i < taps && quad < a.k_h)
                    (i < 8 ? lo : hi) |= (unsigned long long)b[i] << (8 * (i & 7));
            if (skew != 0) {
                hi = hi << (8 * skew) | lo >> (64 - 8 * skew);
                lo <<= 8 * skew;
            }
            wa[t][e] = v4i{(int)lo, (int)(lo >> 32), (int)hi, 0};
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int ch = 4 * RT * quad + 4 * t + r;
            const int s = a.shift[a.n_shift == 1 ? 0 : ch], bv = a.bias != nullptr ? a.bias[ch] : 0;
            const long long st = (long long)bv + (1ll << ((s - 1) & 31)), mag = st < 0 ? -st : st;
            if (s < 1 || s > 31 || mag + a.bound >= (1ll << 31))
                ok = 0;
            if (s < 8)
                low = 1;
            start[t][r] = bv;
            shift[t][r] = s;
        }
    }
    if (LUT)
        lut_l[tid] = (unsigned char)a.lut[tid ^ 0x80]; // by the byte itself
    const bool fast = __syncthreads_and(ok) != 0, high = fast && __syncthreads_or(low) == 0;
    if (fast)
#pragma unroll
        for (int t = 0; t < RT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                start[t][r] += (1 << ((shift[t][r] - 1) & 31)) - (HE ? 1 : 0);
                shift[t][r] -= high ? 8 : 0;
            }
    const Band band = make_band({a.relu ? 0 : -128, 127}, high);

    // this lane's window: row `quad`, column 2 col (+ 1), its dwords (lane groups past the last filter row meet zero filters)
    const int win0 = min(quad, a.k_h - 1) * a.pitch + 16 + (2 * col * a.s_w - a.pad_left) * a.c - a.skew0;
    const int win1 = min(quad, a.k_h - 1) * a.pitch + 16 + ((2 * col + 1) * a.s_w - a.pad_left) * a.c - a.skew1;
    unsigned char *const my_slab = slab[wave];
    // the pieces of the output this lane writes: piece lane + 64 j of the step
    int o_px[kStores], o_off[kStores];
#pragma unroll
    for (int j = 0; j < kStores; j++) {
        const int i = lane + 64 * j, r = i / (kCols * RT), q = i - r * (kCols * RT);
        o_px[j] = q / RT;
        o_off[j] = r * a.out_row + o_px[j] * a.out_pitch + 16 * (q % RT);
    }

    const auto walk = [&](auto mode_tag) __attribute__((always_inline)) {
        constexpr int MODE = decltype(mode_tag)::value;
        unsigned b_slot = 0;
        for (int step = begin; step < end; step++) {
            int n, x0, y0;
            place(step, n, x0, y0);
            wait_copies<kAhead * (kCopies + kStores) + kStores>(); // this step's input has arrived
            const unsigned char *rows = &ring[wave][0][0] + b_slot;
            b_slot = b_slot + kSlot == kSlots * kSlot ? 0 : b_slot + kSlot;
            v4i X[RS][2];
#pragma unroll
            for (int s = 0; s < RS; s++) {
                const unsigned char *row = rows + s * a.s_h * a.pitch;
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    X[s][0][i] = *reinterpret_cast<const int *>(row + win0 + 4 * i);
                    X[s][1][i] = *reinterpret_cast<const int *>(row + win1 + 4 * i);
                }
                X[s][0][3] = X[s][0][2]; // (meets zero filters)
                X[s][1][3] = X[s][1][2];
            }
            feed();
#pragma unroll
            for (int s = 0; s < RS; s++)
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    int words[RT];
#pragma unroll
                    for (int t = 0; t < RT; t++) {
                        const v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa[t][e], X[s][e], start[t], 0, 0, 0);
                        int w = finish4<MODE, HE>(acc, shift[t], band);
                        if constexpr (LUT) {
                            const unsigned u = (unsigned)w;
                            w = (int)((unsigned)lut_l[u & 255] | (unsigned)lut_l[(u >> 16) & 255] << 16) |
                                (int)((unsigned)lut_l[(u >> 8) & 255] | (unsigned)lut_l[u >> 24] << 16) << 8;
                        }
                        words[t] = w;
                    }
                    unsigned char *to = my_slab + (s * kCols + 2 * col + e) * kPx + 4 * RT * quad;
                    if constexpr (RT == 4)
                        *reinterpret_cast<v4i *>(to) = v4i{words[0], words[1], words[2], words[3]};
                    else
#pragma unroll
                        for (int t = 0; t < RT; t++)
                            reinterpret_cast<int *>(to)[t] = words[t];
                }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const long long at = (long long)n * a.out_img + (long long)y0 * a.out_row;
            const __amdgpu_buffer_rsrc_t rs = rsrc_of(a.out + at, __builtin_amdgcn_readfirstlane((a.out_h - y0) * a.out_row)); // (rows past the last: dropped)
#pragma unroll
            for (int j = 0; j < kStores; j++) {
                const v4i v = *reinterpret_cast<const v4i *>(my_slab + 16 * (lane + 64 * j));
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), rs, x0 + o_px[j] < a.out_w ? o_off[j] + x0 * a.out_pitch : kParked, 0, 0);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    };
    if (!fast)
        walk(std::integral_constant<int, 2>{});
    else if (high)
        walk(std::integral_constant<int, 0>{});
    else
        walk(std::integral_constant<int, 1>{});
}

struct StemWalkPlan {
    bool ok;
    int rt, rs;
    StemWalkArgs a;
};

StemWalkPlan stem_walk_plan(const ConvGeom &g, const void *in, const void *out, const void *residual, int cus)
{
    StemWalkPlan plan = {};
    const long long seg = (long long)g.k_w * g.in_c, in_row = (long long)g.in_w * g.in_c;
    if (residual != nullptr || g.in_pitch != g.in_c || g.dil_h != 1 || g.dil_w != 1 || g.batch <= 0 || g.out_h <= 0 || g.out_w <= 0)
        return plan;
    plan.rt = g.out_c / 16;
    if (g.out_c % 16 != 0 || (plan.rt != 1 && plan.rt != 2 && plan.rt != 4) || g.out_pitch % 4 != 0 ||
        ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 3) != 0)
        return plan;
    // a filter row and what lies in front of it in 12 bytes, every second column at the same distance from a dword, image rows
    // of whole pieces, the padding in front of a row at most one
    const int skew0 = -g.pad_left * g.in_c & 3, skew1 = (g.stride_w - g.pad_left) * g.in_c & 3;
    if (g.k_h > 4 || seg + std::max(skew0, skew1) > 12 || ((long long)g.stride_w * g.in_c) % 2 != 0 || in_row % 16 != 0 ||
        g.pad_left * g.in_c + 3 > 16 || g.stride_w > 8 || g.stride_h > 8)
        return plan;
    StemWalkArgs &a = plan.a;
    const int bytes = 16 + 31 * g.stride_w * g.in_c + 12 + 3; // of a copied row: to the end of the last window's dwords
    a.pieces = (bytes + 15) / 16;
    a.pitch = 16 * a.pieces;
    for (plan.rs = 4; plan.rs >= 2 && ((plan.rs - 1) * g.stride_h + g.k_h) * a.pieces > 64 * kCopies; plan.rs /= 2)
        ;
    const long long in_img = in_row * g.in_h, out_row = (long long)g.out_w * g.out_pitch;
    const long long strips = (g.out_w + kCols - 1) / kCols;
    if (plan.rs < 2 || in_img > 0x7f000000ll || (g.out_h + 4) * out_row > 0x7f000000ll)
        return plan;
    const long long steps = (g.out_h + plan.rs - 1) / plan.rs, total = (long long)g.batch * strips * steps;
    if (total > (1ll << 30))
        return plan;
    a.img_h = g.in_h;
    a.c = g.in_c;
    a.out_h = g.out_h;
    a.out_w = g.out_w;
    a.n = g.out_c;
    a.k_h = g.k_h;
    a.k_w = g.k_w;
    a.s_h = g.stride_h;
    a.s_w = g.stride_w;
    a.pad_top = g.pad_top;
    a.pad_left = g.pad_left;
    a.n_shift = g.n_shift;
    a.relu = g.relu;
    a.out_pitch = g.out_pitch;
    a.in_row = (int)in_row;
    a.in_img = (int)in_img;
    a.out_row = (int)out_row;
    a.out_img = out_row * g.out_h;
    a.strips = (int)strips;
    a.steps = (int)steps;
    a.total = (int)total;
    a.skew0 = skew0;
    a.skew1 = skew1;
    a.bound = (int)(g.k_h * seg * 16384);
    a.fd_steps = make_fastdiv((unsigned)steps);
    a.fd_strips = make_fastdiv((unsigned)strips);
    a.fd_pieces = make_fastdiv((unsigned)a.pieces);
    // two workgroups per compute unit, each wavefront with the same number of steps of the strips laid end to end (four, of
    // which two fit at 32 and 64 filters: 19.5 against 15.9 us on 64 images of 224 x 224 x 3 under 32 filters, the same at 16)
    const long long waves = (long long)std::max(8, 2 * cus / 8 * 8) * kWaves;
    a.per_wave = (int)((total + waves - 1) / waves);
    const long long groups = (total + (long long)a.per_wave * kWaves - 1) / ((long long)a.per_wave * kWaves);
    a.n_groups = (int)((groups + 7) / 8 * 8);
    plan.ok = true;
    return plan;
}

template <int RT, int RS>
hipError_t launch_one(const StemWalkPlan &plan, bool half_even, hipStream_t stream)
{
    const dim3 grid((unsigned)plan.a.n_groups), block(kThreads);
    const auto kernel = half_even ? (plan.a.lut ? conv2d_s8_walk_stem_kernel<RT, RS, true, true> : conv2d_s8_walk_stem_kernel<RT, RS, true, false>)
                                  : (plan.a.lut ? conv2d_s8_walk_stem_kernel<RT, RS, false, true> : conv2d_s8_walk_stem_kernel<RT, RS, false, false>);
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, plan.a);
    return hipGetLastError();
}

} // namespace

bool conv2d_s8_walk_stem_supports(const ConvGeom &g, const void *in, const void *out, const void *residual)
{
    return stem_walk_plan(g, in, out, residual, 256).ok;
}

hipError_t launch_conv2d_s8_walk_stem(const ConvGeom &g, const int8_t *in, const int8_t *filter, const int32_t *bias, const int32_t *shift,
                                      const int8_t *lut, const int8_t *residual, int8_t *out, int cu_count, hipStream_t stream)
{
    StemWalkPlan plan = stem_walk_plan(g, in, out, residual, cu_count > 0 ? cu_count : 256);
    if (!plan.ok)
        return hipErrorInvalidValue;
    plan.a.in = in;
    plan.a.w = filter;
    plan.a.lut = lut;
    plan.a.bias = bias;
    plan.a.shift = shift;
    plan.a.out = out;
    const bool he = g.half_even != 0;
    if (plan.rs == 4)
        return plan.rt == 1 ? launch_one<1, 4>(plan, he, stream) : (plan.rt == 2 ? launch_one<2, 4>(plan, he, stream) : launch_one<4, 4>(plan, he, stream));
    return plan.rt == 1 ? launch_one<1, 2>(plan, he, stream) : (plan.rt == 2 ? launch_one<2, 2>(plan, he, stream) : launch_one<4, 2>(plan, he, stream));
}

} // namespace espdl
