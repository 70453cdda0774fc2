// Depthwise 3 x 3 int8 convolution (stride 1 or 2 in x, any in y, dilation 1) over any number of channels from 4 on, gfx950.
//
// A thread owns four channels (one dword) of four neighbouring output columns and walks down a strip of output rows.
// Of every input row it loads the six (stride 2: nine) pixels its columns see, one dword each, and turns them with byte
// permutes into dwords of four neighbouring pixels of one channel, so that one v_dot4_i32_i8 forms the three products
// of a filter row (the filter's fourth byte is zero): 48 of them per 16 outputs and no other multiply.  The turned rows
// stay in registers for the three output rows that see them; the next row is requested one row ahead.
//
// Channel counts that are no multiple of 4: the last thread of a pixel takes the last four channels, some of which its
// neighbour has too; both write the same bytes.  Pixels outside the image are loads behind the descriptor's end (zeros),
// outputs that do not exist stores behind it (dropped), so the walk has no branches.
//
// Bound by memory on large layers: 256 images of 56 x 56 x 144 (231 MB in and out) take 59 us when the tensors come from HBM
// (3.9 TB/s), as they do inside a program (61 us in a chain of operators), and 44 us when one pair of tensors, which the
// last-level cache holds in part, is used again and again; tiles staged through LDS for the matrix cores took 60 (66 in
// that chain) and 54 us.  So the gain is in what the staged form spends on its tiles: 256 images of 14 x 14 x 384 14.5 us (19 us
// before, 7 us at the copy rate; strips of few rows and rounds of wavefronts lie between), one image of 56 x 56 x 144 4.8 us
// (15 us), and 61 channels, which that form does not take, over 256 images of 28 x 28: 16 us (107 us).
//
// Strides of 3 and more in y (a recognizer that folds its last rows): three fresh rows per output row.  512 images of
// 3 x 40 x 120 at stride (3, 1) 6.8 us (9.7 on the kernel without strips, 13.2 inside the recognizer), 256 of 28 x 28 x 192
// 14.5 (18.4), one of 56 x 56 x 144 4.3 (9.3).
//
// Restates depthwise_conv2d_33c1 (esp-dl/dl/base/dl_base_depthwise_conv2d.cpp:9-65) under dwconv_operation_shell's window
// clipping (esp-dl/dl/base/dl_base.hpp:1852-2102); filter memory is [3][3][c].
#include "conv_window.h"

namespace espdl {
namespace {

constexpr int kThreads = 256;
constexpr int kParkedRow = 0x40000000; // a row outside the image; with a parked column still behind every tensor

struct StripArgs {
    const int8_t *in, *w;
    const int32_t *bias, *shift;
    const int8_t *lut;
    int8_t *out;
    int in_bytes, out_bytes; // below 2^30
    int in_h, in_w, c, out_h, out_w, stride_h, pad_top, pad_left, n_shift, relu, half_even;
    int rows; // output rows per strip
    int through; // results go through the L2 caches as they are stored
    FastDiv fd_cq, fd_xs, fd_ys;
    unsigned total;   // threads
    unsigned per_xcd; // workgroups of a contiguous part of the rows, 0: parts dealt to the XCDs in turn
};

// One input row as the filter sees it, per channel: the three pixels of output columns 0 .. 3 in the low bytes.  At stride 1
// column 1 uses column 0's dword with the filter moved up a byte.
template <int SW>
struct Row {
    int win[SW == 1 ? 3 : 4][4];
};

template <int SW>
__device__ __forceinline__ Row<SW> turn(const int (&px)[3 + 3 * SW])
{
    Row<SW> r;
    const auto perm = [](int hi, int lo, unsigned sel) { return (int)__builtin_amdgcn_perm((unsigned)hi, (unsigned)lo, sel); };
    const auto turn4 = [&](int a, int b, int c, int d, int (&t)[4]) {
        const int ab0 = perm(b, a, 0x05010400u), ab1 = perm(b, a, 0x07030602u);
        const int cd0 = perm(d, c, 0x05010400u), cd1 = perm(d, c, 0x07030602u);
        t[0] = perm(cd0, ab0, 0x05040100u);
        t[1] = perm(cd0, ab0, 0x07060302u);
        t[2] = perm(cd1, ab1, 0x05040100u);
        t[3] = perm(cd1, ab1, 0x07060302u);
    };
    turn4(px[0], px[1], px[2], px[3], r.win[0]);
    if constexpr (SW == 1) {
        const int lo = perm(px[5], px[4], 0x05010400u), hi = perm(px[5], px[4], 0x07030602u); // pixels 4, 5 of channels 0 1, 2 3
#pragma unroll
        for (int ch = 0; ch < 4; ch++) {
            const int next = ch < 2 ? lo : hi;
            const unsigned at = 4 + 2 * (ch & 1);
            r.win[1][ch] = perm(next, r.win[0][ch], 0x0c000302u | at << 16);              // pixels 2 3 4
            r.win[2][ch] = perm(next, r.win[0][ch], 0x0c000003u | (at | (at + 1) << 8) << 8); // pixels 3 4 5
        }
    } else {
        turn4(px[4], px[5], px[6], px[7], r.win[2]);
#pragma unroll
        for (int ch = 0; ch < 4; ch++) {
            r.win[1][ch] = perm(r.win[2][ch], r.win[0][ch], 0x0c040302u);                  // pixels 2 3 4
            r.win[3][ch] = perm(px[8], r.win[2][ch], 0x0c000302u | (4u + ch) << 16);       // pixels 6 7 8
        }
    }
    return r;
}

// SH: 1, 2, or 3 for every stride in y that leaves output rows no input row in common.
template <int SH, int SW>
__global__ __launch_bounds__(kThreads) void depthwise_s8_strip_kernel(const StripArgs a)
{
    constexpr int kPx = 3 + 3 * SW;
    __shared__ int8_t table[256];
    if (a.lut != nullptr) {
        table[threadIdx.x] = a.lut[threadIdx.x];
        __syncthreads();
    }
    unsigned id = (a.per_xcd ? (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3) : blockIdx.x) * kThreads + threadIdx.x;
    const bool mine = id < a.total;
    if (!__any(mine))
        return;
    if (!mine)
        id = 0; // goes along (the choice of the epilogue is the wavefront's), writes nothing
    const unsigned q0 = fastdiv(id, a.fd_cq);
    const int c0 = min(4 * (int)(id - q0 * a.fd_cq.d), a.c - 4);
    const unsigned q1 = fastdiv(q0, a.fd_xs);
    const int ox0 = 4 * (int)(q0 - q1 * a.fd_xs.d);
    const unsigned n = fastdiv(q1, a.fd_ys);
    const int oy0 = (int)(q1 - n * a.fd_ys.d) * a.rows;

    const __amdgpu_buffer_rsrc_t in = window::tensor_rsrc(a.in, a.in_bytes);
    const __amdgpu_buffer_rsrc_t out = window::tensor_rsrc(a.out, a.out_bytes);

    int col[kPx];
#pragma unroll
    for (int i = 0; i < kPx; i++) {
        const int ix = ox0 * SW - a.pad_left + i;
        col[i] = (unsigned)ix < (unsigned)a.in_w ? ix * a.c + c0 : window::kParked;
    }
    const int in_row = a.in_w * a.c, in_image = (int)n * a.in_h * in_row;
    const auto load = [&](int iy, int (&px)[kPx]) {
        const int row = (unsigned)iy < (unsigned)a.in_h ? in_image + iy * in_row : kParkedRow;
#pragma unroll
        for (int i = 0; i < kPx; i++)
            px[i] = __builtin_amdgcn_raw_buffer_load_b32(in, col[i] + row, 0, 0);
    };
    int iy = oy0 * (SH == 3 ? a.stride_h : SH) - a.pad_top;
    int px[SH][kPx], first[2][kPx];
    load(iy, first[0]);
    if constexpr (SH != 2)
        load(iy + 1, first[1]);

    // filter rows per channel: bytes kx = 0, 1, 2 and a zero; requantization constants of the four channels
    int w[3][4];
#pragma unroll
    for (int ky = 0; ky < 3; ky++) {
        int k[3];
#pragma unroll
        for (int kx = 0; kx < 3; kx++)
            k[kx] = *reinterpret_cast<const int_unaligned *>(a.w + (ky * 3 + kx) * a.c + c0);
#pragma unroll
        for (int ch = 0; ch < 4; ch++) {
            const unsigned two = __builtin_amdgcn_perm((unsigned)k[1], (unsigned)k[0], 0x0c0c0400u + 0x0101u * ch);
            w[ky][ch] = (int)__builtin_amdgcn_perm((unsigned)k[2], two, 0x0c040100u + 0x010000u * ch);
        }
    }
    v4i start, lsh, rsh, shift;
    bool fast = true;
#pragma unroll
    for (int ch = 0; ch < 4; ch++) {
        const int b = a.bias != nullptr ? a.bias[c0 + ch] : 0, s = a.shift[a.n_shift == 1 ? 0 : c0 + ch];
        fast = fast && s >= 1 && s <= 31;
        const int sc = min(max(s, 1), 31);
        const long long first_value = (long long)b + (1ll << (sc - 1)) - (a.half_even ? 1 : 0);
        fast = fast && (first_value < 0 ? -first_value : first_value) + 9ll * 16384 < (1ll << (31 - max(0, 8 - sc)));
        shift[ch] = s;
        start[ch] = (int)first_value;
        lsh[ch] = max(0, 8 - sc);
        rsh[ch] = max(0, sc - 8);
    }
    fast = __all(fast);
    if (!fast) {
#pragma unroll
        for (int ch = 0; ch < 4; ch++)
            start[ch] = a.bias != nullptr ? a.bias[c0 + ch] : 0;
    } else if (!a.half_even) { // pack_fast4<4> takes the left shifts as packed multipliers
        lsh = v4i{(1 << lsh[0]) | (1 << lsh[1]) << 16, (1 << lsh[2]) | (1 << lsh[3]) << 16, 0, 0};
    }
    const int floor_pk = a.relu ? 0 : (int)0x80008000u;

    const int out_row = a.out_w * a.c;
    int to = mine ? ((int)n * a.out_h + oy0) * out_row + ox0 * a.c + c0 : 0;
    int rows_left = mine ? min(a.rows, a.out_h - oy0) : 0;
    const int cols = a.out_w - ox0;
    const auto finish = [&](const Row<SW> &r0, const Row<SW> &r1, const Row<SW> &r2) {
        v4i acc[4] = {start, start, start, start};
#pragma unroll
        for (int ky = 0; ky < 3; ky++) {
            const Row<SW> &r = ky == 0 ? r0 : ky == 1 ? r1 : r2;
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const int at = SW == 2 ? x : x == 0 ? 0 : x - 1;
#pragma unroll
                for (int ch = 0; ch < 4; ch++)
                    acc[x][ch] = __builtin_amdgcn_sdot4(r.win[at][ch], SW == 1 && x == 1 ? w[ky][ch] << 8 : w[ky][ch], acc[x][ch], false);
            }
        }
#pragma unroll
        for (int x = 0; x < 4; x++) {
            int word;
            if (fast) {
                word = a.half_even ? pack_fast4<5>(acc[x], lsh, rsh, floor_pk) : pack_fast4<4>(acc[x], lsh, rsh, floor_pk);
            } else {
                int q[4];
#pragma unroll
                for (int ch = 0; ch < 4; ch++)
                    q[ch] = requant_s8(acc[x][ch], shift[ch], a.relu != 0, a.half_even != 0);
                word = pack4_s8(q[0], q[1], q[2], q[3]);
            }
            if (a.lut != nullptr) {
                const unsigned i = (unsigned)word ^ 0x80808080u;
                word = pack4_s8(table[i & 255], table[(i >> 8) & 255], table[(i >> 16) & 255], table[i >> 24]);
            }
            const int at = rows_left > 0 && x < cols ? to + x * a.c : window::kParked;
            if (a.through) // uniform
                __builtin_amdgcn_raw_buffer_store_b32(word, out, at, 0, kWriteThrough);
            else
                __builtin_amdgcn_raw_buffer_store_b32(word, out, at, 0, 0);
        }
        to += out_row;
        rows_left--;
    };

    if constexpr (SH == 1) {
        Row<SW> r[3];
        r[0] = turn<SW>(first[0]);
        load(iy + 2, px[0]);
        r[1] = turn<SW>(first[1]);
        iy += 3;
        for (int left = a.rows; left > 0; left -= 3) {
#pragma unroll
            for (int u = 0; u < 3; u++) {
                if (u < left) {
                    r[(u + 2) % 3] = turn<SW>(px[0]);
                    load(iy++, px[0]); // (the last one is not used)
                    finish(r[u], r[(u + 1) % 3], r[(u + 2) % 3]);
                }
            }
        }
    } else if constexpr (SH == 3) {
#pragma unroll
        for (int i = 0; i < kPx; i++) {
            px[0][i] = first[0][i];
            px[1][i] = first[1][i];
        }
        load(iy + 2, px[2]);
        for (int left = a.rows; left > 0; left--) {
            Row<SW> r[3];
            iy += a.stride_h;
#pragma unroll
            for (int ky = 0; ky < 3; ky++) {
                r[ky] = turn<SW>(px[ky]);
                load(iy + ky, px[ky]); // (the last three are not used)
            }
            finish(r[0], r[1], r[2]);
        }
    } else {
        Row<SW> r[2];
        load(iy + 1, px[0]);
        load(iy + 2, px[1]);
        r[0] = turn<SW>(first[0]);
        iy += 3;
        for (int left = a.rows; left > 0; left -= 2) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                if (u < left) {
                    const Row<SW> middle = turn<SW>(px[0]);
                    r[1 - u] = turn<SW>(px[1]);
                    load(iy++, px[0]);
                    load(iy++, px[1]);
                    finish(r[u], middle, r[1 - u]);
                }
            }
        }
    }
}

// Strips per image.  A strip of R rows turns R + 2 of them and starts once (2.5 rows' worth), and the rounds of wavefronts
// (four fit a SIMD) should come out even; few rows where there are few wavefronts.  Within 10 % of the best of 1 to 56 rows
// on sixteen layers from 8 to 300 MB.  Of the strip counts with the same number of rows only the smallest counts, which
// leaves 2 sqrt(out_h) of them, and from where even rounds would cost more than the best found no later one is better: at
// most some microseconds on a layer of a million rows (one count after the other: 5 ms).
int strip_count(long long per_strip, int out_h, int cu_count)
{
    const double capacity = 64.0 * 4 * 4 * std::max(1, cu_count);
    int strips = 1;
    double best = 0;
    for (int s = 1;;) {
        const int rows = (out_h + s - 1) / s;
        const double cost = std::ceil(per_strip * s / capacity) * (rows + 2.5);
        if (s == 1 || cost < best) {
            best = cost;
            strips = s;
        }
        if (rows == 1 || per_strip / capacity * (out_h + 2.5 * s) > best)
            return strips;
        s = (out_h + rows - 2) / (rows - 1);
    }
}

} // namespace

bool depthwise_s8_strip_supports(const ConvGeom &g)
{
    return g.k_h == 3 && g.k_w == 3 && g.dil_h == 1 && g.dil_w == 1 && g.in_c >= 4 && g.stride_h < (1 << 20) &&
        (g.stride_w == 1 || g.stride_w == 2) && (long long)g.in_h * g.in_w * g.in_c < (1ll << 30) - 64 &&
        (long long)g.out_h * g.out_w * g.in_c < (1ll << 30) - 64;
}

hipError_t launch_depthwise_s8_strip(const ConvGeom &g, const int8_t *in, const int8_t *filter, const int32_t *bias,
                                     const int32_t *shift, const int8_t *lut, int8_t *out, int cu_count, hipStream_t stream)
{
    const long long in_image = (long long)g.in_h * g.in_w * g.in_c, out_image = (long long)g.out_h * g.out_w * g.in_c;
    if (g.batch * out_image == 0)
        return hipSuccess;
    StripArgs a;
    a.through = writes_through((long long)g.batch * g.out_h * g.out_w * g.out_c);
    a.w = filter;
    a.bias = bias;
    a.shift = shift;
    a.lut = lut;
    a.in_h = g.in_h;
    a.in_w = g.in_w;
    a.c = g.in_c;
    a.out_h = g.out_h;
    a.stride_h = g.stride_h;
    a.out_w = g.out_w;
    a.pad_top = g.pad_top;
    a.pad_left = g.pad_left;
    a.n_shift = g.n_shift;
    a.relu = g.relu;
    a.half_even = g.half_even;
    const int quads = (g.in_c + 3) / 4, xs = (g.out_w + 3) / 4;
    a.fd_cq = make_fastdiv((unsigned)quads);
    a.fd_xs = make_fastdiv((unsigned)xs);
    // offsets of a launch stay below 2^30: parts of the batch
    const int most = (int)std::max(1ll, ((1ll << 30) - 64) / std::max(in_image, out_image));
    for (int n0 = 0; n0 < g.batch; n0 += most) {
        const int n = std::min(most, g.batch - n0);
        const long long per_strip = (long long)n * xs * quads;
        const int strips = strip_count(per_strip, g.out_h, cu_count);
        a.rows = (g.out_h + strips - 1) / strips;
        a.fd_ys = make_fastdiv((unsigned)strips);
        a.in = in + n0 * in_image;
        a.out = out + n0 * out_image;
        a.in_bytes = (int)(n * in_image);
        a.out_bytes = (int)(n * out_image);
        a.total = (unsigned)(per_strip * strips);
        // Each XCD a contiguous part where the input is far larger than the L2s (115 MB: 60 against 62 us); in turn below,
        // where what the layer in front left in an L2 is still there (20 x 80 x 24, 512 images: 8.5 against 10 us)
        unsigned blocks = (a.total + kThreads - 1) / kThreads;
        a.per_xcd = a.in_bytes >= (64 << 20) ? (blocks + 7) / 8 : 0;
        if (a.per_xcd)
            blocks = 8 * a.per_xcd;
        const dim3 grid(blocks);
        const auto kernel = g.stride_h == 1
            ? (g.stride_w == 1 ? depthwise_s8_strip_kernel<1, 1> : depthwise_s8_strip_kernel<1, 2>)
            : g.stride_h == 2 ? (g.stride_w == 1 ? depthwise_s8_strip_kernel<2, 1> : depthwise_s8_strip_kernel<2, 2>)
                              : (g.stride_w == 1 ? depthwise_s8_strip_kernel<3, 1> : depthwise_s8_strip_kernel<3, 2>);
        hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

} // namespace espdl
