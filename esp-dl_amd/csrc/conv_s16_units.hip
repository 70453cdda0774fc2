// Dense int16 convolution / Gemm for gfx950 on the int8 matrix pipe, any channel count, any window.
//
// What it computes is conv2d_11cn / _33cn / _hwcn for int16 (esp-dl/dl/base/dl_base_conv2d.cpp:9-163 with
// feature_t = int16_t, buffer_t = int64_t) under conv_operation_shell's window clipping
// (esp-dl/dl/base/dl_base.hpp:940-1191): an exact 64-bit sum of int16 x int16 products, plus the int64 bias, shifted and
// rounded, saturated to int16.
//
// There is no int16 MFMA, so both operands are cut into two signed bytes that the int8 MFMA multiplies exactly.
// With h = the high byte of a 16-bit value v (signed) and l = its low byte xor 0x80 (signed, the low byte minus
// 128):  v = 256 h + l + 128.  For a pixel x = A + 128 and a weight w = B + 128 (A = 256 xh + xl, B = 256 wh + wl):
//   sum_k x w = sum_k A B + 128 sum_k A + 128 sum_k B + 16384 K
//             = 65536 HH + 256 (HL + LH) + LL  +  128 (256 sum_k xh + sum_k xl)  +  128 (256 sum_k wh + sum_k wl)  +  16384 K
// with HH = sum_k xh wh and so on: four MFMA products per step into three int32 accumulators (HL and LH share
// one; none can overflow for K < 65536), and the byte sums of the pixels' windows and of the filters (two dot-product
// instructions per loaded dword pair).
//
// The reduction axis is that of conv_window.h: units of 16 channels of one tap, four units per step, K = 64 steps.
// Every position of every step counts in K, whether it exists or not: a tap outside the image, a unit past the last
// tap and a channel past the last one have w = 0 or x = 0, i.e. bytes (0, -128), and x w = 0 comes out of the formula
// like any other product (where w = 0, x may be anything).  So nothing is special but the filter's bytes behind a
// tap's last channel, which are cleared.
//
// X8 builds: the input is an int8 tensor that a RequantizeLinear would have multiplied by 256, so its low bytes are zero
// and its high bytes the int8 values themselves:  sum_k x w = 65536 sum x8 wh + 256 sum x8 l + 32768 sum x8 (l as above).
// Two products per step instead of four, no cutting of pixels, half the input, no RequantizeLinear and no int16 copy.
// They also take an int16 table behind the result (the nearest-entry LUT of esp-dl/dl/base/dl_base_lut.cpp:49-77).
// 80 x 80 x 64 -> 64, 3 x 3, batch 64: 75 us where the three operators took 135 us (51 us as a walk down the image, which
// takes the 3 x 3 layers that fill the device: conv2d_s16_x8_walk.hip).
//
// Two kernels, chosen by their measured cost (see the launch).  Against the one-wavefront-per-pixel-tile kernel
// (conv_s16_mfma.hip) and the 64-bit multiply-add kernel (conv_s16.hip): 80 x 80 x 64 -> 64, 3 x 3, batch 64 98 -> 90 us,
// batch 8 22 -> 16 us, one image 13.4 -> 8.3 us; 40 x 40 x 128 -> 128, batch 64 147 -> 85 us; 22 x 12 x 122 -> 252, 3 x 3,
// batch 57 2764 -> 31 us.
//   * the tiled one: 64 PT pixels x 64 filters per workgroup, both operands global -> registers (two steps ahead) ->
//     cut into bytes -> LDS (two buffers), so that a value is cut once per workgroup;
//   * the narrow one for few outputs: 16 pixels x 16 NT filters per workgroup, its four wavefronts split the reduction
//     axis and read both operands straight from memory in the matrix instruction's layout; the partial sums meet in LDS.
#include <algorithm>
#include <type_traits>

#include "conv_window.h"

namespace espdl {
namespace {

using namespace window;

constexpr int kThreads = 256;
constexpr int kRow = 96; // LDS row of one byte plane: 64 k positions + padding, conflict-free 16-byte reads

struct S16Args {
    WindowArgs win; // byte offsets: in_c and the pitch are in bytes, two per channel, a unit is 32 bytes
    const int64_t *bias;
    const int32_t *shift;
    int16_t *out;
    int n_pix, out_c, ksteps;
    int relu, half_even, n_shift;
    const int16_t *table; // X8: applied to the result, or nullptr
    int table_size, table_shift;
};
constexpr int kMostTable = 4097; // entries

// The table's entry nearest to sample point v; ties as the rounding mode has them.
__device__ __forceinline__ int nearest_entry(int v, int shift, bool half_even)
{
    const int x = (v & 0xffff) ^ 0x8000, half = 1 << (shift - 1);
    return (half_even ? x + half - 1 + ((x >> shift) & 1) : x + half) >> shift;
}

// The 16 values of a unit: two 16-byte loads through the descriptor, zeros where nothing exists.
struct Unit16 {
    v4i lo, hi;
};
template <bool ALIGNED>
__device__ __forceinline__ Unit16 load_unit16(__amdgpu_buffer_rsrc_t rsrc, int off, int bytes)
{
    Unit16 u;
    u.lo = load16<ALIGNED>(rsrc, off, bytes);
    const int next = off + 16; // a parked offset stays parked
    u.hi = load16<ALIGNED>(rsrc, !ALIGNED && next >= bytes ? kParked : next, bytes);
    return u;
}
template <bool ALIGNED>
__device__ __forceinline__ Unit16 load_pixel16(const WindowArgs &a, __amdgpu_buffer_rsrc_t rsrc, const PixelWindow &p, const Unit &u)
{
    const bool ok = u.n > 0 && (unsigned)(p.iy + u.dy) < (unsigned)a.in_h && (unsigned)(p.ix + u.dx) < (unsigned)a.in_w;
    return load_unit16<ALIGNED>(rsrc, ok ? p.base + u.in_off : kParked, a.in_bytes);
}
template <bool ALIGNED>
__device__ __forceinline__ Unit16 load_filter16(const WindowArgs &a, __amdgpu_buffer_rsrc_t rsrc, int row, const Unit &u)
{
    return load_unit16<ALIGNED>(rsrc, u.n > 0 ? row + u.w_off : kParked, a.w_bytes);
}

// locate_unit for 32-byte units
__device__ __forceinline__ Unit locate_unit16(const WindowArgs &a, int u)
{
    const unsigned tap = fastdiv((unsigned)u, a.fd_upt);
    const int j = u - (int)(tap * a.fd_upt.d);
    const unsigned ky = fastdiv(tap, a.fd_kw);
    Unit r;
    r.dy = (int)ky * a.dil_h;
    r.dx = (int)(tap - ky * a.fd_kw.d) * a.dil_w;
    r.in_off = (r.dy * a.in_w + r.dx) * a.in_pitch + 32 * j;
    r.w_off = (int)tap * a.in_c + 32 * j;
    r.n = u < a.n_units ? a.in_c - 32 * j : 0; // bytes
    return r;
}

// X8: a unit is 16 bytes of the input and 32 of the filter (in_c and the pitch count int8 channels).
__device__ __forceinline__ Unit locate_unit_x8(const WindowArgs &a, int u)
{
    const unsigned tap = fastdiv((unsigned)u, a.fd_upt);
    const int j = u - (int)(tap * a.fd_upt.d);
    const unsigned ky = fastdiv(tap, a.fd_kw);
    Unit r;
    r.dy = (int)ky * a.dil_h;
    r.dx = (int)(tap - ky * a.fd_kw.d) * a.dil_w;
    r.in_off = (r.dy * a.in_w + r.dx) * a.in_pitch + 16 * j;
    r.w_off = 2 * (int)tap * a.in_c + 32 * j;
    r.n = u < a.n_units ? 2 * (a.in_c - 16 * j) : 0; // filter bytes
    return r;
}
__device__ __forceinline__ int byte_sum(const v4i &v, int sum)
{
#pragma unroll
    for (int d = 0; d < 4; d++)
        sum = __builtin_amdgcn_sdot4(v[d], 0x01010101, sum, false);
    return sum;
}

// High bytes and low bytes xor 0x80 of half a unit or a unit, in k order, and the running sums of both.
struct Halves {
    v2i h, l;
};
__device__ __forceinline__ Halves cut8(const v4i &v, int &sum_h, int &sum_l)
{
    Halves p;
#pragma unroll
    for (int q = 0; q < 2; q++) {
        p.h[q] = (int)__builtin_amdgcn_perm((unsigned)v[2 * q + 1], (unsigned)v[2 * q], 0x07050301u);
        p.l[q] = (int)__builtin_amdgcn_perm((unsigned)v[2 * q + 1], (unsigned)v[2 * q], 0x06040200u) ^ (int)0x80808080u;
        sum_h = __builtin_amdgcn_sdot4(p.h[q], 0x01010101, sum_h, false);
        sum_l = __builtin_amdgcn_sdot4(p.l[q], 0x01010101, sum_l, false);
    }
    return p;
}
struct Planes {
    v4i h, l;
};
__device__ __forceinline__ Planes cut(const Unit16 &u, int &sum_h, int &sum_l)
{
    const Halves a = cut8(u.lo, sum_h, sum_l), b = cut8(u.hi, sum_h, sum_l);
    return Planes{v4i{a.h[0], a.h[1], b.h[0], b.h[1]}, v4i{a.l[0], a.l[1], b.l[0], b.l[1]}};
}

// The same for a filter unit of which `n` bytes exist.
template <bool ALIGNED>
__device__ __forceinline__ Planes cut_filter(Unit16 u, int n, int &sum_h, int &sum_l)
{
    u.lo = mask_unit<ALIGNED>(u.lo, n);
    u.hi = mask_unit<ALIGNED>(u.hi, n - 16);
    return cut(u, sum_h, sum_l);
}

__device__ __forceinline__ long long byte_term(int sum_h, int sum_l)
{
    return 128ll * (256ll * sum_h + sum_l);
}

__device__ __forceinline__ long long combine(int hh, int mid, int ll)
{
    return ((long long)hh << 16) + ((long long)mid << 8) + (long long)ll;
}

// PT: pixel tiles of 16 per wavefront; FT: filter tiles of 16 per workgroup.
template <int PT, int FT, bool ALIGNED, bool X8 = false>
__global__ __launch_bounds__(kThreads) void conv2d_s16_gemm_kernel(const S16Args a)
{
    constexpr int kTileM = 64 * PT;
    constexpr int kSums = X8 ? 2 : 3; // accumulators of a value
    __shared__ __align__(16) unsigned char b_l[2][X8 ? 1 : 2][kTileM * kRow]; // [buffer][high, low]
    [[maybe_unused]] __shared__ __align__(16) int16_t table_l[X8 ? kMostTable + 7 : 1];
    __shared__ __align__(16) unsigned char a_l[2][2][16 * FT * kRow];
    __shared__ long long pix_term[kTileM];
    __shared__ long long cst[16 * FT];
    __shared__ v2i fast_cst[16 * FT];
    __shared__ int shf[16 * FT];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 15, quad = lane >> 4;
    const int m0 = blockIdx.x * kTileM;
    const int n0 = blockIdx.y * 16 * FT;
    const int my_row = tid >> 2, q4 = tid & 3; // this thread's tile row (+ 64 per pixel piece) and unit of a step

    const __amdgpu_buffer_rsrc_t in_rsrc = tensor_rsrc(a.win.in, a.win.in_bytes);
    const __amdgpu_buffer_rsrc_t w_rsrc = tensor_rsrc(a.win.w, a.win.w_bytes);
    PixelWindow px[PT];
#pragma unroll
    for (int j = 0; j < PT; j++)
        px[j] = pixel_window(a.win, m0 + 64 * j + my_row, a.n_pix);
    // (a filter past the last one reads the last one again: its results are not stored)
    const int w_row = min(n0 + my_row, a.out_c - 1) * a.win.w_len;

    struct Pieces {
        std::conditional_t<X8, v4i, Unit16> b[PT];
        Unit16 w;
        int n;
    };
    auto fetch = [&](int ks, Pieces &p) {
        const Unit u = X8 ? locate_unit_x8(a.win, 4 * ks + q4) : locate_unit16(a.win, 4 * ks + q4);
        p.n = u.n;
#pragma unroll
        for (int j = 0; j < PT; j++) {
            if constexpr (X8)
                p.b[j] = load_pixel_unit<ALIGNED>(a.win, in_rsrc, px[j], u);
            else
                p.b[j] = load_pixel16<ALIGNED>(a.win, in_rsrc, px[j], u);
        }
        if (FT == 4 || my_row < 16 * FT)
            p.w = load_filter16<ALIGNED>(a.win, w_rsrc, w_row, u);
    };
    int bsum_h[PT] = {}, bsum_l[PT] = {}, wsum_h = 0, wsum_l = 0;
    auto stash = [&](int buf, const Pieces &p) {
        const int at = my_row * kRow + 16 * q4;
#pragma unroll
        for (int j = 0; j < PT; j++) {
            if constexpr (X8) {
                bsum_h[j] = byte_sum(p.b[j], bsum_h[j]);
                *reinterpret_cast<v4i *>(&b_l[buf][0][at + 64 * j * kRow]) = p.b[j];
            } else {
                const Planes c = cut(p.b[j], bsum_h[j], bsum_l[j]);
                *reinterpret_cast<v4i *>(&b_l[buf][0][at + 64 * j * kRow]) = c.h;
                *reinterpret_cast<v4i *>(&b_l[buf][1][at + 64 * j * kRow]) = c.l;
            }
        }
        if (FT == 4 || my_row < 16 * FT) {
            const Planes c = cut_filter<ALIGNED>(p.w, p.n, wsum_h, wsum_l);
            *reinterpret_cast<v4i *>(&a_l[buf][0][at]) = c.h;
            *reinterpret_cast<v4i *>(&a_l[buf][1][at]) = c.l;
        }
    };

    Pieces p0, p1;
    fetch(0, p0);
    if (a.ksteps > 1)
        fetch(1, p1);
    if (tid < 16 * FT) {
        const int n = min(n0 + tid, a.out_c - 1);
        cst[tid] = (a.bias != nullptr ? a.bias[n] : 0) + (X8 ? 0 : 16384ll * 64 * a.ksteps);
        shf[tid] = a.shift[a.n_shift == 1 ? 0 : n];
    }
    if constexpr (X8) {
        if (a.table != nullptr)
            for (int i = tid; i < a.table_size; i += kThreads)
                table_l[i] = a.table[i];
    }
    stash(0, p0);
    if (a.ksteps > 2)
        fetch(2, p0);
    __syncthreads();

    v4i acc[PT][FT][kSums]; // HH, HL + LH, LL
#pragma unroll
    for (int c = 0; c < PT; c++)
#pragma unroll
        for (int t = 0; t < FT; t++)
#pragma unroll
            for (int s = 0; s < kSums; s++)
                acc[c][t][s] = v4i{0, 0, 0, 0};
    // row i of filter tile t is filter 4 FT (i / 4) + 4 t + i % 4: a lane ends up with 4 FT consecutive channels
    const int a_row0 = 4 * FT * (col >> 2) + (col & 3);
    auto products = [&](int buf) {
        v4i xh[PT], xl[PT];
#pragma unroll
        for (int c = 0; c < PT; c++) {
            const int at = (16 * PT * wave + 16 * c + col) * kRow + 16 * quad;
            xh[c] = *reinterpret_cast<const v4i *>(&b_l[buf][0][at]);
            if constexpr (!X8)
                xl[c] = *reinterpret_cast<const v4i *>(&b_l[buf][1][at]);
        }
#pragma unroll
        for (int t = 0; t < FT; t++) {
            const int at = (a_row0 + 4 * t) * kRow + 16 * quad;
            const v4i wh = *reinterpret_cast<const v4i *>(&a_l[buf][0][at]);
            const v4i wl = *reinterpret_cast<const v4i *>(&a_l[buf][1][at]);
#pragma unroll
            for (int c = 0; c < PT; c++) {
                acc[c][t][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wh, xh[c], acc[c][t][0], 0, 0, 0);
                acc[c][t][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wl, xh[c], acc[c][t][1], 0, 0, 0);
                if constexpr (!X8) {
                    acc[c][t][2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wl, xl[c], acc[c][t][2], 0, 0, 0);
                    acc[c][t][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wh, xl[c], acc[c][t][1], 0, 0, 0);
                }
            }
        }
    };
    // one barrier per step, as in the int8 kernel (conv2d_s8_pwgemm.hip): step ks reads buffer ks & 1, its end fills
    // the other one from the registers requested two steps before
    for (int ks = 0; ks < a.ksteps; ks += 2) {
        products(0);
        if (ks + 1 < a.ksteps) {
            stash(1, p1);
            if (ks + 3 < a.ksteps)
                fetch(ks + 3, p1);
            __syncthreads();
            products(1);
            if (ks + 2 < a.ksteps) {
                stash(0, p0);
                if (ks + 4 < a.ksteps)
                    fetch(ks + 4, p0);
                __syncthreads();
            }
        }
    }
    // the byte sums: four threads share a row
    auto row_term = [&](int h, int l) {
#pragma unroll
        for (int d = 1; d < 4; d *= 2) {
            h += __shfl_xor(h, d);
            l += __shfl_xor(l, d);
        }
        return byte_term(h, l);
    };
#pragma unroll
    for (int j = 0; j < PT; j++) {
        const long long t = row_term(bsum_h[j], bsum_l[j]);
        if (q4 == 0)
            pix_term[64 * j + my_row] = t;
    }
    if constexpr (!X8) {
        const long long t = row_term(wsum_h, wsum_l);
        if (q4 == 0 && my_row < 16 * FT)
            cst[my_row] += t; // (the first barrier lies behind the start value)
    }
    __syncthreads();

    // Epilogue.  With C the sum of all constants of a value (filter, pixel, and 2^(s-1) for the rounding),
    //   floor((65536 HH + 256 M + LL + C) / 65536) = HH + Ch + floor((M + floor((LL + Cl) / 256)) / 256),  C = 65536 Ch + Cl
    // in 32-bit arithmetic, so a shift of 16 or more is that number shifted by the rest: about nine vector
    // instructions per value where 64-bit arithmetic takes some fifty (80 x 80 x 64 -> 64, 1 x 1, batch 64: 45 -> 34 us).
    // A shift below 16 takes the low half of the sum as well; where the number does not fit 16 bits such a
    // shift saturates anyway.  The fast form needs half-up rounding, shifts of 1 to 44, filter constants
    // below 2^45 and fewer than 1000 steps: no 32-bit sum can then overflow.
    int fine = 1, low = 0;
    if (tid < 16 * FT) {
        const long long c = cst[tid];
        const int s = shf[tid];
        fine = !a.half_even && a.ksteps < 1000 && s >= 1 && s <= 44 && c < (1ll << 45) && c > -(1ll << 45);
        low = s < 16;
        if (fine) {
            const long long r = c + (1ll << (s - 1));
            fast_cst[tid] = v2i{(int)(r >> 16), (int)(r & 0xffff)};
        }
    }
    const bool fast = __syncthreads_and(fine) != 0;
    const bool any_low = __syncthreads_or(low) != 0;
    const int n = n0 + 4 * FT * quad; // this lane: channels n .. n + 4 FT - 1
    auto write = [&](int c, int(&words)[2 * FT]) {
        if constexpr (X8) {
            if (a.table != nullptr) {
#pragma unroll
                for (int i = 0; i < 2 * FT; i++) {
                    const int lo = nearest_entry(words[i], a.table_shift, a.half_even != 0);
                    const int hi = nearest_entry(words[i] >> 16, a.table_shift, a.half_even != 0);
                    words[i] = (int)(unsigned short)table_l[lo] | (table_l[hi] << 16);
                }
            }
        }
        const int row = 16 * PT * wave + 16 * c + col;
        if (m0 + row >= a.n_pix || n >= a.out_c)
            return;
        int16_t *dst = a.out + (long long)(m0 + row) * a.out_c + n;
        if (n + 4 * FT <= a.out_c) {
            if constexpr (FT == 1) {
                *reinterpret_cast<v2i_unaligned *>(dst) = v2i{words[0], words[1]};
            } else {
#pragma unroll
                for (int i = 0; i < FT / 2; i++)
                    *reinterpret_cast<v4i_unaligned *>(dst + 8 * i) =
                        v4i{words[4 * i], words[4 * i + 1], words[4 * i + 2], words[4 * i + 3]};
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4 * FT; i++)
                if (n + i < a.out_c)
                    dst[i] = (int16_t)(words[i >> 1] >> (16 * (i & 1)));
        }
    };
    auto quick = [&](auto low_tag) {
        constexpr bool LOW = decltype(low_tag)::value;
        const v2s floor2 = __builtin_bit_cast(v2s, a.relu != 0 ? 0 : (int)0x80008000u);
        int ph[PT], pl[PT];
#pragma unroll
        for (int c = 0; c < PT; c++) {
            const long long pt = pix_term[16 * PT * wave + 16 * c + col];
            ph[c] = (int)(pt >> 16);
            pl[c] = (int)(pt & 0xffff);
        }
        int words[PT][2 * FT];
#pragma unroll
        for (int t = 0; t < FT; t++) {
            int q[PT][4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int f = 4 * FT * quad + 4 * t + r;
                const int fh = fast_cst[f][0], fl = fast_cst[f][1];
                const int s = shf[f];
#pragma unroll
                for (int c = 0; c < PT; c++) {
                    const int l = (X8 ? 0 : acc[c][t][kSums - 1][r]) + fl + pl[c];
                    const int mid = acc[c][t][1][r] + (l >> 8);
                    const int x = acc[c][t][0][r] + fh + ph[c] + (mid >> 8);
                    if constexpr (LOW) {
                        const int top = min(max(x, -32768), 32767);
                        const int v = (top << 16) | ((mid & 255) << 8) | (l & 255);
                        q[c][r] = s < 16 ? v >> s : x >> (s - 16);
                    } else {
                        q[c][r] = x >> (s - 16);
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < PT; c++) {
                words[c][2 * t] = __builtin_bit_cast(int, __builtin_elementwise_max(__builtin_amdgcn_cvt_pk_i16(q[c][0], q[c][1]), floor2));
                words[c][2 * t + 1] = __builtin_bit_cast(int, __builtin_elementwise_max(__builtin_amdgcn_cvt_pk_i16(q[c][2], q[c][3]), floor2));
            }
        }
#pragma unroll
        for (int c = 0; c < PT; c++)
            write(c, words[c]);
    };
    if (fast) {
        if (any_low)
            quick(std::true_type{});
        else
            quick(std::false_type{});
        return;
    }
    const bool relu = a.relu != 0, half_even = a.half_even != 0;
#pragma unroll
    for (int c = 0; c < PT; c++) {
        const long long pt = pix_term[16 * PT * wave + 16 * c + col];
        int words[2 * FT];
#pragma unroll
        for (int t = 0; t < FT; t++) {
            int q[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int f = 4 * FT * quad + 4 * t + r;
                const int s = shf[f];
                const long long v = cst[f] + pt + combine(acc[c][t][0][r], acc[c][t][1][r], X8 ? 0 : acc[c][t][kSums - 1][r]);
                q[r] = requant_s16(v, s, relu, half_even);
            }
            words[2 * t] = (q[0] & 0xffff) | (q[1] << 16);
            words[2 * t + 1] = (q[2] & 0xffff) | (q[3] << 16);
        }
        write(c, words);
    }
}

// (The arguments by value: by reference the compiler fetches some of them behind the loop's branches, 50 instructions more; 5 x 5 over 160
// channels and 228 pixels -> 16 6.0 -> 6.5 us, 900 layers 0.9 % longer.)
template <int NT, bool ALIGNED, bool X8>
__device__ __forceinline__ void narrow16_tile(const S16Args a, int bx, int by)
{
    constexpr int G = 2; // steps per batch of loads
    constexpr int kSums = X8 ? 2 : 3;
    __shared__ v4i part[4][NT][kSums][64];
    __shared__ long long pix_part[4][16], flt_part[4][NT][16];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int m = bx * 16 + col;
    const int n0 = by * 16 * NT;

    const __amdgpu_buffer_rsrc_t in_rsrc = tensor_rsrc(a.win.in, a.win.in_bytes);
    const __amdgpu_buffer_rsrc_t w_rsrc = tensor_rsrc(a.win.w, a.win.w_bytes);
    const PixelWindow px = pixel_window(a.win, m, a.n_pix);
    int row[NT]; // row i of tile t is filter 4 NT (i / 4) + 4 t + i % 4
#pragma unroll
    for (int t = 0; t < NT; t++)
        row[t] = min(n0 + 4 * NT * (col >> 2) + 4 * t + (col & 3), a.out_c - 1) * a.win.w_len;

    struct Batch {
        std::conditional_t<X8, v4i, Unit16> b[G];
        Unit16 w[G][NT];
        int n[G];
    };
    auto request = [&](int s0, Batch &t) {
#pragma unroll
        for (int i = 0; i < G; i++) {
            const int at = 4 * (wave + 4 * (s0 + i)) + quad;
            const Unit u = X8 ? locate_unit_x8(a.win, at) : locate_unit16(a.win, at);
            t.n[i] = u.n;
            if constexpr (X8)
                t.b[i] = load_pixel_unit<ALIGNED>(a.win, in_rsrc, px, u);
            else
                t.b[i] = load_pixel16<ALIGNED>(a.win, in_rsrc, px, u);
#pragma unroll
            for (int f = 0; f < NT; f++)
                t.w[i][f] = load_filter16<ALIGNED>(a.win, w_rsrc, row[f], u);
        }
    };
    const int steps = (a.ksteps - wave + 3) >> 2; // of this wavefront (none for the last ones of a short reduction)
    Batch cur, nxt;
    request(0, cur);

    // what the epilogue needs: wavefront t finishes filter tile t
    const bool finisher = wave < NT;
    const int f0 = n0 + 4 * NT * quad + 4 * wave;
    long long bias[4];
    int shift[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int n = min(f0 + r, a.out_c - 1);
        bias[r] = (finisher && a.bias != nullptr) ? a.bias[n] : 0;
        shift[r] = finisher ? a.shift[a.n_shift == 1 ? 0 : n] : 0;
    }

    v4i acc[NT][kSums];
    int bh = 0, bl = 0, wh_s[NT] = {}, wl_s[NT] = {};
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int s = 0; s < kSums; s++)
            acc[t][s] = v4i{0, 0, 0, 0};
    auto products = [&](const Batch &t, int left) {
#pragma unroll
        for (int i = 0; i < G; i++)
            if (i < left) { // uniform
                v4i xh, xl;
                if constexpr (X8) {
                    xh = t.b[i];
                    bh = byte_sum(xh, bh);
                } else {
                    const Planes x = cut(t.b[i], bh, bl);
                    xh = x.h;
                    xl = x.l;
                }
#pragma unroll
                for (int f = 0; f < NT; f++) {
                    const Planes w = cut_filter<ALIGNED>(t.w[i][f], t.n[i], wh_s[f], wl_s[f]);
                    acc[f][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w.h, xh, acc[f][0], 0, 0, 0);
                    acc[f][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w.l, xh, acc[f][1], 0, 0, 0);
                    if constexpr (!X8) {
                        acc[f][2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w.l, xl, acc[f][2], 0, 0, 0);
                        acc[f][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w.h, xl, acc[f][1], 0, 0, 0);
                    }
                }
            }
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
    // the four 16-lane groups hold different units of the same pixel and filter rows
    bh += __shfl_xor(bh, 16);
    bl += __shfl_xor(bl, 16);
    bh += __shfl_xor(bh, 32);
    bl += __shfl_xor(bl, 32);
    if (quad == 0)
        pix_part[wave][col] = byte_term(bh, bl);
#pragma unroll
    for (int t = 0; t < NT; t++) {
        int h = wh_s[t], l = wl_s[t];
        h += __shfl_xor(h, 16);
        l += __shfl_xor(l, 16);
        h += __shfl_xor(h, 32);
        l += __shfl_xor(l, 32);
        if (quad == 0)
            flt_part[wave][t][col] = byte_term(h, l);
#pragma unroll
        for (int s = 0; s < kSums; s++)
            part[wave][t][s][lane] = acc[t][s];
    }
    __syncthreads();
    if (!finisher || m >= a.n_pix || f0 >= a.out_c)
        return;
    v4i sum[3];
    sum[2] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < kSums; s++)
        sum[s] = part[0][wave][s][lane] + part[1][wave][s][lane] + part[2][wave][s][lane] + part[3][wave][s][lane];
    // every wavefront counted its own steps: 64 positions each
    const long long common = pix_part[0][col] + pix_part[1][col] + pix_part[2][col] + pix_part[3][col] +
        (X8 ? 0 : 16384ll * 64 * a.ksteps);
    int q[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int i = 4 * quad + r; // filter row of the tile
        const long long flt =
            X8 ? 0 : flt_part[0][wave][i] + flt_part[1][wave][i] + flt_part[2][wave][i] + flt_part[3][wave][i];
        q[r] = requant_s16(bias[r] + common + flt + combine(sum[0][r], sum[1][r], sum[2][r]), shift[r], a.relu != 0,
                           a.half_even != 0);
        if (X8 && a.table != nullptr)
            q[r] = a.table[nearest_entry(q[r], a.table_shift, a.half_even != 0)];
    }
    int16_t *dst = a.out + (long long)m * a.out_c + f0;
    if (f0 + 4 <= a.out_c) {
        *reinterpret_cast<v2i_unaligned *>(dst) = v2i{(q[0] & 0xffff) | (q[1] << 16), (q[2] & 0xffff) | (q[3] << 16)};
    } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (f0 + r < a.out_c)
                dst[r] = (int16_t)q[r];
    }
}

template <int NT, bool ALIGNED, bool X8>
__global__ __launch_bounds__(kThreads) void conv2d_s16_narrow_kernel(const S16Args a)
{
    narrow16_tile<NT, ALIGNED, X8>(a, (int)blockIdx.x, (int)blockIdx.y);
}

// Several layers that do not depend on one another in one launch, as in conv2d_s8_narrow.hip (64 -> 64 over 52, 26 and 13 pixels
// square, 3 x 3 on int8 inputs: 18 us one by one, 9 together; 1 x 1: 16 and 7).
struct S16Group {
    S16Args layer[kMostGrouped];
    int first[kMostGrouped];       // first workgroup of a layer
    FastDiv columns[kMostGrouped]; // workgroups of a row of its grid
};
template <bool X8>
__global__ __launch_bounds__(kThreads) void conv2d_s16_narrow_group_kernel(const S16Group g)
{
    int i = 0;
#pragma unroll
    for (int k = 1; k < kMostGrouped; k++)
        i += (int)blockIdx.x >= g.first[k] ? 1 : 0;
    const unsigned at = blockIdx.x - g.first[i];
    const unsigned by = fastdiv(at, g.columns[i]);
    narrow16_tile<1, true, X8>(g.layer[i], (int)(at - by * g.columns[i].d), (int)by);
}

template <bool X8>
void launch_narrow16(const S16Args &a, bool two, bool aligned, hipStream_t stream)
{
    const dim3 grid((unsigned)((a.n_pix + 15) / 16), (unsigned)(two ? (a.out_c + 31) / 32 : (a.out_c + 15) / 16));
    if (two && aligned)
        hipLaunchKernelGGL((conv2d_s16_narrow_kernel<2, true, X8>), grid, dim3(kThreads), 0, stream, a);
    else if (two)
        hipLaunchKernelGGL((conv2d_s16_narrow_kernel<2, false, X8>), grid, dim3(kThreads), 0, stream, a);
    else if (aligned)
        hipLaunchKernelGGL((conv2d_s16_narrow_kernel<1, true, X8>), grid, dim3(kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((conv2d_s16_narrow_kernel<1, false, X8>), grid, dim3(kThreads), 0, stream, a);
}

template <int FT, bool X8>
void launch_gemm(const S16Args &a, bool aligned, int cus, hipStream_t stream)
{
    // 128-pixel tiles unless that leaves fewer than 1.5 workgroups per compute unit
    const unsigned gy = (unsigned)((a.out_c + 16 * FT - 1) / (16 * FT));
    const long long tiles128 = (a.n_pix + 127) / 128;
    const bool small = tiles128 * gy * 2 < 3ll * cus;
    const dim3 grid(small ? (unsigned)((a.n_pix + 63) / 64) : (unsigned)tiles128, gy);
    if (small && aligned)
        hipLaunchKernelGGL((conv2d_s16_gemm_kernel<1, FT, true, X8>), grid, dim3(kThreads), 0, stream, a);
    else if (small)
        hipLaunchKernelGGL((conv2d_s16_gemm_kernel<1, FT, false, X8>), grid, dim3(kThreads), 0, stream, a);
    else if (aligned)
        hipLaunchKernelGGL((conv2d_s16_gemm_kernel<2, FT, true, X8>), grid, dim3(kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((conv2d_s16_gemm_kernel<2, FT, false, X8>), grid, dim3(kThreads), 0, stream, a);
}

// The geometry in bytes, as conv_window.h counts: a pixel of in_c channels is 2 in_c bytes.
ConvGeom byte_geometry(ConvGeom g)
{
    g.in_c *= 2;
    g.in_pitch = g.in_c;
    return g;
}

int steps_of(const ConvGeom &g)
{
    return (g.k_h * g.k_w * ((g.in_c + 15) / 16) + 3) / 4;
}

// Expected times of the two kernels, straight lines in their work fitted to 97 layers of 56 to 720 K output pixels
// (within 10 to 17 %): launch, the steps of one wavefront or workgroup, all of them over the device.
struct S16Choice {
    float gemm_us, narrow_us;
    int ft;   // filter tiles of a workgroup of the GEMM form
    bool two; // the narrow form's wavefronts take two
    bool narrow() const { return narrow_us < gemm_us; }
    // In a group of layers the narrow form saves the launch and the time between two.
    bool groups() const { return narrow_us < gemm_us + 1.2f; }
};
S16Choice choose(const ConvGeom &g, bool aligned, int cus)
{
    S16Choice c;
    const long long n_pix = (long long)g.batch * g.out_h * g.out_w;
    c.ft = g.out_c <= 16 ? 1 : (g.out_c <= 32 ? 2 : 4);
    const int ksteps = steps_of(g);
    const float steps = (float)ksteps;
    const float tiles = 1e-3f * (float)((n_pix + 63) / 64 * ((g.out_c + 16 * c.ft - 1) / (16 * c.ft)));
    c.gemm_us = aligned ? 3.0f + 0.385f * steps + tiles * (0.227f * steps * (float)(1 + c.ft) + 0.644f * (float)(2 + c.ft))
                        : 3.26f + 0.68f * steps + tiles * (0.158f * steps * (float)(1 + c.ft) + 1.05f * (float)(2 + c.ft));
    const unsigned tiles16 = (unsigned)((n_pix + 15) / 16);
    c.two = g.out_c > 16 && (long long)tiles16 * ((g.out_c + 31) / 32) >= 2ll * cus;
    const unsigned ny = (unsigned)(c.two ? (g.out_c + 31) / 32 : (g.out_c + 15) / 16);
    const float waves = 4e-3f * (float)tiles16 * (float)ny, own = (float)((ksteps + 3) / 4), nt = c.two ? 2.f : 1.f;
    c.narrow_us = aligned ? 3.15f + 0.09f * own + waves * (0.157f + 0.336f * own * nt)
                          : 3.44f + 0.21f * own + waves * (0.51f + 0.277f * own * nt);
    return c;
}

// A layer's launch: the one that is expected to be faster.
template <bool X8>
void launch_one(const S16Args &a, const S16Choice &c, bool aligned, int cus, hipStream_t stream)
{
    if (c.narrow())
        launch_narrow16<X8>(a, c.two, aligned, stream);
    else if (c.ft == 1)
        launch_gemm<1, X8>(a, aligned, cus, stream);
    else if (c.ft == 2)
        launch_gemm<2, X8>(a, aligned, cus, stream);
    else
        launch_gemm<4, X8>(a, aligned, cus, stream);
}

// A launch held back in this thread's open group.
struct Held {
    S16Args args;
    S16Choice choice;
    bool x8;
    int cus;
    hipStream_t stream;
};
thread_local Held held[kMostGrouped];
thread_local int n_held = 0;

// The kernel for a layer and its launch; a.win holds the input and the filter.
template <bool X8>
hipError_t launch_units(const ConvGeom &g, S16Args &a, const int64_t *bias, const int32_t *shift, int16_t *out, int cu_count,
                        hipStream_t stream)
{
    a.win.upt = (g.in_c + 15) / 16; // units of 16 channels
    a.win.n_units = g.k_h * g.k_w * a.win.upt;
    a.win.fd_upt = make_fastdiv((unsigned)a.win.upt);
    a.bias = bias;
    a.shift = shift;
    a.out = out;
    a.n_pix = g.batch * g.out_h * g.out_w;
    a.out_c = g.out_c;
    a.ksteps = steps_of(g);
    a.relu = g.relu;
    a.half_even = g.half_even;
    a.n_shift = g.n_shift;
    if (a.n_pix == 0)
        return hipSuccess;
    const bool aligned = (g.in_c & 15) == 0 &&
        ((reinterpret_cast<uintptr_t>(a.win.in) | reinterpret_cast<uintptr_t>(a.win.w)) & 15) == 0;
    const int cus = cu_count > 0 ? cu_count : 256;
    const S16Choice c = choose(g, aligned, cus);
    if constexpr (X8) { // 3 x 3 layers of whole units as a walk down the image, once their rows fill the device
        const int8_t *in = static_cast<const int8_t *>(a.win.in);
        if (1.1f * conv2d_s16_x8_walk_us(g, in, out, a.table_size, cus) < std::min(c.narrow_us, c.gemm_us)) // (56 x 56 x 16, batch 64: 11.9 against 10.6 us)
            return launch_conv2d_s16_x8_walk(g, in, reinterpret_cast<const int16_t *>(a.win.w), bias, shift, a.table, a.table_size, a.table_shift,
                                             out, cus, stream);
    }
    if (group_open && aligned && c.groups() && n_held < kMostGrouped)
        held[n_held++] = Held{a, c, X8, cus, stream};
    else
        launch_one<X8>(a, c, aligned, cus, stream);
    return hipGetLastError();
}

} // namespace

bool conv2d_s16_units_supports(const ConvGeom &g)
{
    return steps_of(g) < 1024 && window_supports(byte_geometry(g)); // K = 64 steps: the int32 accumulators stay exact
}

hipError_t launch_conv2d_s16_units(const ConvGeom &g, const int16_t *in, const int16_t *filter, const int64_t *bias,
                                   const int32_t *shift, int16_t *out, int cu_count, hipStream_t stream)
{
    S16Args a = {};
    a.win = window_args(byte_geometry(g), reinterpret_cast<const int8_t *>(in), reinterpret_cast<const int8_t *>(filter));
    return launch_units<false>(g, a, bias, shift, out, cu_count, stream);
}

bool conv2d_s16_x8_supports(const ConvGeom &g, int table_size)
{
    return conv2d_s16_units_supports(g) && window_supports(g) && table_size <= kMostTable;
}

hipError_t launch_conv2d_s16_x8(const ConvGeom &g, const int8_t *in, const int16_t *filter, const int64_t *bias,
                                const int32_t *shift, const int16_t *table, int table_size, int16_t *out, int cu_count,
                                hipStream_t stream)
{
    S16Args a = {};
    a.win = window_args(g, in, reinterpret_cast<const int8_t *>(filter));
    a.win.w_len *= 2;
    a.win.w_bytes *= 2;
    a.table = table;
    a.table_size = table_size;
    for (a.table_shift = 0; table != nullptr && ((table_size - 1) << a.table_shift) < 65536;)
        a.table_shift++;
    return launch_units<true>(g, a, bias, shift, out, cu_count, stream);
}

// Which of a group's launches a layer takes (0: none), for tensors at aligned addresses.
int conv2d_s16_group_kind(const ConvGeom &g, bool x8, int table_size, int cu_count)
{
    const S16Choice c = choose(g, true, cu_count > 0 ? cu_count : 256);
    const void *aligned = reinterpret_cast<const void *>(uintptr_t(256));
    if ((g.in_c & 15) != 0 || !c.groups() ||
        (x8 && 1.1f * conv2d_s16_x8_walk_us(g, aligned, aligned, table_size, cu_count > 0 ? cu_count : 256) < std::min(c.narrow_us, c.gemm_us)))
        return 0;
    return x8 ? 6 : 5;
}

// The launches held back since the group was opened: those of one build together.
hipError_t flush_conv2d_s16_units()
{
    const int n = n_held;
    n_held = 0;
    bool done[kMostGrouped] = {};
    for (int i = 0; i < n; i++) {
        if (done[i])
            continue;
        const Held &h = held[i];
        S16Group group;
        long long blocks = 0;
        int members = 0;
        for (int j = i; j < n; j++) {
            const Held &o = held[j];
            if (o.x8 != h.x8 || o.stream != h.stream)
                continue;
            const unsigned columns = (unsigned)((o.args.n_pix + 15) / 16);
            done[j] = true;
            group.layer[members] = o.args;
            group.first[members] = (int)blocks;
            group.columns[members] = make_fastdiv(columns);
            blocks += (long long)columns * ((o.args.out_c + 15) / 16);
            members++;
        }
        if (members == 1 || blocks > 1 << 20) { // (a group's layers are small)
            for (int j = i; j < n; j++)
                if (held[j].x8 == h.x8 && held[j].stream == h.stream) {
                    if (h.x8)
                        launch_one<true>(held[j].args, held[j].choice, true, held[j].cus, h.stream);
                    else
                        launch_one<false>(held[j].args, held[j].choice, true, held[j].cus, h.stream);
                }
        } else {
            for (int k = members; k < kMostGrouped; k++) {
                group.layer[k] = group.layer[0];
                group.first[k] = (int)blocks;
                group.columns[k] = group.columns[0];
            }
            const auto kernel = h.x8 ? conv2d_s16_narrow_group_kernel<true> : conv2d_s16_narrow_group_kernel<false>;
            hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kThreads), 0, h.stream, group);
        }
    }
    return n > 0 ? hipGetLastError() : hipSuccess;
}

} // namespace espdl
