// Reading a convolution window as rows of a matrix product, for any channel count (int8).
//
// The reduction axis is cut into UNITS of 16 positions: unit u is channels [16 j, 16 j + 16) of tap t with
// u = t * upt + j and upt = ceil(in_c / 16).  Where in_c is not a multiple of 16 the last unit of a tap covers
// fewer channels than it has positions: operand A (the filter) is zero there, so it does not matter that operand
// B (the pixels) holds the first channels of the pixel behind.  Taps outside the image are zeros, which is
// conv_operation_shell's window clipping (esp-dl/dl/base/dl_base.hpp:940-1191).
//
// Every unit is one 16-byte load at whatever address it has, through a buffer descriptor of the tensor: a unit that
// does not exist is given an offset past the descriptor's end and comes back as zeros without a branch or a select,
// so that loads requested ahead stay in flight.  A unit that would end behind the tensor (the last pixel's last
// channels) is read as the tensor's last 16 bytes and shifted down: nothing outside the tensor is touched.
#pragma once

#include "espdl_device.h"
#include "espdl_kernels.h"

namespace espdl {
namespace window {

struct WindowArgs {
    const int8_t *in, *w;
    int in_bytes, w_bytes; // sizes of the two tensors (below 2^31), at least 16 each
    int in_h, in_w, in_c, in_pitch;
    int w_len;   // bytes of one filter
    int upt;     // units per tap
    int n_units; // taps * upt
    int stride_h, stride_w, dil_h, dil_w, pad_top, pad_left;
    FastDiv fd_upt, fd_kw, fd_ow, fd_ohw;
};

// Whether the loads of this header can serve the layer in one launch: tensors of 16 bytes to 2 GiB.
inline bool window_supports(const ConvGeom &g)
{
    const long long in_bytes = ((long long)g.batch * g.in_h * g.in_w - 1) * g.in_pitch + g.in_c;
    const long long w_bytes = (long long)g.out_c * g.k_h * g.k_w * g.in_c;
    return in_bytes >= 16 && w_bytes >= 16 && in_bytes < (1ll << 31) - 64 && w_bytes < (1ll << 31) - 64 &&
        (long long)g.batch * g.out_h * g.out_w < (1ll << 31) - 256;
}
// Every unit is whole and 16-byte aligned.
inline bool window_aligned(const ConvGeom &g, const void *in, const void *filter)
{
    return (g.in_c & 15) == 0 && (g.in_pitch & 15) == 0 &&
        ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(filter)) & 15) == 0;
}
inline WindowArgs window_args(const ConvGeom &g, const int8_t *in, const int8_t *filter)
{
    WindowArgs a;
    a.in = in;
    a.w = filter;
    a.in_bytes = (int)(((long long)g.batch * g.in_h * g.in_w - 1) * g.in_pitch + g.in_c);
    a.w_len = g.k_h * g.k_w * g.in_c;
    a.w_bytes = (int)((long long)g.out_c * a.w_len);
    a.in_h = g.in_h;
    a.in_w = g.in_w;
    a.in_c = g.in_c;
    a.in_pitch = g.in_pitch;
    a.upt = (g.in_c + 15) / 16;
    a.n_units = g.k_h * g.k_w * a.upt;
    a.stride_h = g.stride_h;
    a.stride_w = g.stride_w;
    a.dil_h = g.dil_h;
    a.dil_w = g.dil_w;
    a.pad_top = g.pad_top;
    a.pad_left = g.pad_left;
    a.fd_upt = make_fastdiv((unsigned)a.upt);
    a.fd_kw = make_fastdiv((unsigned)g.k_w);
    a.fd_ow = make_fastdiv((unsigned)g.out_w);
    a.fd_ohw = make_fastdiv((unsigned)(g.out_h * g.out_w));
    return a;
}

constexpr int kParked = (int)0x80000000u; // past the end of any tensor: the load returns zeros

// Where the window of output pixel m starts: byte offset of its first tap (possibly outside the tensor) and that
// tap's row and column.  A pixel that does not exist has every tap outside the image.
struct PixelWindow {
    int base, iy, ix;
};
__device__ __forceinline__ PixelWindow pixel_window(const WindowArgs &a, int m, int n_pix)
{
    PixelWindow p = {0, -0x40000000, 0};
    if (m < n_pix) {
        const unsigned n = fastdiv((unsigned)m, a.fd_ohw);
        const unsigned rem = (unsigned)m - n * a.fd_ohw.d;
        const unsigned oy = fastdiv(rem, a.fd_ow);
        const unsigned ox = rem - oy * a.fd_ow.d;
        p.iy = (int)oy * a.stride_h - a.pad_top;
        p.ix = (int)ox * a.stride_w - a.pad_left;
        p.base = (((int)n * a.in_h + p.iy) * a.in_w + p.ix) * a.in_pitch;
    }
    return p;
}

// Tap and channels of a unit: row and column of the tap inside the window, byte offsets from the window's first tap
// and from the filter's first byte, channels the unit holds (<= 0: the unit does not exist).
struct Unit {
    int dy, dx, in_off, w_off, n;
};
__device__ __forceinline__ Unit locate_unit(const WindowArgs &a, int u)
{
    const unsigned tap = fastdiv((unsigned)u, a.fd_upt);
    const int j = u - (int)(tap * a.fd_upt.d);
    const unsigned ky = fastdiv(tap, a.fd_kw);
    Unit r;
    r.dy = (int)ky * a.dil_h;
    r.dx = (int)(tap - ky * a.fd_kw.d) * a.dil_w;
    r.in_off = (r.dy * a.in_w + r.dx) * a.in_pitch + 16 * j;
    r.w_off = (int)tap * a.in_c + 16 * j;
    r.n = u < a.n_units ? a.in_c - 16 * j : 0;
    return r;
}

// 128 bits moved down by `n` bytes (0 .. 15), zeros above.
__device__ __forceinline__ v4i shift_down(const v4i &v, int n)
{
    unsigned long long lo = (unsigned)v[0] | ((unsigned long long)(unsigned)v[1] << 32);
    unsigned long long hi = (unsigned)v[2] | ((unsigned long long)(unsigned)v[3] << 32);
    if (n >= 8) {
        lo = hi;
        hi = 0;
        n -= 8;
    }
    if (n > 0) {
        lo = (lo >> (8 * n)) | (hi << (64 - 8 * n));
        hi >>= 8 * n;
    }
    return v4i{(int)(unsigned)lo, (int)(unsigned)(lo >> 32), (int)(unsigned)hi, (int)(unsigned)(hi >> 32)};
}

// The 16 bytes at offset `off` of a tensor of `bytes` bytes, zeros for a negative (parked) offset.
template <bool ALIGNED>
__device__ __forceinline__ v4i load16(__amdgpu_buffer_rsrc_t rsrc, int off, int bytes)
{
    if constexpr (ALIGNED)
        return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
    const int last = bytes - 16;
    v4i v = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off > last ? last : off, 0, 0));
    if (off > last) // (a parked offset is negative)
        v = shift_down(v, off - last);
    return v;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tensor_rsrc(const int8_t *p, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(p), (short)0, bytes, 0x00020000);
}

// Operand B: a unit of the window of one pixel.
template <bool ALIGNED>
__device__ __forceinline__ v4i load_pixel_unit(const WindowArgs &a, __amdgpu_buffer_rsrc_t rsrc, const PixelWindow &p, const Unit &u)
{
    const bool ok = u.n > 0 && (unsigned)(p.iy + u.dy) < (unsigned)a.in_h && (unsigned)(p.ix + u.dx) < (unsigned)a.in_w;
    return load16<ALIGNED>(rsrc, ok ? p.base + u.in_off : kParked, a.in_bytes);
}

// Operand A: a unit of the filter whose first byte is at offset `row`.  The positions of a unit that hold no channel
// are not zeroed here: mask_unit does that, right in front of the product, so that the load stays in flight.
template <bool ALIGNED>
__device__ __forceinline__ v4i load_filter_unit(const WindowArgs &a, __amdgpu_buffer_rsrc_t rsrc, int row, const Unit &u)
{
    return load16<ALIGNED>(rsrc, u.n > 0 ? row + u.w_off : kParked, a.w_bytes);
}
template <bool ALIGNED>
__device__ __forceinline__ v4i mask_unit(v4i v, int n)
{
    if constexpr (ALIGNED)
        return v;
    if (n < 16) {
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const int keep = min(max(n - 4 * d, 0), 4);
            v[d] = keep >= 4 ? v[d] : (int)((unsigned)v[d] & ((1u << (8 * keep)) - 1u));
        }
    }
    return v;
}

} // namespace window
} // namespace espdl
