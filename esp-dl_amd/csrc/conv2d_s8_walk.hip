// Planner of the walking convolution kernel (conv2d_s8_walk_kernel.h).
#include "conv2d_s8_walk_kernel.h"

namespace espdl {

namespace {

using namespace walk;

// Layer -> kernel arguments (without pointers).  False: a layer that no build takes.
bool walk_layer(const ConvGeom &g, bool residual, WalkArgs *out, WalkLaunch *launch)
{
    if (g.in_c < 16 || g.out_c < 4 || g.in_c > 256 || g.half_even)
        return false;
    if (residual && ((g.out_c & 15) || (g.res_pitch & 15) || g.res_shift != 0))
        return false;
    if (g.k_h != g.k_w || (g.k_h != 1 && g.k_h != 3 && g.k_h != 5) || g.stride_h != g.stride_w || g.stride_w > 2 || g.dil_h != 1 ||
        g.dil_w != 1)
        return false;
    // offsets into the tensors are 31-bit
    const long long px = (long long)g.batch * g.in_h * g.in_w, po = (long long)g.batch * g.out_h * g.out_w;
    const long long most = (1ll << 31) - 65536; // (the last row of a sequence of pixels may end a workgroup's width past it)
    if (px * g.in_pitch >= most || po * g.out_pitch >= most || (residual && po * g.res_pitch >= most))
        return false;
    WalkArgs a = {};
    a.in_bytes = (int)((px - 1) * g.in_pitch + g.in_c);
    a.last = g.in_c - 16;
    a.w_len = g.k_h * g.k_w * g.in_c;
    a.w_bytes = (int)std::min<long long>((long long)g.out_c * a.w_len, most);
    if ((long long)g.out_c * a.w_len >= most)
        return false;
    a.out_bytes = (int)((po - 1) * g.out_pitch + g.out_c);
    a.res_bytes = residual ? (int)((po - 1) * g.res_pitch + g.out_c) : 0;
    a.in_pitch = g.in_pitch;
    a.out_pitch = g.out_pitch;
    a.res_pitch = g.res_pitch;
    a.out_c = g.out_c;
    a.n_shift = g.n_shift;
    a.relu = g.relu;
    a.through = writes_through((long long)po * g.out_c);
    a.mac_bound = (long long)g.k_h * g.k_w * g.in_c * 16384;
    WalkLaunch l = {};
    l.out_bytes = po * g.out_c;
    if (g.k_h == 1 && g.stride_w == 1 && g.pad_top == 0 && g.pad_left == 0 && g.out_h == g.in_h && g.out_w == g.in_w) {
        a.batch = 1;
        l.flat = true;
        l.out_cols = px;
        *out = a;
        *launch = l;
        return true;
    }
    int s = g.stride_w;
    a.in_h = g.in_h;
    a.in_w = g.in_w;
    a.in_row = g.in_w * g.in_pitch;
    a.in_img = a.in_row * g.in_h;
    if (g.k_h == 1 && s == 2) { // every second pixel of every second row, as an image of its own
        if ((g.pad_top | g.pad_left) & 1)
            return false;
        a.in_h = (g.in_h + 1) / 2;
        a.in_w = (g.in_w + 1) / 2;
        a.in_pitch *= 2;
        a.in_row *= 2;
        a.pad_top = g.pad_top / 2;
        a.pad_left = g.pad_left / 2;
        s = 1;
    } else {
        a.pad_top = g.pad_top;
        a.pad_left = g.pad_left;
    }
    a.out_w = g.out_w;
    a.out_h = g.out_h;
    a.batch = g.batch;
    a.out_row = g.out_w * g.out_pitch;
    a.out_img = a.out_row * g.out_h;
    a.res_row = g.out_w * g.res_pitch;
    a.res_img = a.res_row * g.out_h;
    // images side by side: between two of them as many columns as the windows reach past an image on either side
    const long long over = (long long)(g.out_w - 1) * s + g.k_w - 1 - a.pad_left - (a.in_w - 1);
    long long pitch = std::max<long long>(a.in_w + std::max<long long>({0, a.pad_left, over}), (long long)g.out_w * s);
    pitch = (pitch + s - 1) / s * s;
    l.out_cols = (g.batch - 1) * (pitch / s) + g.out_w;
    const long long width = 4096; // more than a workgroup's columns, input columns included
    if ((long long)g.batch * pitch + width >= most || (l.out_cols / 16 + width) * g.out_h >= most)
        return false;
    a.fd_p = make_fastdiv((unsigned)pitch);
    a.fd_po = make_fastdiv((unsigned)(pitch / s));
    a.fd_oh = make_fastdiv((unsigned)a.out_h);
    *out = a;
    *launch = l;
    return true;
}

hipError_t walk_launch(const ConvGeom &g, int nt, WalkArgs &a, const WalkLaunch &l)
{
    const int cu = (g.in_c + 15) / 16;
    if ((g.in_c | g.in_pitch) & 3) // pieces that are no whole dwords of memory
        return g.k_h == 1                   ? launch_raw_1x1(cu, nt, a, l)
            : g.k_h == 3 && g.stride_w == 1 ? launch_raw_3x3(cu, nt, a, l)
                                            : hipErrorInvalidValue;
    if (g.k_h == 1)
        return launch_1x1(cu, nt, a, l);
    if (g.k_h == 3)
        return g.stride_w == 1 ? launch_3x3(cu, nt, a, l) : launch_3x3_s2(cu, nt, a, l);
    return launch_5x5(cu, g.stride_w, nt, a, l);
}

// The filter tiles of a wavefront with the smallest expected time; 0: no build.
int walk_tiles(const ConvGeom &g, const WalkArgs &args, WalkLaunch l, float *us)
{
    int best = 0;
    *us = 1e30f;
    for (int nt : {1, 2, 3, 4, 8}) {
        if (16 * nt >= 2 * g.out_c && nt > 1) // half of the filters would not exist
            continue;
        if (g.out_c < (nt == 8 ? 16 : 4 * nt)) // (a lane's channels)
            continue;
        if (nt == 3 && g.out_c % 16 == 0 && g.out_c % 48 != 0) // (whole tiles: the other counts leave no lane with a part)
            continue;
        WalkArgs a = args;
        float t = 0.f;
        l.us = &t;
        if (walk_launch(g, nt, a, l) == hipSuccess && t < *us) {
            *us = t;
            best = nt;
        }
    }
    return best;
}

} // namespace

float conv2d_s8_walk_us(const ConvGeom &g, const void *in, const void *filter, const void *residual, const void *out, int cu_count)
{
    WalkArgs a;
    WalkLaunch l;
    if (((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(filter) | reinterpret_cast<uintptr_t>(residual) |
          reinterpret_cast<uintptr_t>(out)) & 15) != 0 || !walk_layer(g, residual != nullptr, &a, &l))
        return 1e30f;
    a.res = static_cast<const int8_t *>(residual);
    l.cus = cu_count > 0 ? cu_count : 256;
    float us;
    walk_tiles(g, a, l, &us);
    return us;
}

hipError_t launch_conv2d_s8_walk(const ConvGeom &g, const int8_t *in, const int8_t *filter, const int32_t *bias,
                                 const int32_t *shift, const int8_t *lut, const int8_t *residual, int8_t *out,
                                 int cu_count, hipStream_t stream)
{
    WalkArgs a;
    WalkLaunch l;
    if (!walk_layer(g, residual != nullptr, &a, &l))
        return hipErrorInvalidValue;
    a.in = in;
    a.w = filter;
    a.bias = bias;
    a.shift = shift;
    a.lut = lut;
    a.res = residual;
    a.out = out;
    l.cus = cu_count > 0 ? cu_count : 256;
    l.stream = stream;
    float us;
    const int nt = walk_tiles(g, a, l, &us);
    return nt > 0 ? walk_launch(g, nt, a, l) : hipErrorInvalidValue;
}

} // namespace espdl
