// int8 MaxPool over K x K windows at stride 1 (the pools of SPP / SPPF blocks: 5 x 5, stride 1, padding 2),
// base::max_pool2d of esp-dl/dl/base/dl_base_max_pool2d.cpp:9-29 over the window clipped to the image.
//
// The hardware has no byte-wise maximum, and widening every byte to 32 bits costs several vector-ALU
// operations per byte and window position, which is what bounds a straightforward kernel (a tenth of the
// HBM rate on 5 x 5 windows).  Here the maximum works on int16 pairs (v_pk_max_i16):
//   - of a loaded dword the raw bits serve as the "odd bytes" operand: each 16-bit half orders like its high
//     byte (a signed byte), the low byte below it only breaks ties between equal high bytes, and only the
//     high byte of the result is kept;
//   - the dword shifted left by 8 is the "even bytes" operand in the same way;
//   - one byte permute puts the two results together.
// That is one shift per loaded dword, two packed maxima per dword and window position, one permute per result.
//
// The window is separable: a thread owns two neighbouring output columns and one 16-byte channel vector, walks
// down a strip of output rows, takes the horizontal maxima of each input row once (K + 1 loaded pixels, K
// maxima for the two columns since their windows share K - 1 pixels), keeps the last K of them in registers
// (joined back into bytes, which halves their registers) and takes the vertical maximum for each output row.  A pixel
// outside the image is replaced by the nearest one inside, which the same window holds (every window of a valid geometry
// holds at least one): no load is conditional, and a row's loads are requested while the row before it is worked on.
//
// Bound by memory, at the number of rows in flight: with conditional loads, none of them early, 256 images of 56 x 56 x 144
// took 69 us (3 x 3: 61), 100 of 80 x 80 x 96 44 us and 64 of 20 x 20 x 128 6.9 us; a row ahead 63 (61), 42 and 5.8 us,
// 3.7 TB/s in and out.  Pixels that are not whole dwords apart are taken apart by the memory pipeline, and there the up to five
// rows that a strip requests and does not use cost more than a row ahead gives (17 x 14 x 198, 5 x 5, batch 144: 13.1 us with
// conditional loads, 15.4 with them); the builds for those ask before every row, which costs the others (2 x 17 x 76 x 112,
// 5 x 5: 4.05 -> 4.86).
// Input and output may be channel slices of wider tensors (pitches in bytes).  Where the channels are no multiple of
// the vector, the last one of a pixel reaches back over its neighbour's channels and both write the same bytes: 36 x 8 x
// 194, 128 images take 13.4 us, one byte per thread took 101 us.
#include "espdl_kernels.h"
#include "espdl_device.h"

namespace espdl {

namespace {

constexpr int kThreads = 256;

struct WindowPoolArgs {
    const char *in;
    char *out;
    int h, w, out_h, out_w, pad_top, pad_left;
    int c;      // channels, at least 4 * D
    int cv;     // channel vectors (of D dwords) per pixel
    int rows;   // output rows per strip
    int strips; // strips per image
    int xpairs; // column pairs per row
    long long in_pitch, out_pitch; // bytes from pixel to pixel
    FastDiv fd_cv, fd_xpairs, fd_strips;
    unsigned total; // threads
};

// D dwords of one pixel
template <int D>
struct Vec {
    int d[D];
};

template <int D>
__device__ __forceinline__ Vec<D> load_vec(const char *p)
{
    Vec<D> r;
    if constexpr (D == 4) {
        const v4i x = *reinterpret_cast<const v4i_unaligned *>(p);
        r.d[0] = x[0], r.d[1] = x[1], r.d[2] = x[2], r.d[3] = x[3];
    } else {
        const v2i x = *reinterpret_cast<const v2i_unaligned *>(p);
        r.d[0] = x[0], r.d[1] = x[1];
    }
    return r;
}

template <int D>
__device__ __forceinline__ void store_vec(char *p, const Vec<D> &r)
{
    if constexpr (D == 4)
        *reinterpret_cast<v4i_unaligned *>(p) = v4i{r.d[0], r.d[1], r.d[2], r.d[3]};
    else
        *reinterpret_cast<v2i_unaligned *>(p) = v2i{r.d[0], r.d[1]};
}

template <int D>
__device__ __forceinline__ Vec<D> pkmax(const Vec<D> &a, const Vec<D> &b)
{
    Vec<D> r;
#pragma unroll
    for (int i = 0; i < D; i++)
        r.d[i] = pk_max_i16(a.d[i], b.d[i]);
    return r;
}

// the bytes of each dword moved up by one: the even bytes where packed int16 maxima order by them
template <int D>
__device__ __forceinline__ Vec<D> shifted(const Vec<D> &a)
{
    Vec<D> r;
#pragma unroll
    for (int i = 0; i < D; i++)
        r.d[i] = a.d[i] << 8;
    return r;
}

// bytes [even.1, odd.1, even.3, odd.3] of each dword: the maxima of the odd-byte and even-byte operands as bytes
template <int D>
__device__ __forceinline__ Vec<D> join(const Vec<D> &odd, const Vec<D> &even)
{
    Vec<D> r;
#pragma unroll
    for (int i = 0; i < D; i++)
        r.d[i] = (int)__builtin_amdgcn_perm((unsigned)odd.d[i], (unsigned)even.d[i], 0x07030501u);
    return r;
}

// K x K window, D dwords of channels per thread.  SHORT: rows that the strip does not use are not requested.
template <int K, int D, bool SHORT>
__global__ __launch_bounds__(kThreads) void max_pool_s8_window_kernel(const WindowPoolArgs a)
{
    typedef Vec<D> V;
    const unsigned tid = blockIdx.x * kThreads + threadIdx.x;
    if (tid >= a.total)
        return;
    const unsigned q0 = fastdiv(tid, a.fd_cv);
    const unsigned v = tid - q0 * a.fd_cv.d;
    const unsigned q1 = fastdiv(q0, a.fd_xpairs);
    const unsigned xp = q0 - q1 * a.fd_xpairs.d;
    const unsigned n = fastdiv(q1, a.fd_strips);
    const unsigned strip = q1 - n * a.fd_strips.d;
    const int x0 = 2 * (int)xp, y0 = (int)strip * a.rows;
    const int c0 = min((int)v * 4 * D, a.c - 4 * D);
    const char *img_in = a.in + (long long)n * a.h * a.w * a.in_pitch + c0;
    char *img_out = a.out + (long long)n * a.out_h * a.out_w * a.out_pitch + c0;

    // The K + 1 input columns under the two windows.  A column or row outside the image is replaced by the nearest one inside:
    // the window holds that one too, so its maximum stays the same and every load is unconditional.
    long long col_off[K + 1];
#pragma unroll
    for (int c = 0; c <= K; c++)
        col_off[c] = (long long)min(max(x0 - a.pad_left + c, 0), a.w - 1) * a.in_pitch;
    const bool second = x0 + 1 < a.out_w;
    const long long row_pitch = (long long)a.w * a.in_pitch;

    // the K + 1 pixels of input row `r` of the strip
    auto load_row = [&](int r, V (&px)[K + 1]) {
        const char *row = img_in + min(max(y0 - a.pad_top + r, 0), a.h - 1) * row_pitch;
#pragma unroll
        for (int c = 0; c <= K; c++)
            px[c] = load_vec<D>(row + col_off[c]);
    };

    // horizontal maxima of the last K input rows, as bytes again: [row][column of the pair]
    V hist[K][2];
    const int nrows = a.rows + K - 1;
    V next[K + 1];
    load_row(0, next);
    for (int base = 0; base < nrows; base += K) {
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int r = base + j;
            V odd[K + 1], even[K + 1];
#pragma unroll
            for (int c = 0; c <= K; c++) {
                odd[c] = next[c];
                even[c] = shifted(odd[c]);
            }
            if (!SHORT || r + 1 < nrows) // uniform
                load_row(r + 1, next);
            // columns 1 .. K-1 are under both windows
            V both_odd = odd[1], both_even = even[1];
#pragma unroll
            for (int c = 2; c < K; c++) {
                both_odd = pkmax(both_odd, odd[c]);
                both_even = pkmax(both_even, even[c]);
            }
            hist[j][0] = join(pkmax(odd[0], both_odd), pkmax(even[0], both_even));
            hist[j][1] = join(pkmax(both_odd, odd[K]), pkmax(both_even, even[K]));
            const int y = y0 + r - (K - 1);
            if (r >= K - 1 && r < nrows && y < a.out_h) {
#pragma unroll
                for (int o = 0; o < 2; o++) {
                    V best_odd = hist[0][o], best_even = shifted(hist[0][o]);
#pragma unroll
                    for (int k = 1; k < K; k++) {
                        best_odd = pkmax(best_odd, hist[k][o]);
                        best_even = pkmax(best_even, shifted(hist[k][o]));
                    }
                    if (o == 0 || second)
                        store_vec<D>(img_out + ((long long)y * a.out_w + x0 + o) * a.out_pitch, join(best_odd, best_even));
                }
            }
        }
    }
}

// Strips of one row, which is what few outputs are cut into: all rows of the window are requested at once, where the walk waits
// for one after the other.  5 x 5, launch to launch in a graph: 13 x 13 x 128, one image, 3.2 -> 2.9 us, 30 x 30 x 198 4.8 -> 2.9, 17 x 14 x 61,
// three images, 5.4 -> 3.0, 20 x 20 x 128, 64 images, 4.8 -> 4.4; images of one row, 512 of 40 x 480, 9.5 -> 8.9; 3 x 3 and 2 x 2 as much.
template <int K, int D>
__global__ __launch_bounds__(kThreads) void max_pool_s8_window_row_kernel(const WindowPoolArgs a)
{
    typedef Vec<D> V;
    const unsigned tid = blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= a.total)
        return;
    const unsigned q0 = fastdiv(tid, a.fd_cv);
    const unsigned v = tid - q0 * a.fd_cv.d;
    const unsigned q1 = fastdiv(q0, a.fd_xpairs);
    const unsigned xp = q0 - q1 * a.fd_xpairs.d;
    const unsigned n = fastdiv(q1, a.fd_strips);
    const int x0 = 2 * (int)xp, y = (int)(q1 - n * a.fd_strips.d);
    const int c0 = min((int)v * 4 * D, a.c - 4 * D);
    const char *img_in = a.in + (long long)n * a.h * a.w * a.in_pitch + c0;
    const long long row_pitch = (long long)a.w * a.in_pitch;

    // (columns and rows outside the image: the nearest one inside, as above)
    V px[K][K + 1];
#pragma unroll
    for (int r = 0; r < K; r++) {
        const char *row = img_in + min(max(y - a.pad_top + r, 0), a.h - 1) * row_pitch;
#pragma unroll
        for (int c = 0; c <= K; c++)
            px[r][c] = load_vec<D>(row + (long long)min(max(x0 - a.pad_left + c, 0), a.w - 1) * a.in_pitch);
    }
    char *dst = a.out + (((long long)n * a.out_h + y) * a.out_w + x0) * a.out_pitch + c0;
    // down the columns first: what is left of columns 1 .. K - 1 is under both windows
    V odd[K + 1], even[K + 1];
#pragma unroll
    for (int r = 0; r < K; r++)
#pragma unroll
        for (int c = 0; c <= K; c++) {
            odd[c] = r == 0 ? px[r][c] : pkmax(odd[c], px[r][c]);
            even[c] = r == 0 ? shifted(px[r][c]) : pkmax(even[c], shifted(px[r][c]));
        }
    V both_odd = odd[1], both_even = even[1];
#pragma unroll
    for (int c = 2; c < K; c++) {
        both_odd = pkmax(both_odd, odd[c]);
        both_even = pkmax(both_even, even[c]);
    }
    store_vec<D>(dst, join(pkmax(odd[0], both_odd), pkmax(even[0], both_even)));
    if (x0 + 1 < a.out_w)
        store_vec<D>(dst + a.out_pitch, join(pkmax(both_odd, odd[K]), pkmax(both_even, even[K])));
}

template <int K, int D>
hipError_t launch_window(const WindowPoolArgs &a, bool whole, int cus, hipStream_t stream)
{
    const dim3 grid((a.total + kThreads - 1) / kThreads);
    // One wavefront to a workgroup up to two of them per compute unit, for the loads of a compute unit's wavefronts take turns (30 of
    // 16 bytes each); beyond that wavefronts side by side, whose windows overlap, stay in one workgroup and on one XCD.  Of 1200 pools
    // on the row kernel single wavefronts take 0.51 to 1.06 of the time of four to a workgroup up to 64 workgroups of four, 0.72 to 1.18
    // up to 128, from there 0.87 to 1.34 (12 images of 96 x 54 x 32, 3 x 3: 4.67 and 3.6 us, the walk 3.7).
    if (a.rows == 1 && 2 * (long long)grid.x <= cus)
        hipLaunchKernelGGL((max_pool_s8_window_row_kernel<K, D>), dim3(grid.x * (kThreads / 64)), dim3(64), 0, stream, a);
    else if (a.rows == 1)
        hipLaunchKernelGGL((max_pool_s8_window_row_kernel<K, D>), grid, dim3(kThreads), 0, stream, a);
    else if (whole)
        hipLaunchKernelGGL((max_pool_s8_window_kernel<K, D, false>), grid, dim3(kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((max_pool_s8_window_kernel<K, D, true>), grid, dim3(kThreads), 0, stream, a);
    return hipGetLastError();
}

} // namespace

bool max_pool_s8_window_supports(int h, int w, int c, int k_h, int k_w, int stride_h, int stride_w, int pad_top,
                                 int pad_left, int out_h, int out_w)
{
    if (k_h != k_w || (k_h != 2 && k_h != 3 && k_h != 5) || stride_h != 1 || stride_w != 1)
        return false;
    if (c < 8)
        return false;
    // every window must hold a pixel of the image
    if (pad_top >= k_h || pad_left >= k_w || out_h - 1 - pad_top >= h || out_w - 1 - pad_left >= w)
        return false;
    return true;
}

hipError_t launch_max_pool_s8_window(const void *in, int batch, int h, int w, int c, int k, int pad_top, int pad_left,
                                     int out_h, int out_w, long long in_pitch, long long out_pitch, void *out,
                                     int cu_count, hipStream_t stream)
{
    WindowPoolArgs a;
    a.in = static_cast<const char *>(in);
    a.out = static_cast<char *>(out);
    a.h = h;
    a.w = w;
    a.out_h = out_h;
    a.out_w = out_w;
    a.pad_top = pad_top;
    a.pad_left = pad_left;
    // 16 bytes of channels per thread, at any address; 8 below 16 channels, and for 24 of them, where the second
    // 16 would repeat half of the first
    const int dwords = c >= 16 && c != 24 ? 4 : 2;
    a.c = c;
    a.cv = (c + 4 * dwords - 1) / (4 * dwords);
    a.in_pitch = in_pitch;
    a.out_pitch = out_pitch;
    a.xpairs = (out_w + 1) / 2;
    // Strips per image.  Long strips read each input row once; a strip of `rows` rows reads k - 1 rows more
    // (mostly from cache, but the horizontal maxima are taken again).  Short strips give small tensors enough
    // wavefronts, and the count decides how evenly the last round of wavefronts fills the chip, counted at four
    // wavefronts per SIMD.
    const long long per_row = (long long)batch * a.xpairs * a.cv;
    const int cus = cu_count > 0 ? cu_count : 256;
    const double capacity = (double)cus * 4 * 4;
    int best_strips = 1;
    double best_score = -1.0;
    for (int strips = 1;;) { // of the counts with one strip height only the smallest: 2 sqrt(out_h) of them
        const int rows = (out_h + strips - 1) / strips;
        const double waves = (double)per_row * strips / 64.0;
        const double rounds = waves / capacity;
        const double fill = rounds / (double)(long long)(rounds + 0.999999);
        const double score = fill / (1.0 + 0.5 * (k - 1) / rows);
        if (score > best_score * 1.02) { // ties go to the longer strips
            best_score = score;
            best_strips = strips;
        }
        if (rows <= 1)
            break;
        strips = (out_h + rows - 2) / (rows - 1);
    }
    a.strips = best_strips;
    a.rows = (out_h + best_strips - 1) / best_strips;
    const long long total = per_row * a.strips;
    if (total <= 0)
        return hipSuccess;
    if (total > 0x7fffffffll)
        return hipErrorInvalidValue;
    a.total = (unsigned)total;
    a.fd_cv = make_fastdiv((unsigned)a.cv);
    a.fd_xpairs = make_fastdiv((unsigned)a.xpairs);
    a.fd_strips = make_fastdiv((unsigned)a.strips);
    // (2 x 2 reads a third more rows than it uses: up to some 3 MB 5 % less time all the same, above that 5 % more)
    const bool whole = ((reinterpret_cast<uintptr_t>(in) | (uintptr_t)in_pitch | (uintptr_t)c) & 3) == 0 &&
        (k != 2 || (long long)batch * h * w * c <= (3 << 20));
    switch (k) {
    case 2:
        return dwords == 4 ? launch_window<2, 4>(a, whole, cus, stream) : launch_window<2, 2>(a, whole, cus, stream);
    case 3:
        return dwords == 4 ? launch_window<3, 4>(a, whole, cus, stream) : launch_window<3, 2>(a, whole, cus, stream);
    default:
        return dwords == 4 ? launch_window<5, 4>(a, whole, cus, stream) : launch_window<5, 2>(a, whole, cus, stream);
    }
}

} // namespace espdl
