// The first block of a MobileNetV2-style network - a dense k x k convolution over the few channels of an image, a 3x3
// depthwise convolution, a 1x1 project convolution - as a walk down the image, after the scheme of
// mbconv_s8_walk_kernel.h.  What differs is the expand stage:
//   operand B  a lane group reads one filter row: the at most 13 bytes under it, by a direct-to-LDS copy of the 16 bytes from
//              the dword that the first one lies in.  How far into that dword they start is the same for every second
//              column, so a tile is 16 even or 16 odd columns and the distance goes into operand A (zeros in front of the
//              filter row) instead of a byte shift of the pixels,
//   columns    an even and an odd tile side by side are 32 expanded columns and 30 of the output; the neighbours of an even
//              column are the odd tile's words of the same lane and of the lane before,
//   padding    above and below the image whole lane groups read zeros; at its sides the bytes outside it are masked, in
//              strips that hold a side; the pixels whose 16 bytes would begin in front of the tensor or end behind it (the
//              first of the first row, the last ones of the last) are gathered byte by byte.
//
// Bound by issue: a step (two rows of 30 columns) of two chunks is 36 MFMAs at 16 cycles and 275 vector instructions at
// 4, which one after the other would fill 95 % of the launch's cycles (180 of the 275 round and pack).  224 x 224 x 3, 3x3 stride 2 to 32, project
// to 16, batch 256: 62 us against 98 us on the tile kernel, which builds operand B from bytes; with 48 expanded channels at
// 192 x 200, batch 64, 28 against 75.  Three wavefronts per SIMD instead of two: 62 us too, and coarser strips.
//
// Reference: esp-dl/dl/module/include (dl_module_conv.hpp).
#include "mbconv_s8_walk_kernel.h"

namespace espdl {
namespace {
using namespace mbwalk;

struct StemArgs : MbWalkArgs { // in_row, in_img, in_bytes: of the image
    int skew0, skew1; // bytes between the copied dword's first and the filter row's first byte: even tile, odd tile
};

constexpr int kStemWaves = 8;
constexpr int kStemOut = 30;
constexpr int kStemAhead = 1;
constexpr int kBias = 64; // bytes added to a lane's offset and taken from the base: offsets stay positive

template <int CE, int RT, bool HE>
__global__ __launch_bounds__(64 * kStemWaves, kStemWaves / 4) void mbconv_s8_walk_stem_kernel(const StemArgs a)
{
    constexpr int kWaves = kStemWaves, kThreads = 64 * kWaves, AHEAD = kStemAhead, kSlots = AHEAD + 2;
    constexpr int kXTile = 768, kSlot = 4 * kXTile, kCopies = 4, kStores = 4;
    constexpr int NC = 16 * (2 * CE + RT), TE = 0, TD = 16 * CE, TP = 32 * CE;
    static_assert(CE <= 4);
    // The ring, and behind it [0: zeros, 1 / 2: even / odd tile][column] what the start values are multiplied with: a lane group
    // reads one or the other by the same instruction, so both have to be one object to the compiler.
    constexpr int kOnes = kSlots * kSlot;
    __shared__ __align__(16) unsigned char ring[kWaves][kOnes + 3 * 256];
    __shared__ v4i we_l[CE][2][64], wd_l[CE][3][64], wp_l[RT][64];
    __shared__ __align__(16) int start_l[NC], shift_l[NC];

    const MbconvParams &p = a.p;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int group = (int)(blockIdx.x & 7u) * (a.n_groups >> 3) + (int)(blockIdx.x >> 3);
    const int r_begin = group * a.rows_per_group, r_end = min(a.rows_total, r_begin + a.rows_per_group);

    const auto skew_of = [&](int e) __attribute__((always_inline)) { return e != 0 ? a.skew1 : a.skew0; };
    // expanded column of lane column m in tile e, as image and column inside it
    auto mid_pixel = [&](int v0, int m, int e, int &n, int &x) __attribute__((always_inline)) {
        const int q = v0 + 2 * m + e - p.pad_left;
        n = (int)fastdiv((unsigned)max(q, 0), a.fd_p);
        x = q - n * (int)a.fd_p.d;
        return q >= 0 && n < p.batch && x < p.in_w;
    };

    // ---- copies, AHEAD steps in front of the computation
    const unsigned ring0 = (unsigned)reinterpret_cast<uintptr_t>(&ring[wave][0]);
    int vin[2] = {kParked, kParked};
    int f_r = r_begin, f_row = 0, f_left = 0;
    unsigned f_slot = 0;
    auto feed_segment = [&]() __attribute__((always_inline)) {
        const int g = (int)fastdiv((unsigned)f_r, a.fd_seg);
        const int k0 = f_r - g * a.seg_rows;
        const int rows = min(a.seg_rows - k0, r_end - f_r);
        f_r += rows;
        f_left = rows + 1;
        f_row = 2 * k0 - p.pad_top;
        int lane_now = lane;
        asm volatile("" : "+v"(lane_now));
#pragma unroll
        for (int e = 0; e < 2; e++) {
            int n, x;
            const bool ok = mid_pixel((g * kWaves + wave) * kStemOut, lane_now & 15, e, n, x);
            vin[e] = ok ? kBias + n * a.in_img + (lane_now >> 4) * a.in_row + (x * p.es_w - p.epad_left) * p.in_c - skew_of(e) : kParked;
        }
    };
    auto feed = [&]() __attribute__((always_inline)) { // one step; past the last one nothing is read (the counts stay the same)
        if (f_left == 0 && f_r < r_end)
            feed_segment();
        const bool live = f_left > 0;
        const unsigned base = __builtin_amdgcn_readfirstlane(ring0 + f_slot);
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const bool ok = live && (unsigned)(f_row + s) < (unsigned)p.in_h;
            const int row = (f_row + s) * p.es_h - p.epad_top; // image row of lane group 0
            const int off = __builtin_amdgcn_readfirstlane((ok ? row * a.in_row : 0) - kBias);
            const int left = __builtin_amdgcn_readfirstlane(a.in_bytes - off); // bytes behind the base
            const __amdgpu_buffer_rsrc_t rs = rsrc_of(p.in + off, __builtin_amdgcn_readfirstlane(ok ? left : 0));
            int v[2] = {vin[0], vin[1]};
            if (ok && (row < 1 || row + p.ek_h >= p.img_h)) { // lane groups outside the image, and the ends of the tensor
                const bool in_image = (unsigned)(row + quad) < (unsigned)p.img_h;
#pragma unroll
                for (int e = 0; e < 2; e++)
                    v[e] = (in_image && v[e] >= -off && v[e] <= left - 16) ? v[e] : kParked;
            }
#pragma unroll
            for (int e = 0; e < 2; e++)
                if (quad < p.ek_h)
                    copy16(base + (2 * s + e) * kXTile, v[e], rs);
        }
        f_row += 2;
        f_left -= live ? 1 : 0;
        f_slot = f_slot + kSlot == kSlots * kSlot ? 0 : f_slot + kSlot;
    };
    auto no_stores = [&]() __attribute__((always_inline)) { // dropped: the number of instructions behind a copy is known in every step
#pragma unroll
        for (int i = 0; i < kStores; i++)
            asm volatile("s_nop 4\n\tbuffer_store_byte %0, %0, %1, 0 offen" ::"v"(kParked), "s"(rsrc_of(p.out, 0)) : "memory");
    };

    // ---- set-up: the first copies, filters into LDS in operand order, tables
#pragma unroll
    for (int i = 0; i <= AHEAD; i++) {
        feed();
        no_stores();
    }
    const int taps = p.ek_w * p.in_c; // bytes of a filter row
    {
        constexpr int N = (2 * CE + kWaves - 1) / kWaves;
        unsigned b[N][16];
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int k = wave + i * kWaves, skew = skew_of(k & 1);
            const int8_t *src = p.w_expand + (min(16 * (k >> 1) + col, p.exp_c - 1) * p.ek_h + min(quad, p.ek_h - 1)) * taps;
#pragma unroll
            for (int t = 0; t < 16; t++)
                b[i][t] = (unsigned char)src[min(max(t - skew, 0), taps - 1)];
        }
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int k = wave + i * kWaves, j = k >> 1, skew = skew_of(k & 1);
            v4i w = {0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < 16; t++)
                w[t >> 2] |= t >= skew && t < skew + taps ? (int)(b[i][t] << (8 * (t & 3))) : 0;
            if (quad >= p.ek_h || 16 * j >= p.exp_c)
                w = v4i{0, 0, 0, 0};
            if (j < CE)
                we_l[j][k & 1][lane] = w;
        }
    }
    load_depthwise<CE, kWaves>(p, wd_l, wave, lane);
    load_project<1, RT, kWaves>(p, wp_l, wave, lane);
    const Range range_e = expand_range(p), range_d = depthwise_range(p);
    const Tables tab = make_tables<CE, RT, HE, kThreads>(a, start_l, shift_l, tid);
    const bool fast = tab.fast;
    if (fast && tid < TD)
        we_l[tid >> 4][0][48 + (tid & 15)] = we_l[tid >> 4][1][48 + (tid & 15)] = start_digits(tab.start);
    if (lane < 16)
        *reinterpret_cast<v4i *>(&ring[wave][kOnes + 16 * lane]) = v4i{0, 0, 0, 0};
    __syncthreads();
    const Band band_e = make_band(range_e, tab.high), band_d = make_band(range_d, tab.high), band_p = make_band(project_range(p), tab.high);

    const int c_of = 4 * quad;
    unsigned b_slot = 0;
    const unsigned char *my_ring = &ring[wave][0];
    const bool constant = fast && quad == 3;
    const int xoff = min(quad, 2) * 256 + col * 16;
    const int one_off = kOnes + col * 16;

    int c_r = r_begin, c_left = 0, c_row = 0, c_k = 0, c_v0 = 0; // c_row: first expanded row of the step; c_k: output row it finishes first
    int vout[2] = {kParked, kParked};
    int emask[2] = {0, 0};
    v4i side[2];                     // bytes inside the image
    bool has_side = false, has_end = false; // wave-uniform: the strip holds a side of an image; an end of the tensor
    auto segment = [&]() __attribute__((always_inline)) {
        const int g = (int)fastdiv((unsigned)c_r, a.fd_seg);
        const int k0 = c_r - g * a.seg_rows;
        const int rows = min(a.seg_rows - k0, r_end - c_r);
        c_r += rows;
        c_left = rows + 1;
        c_row = 2 * k0 - p.pad_top;
        c_k = -2;
        int lane_now = lane;
        asm volatile("" : "+v"(lane_now));
        const int m = lane_now & 15;
        c_v0 = (g * kWaves + wave) * kStemOut;
        bool cut = false, end = false;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            int n, x;
            const bool ok = mid_pixel(c_v0, m, e, n, x);
            emask[e] = ok ? -1 : 0;
            if (lane < 16)
                *reinterpret_cast<v4i *>(&ring[wave][kOnes + 256 * (1 + e) + 16 * lane]) = start_factors(emask[e]);
            const int x0 = x * p.es_w - p.epad_left;               // image column of the filter's first
            const int lo = max(0, -x0) * p.in_c + skew_of(e);       // bytes [lo, hi) of the copied ones lie inside
            const int hi = (p.img_w - x0) * p.in_c + skew_of(e);
            cut |= ok && (x0 < 0 || x0 + p.ek_w > p.img_w);
            end |= ok && ((n == 0 && x0 * p.in_c < skew_of(e)) || (n == p.batch - 1 && x0 * p.in_c - skew_of(e) + 16 > a.in_row));
#pragma unroll
            for (int i = 0; i < 4; i++) {
                unsigned w = 0;
#pragma unroll
                for (int b = 0; b < 4; b++)
                    w |= (4 * i + b >= lo && 4 * i + b < hi) ? 0xffu << (8 * b) : 0u;
                side[e][i] = (int)w;
            }
            if (constant)
                side[e] = v4i{-1, -1, -1, -1};
            const int t = 2 * m + e - 1, v = c_v0 + max(t, 0);
            const int no = (int)fastdiv((unsigned)v, a.fd_po);
            const int xo = v - no * (int)a.fd_po.d;
            const int oc = 4 * RT * (lane_now >> 4);
            vout[e] = (t >= 0 && t < kStemOut && no < p.batch && xo < p.out_w && oc < p.out_c) ? no * a.out_img + xo * p.out_c + oc : kParked;
        }
        has_side = __any(cut);
        has_end = __any(end);
    };
    v4i X[2][2];
    // the pixels whose 16 bytes do not lie inside the tensor
    auto gather = [&](v4i &dst, int e, int row) __attribute__((always_inline)) {
        int n, x, lane_now = lane;
        asm volatile("" : "+v"(lane_now));
        const int q = lane_now >> 4;
        if (!mid_pixel(c_v0, lane_now & 15, e, n, x) || q >= p.ek_h || (unsigned)(row + q) >= (unsigned)p.img_h)
            return;
        const long long at = (long long)n * a.in_img + (long long)(row + q) * a.in_row + (x * p.es_w - p.epad_left) * p.in_c - skew_of(e);
        if (at >= 0 && at + 16 <= a.in_bytes)
            return;
        v4i w = {0, 0, 0, 0};
#pragma unroll
        for (int b = 0; b < 16; b++)
            if (at + b >= 0 && at + b < a.in_bytes)
                w[b >> 2] |= (int)((unsigned)(unsigned char)p.in[at + b] << (8 * (b & 3)));
        dst = w;
    };
    auto read_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const bool exists = (unsigned)(c_row + s) < (unsigned)p.in_h;
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int at = constant ? one_off + (exists ? 256 * (1 + e) : 0) : (int)b_slot + xoff + (2 * s + e) * kXTile;
                X[s][e] = *reinterpret_cast<const v4i *>(my_ring + at);
            }
        }
        b_slot = b_slot + kSlot == kSlots * kSlot ? 0 : b_slot + kSlot;
        if (has_end) {
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const int row = (c_row + s) * p.es_h - p.epad_top;
                if ((unsigned)(c_row + s) < (unsigned)p.in_h && (row < 1 || row + p.ek_h >= p.img_h)) {
                    gather(X[s][0], 0, row);
                    gather(X[s][1], 1, row);
                }
            }
        }
        if (has_side) {
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int e = 0; e < 2; e++)
                    X[s][e] &= side[e];
        }
    };

    v4i U[CE][2][2]; // [chunk][tile][row]
#pragma unroll
    for (int j = 0; j < CE; j++)
#pragma unroll
        for (int e = 0; e < 2; e++)
            U[j][e][0] = U[j][e][1] = v4i{0, 0, 0, 0};
    side[0] = side[1] = v4i{0, 0, 0, 0};

    int left = 0;
    for (int r = r_begin; r < r_end;) {
        const int g = (int)fastdiv((unsigned)r, a.fd_seg);
        const int e = min(r_end, (g + 1) * a.seg_rows);
        left += e - r + 1;
        r = e;
    }
    auto walk = [&](auto mode_tag) __attribute__((always_inline)) {
        constexpr int MODE = decltype(mode_tag)::value;
        constexpr bool FOLD = MODE != 2;
        for (; left > 0; left--) {
            if (c_left == 0)
                segment();
            c_left--;
            wait_copies<AHEAD * (kCopies + kStores) + kStores>(); // this step's input has arrived
            read_x();
            feed();
            const int out_y = c_row + p.pad_top - 2;
            v4i D[2][2]; // [row][tile]: operand B of the project stage, a dword per chunk
#pragma unroll
            for (int j = 0; j < CE; j++) {
                const v4i she = *reinterpret_cast<const v4i *>(&shift_l[TE + 16 * j + c_of]);
                v4i se = {0, 0, 0, 0};
                if constexpr (!FOLD)
                    se = *reinterpret_cast<const v4i *>(&start_l[TE + 16 * j + c_of]);
                v4i E[2][2]; // [row][tile]
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    int w[2];
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(we_l[j][e][lane], X[s][e], se, 0, 0, 0);
                        w[e] = finish4<MODE, HE>(acc, she, band_e);
                        if constexpr (!FOLD)
                            w[e] &= (unsigned)(c_row + s) < (unsigned)p.in_h ? emask[e] : 0;
                    }
                    // the window's three columns (the fourth dword meets zero weights)
                    E[s][0][0] = __builtin_amdgcn_update_dpp(0, w[1], 0x111, 0xf, 0xf, true); // row_shr:1
                    E[s][0][1] = w[0];
                    E[s][0][2] = E[s][0][3] = w[1];
                    E[s][1][0] = w[0];
                    E[s][1][1] = w[1];
                    E[s][1][2] = E[s][1][3] = __builtin_amdgcn_update_dpp(0, w[0], 0x101, 0xf, 0xf, true); // row_shl:1
                }
                v4i d[3];
#pragma unroll
                for (int ky = 0; ky < 3; ky++)
                    d[ky] = wd_l[j][ky][lane];
                const v4i sd = *reinterpret_cast<const v4i *>(&start_l[TD + 16 * j + c_of]);
                const v4i shd = *reinterpret_cast<const v4i *>(&shift_l[TD + 16 * j + c_of]);
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const v4i p0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[2], E[0][e], U[j][e][0], 0, 0, 0);
                    v4i p1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[1], E[0][e], U[j][e][1], 0, 0, 0);
                    U[j][e][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[0], E[0][e], sd, 0, 0, 0);
                    p1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[2], E[1][e], p1, 0, 0, 0);
                    U[j][e][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[1], E[1][e], U[j][e][0], 0, 0, 0);
                    U[j][e][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[0], E[1][e], sd, 0, 0, 0);
                    D[0][e][j] = finish4<MODE, HE>(p0, shd, band_d);
                    D[1][e][j] = finish4<MODE, HE>(p1, shd, band_d);
                }
            }
#pragma unroll
            for (int j = CE; j < 4; j++)
#pragma unroll
                for (int e = 0; e < 2; e++)
                    D[0][e][j] = D[1][e][j] = 0;
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const bool live = c_k >= 0 && out_y + s < p.out_h;
                const int off = __builtin_amdgcn_readfirstlane(live ? (out_y + s) * a.out_row : 0);
                const __amdgpu_buffer_rsrc_t rs = rsrc_of(p.out + off, __builtin_amdgcn_readfirstlane(live ? a.out_bytes - off : 0));
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    int words[RT];
#pragma unroll
                    for (int t = 0; t < RT; t++) {
                        const v4i sp = *reinterpret_cast<const v4i *>(&start_l[TP + 4 * RT * quad + 4 * t]);
                        const v4i shp = *reinterpret_cast<const v4i *>(&shift_l[TP + 4 * RT * quad + 4 * t]);
                        const v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wp_l[t][lane], D[s][e], sp, 0, 0, 0);
                        words[t] = finish4<MODE, HE>(acc, shp, band_p);
                    }
                    if constexpr (RT == 2)
                        __builtin_amdgcn_raw_buffer_store_b64(v2u{(unsigned)words[0], (unsigned)words[1]}, rs, vout[e], 0, 0);
                    else
                        __builtin_amdgcn_raw_buffer_store_b32((unsigned)words[0], rs, vout[e], 0, 0);
                }
            }
            c_row += 2;
            c_k += 2;
        }
    };
    if (!fast)
        walk(std::integral_constant<int, 2>{});
    else if (tab.high)
        walk(std::integral_constant<int, 0>{});
    else
        walk(std::integral_constant<int, 1>{});
}

struct StemPlan {
    bool ok;
    int ce, rt;
    StemArgs a;
};

StemPlan stem_plan(const MbconvParams &p, int cus)
{
    StemPlan plan = {};
    if (p.w_expand == nullptr || mbconv_expand_is_pointwise(p) || p.k_h != 3 || p.k_w != 3 || p.dil_h != 1 || p.dil_w != 1 ||
        p.stride_h != 1 || p.stride_w != 1 || p.batch <= 0 || p.residual != nullptr)
        return plan;
    plan.rt = p.out_c % 4 == 0 && p.out_c <= 16 ? 1 : (p.out_c % 8 == 0 && p.out_c <= 32 ? 2 : 0);
    plan.ce = (p.exp_c + 15) / 16;
    if (plan.rt == 0 || p.exp_c % 16 != 0 || plan.ce > 3)
        return plan;
    // a filter row in 13 bytes (up to three in front of it), three of them, and every second column at the same distance
    // from a dword; no window begins outside the image by its whole width
    if (p.ek_h > 3 || p.ek_w * p.in_c > 13 || (p.es_w * p.in_c) % 2 != 0 || (p.img_w * p.in_c) % 4 != 0 || p.img_w * p.in_c < 64 ||
        p.epad_left >= p.ek_w || p.epad_top >= p.ek_h || (p.in_w - 1) * p.es_w - p.epad_left >= p.img_w ||
        (p.in_h - 1) * p.es_h - p.epad_top >= p.img_h)
        return plan;
    StemArgs &a = plan.a;
    a.p = p;
    a.skew0 = (-p.pad_left * p.es_w - p.epad_left) * p.in_c & 3;
    a.skew1 = ((1 - p.pad_left) * p.es_w - p.epad_left) * p.in_c & 3;
    // columns from image to image: the padding between them at least once, an even number
    const long long over = (long long)(p.out_w - 1) + 2 - p.pad_left - (p.in_w - 1);
    long long pitch = std::max<long long>(p.in_w + std::max<long long>({0, p.pad_left, over}), (long long)p.out_w);
    pitch = (pitch + 1) / 2 * 2;
    const long long cols = (p.batch - 1) * pitch + p.out_w;
    const long long in_bytes = (long long)p.batch * p.img_h * p.img_w * p.in_c, out_bytes = (long long)p.batch * p.out_h * p.out_w * p.out_c;
    const long long seg_rows = (p.out_h + 1) / 2;
    const int width = kStemOut * kStemWaves;
    const long long strips = (cols + width - 1) / width;
    if (in_bytes > 0x7f000000ll || out_bytes > 0x7f000000ll || (long long)p.img_w * p.in_c * p.ek_h > 0x400000 ||
        pitch * (p.batch + 1) > (1ll << 30) || strips * seg_rows > (1ll << 30))
        return plan;
    a.in_row = p.img_w * p.in_c;
    a.in_img = a.in_row * p.img_h;
    a.in_bytes = (int)in_bytes;
    a.out_row = p.out_w * p.out_c;
    a.out_img = a.out_row * p.out_h;
    a.out_bytes = (int)out_bytes;
    a.bound_e = (long long)p.ek_h * p.ek_w * p.in_c * 16384;
    a.bound_d = 9ll * 16384;
    a.bound_p = (long long)p.exp_c * 16384;
    a.fd_p = make_fastdiv((unsigned)pitch);
    a.fd_po = make_fastdiv((unsigned)pitch);
    a.seg_rows = (int)seg_rows;
    a.rows_total = (int)(strips * seg_rows);
    const int want = std::max(8, cus / 8 * 8);
    a.rows_per_group = (a.rows_total + want - 1) / want;
    a.n_groups = ((a.rows_total + a.rows_per_group - 1) / a.rows_per_group + 7) / 8 * 8;
    a.fd_seg = make_fastdiv((unsigned)a.seg_rows);
    plan.ok = true;
    return plan;
}

template <int CE, bool HE>
hipError_t launch_ce(const StemPlan &plan, hipStream_t stream)
{
    const dim3 grid((unsigned)plan.a.n_groups), block(64 * kStemWaves);
    if (plan.rt == 1)
        hipLaunchKernelGGL((mbconv_s8_walk_stem_kernel<CE, 1, HE>), grid, block, 0, stream, plan.a);
    else
        hipLaunchKernelGGL((mbconv_s8_walk_stem_kernel<CE, 2, HE>), grid, block, 0, stream, plan.a);
    return hipGetLastError();
}

template <bool HE>
hipError_t launch_he(const StemPlan &plan, hipStream_t stream)
{
    return plan.ce == 1 ? launch_ce<1, HE>(plan, stream) : (plan.ce == 2 ? launch_ce<2, HE>(plan, stream) : launch_ce<3, HE>(plan, stream));
}

} // namespace

bool mbconv_s8_walk_stem_supports(const MbconvParams &p, int cu_count)
{
    return stem_plan(p, cu_count > 0 ? cu_count : 256).ok;
}

hipError_t launch_mbconv_s8_walk_stem(const MbconvParams &p, int cu_count, hipStream_t stream)
{
    const StemPlan plan = stem_plan(p, cu_count > 0 ? cu_count : 256);
    if (!plan.ok)
        return hipErrorInvalidValue;
    return p.half_even ? launch_he<true>(plan, stream) : launch_he<false>(plan, stream);
}

} // namespace espdl
