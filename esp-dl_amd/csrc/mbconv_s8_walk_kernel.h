// MobileNetV2-style inverted residual block (1x1 expand convolution, 3x3 depthwise convolution, 1x1 project convolution
// and, with RES, the block input added to the result) as a walk down the image.  One workgroup per compute unit, eight
// wavefronts; a wavefront owns 14 output columns (stride 2: 15) and goes down them two input rows per step.  Nothing of the
// expanded tensor leaves its registers:
//   expand     a 16-channel chunk of 16 input columns is one MFMA; the four values of a lane (one pixel, the four channels
//              of its quad) are rounded and packed into one dword,
//   depthwise  that dword and the two neighbouring lanes' (two DPP moves) are already an operand B: its reduction runs over
//              (column of the window, channel), operand A holds the weight of filter i in channel i's byte and zeros
//              elsewhere.  One MFMA per window row; the rows that a step does not finish stay behind as accumulators U, so
//              no expanded row is computed twice down a segment,
//   project    the rounded depthwise dwords of four chunks are operand B of the next MFMA as they lie.
// The images of a batch stand side by side in one row of columns with the padding's width between them, so a strip of 14
// or 15 columns crosses from image to image and no tile is nearly empty.  The start value of the expand stage (bias and
// rounding) is folded into the reduction's last lane group, which the block's at most 48 input channels leave free: its
// operand B is a constant where the pixel exists and zeros where it does not, so padding needs no masks.  Input rows come
// by direct-to-LDS copies asked for AHEAD steps early.
//
// Bound by issue: a step (two rows of 16 columns) at stride 1 is 8 MFMAs and about 46 vector instructions per chunk, and
// the two share the SIMD: a third wavefront per SIMD, one instead of two workgroups' worth of wavefronts, or the expand
// filters read from LDS instead of held in registers move the time by 3 % at most (at stride 2 reading them is 7 % faster).
// LDS is active a quarter of the time.  The tile kernel that these blocks took before expands its halo again per tile and
// moves the expanded patch through LDS.  Batch 256, this one against that one: 56 x 56, 24 -> 144 -> 24 with Add 64 against
// 77 us; 112 x 112, 16 -> 96 -> 24, stride 2, 61 against 76 us; 56 x 56, 24 -> 144 -> 32, stride 2, 29 against 38 us.
//
// Reference: the Conv / DepthwiseConv / Add modules of esp-dl/dl/module/include (dl_module_conv.hpp, dl_module_add.hpp).
#pragma once

#include <algorithm>
#include <type_traits>

#include "espdl_device.h"
#include "espdl_kernels.h"

namespace espdl {
namespace mbwalk {

constexpr int kParked = (int)0x80000000u;

typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));

constexpr int kUnits = 3; // units of 16 input channels at most
constexpr int kLdsLimit = 160 * 1024;

struct MbWalkArgs {
    MbconvParams p;
    int in_bytes, out_bytes, in_row, in_img, out_row, out_img;
    int n_groups, rows_total, rows_per_group; // in pairs of input rows (stride 1: of output rows too)
    int seg_rows;                             // the same of one column group
    long long bound_e, bound_d, bound_p;
    FastDiv fd_p, fd_po, fd_seg;
};

// CE chunks of 16 expanded channels (fewer are filled up with zero filters), RT tiles of 16 project filters, stride S.
template <int CE, int RT, int S, bool RES>
struct MbShape {
    static constexpr int ET = S;                  // expand tiles of 16 columns: all of them, or the even and the odd ones
    static constexpr int kOut = S == 1 ? 14 : 15; // output columns of a wavefront
    static constexpr int kFirst = S == 1 ? 1 : 0; // lane column of the first of them (the window's centre at stride 1)
    static constexpr int G = (CE + 3) / 4;        // project reduction steps
    static constexpr int NL = S == 1 ? 2 : 1;     // output rows whose depthwise sums live from step to step
    static constexpr int NR = S == 1 ? 2 : 1;     // output rows a step finishes
    static constexpr int kXTile = kUnits * 256;
    static constexpr int kSlot = 2 * ET * kXTile;
    static constexpr int kOnes = (1 + ET) * 256; // what the start values are multiplied with, behind a wavefront's ring
    static constexpr int kResRow = RT * 256;
    static constexpr int kRes = RES ? NR * kResRow : 16; // the residual operand of the step
    static constexpr int kCopies = 2 * ET;
    static constexpr int kStores = NR;
    static constexpr int kTabs = (2 * CE + RT) * 16 * 8;
    static constexpr long lds(int waves, int ahead)
    {
        return (4 * CE + G * RT) * 1024l + kTabs + (long)waves * ((ahead + 2) * kSlot + kOnes + kRes) + 512;
    }
    static constexpr int W = 8; // wavefronts
    static constexpr int AHEAD = lds(W, 2) <= kLdsLimit ? 2 : 1;
    static_assert(lds(W, 1) <= kLdsLimit);
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const int8_t *p, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(p), (short)0, bytes, 0x00020000);
}
__device__ __forceinline__ void copy16(unsigned lds, int voff, __amdgpu_buffer_rsrc_t rsrc)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(voff), "s"(rsrc) : "memory");
}
__device__ __forceinline__ void copy4(unsigned lds, int voff, __amdgpu_buffer_rsrc_t rsrc)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds), "v"(voff), "s"(rsrc) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_copies()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory");
}

// Clamps of a stage's result.
struct Band {
    int lo, hi;   // as values
    int flo, fhi; // as pairs of int16: of the values (MODE 1) or of the values in the high bytes (MODE 0)
};
// Four channels of one pixel.  MODE 0: every shift is at least 8 and only the lower clamp acts (the value sits in bits 8 ..
// of the shifted sum, the saturating convert to int16 saturates it to int8).  1: any shift of 1 .. 31.  2: the general form.
template <int MODE, bool HE>
__device__ __forceinline__ int finish4(const v4i &acc, const v4i &shift, const Band &b)
{
    if constexpr (MODE == 2) {
        int q[4];
#pragma unroll
        for (int r = 0; r < 4; r++)
            q[r] = min(max(requant_s8(acc[r], shift[r], false, HE), b.lo), b.hi);
        return pack4_s8(q[0], q[1], q[2], q[3]);
    } else {
        int v[4];
#pragma unroll
        for (int r = 0; r < 4; r++)
            v[r] = (HE ? half_even_add(acc[r], MODE == 0 ? shift[r] + 8 : shift[r]) : acc[r]) >> shift[r];
        v2s p01 = __builtin_amdgcn_cvt_pk_i16(v[0], v[1]), p23 = __builtin_amdgcn_cvt_pk_i16(v[2], v[3]);
        p01 = __builtin_elementwise_max(p01, __builtin_bit_cast(v2s, b.flo));
        p23 = __builtin_elementwise_max(p23, __builtin_bit_cast(v2s, b.flo));
        if constexpr (MODE == 1) {
            p01 = __builtin_elementwise_min(p01, __builtin_bit_cast(v2s, b.fhi));
            p23 = __builtin_elementwise_min(p23, __builtin_bit_cast(v2s, b.fhi));
        }
        return (int)__builtin_amdgcn_perm((unsigned)__builtin_bit_cast(int, p23), (unsigned)__builtin_bit_cast(int, p01), MODE == 0 ? 0x07050301u : 0x06040200u);
    }
}

// Clamps of the three stages.
struct Range {
    int lo, hi;
};
__device__ __forceinline__ Range expand_range(const MbconvParams &p)
{
    return {max(p.relu_expand ? 0 : -128, p.clip_e ? p.clip_e_lo : -128), p.clip_e ? p.clip_e_hi : 127};
}
__device__ __forceinline__ Range depthwise_range(const MbconvParams &p)
{
    return {max(p.relu_dw ? 0 : -128, p.clip_d ? p.clip_d_lo : -128), p.clip_d ? p.clip_d_hi : 127};
}
__device__ __forceinline__ Range project_range(const MbconvParams &p)
{
    return {p.relu_project ? 0 : -128, 127};
}
__device__ __forceinline__ Band make_band(const Range &r, bool high)
{
    const auto pair = [](int v) { return (v & 0xffff) * 0x00010001; };
    return high ? Band{r.lo, r.hi, pair(r.lo * 256), 0} : Band{r.lo, r.hi, pair(r.lo), pair(r.hi)};
}

// The set-up's loads all read inside their arrays and are selected afterwards: none waits for another.
// Depthwise filters: row i of chunk j in the lane group of its four channels, dword kx holds the weight in its own channel's
// byte.
template <int CE, int WAVES>
__device__ __forceinline__ void load_depthwise(const MbconvParams &p, v4i (*wd)[3][64], int wave, int lane)
{
    constexpr int N = (3 * CE + WAVES - 1) / WAVES;
    const int col = lane & 15, quad = lane >> 4;
    unsigned w[N][3];
#pragma unroll
    for (int i = 0; i < N; i++) {
        const int e = min(wave + i * WAVES, 3 * CE - 1), j = e / 3, ky = e - 3 * j;
        const int8_t *src = p.w_dw + ky * 3 * p.exp_c + min(16 * j + col, p.exp_c - 1);
#pragma unroll
        for (int kx = 0; kx < 3; kx++)
            w[i][kx] = (unsigned char)src[kx * p.exp_c];
    }
#pragma unroll
    for (int i = 0; i < N; i++) {
        const int e = wave + i * WAVES, j = e / 3;
        const bool own = quad == (col >> 2) && 16 * j < p.exp_c;
        const int at = 8 * (col & 3);
        if (e < 3 * CE)
            wd[j][e - 3 * j][lane] = own ? v4i{(int)(w[i][0] << at), (int)(w[i][1] << at), (int)(w[i][2] << at), 0} : v4i{0, 0, 0, 0};
    }
}

// Project filters: byte 4 jj + r of lane group q in step g is channel 16 (4 g + jj) + 4 q + r, as the depthwise results lie.
template <int G, int RT, int WAVES>
__device__ __forceinline__ void load_project(const MbconvParams &p, v4i (*wp)[64], int wave, int lane)
{
    constexpr int N = (G * RT + WAVES - 1) / WAVES;
    const int col = lane & 15, quad = lane >> 4;
    v4i w[N];
#pragma unroll
    for (int i = 0; i < N; i++) {
        const int e = min(wave + i * WAVES, G * RT - 1), g = e / RT, t = e - g * RT;
        const int oc = min(4 * RT * (col >> 2) + 4 * t + (col & 3), p.out_c - 1);
#pragma unroll
        for (int jj = 0; jj < 4; jj++)
            w[i][jj] = *reinterpret_cast<const int *>(p.w_project + oc * p.exp_c + min(16 * (4 * g + jj), p.exp_c - 16) + 4 * quad);
    }
#pragma unroll
    for (int i = 0; i < N; i++) {
        const int e = wave + i * WAVES, g = e / RT, t = e - g * RT;
        const bool filter = 4 * RT * (col >> 2) + 4 * t + (col & 3) < p.out_c;
#pragma unroll
        for (int jj = 0; jj < 4; jj++)
            w[i][jj] = filter && 16 * (4 * g + jj) < p.exp_c ? w[i][jj] : 0;
        if (e < G * RT)
            wp[e][lane] = w[i];
    }
}

// Start values and shifts of all stages (expand, depthwise, project) in LDS, and what their ranges allow: one table entry
// per thread of a whole workgroup.
struct Tables {
    bool fast; // start values with the rounding added, all of them within the folded form, and no sum overflows
    bool high; // fast, every shift at least 8, and no stage but a ReLU clamps: MODE 0
    int start; // of this thread's entry
};
template <int CE, int RT, bool HE, int THREADS>
__device__ __forceinline__ Tables make_tables(const MbWalkArgs &a, int *start, int *shift, int tid)
{
    constexpr int NC = 16 * (2 * CE + RT), TD = 16 * CE, TP = 32 * CE;
    static_assert(NC <= THREADS);
    const MbconvParams &p = a.p;
    const int c = tid, stage = c < TD ? 0 : (c < TP ? 1 : 2);
    const int ch = c - (stage == 0 ? 0 : (stage == 1 ? TD : TP)), n = stage == 2 ? p.out_c : p.exp_c;
    const int32_t *sp = stage == 0 ? p.s_expand : (stage == 1 ? p.s_dw : p.s_project);
    const int32_t *bp = stage == 0 ? p.b_expand : (stage == 1 ? p.b_dw : p.b_project);
    const bool one = (stage == 0 ? p.n_s_expand : (stage == 1 ? p.n_s_dw : p.n_s_project)) == 1;
    const long long bound = stage == 0 ? a.bound_e : (stage == 1 ? a.bound_d : a.bound_p);
    int s = 8, b = 0;
    const Range re = expand_range(p), rd = depthwise_range(p);
    int ok = re.lo <= 0 && re.hi >= 0, high = re.hi == 127 && rd.hi == 127;
    if (c < NC && ch < n) {
        s = sp[one ? 0 : ch];
        b = bp ? bp[ch] : 0;
        const long long st = (long long)b + (1ll << ((s - 1) & 31)), mag = st < 0 ? -st : st;
        if (s < 1 || s > 31 || mag + bound >= (1ll << 31) || (stage == 0 && mag > 240000))
            ok = 0;
        if (s < 8)
            high = 0;
    }
    Tables t;
    t.fast = __syncthreads_and(ok) != 0;
    t.high = __syncthreads_and(high) != 0 && t.fast;
    t.start = t.fast ? b + (1 << ((s - 1) & 31)) - (HE ? 1 : 0) : b;
    if (c < NC) {
        start[c] = t.start;
        shift[c] = t.high ? s - 8 : s;
    }
    return t;
}

// A start value b as d0 + 127 (d1 + .. + d15): operand A of sixteen products whose operand B is 1 and fifteen times 127 where
// the pixel exists and zeros where it does not.
__device__ __forceinline__ v4i start_digits(int b)
{
    int t = (b + (b < 0 ? -63 : 63)) / 127;
    int d[16];
    d[0] = b - 127 * t;
#pragma unroll
    for (int i = 1; i < 16; i++) {
        d[i] = min(max(t, -127), 127);
        t -= d[i];
    }
    v4i w;
#pragma unroll
    for (int i = 0; i < 4; i++)
        w[i] = pack4_s8(d[4 * i], d[4 * i + 1], d[4 * i + 2], d[4 * i + 3]);
    return w;
}
__device__ __forceinline__ v4i start_factors(int mask)
{
    return v4i{mask & 0x7f7f7f01, mask & 0x7f7f7f7f, mask & 0x7f7f7f7f, mask & 0x7f7f7f7f};
}

template <int CE, int RT, int S, bool HE, bool RES>
__global__ __launch_bounds__((64 * MbShape<CE, RT, S, RES>::W), 2) void mbconv_s8_walk_kernel(const MbWalkArgs a)
{
    static_assert(RT == 2 || RT == 4);
    using Shape = MbShape<CE, RT, S, RES>;
    constexpr int ET = Shape::ET, G = Shape::G, NL = Shape::NL, NR = Shape::NR, kWaves = Shape::W, kThreads = 64 * kWaves;
    constexpr int AHEAD = Shape::AHEAD, kSlot = Shape::kSlot, kSlots = AHEAD + 2, kCopies = Shape::kCopies, kStores = Shape::kStores;
    constexpr int NC = 16 * (2 * CE + RT); // channels of all tables: expand, depthwise, project
    constexpr int TE = 0, TD = 16 * CE, TP = 32 * CE;
    // The ring, and behind it [0: zeros, else expand tile][column] what the start values are multiplied with: a lane group reads
    // one or the other by the same instruction, so both have to be one object to the compiler.
    constexpr int kOnes = kSlots * kSlot;
    __shared__ __align__(16) unsigned char ring[kWaves][kOnes + Shape::kOnes];
    __shared__ __align__(16) unsigned char res_l[kWaves][Shape::kRes];
    __shared__ v4i we_l[CE][64], wd_l[CE][3][64], wp_l[G * RT][64];
    __shared__ __align__(16) int start_l[NC], shift_l[NC];

    const MbconvParams &p = a.p;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int group = (int)(blockIdx.x & 7u) * (a.n_groups >> 3) + (int)(blockIdx.x >> 3);
    const int r_begin = group * a.rows_per_group, r_end = min(a.rows_total, r_begin + a.rows_per_group);
    const int c0 = p.in_c, units = (c0 + 15) >> 4;

    // ---- copies, AHEAD steps in front of the computation
    const unsigned ring0 = (unsigned)reinterpret_cast<uintptr_t>(&ring[wave][0]);
    int vin[ET];
    int f_r = r_begin, f_row = 0, f_left = 0;
    unsigned f_slot = 0;
    // input column of lane column m in expand tile e, as image and column inside it
    auto in_pixel = [&](int v0, int m, int e, int &n, int &x) {
        const int q = (v0 + m) * S - p.pad_left + e;
        n = (int)fastdiv((unsigned)max(q, 0), a.fd_p);
        x = q - n * (int)a.fd_p.d;
        return q >= 0 && n < p.batch && x < p.in_w;
    };
    auto feed_segment = [&]() {
        const int g = (int)fastdiv((unsigned)f_r, a.fd_seg);
        const int k0 = f_r - g * a.seg_rows;
        const int rows = min(a.seg_rows - k0, r_end - f_r);
        f_r += rows;
        f_left = rows + 1;
        f_row = 2 * k0 - p.pad_top;
        int lane_now = lane; // (through an empty asm statement: nothing of this is kept in registers between segments)
        asm volatile("" : "+v"(lane_now));
#pragma unroll
        for (int e = 0; e < ET; e++) {
            int n, x;
            const bool ok = in_pixel((g * kWaves + wave) * Shape::kOut, lane_now & 15, e, n, x);
            vin[e] = ok ? n * a.in_img + x * c0 + min(16 * (lane_now >> 4), c0 - 16) : kParked;
        }
    };
    auto feed = [&]() { // one step; past the last one nothing is read (the counts stay the same)
        if (f_left == 0 && f_r < r_end)
            feed_segment();
        const bool live = f_left > 0;
        const unsigned base = __builtin_amdgcn_readfirstlane(ring0 + f_slot);
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const bool ok = live && (unsigned)(f_row + s) < (unsigned)p.in_h;
            const int off = __builtin_amdgcn_readfirstlane(ok ? (f_row + s) * a.in_row : 0);
            const __amdgpu_buffer_rsrc_t rs = rsrc_of(p.in + off, __builtin_amdgcn_readfirstlane(ok ? a.in_bytes - off : 0));
#pragma unroll
            for (int e = 0; e < ET; e++)
                if (quad < units)
                    copy16(base + (s * ET + e) * Shape::kXTile, vin[e], rs);
        }
        f_row += 2;
        f_left -= live ? 1 : 0;
        f_slot = f_slot + kSlot == kSlots * kSlot ? 0 : f_slot + kSlot;
    };
    auto no_stores = [&]() { // dropped: the number of instructions behind a copy is known in every step
#pragma unroll
        for (int i = 0; i < kStores; i++)
            asm volatile("s_nop 4\n\tbuffer_store_byte %0, %0, %1, 0 offen" ::"v"(kParked), "s"(rsrc_of(p.out, 0)) : "memory");
    };

    // ---- set-up: the first copies, filters into LDS in operand order, tables
#pragma unroll
    for (int e = 0; e < ET; e++)
        vin[e] = kParked;
#pragma unroll
    for (int i = 0; i <= AHEAD; i++) {
        feed();
        no_stores();
    }
    {
        // expand: row i of chunk j is filter 16 j + i; unit u holds input channels min(16 u, c0 - 16) .. + 15, those that
        // unit u - 1 holds already as zeros
        constexpr int N = (CE + kWaves - 1) / kWaves;
        const int first = min(16 * quad, c0 - 16), skip = (16 * quad - first) >> 2; // bytes, dwords
        v4i w[N];
#pragma unroll
        for (int i = 0; i < N; i++)
            w[i] = *reinterpret_cast<const v4i_unaligned *>(p.w_expand + min(16 * (wave + i * kWaves) + col, p.exp_c - 1) * c0 + first);
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int e = wave + i * kWaves;
#pragma unroll
            for (int d = 0; d < 4; d++)
                w[i][d] = d < skip || quad >= units || 16 * e >= p.exp_c ? 0 : w[i][d];
            if (e < CE)
                we_l[e][lane] = w[i];
        }
    }
    load_depthwise<CE, kWaves>(p, wd_l, wave, lane);
    load_project<G, RT, kWaves>(p, wp_l, wave, lane);
    const Range range_e = expand_range(p), range_d = depthwise_range(p);
    const Tables tab = make_tables<CE, RT, HE, kThreads>(a, start_l, shift_l, tid);
    const bool fast = tab.fast, is_high = tab.high;
    if (fast && tid < TD)
        we_l[tid >> 4][48 + (tid & 15)] = start_digits(tab.start);
    if (lane < 16)
        *reinterpret_cast<v4i *>(&ring[wave][kOnes + 16 * lane]) = v4i{0, 0, 0, 0};
    __syncthreads();
    const Band band_e = make_band(range_e, is_high), band_d = make_band(range_d, is_high), band_p = make_band(project_range(p), is_high);

    const int c_of = 4 * quad; // of this lane's four channels of a chunk
    const Requant4 res_q = make_requant4(p.residual_shift);

    v4i X[2][ET];
    unsigned b_slot = 0;
    const unsigned char *my_ring = &ring[wave][0];
    // lane groups past the last unit meet zero filters, or (folded start values, last group) the constant of the pixel
    const bool constant = fast && quad == 3;
    const int xoff = min(quad, kUnits - 1) * 256 + col * 16;
    const int one_off = kOnes + col * 16;
    auto read_x = [&](int row) { // row: first input row of the step
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const bool exists = (unsigned)(row + s) < (unsigned)p.in_h;
#pragma unroll
            for (int e = 0; e < ET; e++) {
                const int at = constant ? one_off + (exists ? 256 * (1 + e) : 0) : (int)b_slot + xoff + (s * ET + e) * Shape::kXTile;
                X[s][e] = *reinterpret_cast<const v4i *>(my_ring + at);
            }
        }
        b_slot = b_slot + kSlot == kSlots * kSlot ? 0 : b_slot + kSlot;
    };

    int vout = kParked;
    int emask[ET];
    int c_r = r_begin, c_left = 0, c_row = 0, c_k = 0; // c_row: first input row of the step; c_k: output row the step finishes first
    auto segment = [&]() {
        const int g = (int)fastdiv((unsigned)c_r, a.fd_seg);
        const int k0 = c_r - g * a.seg_rows;
        const int rows = min(a.seg_rows - k0, r_end - c_r);
        c_r += rows;
        c_left = rows + 1;
        c_row = 2 * k0 - p.pad_top;
        c_k = -NR;
        int lane_now = lane;
        asm volatile("" : "+v"(lane_now));
        const int v0 = (g * kWaves + wave) * Shape::kOut;
#pragma unroll
        for (int e = 0; e < ET; e++) {
            int n, x;
            emask[e] = in_pixel(v0, lane_now & 15, e, n, x) ? -1 : 0;
            if (lane < 16)
                *reinterpret_cast<v4i *>(&ring[wave][kOnes + 256 * (1 + e) + 16 * lane]) = start_factors(emask[e]);
        }
        const int o = (lane_now & 15) - Shape::kFirst, v = v0 + max(o, 0);
        const int n = (int)fastdiv((unsigned)v, a.fd_po);
        const int x = v - n * (int)a.fd_po.d;
        const int oc = 4 * RT * (lane_now >> 4);
        vout = (o >= 0 && o < Shape::kOut && n < p.batch && x < p.out_w && oc < p.out_c) ? n * a.out_img + x * p.out_c + oc : kParked;
    };
#pragma unroll
    for (int e = 0; e < ET; e++)
        emask[e] = 0;

    v4i U[CE][NL];
#pragma unroll
    for (int j = 0; j < CE; j++)
#pragma unroll
        for (int i = 0; i < NL; i++)
            U[j][i] = v4i{0, 0, 0, 0};
    const unsigned res0 = (unsigned)reinterpret_cast<uintptr_t>(&res_l[wave][0]);

    int left = 0;
    for (int r = r_begin; r < r_end;) {
        const int g = (int)fastdiv((unsigned)r, a.fd_seg);
        const int e = min(r_end, (g + 1) * a.seg_rows);
        left += e - r + 1;
        r = e;
    }
    const auto row_rsrc = [&](const int8_t *t, int y, bool live) { // a row of the output's shape
        const int off = __builtin_amdgcn_readfirstlane(live ? y * a.out_row : 0);
        return rsrc_of(t + off, __builtin_amdgcn_readfirstlane(live ? a.out_bytes - off : 0));
    };

    auto walk = [&](auto mode_tag) {
        constexpr int MODE = decltype(mode_tag)::value;
        constexpr bool FOLD = MODE != 2;
        for (; left > 0; left--) {
            if (c_left == 0)
                segment();
            c_left--;
            wait_copies<AHEAD * (kCopies + kStores) + kStores>(); // this step's input has arrived
            read_x(c_row);
            const int out_y = ((c_row + p.pad_top) >> (S - 1)) - NR; // first output row this step finishes
            if constexpr (RES) { // asked for now, needed at the end of the step
#pragma unroll
                for (int s = 0; s < NR; s++) {
                    const __amdgpu_buffer_rsrc_t rs = row_rsrc(p.residual, out_y + s, c_k >= 0 && out_y + s < p.out_h);
                    const unsigned dst = __builtin_amdgcn_readfirstlane(res0 + s * Shape::kResRow);
#pragma unroll
                    for (int t = 0; t < RT; t++)
                        copy4(dst + 256 * t, vout + 4 * t, rs);
                }
            }
            v4i pacc[NR][RT];
#pragma unroll
            for (int t = 0; t < RT; t++)
#pragma unroll
                for (int s = 0; s < NR; s++)
                    pacc[s][t] = *reinterpret_cast<const v4i *>(&start_l[TP + 4 * RT * quad + 4 * t]);
            v4i D[NR];
#pragma unroll
            for (int j = 0; j < CE; j++) {
                const v4i ae = we_l[j][lane];
                const v4i she = *reinterpret_cast<const v4i *>(&shift_l[TE + 16 * j + c_of]);
                v4i E[2];
                {
                    int w[2][ET];
                    v4i se = {0, 0, 0, 0};
                    if constexpr (!FOLD)
                        se = *reinterpret_cast<const v4i *>(&start_l[TE + 16 * j + c_of]);
#pragma unroll
                    for (int s = 0; s < 2; s++)
#pragma unroll
                        for (int e = 0; e < ET; e++) {
                            const v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(ae, X[s][e], se, 0, 0, 0);
                            w[s][e] = finish4<MODE, HE>(acc, she, band_e);
                            if constexpr (!FOLD)
                                w[s][e] &= (unsigned)(c_row + s) < (unsigned)p.in_h ? emask[e] : 0;
                        }
                    // the window's three columns: the neighbouring lanes' words (the fourth dword meets zero weights)
#pragma unroll
                    for (int s = 0; s < 2; s++) {
                        if constexpr (S == 1) {
                            E[s][0] = __builtin_amdgcn_update_dpp(0, w[s][0], 0x111, 0xf, 0xf, true); // row_shr:1
                            E[s][1] = w[s][0];
                            E[s][2] = __builtin_amdgcn_update_dpp(0, w[s][0], 0x101, 0xf, 0xf, true); // row_shl:1
                        } else {
                            E[s][0] = w[s][0];
                            E[s][1] = w[s][ET - 1];
                            E[s][2] = __builtin_amdgcn_update_dpp(0, w[s][0], 0x101, 0xf, 0xf, true);
                        }
                        E[s][3] = E[s][2];
                    }
                }
                v4i d[3];
#pragma unroll
                for (int ky = 0; ky < 3; ky++)
                    d[ky] = wd_l[j][ky][lane];
                const v4i sd = *reinterpret_cast<const v4i *>(&start_l[TD + 16 * j + c_of]);
                const v4i shd = *reinterpret_cast<const v4i *>(&shift_l[TD + 16 * j + c_of]);
                if constexpr (S == 1) {
                    const v4i p0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[2], E[0], U[j][0], 0, 0, 0);
                    v4i p1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[1], E[0], U[j][NL - 1], 0, 0, 0);
                    U[j][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[0], E[0], sd, 0, 0, 0);
                    p1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[2], E[1], p1, 0, 0, 0);
                    U[j][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[1], E[1], U[j][0], 0, 0, 0);
                    U[j][NL - 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[0], E[1], sd, 0, 0, 0);
                    D[0][j & 3] = finish4<MODE, HE>(p0, shd, band_d);
                    D[NR - 1][j & 3] = finish4<MODE, HE>(p1, shd, band_d);
                } else {
                    const v4i p0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[2], E[0], U[j][0], 0, 0, 0);
                    U[j][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[0], E[0], sd, 0, 0, 0);
                    U[j][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(d[1], E[1], U[j][0], 0, 0, 0);
                    D[0][j & 3] = finish4<MODE, HE>(p0, shd, band_d);
                }
                if ((j & 3) == 3 || j == CE - 1) {
#pragma unroll
                    for (int i = (j & 3) + 1; i < 4; i++)
#pragma unroll
                        for (int s = 0; s < NR; s++)
                            D[s][i] = 0;
#pragma unroll
                    for (int t = 0; t < RT; t++) {
                        const v4i ap = wp_l[(j >> 2) * RT + t][lane];
#pragma unroll
                        for (int s = 0; s < NR; s++)
                            pacc[s][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ap, D[s], pacc[s][t], 0, 0, 0);
                    }
                }
            }
            feed();
            if constexpr (RES)
                wait_copies<kCopies>(); // the residual operand (the copies behind it stay in flight)
#pragma unroll
            for (int s = 0; s < NR; s++) {
                int words[RT];
#pragma unroll
                for (int t = 0; t < RT; t++) {
                    const v4i shp = *reinterpret_cast<const v4i *>(&shift_l[TP + 4 * RT * quad + 4 * t]);
                    words[t] = finish4<MODE, HE>(pacc[s][t], shp, band_p);
                    if constexpr (RES) {
                        const unsigned char *rp = &res_l[wave][s * Shape::kResRow];
                        const int r0 = *reinterpret_cast<const int *>(rp + t * 256 + lane * 4);
                        const int rw = p.residual_shift != 0 ? requant4_s8(r0, res_q) : r0;
                        v2s s01 = __builtin_bit_cast(v2s, (int)__builtin_amdgcn_perm(0u, (unsigned)words[t], 0x010c000cu));
                        v2s s23 = __builtin_bit_cast(v2s, (int)__builtin_amdgcn_perm(0u, (unsigned)words[t], 0x030c020cu));
                        s01 = __builtin_elementwise_add_sat(s01, __builtin_bit_cast(v2s, (int)__builtin_amdgcn_perm(0u, (unsigned)rw, 0x010c000cu)));
                        s23 = __builtin_elementwise_add_sat(s23, __builtin_bit_cast(v2s, (int)__builtin_amdgcn_perm(0u, (unsigned)rw, 0x030c020cu)));
                        words[t] = (int)__builtin_amdgcn_perm((unsigned)__builtin_bit_cast(int, s23),
                                                              (unsigned)__builtin_bit_cast(int, s01), 0x07050301u);
                    }
                }
                const __amdgpu_buffer_rsrc_t rs = row_rsrc(p.out, out_y + s, c_k >= 0 && out_y + s < p.out_h);
                if constexpr (RT == 4)
                    __builtin_amdgcn_raw_buffer_store_b128(v4u{(unsigned)words[0], (unsigned)words[1], (unsigned)words[2], (unsigned)words[3]}, rs, vout, 0, 0);
                else
                    __builtin_amdgcn_raw_buffer_store_b64(v2u{(unsigned)words[0], (unsigned)words[1]}, rs, vout, 0, 0);
            }
            c_row += 2;
            c_k += NR;
        }
    };
    if (!fast)
        walk(std::integral_constant<int, 2>{});
    else if (is_high)
        walk(std::integral_constant<int, 0>{});
    else
        walk(std::integral_constant<int, 1>{});
}

} // namespace mbwalk
} // namespace espdl
