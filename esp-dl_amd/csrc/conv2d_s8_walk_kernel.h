// Dense int8 convolution as a walk down the image with the filters in registers: 1 x 1 at stride 1 and 2, 3 x 3 and
// 5 x 5 at stride 1 and 2, 16 and more input channels, any filter count from 4 on, round half up.
//
// What it computes is conv2d_11cn / _33cn / _hwcn (esp-dl/dl/base/dl_base_conv2d.cpp:9-163) under
// conv_operation_shell's window clipping (esp-dl/dl/base/dl_base.hpp:940-1191) with the n_wise epilogue
// (esp-dl/dl/base/dl_base_activate_buffer.hpp:27-36, 61-72, 173-181, 201-210).  Integer sums do not depend on their
// order, so the result is bit-identical.
//
// The layers of a detector's upper levels move many pixels of few channels: per 16 pixels there are ten to forty matrix
// instructions, and address arithmetic, operand reads and barriers per filter tap cost more than those.  Here a wavefront
// owns PT tiles of 16 output COLUMNS and 16 NT filters and goes down the rows:
//   * operand A - all KH x KS x NT filter tiles - stays in registers for the life of the (persistent) wavefront;
//   * an input row is read once: each reduction step's operand B (16 columns x 64 bytes of the row's window: the taps of a
//     filter row are neighbours in memory) serves the KH output rows it belongs to, whose accumulators are live at the
//     same time and change roles from step to step; 3 x 3 over 64 channels: three operand reads for 36 matrix instructions;
//   * input rows come straight from memory into a ring in the wavefront's own part of LDS (`buffer_load ... lds`, 16
//     bytes per lane, no registers), AHEAD steps in front of the computation; there is no barrier after the set-up.
//     Where a lane's piece comes from does not change on the way down, so a step costs a few scalar instructions;
//     columns and rows outside the image are pieces past the end of the buffer and arrive as zeros;
//   * the columns of all images form one sequence (with gaps as wide as the padding), cut into tiles of 16 without
//     regard to image borders: a 20-column image wastes 1 column in 21 and not 12 in 32;
//   * a pixel whose channels are no multiple of 16 ends with a unit that reaches back over the one before; what both hold
//     counts in the first and meets zeros in the filters of the second (20480 x 120 -> 480, 1 x 1: 12.8 -> 8.7 us;
//     202 x 67 x 42 x 40 -> 13, 3 x 3: 48 -> 13 us, where units are loaded tap by tap from memory).  Where they are no
//     multiple of 4 either, pieces pass through registers on their way to LDS (120 x 73 x 30 x 77 -> 87, 3 x 3: 88 -> 31 us;
//     200 x 19 x 23 x 22 -> 33 11.0 -> 9.9 us);
//   * a workgroup's wavefronts take neighbouring tiles; each workgroup walks the same number of output rows, however
//     many images those touch.
// What bounds it: memory where the reduction is short (160 x 160 x 32 -> 64, 1 x 1, batch 64: 4.2 TB/s), else the matrix
// pipe, which on random bytes sustains about 2 POP/s here (a large library product: 2.1).  Measured at batch 64 against
// the kernels such layers took before, us: 3 x 3 over 160 x 160 x 32 -> 32 47 -> 31, the same with a residual operand
// 77 -> 41; 3 x 3 at stride 2 over 320 x 320 x 16 -> 32 61 -> 38, 160 x 160 x 64 -> 64 49 -> 35; 3 x 3 over
// 80 x 80 x 64 -> 64 28 -> 22, 128 -> 128 90 -> 61; 1 x 1 over 160 x 160 x 32 -> 64 51 -> 37, 80 x 80 x 256 -> 256
// 77 -> 51; 5 x 5 over 80 x 80 x 64 -> 64 58 -> 44; 56 x 56 x 64 -> 64, 3 x 3, batch 256 42 -> 34.
#pragma once

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "espdl_device.h"
#include "espdl_kernels.h"

namespace espdl {
namespace walk {

constexpr int kParked = (int)0x80000000u; // past the end of any tensor: loads return zeros, stores are dropped

struct WalkArgs {
    const int8_t *in, *w;
    const int32_t *bias, *shift;
    const int8_t *lut, *res;
    int8_t *out;
    int in_bytes, w_bytes, out_bytes, res_bytes;
    int in_h, in_w, in_pitch, in_row, in_img;   // columns of a real image row, bytes from row to row and image to image
    int out_h, out_w, out_pitch, out_row, out_img;
    int res_pitch, res_row, res_img;
    int batch, out_c, n_shift, relu;
    int through; // results go through the L2 caches as they are stored
    int pad_top, pad_left;
    int w_len;    // bytes of one filter
    int last;     // first channel of a pixel's last unit, which overlaps the one before where channels are no multiple of 16
    int n_groups;   // workgroups in x
    int rows_total, rows_per_group; // output rows times column groups, and how many one workgroup walks
    long long mac_bound;
    FastDiv fd_p;  // columns an image takes in the input's sequence of columns
    FastDiv fd_po; // ... in the output's
    FastDiv fd_oh;
};

// KH: filter rows and columns; S: stride; CU: 16-byte units of an input pixel; NT: filter tiles (of 16) of a wavefront;
// RES: a residual operand is added.
template <int KH, int S, int CU, int NT, bool RES>
struct WalkShape {
    // pixel tiles (16 output columns) of a wavefront
    static constexpr int PT = KH == 1 ? (CU == 1 && NT <= 2 ? 4 : CU <= 3 ? 2 : 1) : (CU * NT <= 2 || (CU <= 2 && NT <= 2 && S == 2) ? 2 : 1);
    static constexpr int kCols = 16 * PT * S + KH - S; // input columns of a wavefront's tile
    static constexpr int kRowUnits = kCols * CU;
    static constexpr int kRowLoads = (kRowUnits + 63) / 64;
    static constexpr int KS = (KH * CU + 3) / 4;     // reduction steps per filter row
    static constexpr int kLag = (KH - 1) / S;        // steps from an output row's first input rows to its last
    static constexpr int kAcc = kLag + 1;
    static constexpr int kResUnits = RES ? 16 * PT * NT : 0;
    static constexpr int kResLoads = (kResUnits + 63) / 64;
    static constexpr int kCopies = S * kRowLoads + kResLoads; // per step
    static constexpr int kSlot = (S * kRowUnits + kResUnits) * 16;
    static constexpr int kFilterUnits = KH * KS * NT; // of 1 KB
    static constexpr long lds(int waves, int ahead) { return (long)waves * (ahead + 2) * kSlot + kFilterUnits * 1024l + 16 * NT * 11 + 512; }
    // wavefronts of a workgroup, and steps whose input is in flight while one is computed: two workgroups of four where
    // their LDS fits a compute unit, else one of eight
    static constexpr long kHalfCu = 80 * 1024, kCu = 160 * 1024;
    static constexpr bool kTwo = lds(4, 2) <= kHalfCu;
    static constexpr int W = kTwo ? 4 : (lds(8, 1) <= kCu ? 8 : 4);
    static constexpr int AHEAD = lds(W, 3) <= (kTwo ? kHalfCu : kCu) ? 3 : (lds(W, 2) <= (kTwo ? kHalfCu : kCu) ? 2 : 1);
    // physical place of unit j of column i (its place in LDS, see `place`): a read of 16 bytes per lane is served in groups
    // of 8 neighbouring columns x 2 neighbouring units, which must not meet in one of the 16 banks of 16 bytes
    static constexpr int kSwzSh = CU % 16 == 0 ? 0 : (CU % 8 == 0 ? 1 : 2);
    static constexpr int kSwzMask = CU % 16 == 0 ? 7 : (CU % 8 == 0 ? 3 : (CU % 4 == 0 ? 1 : 0));
    static constexpr int kHalf = (kCols + 1) / 2;
    static constexpr int kHeld = kAcc == 2 ? 2 : 3; // steps in registers (RAW), a multiple of the accumulators' roles
    static constexpr int kLaneC = NT == 8 ? 16 : 4 * NT; // neighbouring channels that a lane stores at once
    static __device__ __forceinline__ int swz(int ip) { return ((ip >> kSwzSh) & kSwzMask) << 1; }
    static __device__ __forceinline__ int place(int i) { return S == 1 ? i : (i & 1) * kHalf + (i >> 1); }
    static __device__ __forceinline__ int column(int ip) { return S == 1 ? ip : (ip < kHalf ? 2 * ip : 2 * (ip - kHalf) + 1); }
    // channel of a chunk that row i of filter tile t holds: a lane ends up with 4 NT neighbours (twice 16 for NT = 8)
    static __device__ __forceinline__ int channel(int t, int i)
    {
        return NT == 8 ? 64 * (t >> 2) + 16 * (i >> 2) + 4 * (t & 3) + (i & 3) : 4 * NT * (i >> 2) + 4 * t + (i & 3);
    }
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const int8_t *p, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(p), (short)0, bytes, 0x00020000);
}

// 64 pieces of 16 bytes from memory straight into LDS at `lds` + 16 lane.
__device__ __forceinline__ void copy_to_lds(unsigned lds, int voff, __amdgpu_buffer_rsrc_t rsrc)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(voff), "s"(rsrc)
                 : "memory");
}
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef unsigned v3u __attribute__((ext_vector_type(3)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
template <int AUX>
__device__ __forceinline__ void store_as(const v4u &v, __amdgpu_buffer_rsrc_t rsrc, int voff)
{
    __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, voff, 0, AUX);
}
template <int AUX>
__device__ __forceinline__ void store_as(const v3u &v, __amdgpu_buffer_rsrc_t rsrc, int voff)
{
    __builtin_amdgcn_raw_buffer_store_b96(v, rsrc, voff, 0, AUX);
}
template <int AUX>
__device__ __forceinline__ void store_as(const v2u &v, __amdgpu_buffer_rsrc_t rsrc, int voff)
{
    __builtin_amdgcn_raw_buffer_store_b64(v, rsrc, voff, 0, AUX);
}
template <int AUX>
__device__ __forceinline__ void store_as(unsigned v, __amdgpu_buffer_rsrc_t rsrc, int voff)
{
    __builtin_amdgcn_raw_buffer_store_b32(v, rsrc, voff, 0, AUX);
}
template <typename T>
__device__ __forceinline__ void store(const T &v, __amdgpu_buffer_rsrc_t rsrc, int voff, int through)
{
    if (through != 0) // uniform
        store_as<kWriteThrough>(v, rsrc, voff);
    else
        store_as<0>(v, rsrc, voff);
}
template <int N>
__device__ __forceinline__ void wait_copies()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory"); // (six bits)
}

// RAW: channels or a pitch that are no multiple of 4.  The copies into LDS take whole dwords only, so the pieces pass through
// registers: requested kHeld steps before they are written to the ring, that a step before their operands are read.
template <int KH, int S, int CU, int NT, bool RES, bool RAW = false>
__global__ __launch_bounds__((64 * WalkShape<KH, S, CU, NT, RES>::W), 2) void conv2d_s8_walk_kernel(const WalkArgs a)
{
    static_assert(!(RES && RAW));
    using Shape = WalkShape<KH, S, CU, NT, RES>;
    constexpr int KS = Shape::KS, PT = Shape::PT, AHEAD = Shape::AHEAD, kWaves = Shape::W;
    constexpr int LR = Shape::kRowLoads, RL = Shape::kResLoads, LAG = Shape::kLag, NACC = Shape::kAcc;
    constexpr int kStores = NT == 8 ? 2 * PT : PT; // per step
    constexpr int kSlot = Shape::kSlot, kSlots = AHEAD + 2, kCopies = Shape::kCopies;
    __shared__ __align__(16) unsigned char ring[kWaves][kSlots][kSlot];
    __shared__ __align__(16) struct {
        int start[16 * NT], gen[16 * NT];     // accumulator start values, shifts of the general form
        unsigned short lmul[16 * NT];         // left shifts of the short form as multipliers
        unsigned char rsh[16 * NT];           // its right shifts
    } tab_l;
    __shared__ v4i filt_l[KH * KS * NT][64]; // filters in operand-A order
    __shared__ unsigned char lut_l[256];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int group = (int)(blockIdx.x & 7u) * (a.n_groups >> 3) + (int)(blockIdx.x >> 3); // contiguous parts per XCD
    const int n0 = blockIdx.y * 16 * NT;

    const int r_begin = group * a.rows_per_group, r_end = min(a.rows_total, r_begin + a.rows_per_group);

    // Filter of row c of the chunk.  A lane stores kLaneC neighbouring channels at once; where only a part of them exists it
    // takes the last kLaneC ones of the layer, some of which the lane before has too: both write the same bytes.
    constexpr int kLaneC = Shape::kLaneC;
    const auto filter_of = [&](int c) {
        const int first = n0 + c / kLaneC * kLaneC;
        return (first < a.out_c ? min(first, a.out_c - kLaneC) : first) + c % kLaneC;
    };

    // ---- requests of what the set-up needs: one filter's bias and shift per lane, the workgroup's filters straight into
    // LDS (a part per wavefront) in operand-A order
    const bool has_lut = a.lut != nullptr;
    // (in 500 random 3 x 3 layers of 16 MB at most the choice under three and four filter tiles too gains 0.6 % in the mean, in 400 of one
    // and two it gives 0.5 %; but 56 x 56 x 64 -> 64 at batch 256, whose results it does not concern, pays 33.1 -> 34.9 us, its branches
    // part the epilogue's instructions from the next step's; one unit, 62 x 104 x 16 -> 64 at batch 19: 7.8 -> 7.0 us all the
    // same; beyond 8 units registers spill)
    const int through = KH == 1 || (KH == 3 && CU <= 8 && (NT <= 2 || CU == 1)) ? a.through : 0;
    constexpr int kMine = (16 * NT + 63) / 64; // filters of a lane
    int my_shift[kMine], my_bias[kMine];
#pragma unroll
    for (int i = 0; i < kMine; i++) {
        const int oc = min(filter_of(min(64 * i + lane, 16 * NT - 1)), a.out_c - 1);
        my_shift[i] = a.shift[a.n_shift == 1 ? 0 : oc];
        my_bias[i] = a.bias != nullptr ? a.bias[oc] : 0;
    }
    const unsigned char my_entry = has_lut && tid < 256 ? (unsigned char)a.lut[tid] : 0;
    {
        const __amdgpu_buffer_rsrc_t wr = rsrc_of(a.w, a.w_bytes);
        constexpr int units = KH * CU;
        const unsigned filt0 = (unsigned)reinterpret_cast<uintptr_t>(&filt_l[0][0]);
        const auto unit_at = [&](int e) { // e = (ky * KS + s) * NT + t
            const int t = e % NT, ks = e / NT, ky = ks / KS, u = 4 * (ks - ky * KS) + quad;
            const int oc = filter_of(Shape::channel(t, col)), tap = u / CU;
            return oc < a.out_c && u < units ? oc * a.w_len + (ky * KH + tap) * (a.last + 16) + min(16 * (u - tap * CU), a.last) : kParked;
        };
        constexpr int total = KH * KS * NT, N = (total + kWaves - 1) / kWaves;
        if constexpr (RAW) {
            v4i f[N];
#pragma unroll
            for (int i = 0; i < N; i++)
                f[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, unit_at(min(wave + i * kWaves, total - 1)), 0, 0));
#pragma unroll
            for (int i = 0; i < N; i++)
                if (wave + i * kWaves < total)
                    filt_l[wave + i * kWaves][lane] = f[i];
        } else {
            for (int e = wave; e < total; e += kWaves)
                copy_to_lds(filt0 + e * 1024, unit_at(e), wr);
        }
    }

    // ---- requests: the state of the copies, `AHEAD` steps in front of the computation
    const unsigned ring0 = (unsigned)reinterpret_cast<uintptr_t>(&ring[wave][0][0]);
    int vin[LR], vres[RL > 0 ? RL : 1];
    int f_r = r_begin, f_row = 0, f_left = 0, f_res = 0;
    unsigned f_slot = 0;
    auto feed_segment = [&]() { // the part of a column group that starts at f_r
        const int g = (int)fastdiv((unsigned)f_r, a.fd_oh);
        const int y0 = f_r - g * a.out_h;
        const int rows = min(a.out_h - y0, r_end - f_r);
        f_r += rows;
        f_left = rows + LAG;
        f_row = y0 * S - a.pad_top;
        f_res = y0 - LAG;
        const int c0 = (g * kWaves + wave) * 16 * PT;
        int lane_now = lane; // (through an empty asm statement: nothing of this is kept in registers between segments)
        asm volatile("" : "+v"(lane_now));
#pragma unroll
        for (int j = 0; j < LR; j++) {
            const int e = j * 64 + lane_now;
            const int ip = e / CU;
            const int u = (e - ip * CU) ^ Shape::swz(ip);
            const int i = Shape::column(ip);
            const int q = c0 * S - a.pad_left + i;
            const int n = (int)fastdiv((unsigned)max(q, 0), a.fd_p);
            const int x = q - n * (int)a.fd_p.d;
            const bool ok = q >= 0 && n < a.batch && x < a.in_w;
            vin[j] = ok ? n * a.in_img + x * a.in_pitch + min(16 * u, a.last) : kParked;
        }
        if constexpr (RES) {
#pragma unroll
            for (int j = 0; j < RL; j++) {
                const int e = j * 64 + lane_now, i = e / NT, u = e - i * NT;
                const int v = c0 + i;
                const int n = (int)fastdiv((unsigned)v, a.fd_po);
                const int x = v - n * (int)a.fd_po.d;
                const bool ok = n < a.batch && x < a.out_w && n0 + 16 * u < a.out_c;
                vres[j] = ok ? n * a.res_img + x * a.res_pitch + n0 + 16 * u : kParked;
            }
        }
    };
    auto copy = [&](unsigned lds, int voff, __amdgpu_buffer_rsrc_t rs, int units) {
        if (units >= 64 || lane < units)
            copy_to_lds(lds, voff, rs);
    };
    constexpr int kHeld = Shape::kHeld;
    [[maybe_unused]] v4i held[RAW ? kHeld : 1][RAW ? S : 1][RAW ? LR : 1];
    [[maybe_unused]] unsigned w_slot = 0;
    auto feed = [&](auto held_tag, bool write) __attribute__((always_inline)) { // one step; past the last one nothing is read (the counts stay the same)
        [[maybe_unused]] constexpr int H = decltype(held_tag)::value % kHeld;
        if (f_left == 0 && f_r < r_end)
            feed_segment();
        const bool live = f_left > 0;
        const unsigned base = __builtin_amdgcn_readfirstlane(ring0 + f_slot);
        if constexpr (RAW) {
            if (write) {
#pragma unroll
                for (int s = 0; s < S; s++)
#pragma unroll
                    for (int j = 0; j < LR; j++)
                        if (Shape::kRowUnits - 64 * j >= 64 || lane < Shape::kRowUnits - 64 * j)
                            *reinterpret_cast<v4i *>(&ring[wave][0][0] + w_slot + s * Shape::kRowUnits * 16 + j * 1024 + 16 * lane) = held[H][s][j];
                // Other lanes read these pieces in the next step, and what lay in the slot was read two steps ago at least: one
                // fence a step orders both.  LDS executes a wavefront's instructions in order, so nothing is waited for.
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                w_slot = w_slot + kSlot == kSlots * kSlot ? 0 : w_slot + kSlot;
            }
        }
#pragma unroll
        for (int s = 0; s < S; s++) {
            const bool ok = live && (unsigned)(f_row + s) < (unsigned)a.in_h;
            const int off = __builtin_amdgcn_readfirstlane(ok ? (f_row + s) * a.in_row : 0);
            const __amdgpu_buffer_rsrc_t rs = rsrc_of(a.in + off, __builtin_amdgcn_readfirstlane(ok ? a.in_bytes - off : 0)); // rows outside the image arrive as zeros
#pragma unroll
            for (int j = 0; j < LR; j++) {
                if constexpr (RAW)
                    held[H][s][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs, vin[j], 0, 0));
                else
                    copy(base + s * Shape::kRowUnits * 16 + j * 1024, vin[j], rs, Shape::kRowUnits - 64 * j);
            }
        }
        if constexpr (RES) {
            const bool ok = live && f_res >= 0;
            const int off = __builtin_amdgcn_readfirstlane(ok ? f_res * a.res_row : 0);
            const __amdgpu_buffer_rsrc_t rs = rsrc_of(a.res + off, __builtin_amdgcn_readfirstlane(ok ? a.res_bytes - off : 0));
#pragma unroll
            for (int j = 0; j < RL; j++)
                copy(base + S * Shape::kRowUnits * 16 + j * 1024, vres[j], rs, Shape::kResUnits - 64 * j);
        }
        f_row += S;
        f_res++;
        f_left -= live ? 1 : 0;
        f_slot = f_slot + kSlot == kSlots * kSlot ? 0 : f_slot + kSlot;
    };
    // a step issues its copies, then one store per pixel tile: where it has nothing to store, stores that are dropped, so
    // that the number of instructions behind a copy is known and the wait for it does not wait for what came later
    auto no_stores = [&]() {
#pragma unroll
        for (int p = 0; p < kStores; p++)
            asm volatile("s_nop 4\n\tbuffer_store_byte %0, %0, %1, 0 offen" ::"v"(kParked), "s"(rsrc_of(a.out, 0)) : "memory");
    };
    for (int j = 0; j < LR; j++)
        vin[j] = kParked;
    for (int j = 0; j < RL; j++)
        vres[j] = kParked;
    if constexpr (RAW) { // steps 0 and 1 are in the ring behind it
        feed(std::integral_constant<int, 0>{}, false);
        feed(std::integral_constant<int, 1>{}, false);
        if constexpr (kHeld == 3)
            feed(std::integral_constant<int, 2>{}, false);
        feed(std::integral_constant<int, kHeld>{}, true);
        feed(std::integral_constant<int, kHeld + 1>{}, true);
    } else {
#pragma unroll
        for (int i = 0; i <= AHEAD; i++) {
            feed(std::integral_constant<int, 0>{}, false);
            if (i > 0)
                no_stores();
        }
    }

    // ---- constants of the epilogue; short form when every shift of the chunk lies in 1 .. 31 and the sums fit (as in the
    // other kernels)
    bool fast, use_lsh;
    {
        int ok = 1, low = 0;
#pragma unroll
        for (int i = 0; i < kMine; i++) {
            const int s = my_shift[i];
            if (s < 1 || s > 31) {
                ok = 0;
            } else {
                const long long st = (long long)my_bias[i] + (1ll << (s - 1));
                if ((st < 0 ? -st : st) + a.mac_bound >= (1ll << (31 - max(0, 8 - s))))
                    ok = 0;
            }
            low |= s < 8;
        }
        fast = __all(ok) != 0;
        use_lsh = __any(low) != 0;
        if (wave == 0) {
#pragma unroll
            for (int i = 0; i < kMine; i++) {
                const int s = my_shift[i], c = 64 * i + lane;
                if (c < 16 * NT) {
                    tab_l.start[c] = fast ? my_bias[i] + (1 << (s - 1)) : my_bias[i];
                    tab_l.gen[c] = s;
                    tab_l.lmul[c] = (unsigned short)(fast ? 1 << max(0, 8 - s) : 1);
                    tab_l.rsh[c] = (unsigned char)max(0, s - 8);
                }
            }
        }
    }
    if (has_lut && tid < 256)
        lut_l[(tid + 128) & 255] = my_entry; // by the value's byte, not the value + 128
    const bool relu = a.relu != 0;
    const int floor_pk = relu ? 0 : (int)0x80008000u;

    // ---- operand B: LDS offsets of this lane's units inside a step's input
    int boff[KS];
#pragma unroll
    for (int s = 0; s < KS; s++) {
        const int u = min(4 * s + quad, KH * CU - 1); // (units past the window meet zero filters)
        const int tap = u / CU, j = u - tap * CU, ip = Shape::place(col * S + tap);
        boff[s] = 16 * (ip * CU + (j ^ Shape::swz(ip)));
    }
    if constexpr (!RAW)
        wait_copies<(AHEAD + 1) * kCopies + AHEAD * kStores>(); // this wavefront's part of the filters
    __syncthreads();
    v4i A[KH][KS][NT]; // operand A of the whole reduction, in registers for the life of the wavefront
#pragma unroll
    for (int ky = 0; ky < KH; ky++)
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                A[ky][s][t] = filt_l[(ky * KS + s) * NT + t][lane];
    if (const int twice = 16 * CU - 16 - a.last) // bytes of a last unit that the one before has: counted there
#pragma unroll
        for (int s = 0; s < KS; s++)
            if ((4 * s + quad) % CU == CU - 1)
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const int cut = twice - 4 * d;
                    const int mask = cut <= 0 ? -1 : (cut >= 4 ? 0 : (int)(0xffffffffu << (8 * cut)));
#pragma unroll
                    for (int ky = 0; ky < KH; ky++)
#pragma unroll
                        for (int t = 0; t < NT; t++)
                            A[ky][s][t][d] &= mask;
                }
    const auto c_of = [&](int t) { return Shape::channel(t, 4 * quad); }; // first of this lane's four channels of a filter tile
    unsigned rsh[NT]; // right shifts of the lane's channels, a byte each
#pragma unroll
    for (int t = 0; t < NT; t++) {
        rsh[t] = *reinterpret_cast<const unsigned *>(&tab_l.rsh[c_of(t)]);
    }

    v4i B[S][PT][KS];
    unsigned b_slot = 0; // slot of the step whose operands are read next
    const unsigned char *my_ring = &ring[wave][0][0];
    auto read_b = [&](int s) {
#pragma unroll
        for (int row = 0; row < S; row++)
#pragma unroll
            for (int p = 0; p < PT; p++)
                B[row][p][s] = *reinterpret_cast<const v4i *>(my_ring + (b_slot + boff[s]) + (row * Shape::kRowUnits * 16 + p * 256 * CU));
    };
    auto next_b = [&]() { b_slot = b_slot + kSlot == kSlots * kSlot ? 0 : b_slot + kSlot; };
    if constexpr (!RAW)
        wait_copies<AHEAD * (kCopies + kStores)>();
#pragma unroll
    for (int s = 0; s < KS; s++)
        read_b(s);
    next_b();

    // ---- the walk
    int vout[kStores];
    int c_r = r_begin, c_left = 0, c_y = 0; // c_y: output row that the current step finishes, relative to the segment
    int c_soff = 0;
    int segs = 0;
    for (int r = r_begin; r < r_end;) { // column groups the range touches
        const int g = (int)fastdiv((unsigned)r, a.fd_oh);
        r = min(r_end, (g + 1) * a.out_h);
        segs++;
    }
    int left = max(0, r_end - r_begin) + LAG * segs;
    auto segment = [&]() {
        const int g = (int)fastdiv((unsigned)c_r, a.fd_oh);
        const int y0 = c_r - g * a.out_h;
        const int rows = min(a.out_h - y0, r_end - c_r);
        c_r += rows;
        c_left = rows + LAG;
        c_y = -LAG;
        c_soff = (y0 - LAG) * a.out_row;
        int lane_now = lane;
        asm volatile("" : "+v"(lane_now));
        const int c0 = (g * kWaves + wave) * 16 * PT + (lane_now & 15);
#pragma unroll
        for (int p = 0; p < PT; p++) {
            const int v = c0 + 16 * p;
            const int n = (int)fastdiv((unsigned)v, a.fd_po);
            const int x = v - n * (int)a.fd_po.d;
            const int off = (n < a.batch && x < a.out_w) ? n * a.out_img + x * a.out_pitch : kParked;
#pragma unroll
            for (int i = 0; i < kStores / PT; i++) {
                const int oc = filter_of(Shape::channel(4 * i, 4 * (lane_now >> 4)));
                vout[i * PT + p] = off + oc >= 0 && oc < a.out_c ? off + oc : kParked;
            }
        }
    };
    v4i acc[NACC][PT][NT];
#pragma unroll
    for (int i = 0; i < NACC; i++)
#pragma unroll
        for (int p = 0; p < PT; p++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                acc[i][p][t] = v4i{0, 0, 0, 0};

    auto step = [&](auto tag) {
        constexpr int R = decltype(tag)::value;
        constexpr int NEW = R % NACC, FIN = (R + LAG * (NACC - 1)) % NACC; // (LAG < NACC: LAG roles back)
        if (c_left == 0)
            segment();
        c_left--;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const v4i st = *reinterpret_cast<const v4i *>(&tab_l.start[c_of(t)]);
#pragma unroll
            for (int p = 0; p < PT; p++)
                acc[NEW][p][t] = st;
        }
        if constexpr (!RAW)
            wait_copies<(AHEAD - 1) * kCopies + AHEAD * kStores>(); // the next step's input has arrived
        // residual words of the row that this step finishes sit in this step's slot, one in front of the next one's
        int resw[PT][NT];
        if constexpr (RES) {
            const unsigned prev = b_slot == 0 ? (kSlots - 1) * kSlot : b_slot - kSlot;
#pragma unroll
            for (int p = 0; p < PT; p++) {
                const int *rp = reinterpret_cast<const int *>(my_ring + prev + S * Shape::kRowUnits * 16 + (16 * p + col) * 16 * NT);
#pragma unroll
                for (int t = 0; t < NT; t++)
                    resw[p][t] = rp[Shape::channel(t, 4 * quad) / 4];
            }
        }
#pragma unroll
        for (int s = 0; s < KS; s++) {
#pragma unroll
            for (int ky = KH - 1; ky >= 0; ky--) {
                const int row = ky % S, idx = (R - ky / S + KH * NACC) % NACC;
#pragma unroll
                for (int p = 0; p < PT; p++)
#pragma unroll
                    for (int t = 0; t < NT; t++)
                        acc[idx][p][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[ky][s][t], B[row][p][s], acc[idx][p][t], 0, 0, 0);
            }
            read_b(s);
        }
        next_b();
        // into the slot of the step before (the ring has AHEAD + 2: this step's residual words still lie in its own; RAW: the pieces
        // of the step after the next, requested kHeld steps ago)
        feed(std::integral_constant<int, R + 2>{}, true);
        if (c_y >= 0) {
            const __amdgpu_buffer_rsrc_t out_rs = rsrc_of(a.out + c_soff, a.out_bytes - c_soff);
#pragma unroll
            for (int p = 0; p < PT; p++) {
                int words[NT];
                if (fast) {
                    v2s half[NT][2];
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        int v[4];
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int x = acc[FIN][p][t][r];
                            v[r] = x >> ((rsh[t] >> (8 * r)) & 255u);
                        }
                        half[t][0] = __builtin_amdgcn_cvt_pk_i16(v[0], v[1]);
                        half[t][1] = __builtin_amdgcn_cvt_pk_i16(v[2], v[3]);
                    }
                    if (use_lsh) { // uniform
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            const v2i lm = *reinterpret_cast<const v2i *>(&tab_l.lmul[c_of(t)]);
                            half[t][0] = pk_mul_sat_i16(half[t][0], lm[0]);
                            half[t][1] = pk_mul_sat_i16(half[t][1], lm[1]);
                        }
                    }
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        const v2s p01 = __builtin_elementwise_max(half[t][0], __builtin_bit_cast(v2s, floor_pk));
                        const v2s p23 = __builtin_elementwise_max(half[t][1], __builtin_bit_cast(v2s, floor_pk));
                        words[t] = (int)__builtin_amdgcn_perm((unsigned)__builtin_bit_cast(int, p23),
                                                              (unsigned)__builtin_bit_cast(int, p01), 0x07050301u);
                    }
                } else {
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        int q[4];
                        const v4i sh = *reinterpret_cast<const v4i *>(&tab_l.gen[c_of(t)]);
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            q[r] = requant_s8(acc[FIN][p][t][r], sh[r], relu, false);
                        words[t] = pack4_s8(q[0], q[1], q[2], q[3]);
                    }
                }
                if (has_lut) {
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        const unsigned w = (unsigned)words[t];
                        // bytes 0 and 2, 1 and 3 into the halves of a register each (loads of 16 bits)
                        const v2s even = {(short)lut_l[w & 255u], (short)lut_l[(w >> 16) & 255u]};
                        const v2s odd = {(short)lut_l[(w >> 8) & 255u], (short)lut_l[w >> 24]};
                        words[t] = __builtin_bit_cast(int, odd) << 8 | __builtin_bit_cast(int, even);
                    }
                }
                if constexpr (RES) {
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        v2s s01 = __builtin_bit_cast(v2s, (int)__builtin_amdgcn_perm(0u, (unsigned)words[t], 0x010c000cu));
                        v2s s23 = __builtin_bit_cast(v2s, (int)__builtin_amdgcn_perm(0u, (unsigned)words[t], 0x030c020cu));
                        s01 = __builtin_elementwise_add_sat(s01, __builtin_bit_cast(v2s, (int)__builtin_amdgcn_perm(0u, (unsigned)resw[p][t], 0x010c000cu)));
                        s23 = __builtin_elementwise_add_sat(s23, __builtin_bit_cast(v2s, (int)__builtin_amdgcn_perm(0u, (unsigned)resw[p][t], 0x030c020cu)));
                        words[t] = (int)__builtin_amdgcn_perm((unsigned)__builtin_bit_cast(int, s23),
                                                              (unsigned)__builtin_bit_cast(int, s01), 0x07050301u);
                    }
                }
                if constexpr (NT == 8) {
                    store(v4u{(unsigned)words[0], (unsigned)words[1], (unsigned)words[2], (unsigned)words[3]}, out_rs, vout[p], through);
                    store(v4u{(unsigned)words[4 % NT], (unsigned)words[5 % NT], (unsigned)words[6 % NT], (unsigned)words[7 % NT]}, out_rs, vout[PT + p], through);
                } else if constexpr (NT == 4) {
                    store(v4u{(unsigned)words[0], (unsigned)words[1], (unsigned)words[2], (unsigned)words[3]}, out_rs, vout[p], through);
                } else if constexpr (NT == 3) {
                    store(v3u{(unsigned)words[0], (unsigned)words[1], (unsigned)words[2]}, out_rs, vout[p], through);
                } else if constexpr (NT == 2) {
                    store(v2u{(unsigned)words[0], (unsigned)words[1]}, out_rs, vout[p], through);
                } else {
                    store((unsigned)words[0], out_rs, vout[p], through);
                }
            }
        } else {
            no_stores();
        }
        c_y++;
        c_soff += a.out_row;
    };
    constexpr int kRoles = RAW ? kHeld : NACC; // the accumulators' roles (and the held steps') rotate with the steps
    while (left > 0) {
        step(std::integral_constant<int, 0>{});
        if (--left == 0)
            break;
        if constexpr (kRoles > 1) {
            step(std::integral_constant<int, 1>{});
            if (--left == 0)
                break;
        }
        if constexpr (kRoles > 2) {
            step(std::integral_constant<int, 2>{});
            if (--left == 0)
                break;
        }
        if constexpr (NACC > 3) {
            step(std::integral_constant<int, 3>{});
            if (--left == 0)
                break;
        }
        if constexpr (NACC > 4) {
            step(std::integral_constant<int, 4>{});
            if (--left == 0)
                break;
        }
    }
}

// Whether a build exists: filters and accumulators fit 256 registers with what else a wavefront holds, and its LDS leaves
// a compute unit two wavefronts per SIMD.  With a residual operand 204 fit beside four filter tiles (3 and 4 units; 80 x 80 x 64 -> 64,
// 3 x 3, batch 64, input and results slices of wider tensors: 38.1 us as two chunks of 32 filters, 29.8 as one); beside one tile,
// 15 and 16 units spill 49 registers at that: a row of the input then takes several more loads, each with an address.
template <int KH, int S, int CU, int NT, bool RES, bool RAW>
constexpr bool walk_fits()
{
    using Shape = WalkShape<KH, S, CU, NT, RES>;
    if (RAW && 4 * (KH * Shape::KS * NT + Shape::kAcc * NT * Shape::PT + S * Shape::PT * Shape::KS + Shape::kHeld * S * Shape::kRowLoads) > 204)
        return false;
    return (NT != 8 || KH == 1) && (!RES || (S == 1 && KH <= 3)) &&
        4 * (KH * Shape::KS * NT + Shape::kAcc * NT * Shape::PT + S * Shape::PT * Shape::KS) <= (RES ? (NT == 4 ? 204 : 200) : 208) &&
        (Shape::kTwo || Shape::W == 8 || (S == 2 && Shape::lds(4, 1) <= Shape::kCu));
}

// What the launch needs beyond the kernel's arguments.
struct WalkLaunch {
    int cus;
    bool flat;           // the pixels of all images as one sequence
    long long out_cols;  // columns of all images side by side; flat: pixels
    long long out_bytes; // of the whole result
    hipStream_t stream;
    float *us;           // not null: nothing is launched, the expected time goes here
};

// How a layer is cut: column groups (of a workgroup's tiles), rows they have together, workgroups, rows of each.
struct WalkCut {
    int width, groups, rows, rows_total, per_group, n_groups, chunks;
};
template <int KH, int S, int CU, int NT, bool RES>
WalkCut walk_cut(const WalkArgs &a, const WalkLaunch &l, int per_cu)
{
    using Shape = WalkShape<KH, S, CU, NT, RES>;
    WalkCut c;
    c.width = 16 * Shape::PT * Shape::W;
    c.groups = (int)((l.out_cols + c.width - 1) / c.width);
    c.rows = a.out_h;
    if (l.flat) { // one column group whose rows are a workgroup's pixels
        c.rows = c.groups;
        c.groups = 1;
    }
    c.chunks = (a.out_c + 16 * NT - 1) / (16 * NT);
    c.rows_total = c.groups * c.rows;
    const int want = std::max(8, l.cus * per_cu / c.chunks / 8 * 8);
    c.per_group = (c.rows_total + want - 1) / want;
    c.n_groups = ((c.rows_total + c.per_group - 1) / c.per_group + 7) / 8 * 8;
    return c;
}

// Expected time.  Set-up (the filters among it), then the steps of one wavefront: what the wavefronts of a SIMD spend in
// matrix instructions, epilogue, copies and the rest of a step, one after the other; where that and the memory's time are
// alike they add up in part.  The constants are a fit over 780 random layers of 1 to 260 MB (1641 builds, 8 % root mean
// square).  Filter chunks of one pixel are written by different workgroups: past what the caches hold, their pieces of a
// line reach memory one by one (188 x 63 x 88 x 32 -> 96, 1 x 1: 40 us as one chunk, 66 as pieces of 64 bytes, 81 of 32).
// Many chunks over few pixels: each has eight workgroups at least, idle ones among them, and every workgroup fetches its filters
// before it starts, in as many turns as there are more workgroups than the CUs hold; the workgroups of the chunks beyond 16 cost
// 1.5 ns each (120 channels of 40 pixels -> 6625, 1 x 1: 8.4 us, 4.7 on the pointwise GEMM kernel; 4 x 32 x 96 -> 6576, 3 x 3 at
// stride 2, batch 2: 62, 8 on the narrow one; 1450 layers of 200 to 8192 filters: 0.16 root mean square, 0.21 before).
// RAW builds under 3 x 3 pass their pieces through registers step by step, which takes a fifth longer; those of 11 and 12 units of
// a pixel and the ones of 15 and 16 without RAW spill 24 to 35 registers besides (1600 and 60 layers).  At stride 2 the builds of 6
// units and more, 5 under 5 x 5, take more than 256 registers: one wavefront per SIMD, 1.4 and 2.3 us more whatever the layer's size
// (52 layers of 5 to 82 us; 3 x 3 counts 1, for the unit kernel's line lies as far below its time at 128 channels).  Four filter tiles
// beside a residual operand on 3 and 4 units, the builds that take all registers: of two chunks of 32 filters and one of 64 the smaller
// expected time is more often the one that is too small, and two chunks read a layer's input twice and write halves of its pixels.  With
// 1.2 us in favour of the two and a tenth of the memory's time in favour of the one, 5 of 4000 layers of 33 to 64 channels, slices of wider
// tensors among them, are slower by more than 5 % than without the builds, at 0.963 of that time in the mean (119 layers and 0.961 by the
// expected time alone: 40 x 40 x 64 -> 128, batch 58, 14.2 us as two chunks and 17.4 as one).
template <int KH, int S, int CU, int NT, bool RES, bool RAW>
float walk_us(const WalkArgs &a, const WalkLaunch &l)
{
    using Shape = WalkShape<KH, S, CU, NT, RES>;
    constexpr int kRegs = 44 + 4 * (KH * Shape::KS * NT + Shape::kAcc * NT * Shape::PT + S * Shape::PT * Shape::KS);
    constexpr int kPerCu = std::max(1, std::min({512 / kRegs * 4 / Shape::W, (int)(Shape::kCu / Shape::lds(Shape::W, Shape::AHEAD)), 8}));
    const WalkCut c = walk_cut<KH, S, CU, NT, RES>(a, l, kPerCu);
    const float segments = l.flat ? 1.f : 1.f + (float)(c.per_group - 1) / (float)c.rows;
    const float steps = (float)c.per_group + (float)Shape::kLag * segments;
    const int busy = (c.rows_total + c.per_group - 1) / c.per_group * c.chunks;
    const float waves = (float)(std::min(kPerCu, (busy + l.cus - 1) / l.cus) * Shape::W) * 0.25f; // of a SIMD
    const float cycles = waves * (14.4f * (KH * Shape::KS * NT * Shape::PT) + 86.f * (NT * Shape::PT) + 110.f + 1.95f * (Shape::kSlot / 16));
    const float resident = (float)(l.cus * kPerCu);
    const float walk = steps * cycles * (1.f / 2100.f) * std::max(1.f, (float)busy / resident);
    const float memory = (float)((long long)a.in_bytes + l.out_bytes + a.res_bytes) * (1.f / 9e6f);
    const float set_up = 2.9f + 0.027f * Shape::kFilterUnits + (S == 2 ? 0.25f : 0.f) - (Shape::W == 8 ? 0.36f : 0.f);
    float us = set_up * std::max(1.f, (float)(c.n_groups * c.chunks) / resident) + 1.5e-3f * (float)(c.n_groups * std::max(0, c.chunks - 16)) +
        std::cbrt((walk * std::sqrt(walk) + memory * std::sqrt(memory)) * (walk * std::sqrt(walk) + memory * std::sqrt(memory)));
    if (c.chunks > 1 && l.out_bytes > 80000000)
        us += 12e-6f * (float)l.out_bytes / (float)(16 * NT);
    if constexpr (RAW)
        return KH == 1 ? us + 0.1f : us * (CU <= 3 ? 1.15f : (CU <= 10 ? 1.2f : 1.5f)) + 0.3f;
    if (S == 2 && ((KH == 3 && CU >= 6) || (KH == 5 && CU >= 5)))
        us += KH == 3 ? 1.f : 2.3f;
    if (RES && kRegs > 244)
        us += 1.2f - 0.1f * memory;
    return KH == 3 && S == 1 && CU >= 15 ? 1.5f * us : us;
}

template <int KH, int S, int CU, int NT, bool RES, bool RAW = false>
hipError_t launch_one(WalkArgs &a, const WalkLaunch &l)
{
    if constexpr (!walk_fits<KH, S, CU, NT, RES, RAW>()) {
        return hipErrorInvalidValue;
    } else {
        using Shape = WalkShape<KH, S, CU, NT, RES>;
        if (l.us != nullptr) {
            *l.us = walk_us<KH, S, CU, NT, RES, RAW>(a, l);
            return hipSuccess;
        }
        constexpr int kThreads = 64 * Shape::W;
        const auto kernel = conv2d_s8_walk_kernel<KH, S, CU, NT, RES, RAW>;
        const WalkCut c = walk_cut<KH, S, CU, NT, RES>(a, l, resident_workgroups_per_cu(kernel, kThreads, 0));
        if (l.flat) {
            a.in_w = a.out_w = c.width;
            a.in_h = a.out_h = c.rows;
            a.in_row = c.width * a.in_pitch;
            a.out_row = c.width * a.out_pitch;
            a.res_row = c.width * a.res_pitch;
            a.fd_p = a.fd_po = make_fastdiv((unsigned)c.width);
            a.fd_oh = make_fastdiv((unsigned)a.out_h);
        }
        a.rows_total = c.rows_total;
        a.rows_per_group = c.per_group;
        a.n_groups = c.n_groups;
        hipLaunchKernelGGL(kernel, dim3((unsigned)c.n_groups, (unsigned)c.chunks), dim3(kThreads), 0, l.stream, a);
        return hipGetLastError();
    }
}
template <int KH, int S, int CU, int NT>
hipError_t launch_nt(WalkArgs &a, const WalkLaunch &l)
{
    return a.res != nullptr ? launch_one<KH, S, CU, NT, true>(a, l) : launch_one<KH, S, CU, NT, false>(a, l);
}
template <int KH, int S, int CU>
hipError_t launch_cu(int nt, WalkArgs &a, const WalkLaunch &l)
{
    switch (nt) {
    case 8:
        return launch_nt<KH, S, CU, 8>(a, l);
    case 4:
        return launch_nt<KH, S, CU, 4>(a, l);
    case 3:
        return launch_nt<KH, S, CU, 3>(a, l);
    case 2:
        return launch_nt<KH, S, CU, 2>(a, l);
    default:
        return launch_nt<KH, S, CU, 1>(a, l);
    }
}
template <int KH, int S, int CU>
hipError_t launch_raw(int nt, WalkArgs &a, const WalkLaunch &l)
{
    switch (a.res != nullptr ? 0 : nt) {
    case 4:
        return launch_one<KH, S, CU, 4, false, true>(a, l);
    case 3:
        return launch_one<KH, S, CU, 3, false, true>(a, l);
    case 2:
        return launch_one<KH, S, CU, 2, false, true>(a, l);
    case 1:
        return launch_one<KH, S, CU, 1, false, true>(a, l);
    default:
        return hipErrorInvalidValue;
    }
}
// Per window entry points, each compiled in its own translation unit; hipErrorInvalidValue: no such build.
hipError_t launch_1x1(int cu, int nt, WalkArgs &a, const WalkLaunch &l);
hipError_t launch_3x3(int cu, int nt, WalkArgs &a, const WalkLaunch &l);
hipError_t launch_3x3_s2(int cu, int nt, WalkArgs &a, const WalkLaunch &l);
hipError_t launch_5x5(int cu, int stride, int nt, WalkArgs &a, const WalkLaunch &l);
hipError_t launch_raw_1x1(int cu, int nt, WalkArgs &a, const WalkLaunch &l);
hipError_t launch_raw_3x3(int cu, int nt, WalkArgs &a, const WalkLaunch &l);

} // namespace walk
} // namespace espdl
