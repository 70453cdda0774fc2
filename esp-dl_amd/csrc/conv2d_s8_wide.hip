// Pointwise int8 convolution / Gemm with a short reduction under thousands of filters (a recognizer's 120 -> 6625
// classifier over every position): bound by writing the result, which is fifty times the size of the input.
//
// A wavefront keeps 64 pixels in registers as operand B for its whole walk and takes the filters 64 at a time, which it
// reads as operand A straight from L2 in operand order, a step ahead.  The four wavefronts of a workgroup take
// neighbouring groups of 64 filters of the same pixels, so a step makes 256 neighbouring bytes of each of 64 rows.  (Row i
// of tile t is filter 16 (i / 4) + 4 t + i % 4 of the group: a lane ends with 16 neighbouring filters of one pixel.)
// Rows of an odd length start at any address.  Writing them as the lanes hold them, 16 bytes at odd addresses, ran at
// 1.9 TB/s; so a step's bytes pass through LDS and leave as whole aligned 16-byte pieces of memory, cut out of the bytes
// of this step and the last 16 of the step before, and only the two ends of a row's walk are written by the byte.
//
// 20480 pixels x 120 -> 6625 (136 MB written, 26 us at the copy rate): 44 us inside the recognizer, where the kernel that keeps
// filters in LDS took 71 us.  A step is what bounds it: 330 vector and 32 matrix instructions of each of two wavefronts of a SIMD
// and a barrier, 2.3 us for 32 KB per compute unit.  A workgroup may have several walks, over other pixels under the same filters, so
// that the filters' constants are brought in once (two walks 42.4 us, one each 46.6; where some shift is below 8 46.1 and 49.9).
// Reading the pieces from LDS with one unaligned instruction instead of five words and shifts costs 4 us.
//
// Restates conv2d_11cn (esp-dl/dl/base/dl_base_conv2d.cpp:9-33) with the n_wise epilogue
// (esp-dl/dl/base/dl_base_activate_buffer.hpp:27-36, 61-72, 173-181, 201-210).
#include <atomic>
#include <type_traits>

#include "conv_window.h"

namespace espdl {
namespace {

using namespace window;

typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kRow = 16 + 256; // a row of the output tile in LDS: the 16 bytes in front, then those of the step
constexpr int kTileBytes = 64 * kRow + 16;
constexpr int kMaxSteps = 12; // of a walk

struct WideArgs {
    const int8_t *in, *w;
    const int32_t *bias, *shift;
    int8_t *out;
    int in_bytes, w_bytes;
    int M, K, N, in_pitch, out_pitch;
    int per_walk; // filters of a workgroup, a multiple of 256
    int relu, half_even, n_shift;
};

// WALKS: a workgroup may have several walks, each of which requests its operands itself.  (A build of its own, for with one walk
// they are on their way while the constants are prepared.  Requested there for the first walk and in the loop for the others they
// were live across all five epilogues, and 37 registers of KS 2 spilled: 44.1 instead of 42.4 us, with shifts below 8 51.4 instead of
// 46.1, which was longer than one walk each.)
template <int KS, bool WALKS>
__global__ __launch_bounds__(kThreads, 2) void conv2d_s8_wide_kernel(const WideArgs a)
{
    __shared__ __align__(16) unsigned char tile[2][kTileBytes];
    extern __shared__ __align__(16) int cst[]; // per filter of the walk: start value | right shift | left shift
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int n_begin = blockIdx.y * a.per_walk, n_end = min(a.N, n_begin + a.per_walk);
    int *const c_start = cst, *const c_rsh = cst + a.per_walk, *const c_lsh = cst + 2 * a.per_walk;
    const __amdgpu_buffer_rsrc_t in = tensor_rsrc(a.in, a.in_bytes), w = tensor_rsrc(a.w, a.w_bytes);

    // the pixels of a walk
    v4i b[4][KS];
    const auto pixels = [&](int m0, int col, int quad) {
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int k = 0; k < KS; k++) {
                const int at = 64 * k + 16 * quad, m = m0 + 16 * c + col;
                b[c][k] = load16<false>(in, m < a.M && at < a.K ? m * a.in_pitch + at : kParked, a.in_bytes);
            }
    };
    const auto mask = [&](int quad) { // zeros behind the last channel (operand A may then hold anything there)
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int k = 0; k < KS; k++)
                b[c][k] = mask_unit<false>(b[c][k], max(a.K - (64 * k + 16 * quad), 0));
    };
    if constexpr (!WALKS)
        pixels(blockIdx.x * 64, col, quad);
    // Operand A of step n: rows in lane order, a filter past the last one reads the last one again.  Away from the last
    // filters every piece is whole and the lane's one offset serves all of them.
    const auto fetch = [&](int n, v4i (&p)[4][KS], int col, int quad) {
        const int row_in_group = 16 * (col >> 2) + (col & 3);
        if (n + 64 < a.N) {
            const int row = (n + row_in_group) * a.K + 16 * quad;
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int k = 0; k < KS; k++)
                    p[t][k] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(w, row, 4 * t * a.K + 64 * k, 0));
            return;
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int row = min(n + row_in_group + 4 * t, a.N - 1) * a.K + 16 * quad;
#pragma unroll
            for (int k = 0; k < KS; k++)
                p[t][k] = load16<false>(w, 64 * k + 16 * quad < a.K ? row + 64 * k : kParked, a.w_bytes);
        }
    };
    v4i fa[4][KS];
    if constexpr (!WALKS)
        fetch(n_begin + 64 * wave, fa, col, quad);

    int ok = 1, low = 0; // the short epilogue is exact; some shift is below 8
    for (int i0 = tid; i0 < a.per_walk; i0 += 6 * kThreads) { // six at a time: their loads are in flight together
        int sh[6], bias[6];
#pragma unroll
        for (int u = 0; u < 6; u++) {
            const int n = min(n_begin + i0 + u * kThreads, a.N - 1);
            sh[u] = a.shift[a.n_shift == 1 ? 0 : n];
            bias[u] = a.bias != nullptr ? a.bias[n] : 0;
        }
#pragma unroll
        for (int u = 0; u < 6; u++) {
            const int i = i0 + u * kThreads, s = min(max(sh[u], 1), 31);
            const long long start = (long long)bias[u] + (1ll << (s - 1));
            if (sh[u] != s || (start < 0 ? -start : start) + (long long)a.K * 16384 >= 1ll << (31 - max(0, 8 - s)))
                ok = 0;
            if (s < 8)
                low = 1;
            if (i < a.per_walk) {
                c_start[i] = (int)start - (a.half_even ? 1 : 0);
                c_rsh[i] = max(0, s - 8);
                c_lsh[i] = max(0, 8 - s);
            }
        }
    }
    if constexpr (!WALKS)
        mask(quad);
    const bool fast = __syncthreads_and(ok) != 0, high = __syncthreads_or(low) == 0;

    const int floor_pk = a.relu ? 0 : (int)0x80008000u;
    const int len = n_end - n_begin;
    int turn = 0; // steps so far: the buffer of one is written while the other's bytes leave, also from walk to walk
    const auto walk = [&](auto mode) {
        constexpr int MODE = decltype(mode)::value; // of pack_fast4, -1: the general epilogue
        for (int m0 = 64 * blockIdx.x; m0 < a.M; m0 += 64 * gridDim.x) {
            int tid = (int)threadIdx.x;
            if constexpr (WALKS) // (through an empty asm statement: nothing that follows from it is kept from walk to walk)
                asm volatile("" : "+v"(tid));
            const int col = tid & 15, quad = (tid & 63) >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            if constexpr (WALKS) {
                pixels(m0, col, quad);
                fetch(n_begin + 64 * wave, fa, col, quad);
                mask(quad);
            }
            // The walk's bytes of row r start lead(r) bytes into a 16-byte piece of memory.
            int8_t *const out0 = a.out + (long long)m0 * a.out_pitch + n_begin;
            const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(out0 - 16, (short)0, 0x7ffffff0, 0x00020000);
            const auto lead = [&](int r) { return (int)((reinterpret_cast<uintptr_t>(out0) + (unsigned)(r * a.out_pitch)) & 15); };
            // Pieces of the rows this lane writes: row (tid / 16) + 16 i, piece tid % 16 of a step.
            int from[4], to[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int r = (tid >> 4) + 16 * i, at = 16 * (tid & 15) - lead(r);
                from[i] = r * kRow + 16 + at;
                to[i] = m0 + r < a.M ? 16 + r * a.out_pitch + at : kParked;
            }
            for (int step = 0; 256 * step < len; step++, turn += WALKS ? 1 : 0) {
                const int n = n_begin + 256 * step + 64 * wave;
                const int parity = WALKS ? turn : step;
                unsigned char *buf = tile[parity & 1], *next = tile[~parity & 1];
                v4i acc[4][4]; // [pixel tile][filter tile]
                const int at = n - n_begin + 16 * quad;
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    v4i start;
                    if constexpr (MODE >= 0) {
                        start = *reinterpret_cast<const v4i *>(&c_start[at + 4 * t]);
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            start[r] = a.bias != nullptr ? a.bias[min(n_begin + at + 4 * t + r, a.N - 1)] : 0;
                    }
#pragma unroll
                    for (int c = 0; c < 4; c++)
                        acc[c][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[t][0], b[c][0], start, 0, 0, 0);
                }
#pragma unroll
                for (int k = 1; k < KS; k++)
#pragma unroll
                    for (int t = 0; t < 4; t++)
#pragma unroll
                        for (int c = 0; c < 4; c++)
                            acc[c][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[t][k], b[c][k], acc[c][t], 0, 0, 0);
                if (256 * (step + 1) < len)
                    fetch(n + 256, fa, col, quad);
                int words[4][4];
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const v4i rsh = *reinterpret_cast<const v4i *>(&c_rsh[at + 4 * t]);
                    v4i lsh = {0, 0, 0, 0};
                    if constexpr (MODE != 0 && MODE != 6)
                        lsh = *reinterpret_cast<const v4i *>(&c_lsh[at + 4 * t]);
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        if constexpr (MODE >= 0) {
                            words[c][t] = pack_fast4<MODE>(acc[c][t], lsh, rsh, floor_pk);
                        } else {
                            int q[4];
#pragma unroll
                            for (int r = 0; r < 4; r++)
                                q[r] = requant_s8(acc[c][t][r], a.shift[a.n_shift == 1 ? 0 : min(n_begin + at + 4 * t + r, a.N - 1)], a.relu != 0, a.half_even != 0);
                            words[c][t] = pack4_s8(q[0], q[1], q[2], q[3]);
                        }
                    }
                }
#pragma unroll
                for (int c = 0; c < 4; c++)
                    *reinterpret_cast<v4i *>(buf + (16 * c + col) * kRow + 16 + 64 * wave + 16 * quad) =
                        v4i{words[c][0], words[c][1], words[c][2], words[c][3]};
                __syncthreads(); // one barrier per step: the other buffer was read before this one
                // Out in whole 16-byte pieces of memory: a piece ends lead(r) bytes short of where 16 bytes of the step end, so
                // the first of a step begins with bytes of the step before.
                const bool last = 256 * (step + 1) >= len;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int *src = reinterpret_cast<const int *>(buf + (from[i] & ~3));
                    int d[5];
#pragma unroll
                    for (int k = 0; k < 5; k++)
                        d[k] = src[k];
                    v4i v;
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        v[k] = (int)__builtin_amdgcn_alignbyte((unsigned)d[k + 1], (unsigned)d[k], (unsigned)(from[i] & 3));
                    int at = to[i];
                    if (step == 0 || last) { // pieces of which the walk only has a part
                        const int r = (tid >> 4) + 16 * i, off = lead(r), first = 256 * step + 16 * (tid & 15);
                        if (first < off || first + 16 > off + len)
                            at = kParked;
                    }
                    // (the step's offset is added here: beside one in a scalar register the compiler takes the data as read at once, and
                    // where the next instruction wrote the fourth dword's register, that value was stored now and then)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), out, at + 256 * step, 0, 0);
                }
                // those parts, a byte per lane: in front and behind
                if (step == 0 || last) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int r = (tid >> 4) + 16 * i, byte = tid & 15, off = lead(r), end = off + len, tail = end & ~15;
                        if (m0 + r >= a.M)
                            continue;
                        int8_t *row = out0 + (long long)r * a.out_pitch - off;
                        const unsigned char *bytes = buf + r * kRow + 16 - off;
                        if (step == 0 && byte >= off && byte < end && (off != 0 || end < 16))
                            row[byte] = (int8_t)bytes[byte];
                        if (last && tail != 0 && tail + byte < end)
                            row[tail + byte] = (int8_t)bytes[tail + byte - 256 * step];
                    }
                }
                if (tid < 64) // what the next step's first pieces start with
                    *reinterpret_cast<v4i *>(next + tid * kRow) = *reinterpret_cast<const v4i *>(buf + tid * kRow + 256);
            }
            if constexpr (!WALKS)
                break;
        }
    };
    if (!fast)
        walk(std::integral_constant<int, -1>{});
    else if (a.half_even)
        high ? walk(std::integral_constant<int, 6>{}) : walk(std::integral_constant<int, 5>{});
    else
        high ? walk(std::integral_constant<int, 0>{}) : walk(std::integral_constant<int, 1>{});
}

// The tile and the constants of walks of 10 steps and more are past the 64 KB of LDS that a launch may have unasked
// (twelve steps: 70 KB, two workgroups to a compute unit as before): the limit is raised once per device (bit d: done on
// device d; two threads may both do it).
template <int KS, bool WALKS>
hipError_t allow_lds(size_t dynamic)
{
    if (2 * kTileBytes + dynamic <= 64 * 1024)
        return hipSuccess;
    static std::atomic<unsigned long long> raised{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return e;
    const unsigned long long bit = 1ull << (dev & 63);
    if (dev < 64 && (raised.load(std::memory_order_relaxed) & bit))
        return hipSuccess;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(conv2d_s8_wide_kernel<KS, WALKS>), hipFuncAttributeMaxDynamicSharedMemorySize,
                            3 * (int)sizeof(int) * 256 * kMaxSteps);
    if (e == hipSuccess && dev < 64)
        raised.fetch_or(bit, std::memory_order_relaxed);
    return e;
}

} // namespace

// Rows of the result that are no multiple of 16 bytes long, which the other kernels write in pieces at odd addresses, and
// enough of them: 640 rows of 6625 take 8.5 us either way, 1280 rows 10 against 15 us.  (3000 rows of 2048 from 128: 8.7
// against 6.6 us, 20480 rows of 4096 from 64: 28 against 30 us.)
bool conv2d_s8_wide_supports(const ConvGeom &g, const int8_t *lut, const int8_t *residual)
{
    const bool flat = g.k_h == 1 && g.k_w == 1 && g.stride_h == 1 && g.stride_w == 1 && g.pad_top == 0 && g.pad_left == 0 &&
        g.out_h == g.in_h && g.out_w == g.in_w;
    return flat && lut == nullptr && residual == nullptr && g.in_c >= 16 && g.in_c <= 128 && g.out_c >= 2048 &&
        (g.out_pitch & 15) != 0 && g.out_pitch < (1 << 24) && (long long)g.batch * g.out_h * g.out_w >= 1024 && window_supports(g);
}

hipError_t launch_conv2d_s8_wide(const ConvGeom &g, const int8_t *in, const int8_t *filter, const int32_t *bias,
                                 const int32_t *shift, int8_t *out, int cu_count, hipStream_t stream)
{
    const WindowArgs wa = window_args(g, in, filter);
    WideArgs a;
    a.in = in;
    a.w = filter;
    a.bias = bias;
    a.shift = shift;
    a.out = out;
    a.in_bytes = wa.in_bytes;
    a.w_bytes = wa.w_bytes;
    a.M = g.batch * g.out_h * g.out_w;
    a.K = g.in_c;
    a.N = g.out_c;
    a.in_pitch = g.in_pitch;
    a.out_pitch = g.out_pitch;
    a.relu = g.relu;
    a.half_even = g.half_even;
    a.n_shift = g.n_shift;
    if (a.M == 0)
        return hipSuccess;
    // Steps per walk: rounds of workgroups (two fit a compute unit) times a walk and its start, which costs about four
    // steps; kMaxSteps steps' constants at most lie in LDS.
    const int tiles = (a.M + 63) / 64, steps = (a.N + 255) / 256;
    const long long slots = 2ll * std::max(1, cu_count);
    int per = 1;
    long long best = 0;
    for (int p = 1; p <= std::min(steps, kMaxSteps); p++) {
        const long long cost = ((long long)tiles * ((steps + p - 1) / p) + slots - 1) / slots * (p + 4);
        if (p == 1 || cost < best) {
            best = cost;
            per = p;
        }
    }
    const long long groups = std::max(1ll, slots / ((steps + per - 1) / per)); // that take the same filters
    // More rounds than one become walks of the same workgroups.  Beyond 64 channels, where a step is matrix work too, only if that leaves
    // the busiest compute unit no more tiles than it had, and at most 1.3 times an even share of all steps: 250 random layers 0.87 to
    // 1.06 of the time of a workgroup per walk, 0.95 in the mean; the other 84 up to 1.25.  (Up to 64 channels 59 layers 0.82 to 1.03.)
    int walks = (int)((tiles + groups - 1) / groups);
    const long long cus = std::max(1, cu_count), columns = (steps + per - 1) / per;
    const long long share = ((tiles + walks - 1) / walks * columns + cus - 1) / cus * walks; // walks of the busiest compute unit
    if (a.K > 64 && (share > (tiles * columns + cus - 1) / cus || 10 * share * per * cus > 13ll * tiles * steps))
        walks = 1;
    a.per_walk = 256 * per;
    const dim3 grid((unsigned)((tiles + walks - 1) / walks), (unsigned)((steps + per - 1) / per));
    const size_t lds = (size_t)3 * sizeof(int) * a.per_walk;
    const auto launch = [&](auto ks, auto several) {
        constexpr int KS = decltype(ks)::value;
        constexpr bool WALKS = decltype(several)::value;
        const hipError_t e = allow_lds<KS, WALKS>(lds);
        if (e != hipSuccess)
            return e;
        hipLaunchKernelGGL((conv2d_s8_wide_kernel<KS, WALKS>), grid, dim3(kThreads), lds, stream, a);
        return hipGetLastError();
    };
    const std::integral_constant<int, 1> one;
    const std::integral_constant<int, 2> two;
    if (walks > 1)
        return a.K <= 64 ? launch(one, std::true_type{}) : launch(two, std::true_type{});
    return a.K <= 64 ? launch(one, std::false_type{}) : launch(two, std::false_type{});
}

} // namespace espdl
