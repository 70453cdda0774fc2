// Inverted-residual block (1x1 expand conv -> 3x3 depthwise conv -> 1x1 project conv [-> Add]) for int8 on gfx950 in
// TWO launches: this kernel runs expand -> depthwise and writes the depthwise result to a workspace, the project
// convolution and the Add follow through the dense kernels (conv2d_s8_narrow.hip, conv2d_s8_pwgemm.hip).
//
// The stages compute exactly what the separate operators compute (mbconv_s8_stages.h names the reference functions),
// with the int8 result of every stage materialized before the next one reads it.
//
// Why: the single-launch kernels give a wavefront or a workgroup a whole tile of the block, all its expanded channels
// and the project product behind them.  Such a chain takes 12 to 24 us however few tiles there are, and with few
// images most of the device watches (7 x 7, 160 -> 960 -> 160, one image: ONE workgroup, 21.6 us).  Expanded channels are
// independent up to the project product, so here a workgroup takes a tile and 64 expanded channels of it (one chunk
// of 16 per wavefront), which multiplies the workgroups by up to exp_c / 64; the depthwise result (a few MB at most on
// such images) stays in the caches until the project launch reads it.
//
// The block-input patch of the tile lies in LDS, copied once per workgroup (kept in registers as operand B, as the
// single-launch kernels do, it left two wavefronts per SIMD).  A wavefront requests the filters and constants of its
// next chunk a chunk ahead, builds the requantization constants of its own chunk in LDS (no workgroup tables, no votes
// across wavefronts) and runs expand -> depthwise in a private LDS area.  The four chunks of a group meet in an LDS tile
// [pixel][64 channels] that all wavefronts write out as 64-byte runs.
//
// On few images the launch is the life of one workgroup, instructions and round trips one behind the other (28 x 28, 32 -> 192, one image:
// 0.4 us of arguments and addresses, 0.4 for the patch, 0.95 for constants and a barrier that waited for the next chunk's
// loads, 0.55 expand, 0.85 depthwise, after 1.2 us between launches).  So there a tile has two output rows (one at stride 2)
// instead of seven (four), a workgroup takes one group of 64 channels without a loop around it, barriers order LDS alone, and
// all arguments are fetched at once: 4.6 -> 3.2 us; 7 x 7, 160 -> 960 5.0 -> 3.55; 37 images of 10 x 10, 64 -> 384 5.4 -> 4.8, of 20 x 20, 32 ->
// 192 6.2 -> 5.6.  Requesting the patch before and placing it behind the constants' arithmetic held too many registers (spills from
// 65 input channels on, 14 x 14, 96 -> 576 3.6 -> 4.0 us).
#include <algorithm>
#include <type_traits>

#include "conv_window.h"
#include "mbconv_s8_stages.h"

namespace espdl {

namespace {

using namespace mbstage;

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;

struct SplitArgs {
    MbconvParams p;
    int8_t *mid; // [batch][out_h][out_w][exp_c]
    int through; // results go through the L2 caches as they are stored
    int tiles_x, tiles_y, n_tiles;
    int n_groups;    // groups of 64 expanded channels
    int per_wg;      // groups a workgroup walks
    int parts;       // workgroups per tile
    int in_bytes;
    int units, pitch; // 16-byte pieces of a patch pixel, LDS bytes from pixel to pixel (twice an odd number of pieces)
    FastDiv fd_units, fd_tiles_x, fd_tiles_yx, fd_parts;
};

// Tile of PT x TW output pixels; patch of ((PT - 1) S + 3) x ((TW - 1) S + 3) block-input pixels.
template <int PT, int TW, int S>
struct Tile {
    static constexpr int PH = (PT - 1) * S + 3, PW = (TW - 1) * S + 3;
    static constexpr int NXPT = (PH * PW + 15) / 16;
    // row of patch position p: p / PW in 24 bits (p below 1024, PW 9, 15 or 16)
    static constexpr unsigned kPerPW = (65536u + PW - 1) / PW;
    static __device__ __forceinline__ int patch_row(int p)
    {
        return (int)(__umul24((unsigned)p, kPerPW) >> 16);
    }
    static constexpr int TWP = TW <= 8 ? 8 : 16; // pixel slots per output row in the LDS tile
    // the depthwise stage reads up to one row pair and three columns past the patch (zero weights meet those bytes)
    static constexpr int EXP_BYTES = std::max((PH + 1) * PW + 48, NXPT * 16) * 16;
    static constexpr int DW_BYTES = PT * TWP * kDws;
};

// LOOP: a workgroup walks several groups of 64 expanded channels.  Without it what the loop would keep over its turns (addresses, masks,
// some 170 instructions and scalar spills ahead of the first product) does not exist.
template <int PT, int TW, int S, int KSE, bool HE, bool CLIP, bool LOOP>
__global__ __launch_bounds__(kThreads, 4) void mbconv_s8_expand_dw_kernel(const SplitArgs a)
{
    using T = Tile<PT, TW, S>;
    constexpr int NXPT = T::NXPT;
    __shared__ __align__(16) unsigned char exp_l[kWaves][T::EXP_BYTES];
    __shared__ __align__(16) unsigned char dw_l[T::DW_BYTES];
    __shared__ __align__(16) int tab_l[kWaves][2][3 * 16]; // expand, depthwise: [start value | right shift | left shift]
    extern __shared__ __align__(16) unsigned char patch_l[]; // [NXPT * 16 pixels][pitch] + slack
    const MbconvParams &p = a.p;
    if constexpr (!LOOP) // every argument on its way at once: one round trip of the scalar cache in front of everything
        asm volatile("" ::"s"(p.relu_expand), "s"(p.out_h), "s"(p.out_w), "s"(p.pad_top), "s"(p.n_s_dw), "s"(a.mid), "s"(a.through),
                     "s"(a.pitch), "s"(a.units), "s"(p.b_dw), "s"(p.s_dw));
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, quad = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // all workgroups of a tile on one XCD (they share the patch and the lines of the result)
    int id = blockIdx.x;
    if ((gridDim.x & 7u) == 0)
        id = (int)(blockIdx.x & 7u) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    const unsigned tile = fastdiv((unsigned)id, a.fd_parts);
    const int part = id - (int)(tile * a.fd_parts.d);
    const unsigned n = fastdiv(tile, a.fd_tiles_yx);
    const unsigned rem = tile - n * a.fd_tiles_yx.d;
    const unsigned ty = fastdiv(rem, a.fd_tiles_x);
    const int oy0 = (int)ty * PT, ox0 = (int)(rem - ty * a.fd_tiles_x.d) * TW;
    const int iy0 = oy0 * S - p.pad_top, ix0 = ox0 * S - p.pad_left;
    const int c0 = p.in_c;

    // what a chunk of 16 expanded channels needs, requested one chunk ahead
    struct Chunk {
        v4i aop[KSE];
        int wd0[3], wd1[3];
        int bias, shift; // lanes 0 .. 15: expand channel `col`, lanes 16 .. 31: depthwise channel `col`
    };
    const __amdgpu_buffer_rsrc_t we_rsrc = window::tensor_rsrc(p.w_expand, p.exp_c * c0);
    const bool dw_lane = quad == 1;
    const int32_t *b_src = dw_lane ? p.b_dw : p.b_expand, *s_src = dw_lane ? p.s_dw : p.s_expand;
    const unsigned s_step = (dw_lane ? p.n_s_dw : p.n_s_expand) == 1 ? 0u : 1u;
    auto load_chunk = [&](int sub, Chunk &w) {
        const int ch = min(16 * sub, p.exp_c - 16) + col; // (a chunk past the last reads the last one again)
#pragma unroll
        for (int ks = 0; ks < KSE; ks++) {
            const int left = c0 - 64 * ks - 16 * quad;
            w.aop[ks] = window::load16<true>(we_rsrc, left > 0 ? ch * c0 + 64 * ks + 16 * quad : window::kParked, 0);
        }
#pragma unroll
        for (int kx = 0; kx < 3; kx++) {
            w.wd0[kx] = (int)p.w_dw[(size_t)(unsigned)((min(quad, 2) * 3 + kx) * p.exp_c + ch)];
            w.wd1[kx] = 0;
            if constexpr (S == 1)
                w.wd1[kx] = (int)p.w_dw[(size_t)(unsigned)((max(quad - 1, 0) * 3 + kx) * p.exp_c + ch)];
        }
        w.bias = b_src != nullptr ? b_src[(size_t)(unsigned)ch] : 0;
        w.shift = s_src[(size_t)(s_step * (unsigned)ch)];
    };
    const int g_first = LOOP ? part * a.per_wg : part, g_end = LOOP ? min(g_first + a.per_wg, a.n_groups) : g_first + 1;
    Chunk cur;
    load_chunk(4 * g_first + wave, cur);

    // the block-input patch: operand B of the expand products.  Nothing is zeroed: a pixel outside the image has its
    // expand OUTPUT zeroed through xmask, positions past the last channel meet zeros in operand A
    {
        const __amdgpu_buffer_rsrc_t in_rsrc = window::tensor_rsrc(p.in, a.in_bytes);
        const int img = (int)n * p.in_h * p.in_w;
        const int n_pieces = T::PH * T::PW * a.units;
        for (int first = 0; first < n_pieces; first += 4 * kThreads) {
            v4i v[4];
            int at[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (!LOOP && first + j * kThreads >= n_pieces) // uniform
                    break;
                const int u = first + j * kThreads + tid;
                const int pp = (int)fastdiv((unsigned)u, a.fd_units), unit = u - pp * a.units;
                const int prow = T::patch_row(pp);
                const int iy = iy0 + prow, ix = ix0 + pp - prow * T::PW;
                const bool valid = u < n_pieces && (unsigned)iy < (unsigned)p.in_h && (unsigned)ix < (unsigned)p.in_w;
                at[j] = pp * a.pitch + 16 * unit;
                v[j] = window::load16<true>(in_rsrc, valid ? (img + iy * p.in_w + ix) * c0 + 16 * unit : window::kParked, 0);
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (first + j * kThreads + tid < n_pieces)
                    *reinterpret_cast<v4i *>(patch_l + at[j]) = v[j];
        }
    }
    unsigned xmask = 0;
#pragma unroll
    for (int pt = 0; pt < NXPT; pt++) {
        const int pp = pt * 16 + col;
        const int prow = T::patch_row(pp);
        const int iy = iy0 + prow, ix = ix0 + pp - prow * T::PW;
        xmask |= (unsigned)iy < (unsigned)p.in_h && (unsigned)ix < (unsigned)p.in_w ? 1u << pt : 0u;
    }
    const unsigned char *patch_src = patch_l + col * a.pitch + 16 * quad;
    const int tile_step = 16 * a.pitch;
    // expand stage of a chunk: four pixel tiles at a time
    auto expand = [&](auto mode_tag, const v4i(&aop)[KSE], const StageConsts &c, int floor_pk, int ceil_pk, unsigned char *dst) {
        constexpr int MODE = decltype(mode_tag)::value;
#pragma unroll
        for (int g0 = 0; g0 < NXPT; g0 += 4) {
            v4i acc[4];
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (g0 + j < NXPT) {
                    acc[j] = c.init;
#pragma unroll
                    for (int ks = 0; ks < KSE; ks++)
                        acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                            aop[ks], *reinterpret_cast<const v4i *>(patch_src + (g0 + j) * tile_step + 64 * ks), acc[j], 0, 0, 0);
                }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (g0 + j < NXPT) {
                    int word = wave_pack_tab<MODE, CLIP>(acc[j], c, floor_pk, p.relu_expand != 0, HE, ceil_pk);
                    word &= __builtin_amdgcn_sbfe((int)xmask, g0 + j, 1); // all ones or zero
                    *reinterpret_cast<int *>(dst + (g0 + j) * 256) = word;
                }
        }
    };

    const unsigned bound_e = (unsigned)c0 * 16384u, bound_d = 9u * 16384u;
    // with a Clip behind a stage the lower clamp is its bound (or ReLU's 0 where that is higher)
    auto floor_of = [](int relu, int clip, int lo) {
        const int v = clip ? max(lo, relu ? 0 : -128) : (relu ? 0 : -128);
        return ((v * 256) & 0xffff) | (int)((unsigned)(v * 256) << 16);
    };
    auto ceil_of = [](int clip, int hi) {
        const int v = ((clip ? hi : 127) * 256) | 0xff;
        return (v & 0xffff) | (int)((unsigned)v << 16);
    };
    const int floor_e = floor_of(p.relu_expand, CLIP && p.clip_e, p.clip_e_lo), ceil_e = ceil_of(CLIP && p.clip_e, p.clip_e_hi);
    const int floor_d = floor_of(p.relu_dw, CLIP && p.clip_d, p.clip_d_lo), ceil_d = ceil_of(CLIP && p.clip_d, p.clip_d_hi);
    unsigned char *exp_dst = exp_l[wave] + col * 16 + 4 * quad;
    const unsigned char *exp_src = exp_l[wave] + (quad * T::PW + S * col) * 16;
    unsigned char *dw_dst = dw_l + col * kDws + 16 * wave + 4 * quad;
    int *tab = tab_l[wave][0];
    const bool write_ok = col < TW;

    int gi = g_first;
    do {
        Chunk nxt = cur;
        const int sub = 4 * gi + wave;
        if constexpr (LOOP) // (the last one again in the last turn: a branch here costs 3 %, 4 % on 80 -> 480 at stride 2)
            load_chunk(4 * min(gi + 1, g_end - 1) + wave, nxt);
        // constants of this chunk: the short form where every channel of the stage can take it (see mbconv_s8_stages.h)
        int mode_e, mode_d;
        {
            const int s = cur.shift, b = cur.bias;
            const bool bad = !short_ok(s, b, dw_lane ? bound_d : bound_e);
            const unsigned long long m_bad = __ballot(bad), m_low = __ballot(s < 8);
            auto mode_of = [&](int sh) {
                const unsigned any_bad = (unsigned)(m_bad >> sh) & 0xffffu, any_low = (unsigned)(m_low >> sh) & 0xffffu;
                return any_bad != 0 ? -1 : (HE ? (any_low != 0 ? 5 : 6) : (any_low != 0 ? 1 : 0));
            };
            mode_e = mode_of(0);
            mode_d = mode_of(16);
            const int mode = dw_lane ? mode_d : mode_e;
            if (lane < 32) {
                int *t = tab + 48 * quad + col;
                t[0] = mode < 0 ? b : b + (1 << (s - 1)) - (HE ? 1 : 0);
                t[16] = mode < 0 ? s : max(0, s - 8);
                t[32] = mode < 0 ? 0 : max(0, 8 - s);
            }
        }
        wave_lds_sync();
        v4i aop[KSE];
#pragma unroll
        for (int ks = 0; ks < KSE; ks++)
            aop[ks] = window::mask_unit<false>(cur.aop[ks], c0 - 64 * ks - 16 * quad);
        const StageConsts ce = read_stage_table(tab, 16, 4 * quad, mode_e);
        if (!LOOP || gi == g_first)
            lds_barrier(); // the patch is complete
        {
            if (!HE && ce.mode == 0)
                expand(std::integral_constant<int, 0>{}, aop, ce, floor_e, ceil_e, exp_dst);
            else if (!HE && ce.mode == 1)
                expand(std::integral_constant<int, 1>{}, aop, ce, floor_e, ceil_e, exp_dst);
            else if (HE && ce.mode == 6)
                expand(std::integral_constant<int, 6>{}, aop, ce, floor_e, ceil_e, exp_dst);
            else if (HE && ce.mode == 5)
                expand(std::integral_constant<int, 5>{}, aop, ce, floor_e, ceil_e, exp_dst);
            else
                expand(std::integral_constant<int, -1>{}, aop, ce, floor_e, ceil_e, exp_dst);
        }
        wave_lds_sync();
        if (LOOP && gi != g_first)
            lds_barrier(); // the tile's previous group has been read
        if (16 * sub < p.exp_c) { // uniform
            v4i a0[3], a1[3];
#pragma unroll
            for (int kx = 0; kx < 3; kx++) {
                a0[kx] = diag_operand(quad < 3 ? cur.wd0[kx] : 0, col);
                a1[kx] = diag_operand(quad >= 1 ? cur.wd1[kx] : 0, col);
            }
            const StageConsts cd = read_stage_table(tab + 48, 16, 4 * quad, mode_d);
            const bool relu = p.relu_dw != 0;
            constexpr int row_bytes = T::TWP * kDws;
            if (!HE && cd.mode == 0)
                depthwise_chunk<0, PT, S, true, false, CLIP>(exp_src, PT, T::PW, a0, a1, cd, floor_d, relu, HE, dw_dst, row_bytes, write_ok, ceil_d);
            else if (!HE && cd.mode == 1)
                depthwise_chunk<1, PT, S, true, false, CLIP>(exp_src, PT, T::PW, a0, a1, cd, floor_d, relu, HE, dw_dst, row_bytes, write_ok, ceil_d);
            else if (HE && cd.mode == 6)
                depthwise_chunk<6, PT, S, true, false, CLIP>(exp_src, PT, T::PW, a0, a1, cd, floor_d, relu, HE, dw_dst, row_bytes, write_ok, ceil_d);
            else if (HE && cd.mode == 5)
                depthwise_chunk<5, PT, S, true, false, CLIP>(exp_src, PT, T::PW, a0, a1, cd, floor_d, relu, HE, dw_dst, row_bytes, write_ok, ceil_d);
            else
                depthwise_chunk<-1, PT, S, true, false, CLIP>(exp_src, PT, T::PW, a0, a1, cd, floor_d, relu, HE, dw_dst, row_bytes, write_ok, ceil_d);
        }
        lds_barrier(); // the group's tile is complete
        int8_t *dst = a.mid + (((long long)n * p.out_h + oy0) * p.out_w + ox0) * p.exp_c + 64 * gi;
#pragma unroll
        for (int i = 0; i < (PT * T::TWP * 4 + kThreads - 1) / kThreads; i++) {
            const int u = tid + i * kThreads;
            const int slot = u >> 2, q = u & 3;
            const int row = slot / T::TWP, x = slot % T::TWP;
            if (row < PT && x < TW && oy0 + row < p.out_h && ox0 + x < p.out_w && 64 * gi + 16 * q < p.exp_c)
                store16(dst, (row * p.out_w + x) * p.exp_c + 16 * q, *reinterpret_cast<const v4i *>(dw_l + slot * kDws + 16 * q), a.through);
        }
        cur = nxt;
    } while (LOOP && ++gi < g_end);
}

struct SplitPlan {
    bool ok;
    int pt, tw, kse;
    float us; // expected time
};

// Expected time of tiles of `pt` rows: the launch and one workgroup's chain, which is shorter the fewer rows it has, then the work of
// all workgroups, which grows with the halo (two rows of the patch at stride 1, one at stride 2); the highest tiles lose 2 to 4 us
// where workgroups walk several groups, of which there are fewer and longer ones then.  Fitted to 6700 launches on 1 to 400
// images and 1 KB to 300 MB of results, each tile forced in turn: 4 to 8 % off; the tile it picks takes 0.5 % more than the best one in
// the mean, the largest one 26 %.  (A fit to 1 to 100 images, most of them below 4 MB, had the highest tiles at stride 1 half as expensive
// again as expected beyond that: 48 images of 40 x 40, 24 -> 144, 12.6 us expected, 24.5 measured.)
float split_us(const MbconvParams &p, int kse, int tw, int pt)
{
    const long long tiles = (long long)p.batch * ((p.out_w + tw - 1) / tw) * ((p.out_h + pt - 1) / pt);
    const long long groups = (p.exp_c + 63) / 64;
    const float work = (float)(tiles * groups) * (1.f / 256.f), k = (float)(kse - 1), he = p.half_even ? 1.f : 0.f;
    const float walks = groups > 1 && tiles * groups >= 2048 ? 1.f : 0.f; // several groups to a workgroup of the highest tiles
    if (p.stride_h == 2)
        return pt == 1 ? (3.2f + 0.18f * k + work * (0.431f + 0.04f * k)) * (1.f + 0.056f * he)
            : pt == 2  ? (3.41f + 0.21f * k + work * (0.54f + 0.091f * k)) * (1.f + 0.069f * he)
                       : (3.95f + 0.35f * k + work * (0.696f + 0.208f * k) + 2.3f * walks) * (1.f + 0.077f * he);
    if (tw == 7)
        return pt == 2 ? (3.46f + 0.087f * k + work * (0.476f + 0.054f * k)) * (1.f + 0.017f * he)
            : pt == 4  ? (3.68f + 0.098f * k + work * (0.563f + 0.09f * k)) * (1.f + 0.042f * he)
                       : (4.11f + 0.133f * k + work * (0.661f + 0.158f * k) + 3.5f * walks) * (1.f + 0.062f * he);
    const float wide_pixel = kse == 3 ? 0.21f : 0.f; // its patch leaves a compute unit fewer workgroups
    return pt == 2 ? (3.34f + 0.135f * k + work * (0.513f + 0.071f * k)) * (1.f + 0.058f * he)
        : pt == 4  ? (3.59f + 0.106f * k + work * (0.667f + 0.17f * k)) * (1.f + 0.07f * he)
                   : (4.07f + 0.24f * k + work * (0.867f + 0.213f * k + wide_pixel) + 3.5f * walks) * (1.f + 0.096f * he);
}

SplitPlan split_plan(const MbconvParams &p)
{
    SplitPlan plan = {};
    if (p.w_expand == nullptr || !mbconv_expand_is_pointwise(p) || p.k_h != 3 || p.k_w != 3 || p.dil_h != 1 ||
        p.dil_w != 1 || p.stride_h != p.stride_w || (p.stride_h != 1 && p.stride_h != 2))
        return plan;
    if (p.in_c % 4 != 0 || p.in_c > 192 || p.exp_c % 16 != 0 || p.exp_c < 16 || p.exp_c >= 65536 ||
        (reinterpret_cast<uintptr_t>(p.in) & 3) != 0 || (reinterpret_cast<uintptr_t>(p.w_expand) & 3) != 0)
        return plan;
    if ((long long)p.batch * p.in_h * p.in_w * p.in_c >= (1ll << 31) - 64 || (long long)p.exp_c * p.in_c >= (1ll << 31) ||
        (long long)p.batch * p.out_h * p.out_w * p.exp_c >= (1ll << 31) - 64)
        return plan;
    plan.kse = (p.in_c + 63) / 64;
    // narrow images and strided blocks take tiles of seven columns (a patch of fifteen columns at stride 2), wide
    // images at stride 1 tiles of fourteen
    plan.tw = p.stride_h == 1 && p.out_w > 7 ? 14 : 7;
    // fewer rows while that leaves the launch shorter: few images
    const int rows[2][3] = {{7, 4, 2}, {4, 2, 1}};
    plan.us = 1e30f;
    for (const int pt : rows[p.stride_h - 1]) {
        const float us = split_us(p, plan.kse, plan.tw, pt);
        if (us < plan.us) {
            plan.us = us;
            plan.pt = pt;
        }
    }
    plan.ok = true;
    return plan;
}

template <int PT, int TW, int S, int KSE, bool HE, bool LOOP>
hipError_t launch_tile(const SplitArgs &a, hipStream_t stream)
{
    const dim3 grid((unsigned)(a.n_tiles * a.parts));
    // (the last k step of the last pixel reads up to 64 bytes past its pixel)
    const size_t lds = (size_t)Tile<PT, TW, S>::NXPT * 16 * a.pitch + 256;
    if (a.p.clip_e || a.p.clip_d)
        hipLaunchKernelGGL((mbconv_s8_expand_dw_kernel<PT, TW, S, KSE, HE, true, LOOP>), grid, dim3(kThreads), lds, stream, a);
    else
        hipLaunchKernelGGL((mbconv_s8_expand_dw_kernel<PT, TW, S, KSE, HE, false, LOOP>), grid, dim3(kThreads), lds, stream, a);
    return hipGetLastError();
}

template <int KSE, bool HE>
hipError_t launch_kse(const SplitPlan &plan, const SplitArgs &a, hipStream_t stream)
{
    if (a.per_wg > 1)
        return a.p.stride_h == 2 ? launch_tile<4, 7, 2, KSE, HE, true>(a, stream)
            : plan.tw == 7       ? launch_tile<7, 7, 1, KSE, HE, true>(a, stream)
                                 : launch_tile<7, 14, 1, KSE, HE, true>(a, stream);
    if (a.p.stride_h == 2)
        return plan.pt == 1 ? launch_tile<1, 7, 2, KSE, HE, false>(a, stream)
            : plan.pt == 2  ? launch_tile<2, 7, 2, KSE, HE, false>(a, stream)
                            : launch_tile<4, 7, 2, KSE, HE, false>(a, stream);
    if (plan.tw == 7)
        return plan.pt == 2 ? launch_tile<2, 7, 1, KSE, HE, false>(a, stream)
            : plan.pt == 4  ? launch_tile<4, 7, 1, KSE, HE, false>(a, stream)
                            : launch_tile<7, 7, 1, KSE, HE, false>(a, stream);
    return plan.pt == 2 ? launch_tile<2, 14, 1, KSE, HE, false>(a, stream)
        : plan.pt == 4  ? launch_tile<4, 14, 1, KSE, HE, false>(a, stream)
                        : launch_tile<7, 14, 1, KSE, HE, false>(a, stream);
}

template <bool HE>
hipError_t launch_split(const SplitPlan &plan, const SplitArgs &a, hipStream_t stream)
{
    switch (plan.kse) {
    case 1:
        return launch_kse<1, HE>(plan, a, stream);
    case 2:
        return launch_kse<2, HE>(plan, a, stream);
    default:
        return launch_kse<3, HE>(plan, a, stream);
    }
}

} // namespace

bool mbconv_s8_split_supports(const MbconvParams &p)
{
    return split_plan(p).ok;
}

float mbconv_s8_expand_dw_us(const MbconvParams &p)
{
    return split_plan(p).us;
}

hipError_t launch_mbconv_s8_expand_dw(const MbconvParams &p, int8_t *mid, int cu_count, hipStream_t stream)
{
    const SplitPlan plan = split_plan(p);
    if (!plan.ok)
        return hipErrorInvalidValue;
    SplitArgs a = {};
    a.p = p;
    a.mid = mid;
    a.through = writes_through((long long)p.batch * p.out_h * p.out_w * p.exp_c);
    a.tiles_x = (p.out_w + plan.tw - 1) / plan.tw;
    a.tiles_y = (p.out_h + plan.pt - 1) / plan.pt;
    const long long tiles = (long long)p.batch * a.tiles_x * a.tiles_y;
    a.n_groups = (p.exp_c + 63) / 64;
    if (tiles == 0)
        return hipSuccess;
    // As many groups per workgroup as leave four workgroups per compute unit: the patch is loaded once for all of them.
    const long long cus = cu_count > 0 ? cu_count : 256;
    a.per_wg = (int)std::min<long long>(a.n_groups, std::max<long long>(1, tiles * a.n_groups / (4 * cus)));
    if (plan.pt != (p.stride_h == 1 ? 7 : 4))
        a.per_wg = 1;
    a.parts = (a.n_groups + a.per_wg - 1) / a.per_wg;
    a.per_wg = (a.n_groups + a.parts - 1) / a.parts;
    if (tiles * a.parts > 0x7fffffff)
        return hipErrorInvalidValue;
    a.n_tiles = (int)tiles;
    a.in_bytes = p.batch * p.in_h * p.in_w * p.in_c;
    a.units = (p.in_c + 15) / 16;
    int pitch_units = a.units;
    while (pitch_units > 1 && pitch_units % 4 != 2)
        pitch_units++;
    a.pitch = 16 * pitch_units;
    a.fd_units = make_fastdiv((unsigned)a.units);
    a.fd_tiles_x = make_fastdiv((unsigned)a.tiles_x);
    a.fd_tiles_yx = make_fastdiv((unsigned)(a.tiles_x * a.tiles_y));
    a.fd_parts = make_fastdiv((unsigned)a.parts);
    return p.half_even ? launch_split<true>(plan, a, stream) : launch_split<false>(plan, a, stream);
}

} // namespace espdl
