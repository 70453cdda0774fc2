// Dense 3 x 3 int16 convolution whose input is an int8 tensor that a RequantizeLinear would have multiplied by 256, as a walk
// down the image with the filters in registers.
//
// What it computes is conv2d_33cn for int16 (esp-dl/dl/base/dl_base_conv2d.cpp:35-163 with feature_t = int16_t, buffer_t =
// int64_t) under conv_operation_shell's window clipping (esp-dl/dl/base/dl_base.hpp:940-1191), optionally followed by the
// nearest-entry table of esp-dl/dl/base/dl_base_lut.cpp:49-77.  The arithmetic is that of the X8 builds in
// conv_s16_units.hip: a weight w = 256 h + l + 128 is two signed bytes, an input value 256 x, and
//   sum x w = 65536 sum x h + 256 sum x l + 32768 sum x.
// The walk is that of conv2d_s8_walk_kernel.h at one pixel tile: a wavefront owns 16 output columns and 16 NT filters, both
// byte planes of all of them stay in registers as operand A, and every input row is read once into a ring in LDS by
// direct-to-LDS copies and serves the three output rows it belongs to.  The sums of the input bytes are four dot products
// per operand read.
//
// Bound by the matrix pipe and the epilogue, the table's lookups among it.  Against the tiled kernel, which cuts the filters
// into bytes again in every workgroup and meets a barrier per 64 products: 80 x 80 x 64 -> 64 with a table, batch 64, 51
// against 87 us, 40 x 40 21 against 27; 80 x 80 x 32 -> 32 without one 24 against 33; 40 x 40 x 128 -> 128, batch 32, 29
// against 40.  Half even takes the general epilogue, which the estimate does not know of: of 350 random layers two take more than
// 5 % longer than on the tiled kernel.
#include "conv2d_s8_walk_kernel.h"

namespace espdl {
namespace {
using namespace walk;

constexpr int kTable = 4097; // entries at most
constexpr int kWaves = 8, kThreads = 64 * kWaves;

struct X8WalkArgs {
    const int8_t *in;
    const int16_t *w, *table;
    const int64_t *bias;
    const int32_t *shift;
    int16_t *out;
    int in_bytes, in_h, in_w, in_c, in_row, in_img;
    int out_h, out_w, out_c, out_row, out_img, out_bytes; // bytes
    int batch, n_shift, relu, half_even, pad_top, pad_left, table_size, table_shift;
    int n_groups, rows_total, rows_per_group;
    FastDiv fd_p, fd_oh;
};

// The table's entry nearest to sample point v; ties as the rounding mode has them.
__device__ __forceinline__ int nearest(int v, int shift, bool half_even)
{
    const int x = (v & 0xffff) ^ 0x8000, half = 1 << (shift - 1);
    return (half_even ? x + half - 1 + ((x >> shift) & 1) : x + half) >> shift;
}

template <int CU, int NT>
struct X8Shape {
    using Rows = WalkShape<3, 1, CU, 2 * NT, false>; // two byte planes per filter tile
    static constexpr int kFilters = 3 * Rows::KS * 2 * NT;
    static constexpr long lds(int ahead) { return (long)kWaves * (ahead + 2) * Rows::kRowUnits * 16 + kFilters * 1024l + kTable * 2 + 16 * NT * 32 + 512; }
    static constexpr int AHEAD = lds(2) <= 160 * 1024 ? 2 : 1;
    static_assert(Rows::PT == 1 && lds(1) <= 160 * 1024);
};

template <int CU, int NT>
__global__ __launch_bounds__(kThreads, 2) void conv2d_s16_x8_walk_kernel(const X8WalkArgs a)
{
    using Shape = typename X8Shape<CU, NT>::Rows;
    constexpr int KS = Shape::KS, LR = Shape::kRowLoads, AHEAD = X8Shape<CU, NT>::AHEAD, kSlots = AHEAD + 2;
    constexpr int kSlot = Shape::kRowUnits * 16, LAG = 2, NACC = 3, units = 3 * CU, kStores = 1;
    __shared__ __align__(16) unsigned char ring[kWaves][kSlots][kSlot];
    __shared__ v4i filt_l[X8Shape<CU, NT>::kFilters][64];
    __shared__ __align__(16) long long bias_l[16 * NT];
    __shared__ __align__(16) v2i fast_l[16 * NT];
    __shared__ __align__(16) int shift_l[16 * NT];
    __shared__ __align__(16) int16_t table_l[kTable + 7];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int group = (int)(blockIdx.x & 7u) * (a.n_groups >> 3) + (int)(blockIdx.x >> 3);
    const int n0 = blockIdx.y * 16 * NT;
    const int r_begin = group * a.rows_per_group, r_end = min(a.rows_total, r_begin + a.rows_per_group);

    // ---- copies, AHEAD steps in front of the computation
    const unsigned ring0 = (unsigned)reinterpret_cast<uintptr_t>(&ring[wave][0][0]);
    int vin[LR];
#pragma unroll
    for (int j = 0; j < LR; j++)
        vin[j] = kParked;
    int f_r = r_begin, f_row = 0, f_left = 0;
    unsigned f_slot = 0;
    const auto feed_segment = [&]() __attribute__((always_inline)) {
        const int g = (int)fastdiv((unsigned)f_r, a.fd_oh);
        const int y0 = f_r - g * a.out_h;
        const int rows = min(a.out_h - y0, r_end - f_r);
        f_r += rows;
        f_left = rows + LAG;
        f_row = y0 - a.pad_top;
        const int c0 = (g * kWaves + wave) * 16;
        int lane_now = lane; // (through an empty asm statement: nothing of this is kept in registers between segments)
        asm volatile("" : "+v"(lane_now));
#pragma unroll
        for (int j = 0; j < LR; j++) {
            const int e = j * 64 + lane_now, i = e / CU, u = (e - i * CU) ^ Shape::swz(i);
            const int q = c0 - a.pad_left + i;
            const int n = (int)fastdiv((unsigned)max(q, 0), a.fd_p);
            const int x = q - n * (int)a.fd_p.d;
            vin[j] = q >= 0 && n < a.batch && x < a.in_w ? n * a.in_img + x * a.in_c + 16 * u : kParked;
        }
    };
    const auto feed = [&]() __attribute__((always_inline)) { // one step; past the last one nothing is read (the counts stay the same)
        if (f_left == 0 && f_r < r_end)
            feed_segment();
        const bool live = f_left > 0, ok = live && (unsigned)f_row < (unsigned)a.in_h;
        const unsigned base = __builtin_amdgcn_readfirstlane(ring0 + f_slot);
        const int off = __builtin_amdgcn_readfirstlane(ok ? f_row * a.in_row : 0);
        const __amdgpu_buffer_rsrc_t rs = rsrc_of(a.in + off, __builtin_amdgcn_readfirstlane(ok ? a.in_bytes - off : 0));
#pragma unroll
        for (int j = 0; j < LR; j++)
            if (Shape::kRowUnits - 64 * j >= 64 || lane < Shape::kRowUnits - 64 * j)
                copy_to_lds(base + j * 1024, vin[j], rs);
        f_row++;
        f_left -= live ? 1 : 0;
        f_slot = f_slot + kSlot == kSlots * kSlot ? 0 : f_slot + kSlot;
    };
    const auto no_stores = [&]() __attribute__((always_inline)) { // dropped: the number of instructions behind a copy is known in every step
        asm volatile("s_nop 4\n\tbuffer_store_byte %0, %0, %1, 0 offen" ::"v"(kParked), "s"(rsrc_of(reinterpret_cast<const int8_t *>(a.out), 0)) : "memory");
    };
#pragma unroll
    for (int i = 0; i <= AHEAD; i++) {
        feed();
        no_stores();
    }

    // ---- set-up: byte planes of the filters in operand-A order.  Row i of tile t is filter 4 NT (i / 4) + 4 t + i % 4 of the
    // chunk: a lane ends up with 4 NT neighbouring channels.
    {
        constexpr int total = 3 * KS * NT, N = (total + kWaves - 1) / kWaves;
        v4i lo[N], hi[N];
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int e = min(wave + i * kWaves, total - 1), t = e % NT, ks = e / NT, ky = ks / KS, u = min(4 * (ks - ky * KS) + quad, units - 1);
            const int oc = min(n0 + 4 * NT * (col >> 2) + 4 * t + (col & 3), a.out_c - 1), tap = u / CU;
            const int16_t *src = a.w + ((long long)oc * 9 + ky * 3 + tap) * (16 * CU) + 16 * (u - tap * CU);
            lo[i] = *reinterpret_cast<const v4i_unaligned *>(src);
            hi[i] = *reinterpret_cast<const v4i_unaligned *>(src + 8);
        }
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int e = wave + i * kWaves, t = e % NT, ks = e / NT, s = ks % KS;
            v4i h, l;
#pragma unroll
            for (int d = 0; d < 2; d++) {
                h[d] = (int)__builtin_amdgcn_perm((unsigned)lo[i][2 * d + 1], (unsigned)lo[i][2 * d], 0x07050301u);
                h[d + 2] = (int)__builtin_amdgcn_perm((unsigned)hi[i][2 * d + 1], (unsigned)hi[i][2 * d], 0x07050301u);
                l[d] = (int)__builtin_amdgcn_perm((unsigned)lo[i][2 * d + 1], (unsigned)lo[i][2 * d], 0x06040200u) ^ (int)0x80808080u;
                l[d + 2] = (int)__builtin_amdgcn_perm((unsigned)hi[i][2 * d + 1], (unsigned)hi[i][2 * d], 0x06040200u) ^ (int)0x80808080u;
            }
            if (4 * s + quad >= units) // past the window
                h = l = v4i{0, 0, 0, 0};
            if (e < total) {
                filt_l[ks * 2 * NT + 2 * t][lane] = h;
                filt_l[ks * 2 * NT + 2 * t + 1][lane] = l;
            }
        }
    }
    if (a.table != nullptr)
        for (int i = tid; i < a.table_size; i += kThreads)
            table_l[i] = a.table[i];
    // The short epilogue, as in conv_s16_units.hip: with C = bias + 32768 sum x + 2^(s-1) = 65536 Ch + Cl,
    //   floor((65536 HH + 256 M + C) / 65536) = HH + Ch + floor((M + floor(Cl / 256)) / 256)
    // in 32-bit arithmetic, shifted by the rest where s >= 16.
    int fine = 1, low = 0;
    if (tid < 16 * NT) {
        const int n = min(n0 + tid, a.out_c - 1), s = a.shift[a.n_shift == 1 ? 0 : n];
        const long long c = a.bias != nullptr ? a.bias[n] : 0;
        fine = !a.half_even && s >= 1 && s <= 44 && c < (1ll << 45) && c > -(1ll << 45);
        low = s < 16;
        const long long r = c + (1ll << ((s - 1) & 63));
        bias_l[tid] = c;
        fast_l[tid] = v2i{(int)(r >> 16), (int)(r & 0xffff)};
        shift_l[tid] = s;
    }
    const bool fast = __syncthreads_and(fine) != 0, any_low = __syncthreads_or(low) != 0;
    v4i A[3][KS][2 * NT]; // operand A of the whole reduction, in registers for the life of the wavefront
#pragma unroll
    for (int ky = 0; ky < 3; ky++)
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int t = 0; t < 2 * NT; t++)
                A[ky][s][t] = filt_l[(ky * KS + s) * 2 * NT + t][lane];
    int boff[KS];
#pragma unroll
    for (int s = 0; s < KS; s++) {
        const int u = min(4 * s + quad, units - 1), tap = u / CU, i = col + tap;
        boff[s] = 16 * (i * CU + ((u - tap * CU) ^ Shape::swz(i)));
    }
    const unsigned char *my_ring = &ring[wave][0][0];
    unsigned b_slot = 0;

    // ---- the walk
    int vout = kParked;
    int c_r = r_begin, c_left = 0, c_y = 0; // c_y: output row that the current step finishes, relative to the segment
    int c_soff = 0;
    int left = 0;
    for (int r = r_begin; r < r_end;) {
        const int g = (int)fastdiv((unsigned)r, a.fd_oh), e = min(r_end, (g + 1) * a.out_h);
        left += e - r + LAG;
        r = e;
    }
    const auto segment = [&]() __attribute__((always_inline)) {
        const int g = (int)fastdiv((unsigned)c_r, a.fd_oh);
        const int y0 = c_r - g * a.out_h;
        const int rows = min(a.out_h - y0, r_end - c_r);
        c_r += rows;
        c_left = rows + LAG;
        c_y = -LAG;
        c_soff = (y0 - LAG) * a.out_row;
        int lane_now = lane;
        asm volatile("" : "+v"(lane_now));
        const int v = (g * kWaves + wave) * 16 + (lane_now & 15);
        const int n = (int)fastdiv((unsigned)v, a.fd_p);
        const int x = v - n * (int)a.fd_p.d, oc = n0 + 4 * NT * (lane_now >> 4);
        vout = n < a.batch && x < a.out_w && oc < a.out_c ? n * a.out_img + (x * a.out_c + oc) * 2 : kParked;
    };
    v4i acc[NACC][2 * NT];
    int sum[NACC]; // of the input bytes under the window, this lane's units
#pragma unroll
    for (int i = 0; i < NACC; i++) {
        sum[i] = 0;
#pragma unroll
        for (int t = 0; t < 2 * NT; t++)
            acc[i][t] = v4i{0, 0, 0, 0};
    }
    const auto step = [&](auto tag) __attribute__((always_inline)) {
        constexpr int R = decltype(tag)::value;
        constexpr int NEW = R % NACC, FIN = (R + NACC - LAG) % NACC;
        if (c_left == 0)
            segment();
        c_left--;
#pragma unroll
        for (int t = 0; t < 2 * NT; t++)
            acc[NEW][t] = v4i{0, 0, 0, 0};
        wait_copies<AHEAD * (LR + kStores) + kStores>(); // this step's input has arrived
        const unsigned char *slot = my_ring + b_slot;
        b_slot = b_slot + kSlot == kSlots * kSlot ? 0 : b_slot + kSlot;
        feed();
        int row_sum = 0;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const v4i b = *reinterpret_cast<const v4i *>(slot + boff[s]);
#pragma unroll
            for (int ky = 2; ky >= 0; ky--) {
                const int idx = (R - ky + 3 * NACC) % NACC;
#pragma unroll
                for (int t = 0; t < 2 * NT; t++)
                    acc[idx][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[ky][s][t], b, acc[idx][t], 0, 0, 0);
            }
            const int ones = 4 * s + 3 < units || 4 * s + quad < units ? 0x01010101 : 0;
#pragma unroll
            for (int d = 0; d < 4; d++)
                row_sum = __builtin_amdgcn_sdot4(b[d], ones, row_sum, false);
        }
        sum[NEW] = row_sum;
        sum[(R + 2) % NACC] += row_sum; // row y - 1
        sum[(R + 1) % NACC] += row_sum; // row y - 2
        if (c_y >= 0) {
            int total = sum[FIN];
            total += __shfl_xor(total, 16);
            total += __shfl_xor(total, 32);
            int words[2 * NT];
            const auto finish = [&](auto low_tag) __attribute__((always_inline)) {
                constexpr bool LOW = decltype(low_tag)::value;
                const v2s floor2 = __builtin_bit_cast(v2s, a.relu != 0 ? 0 : (int)0x80008000u);
                const int ph = total >> 1, pl = (total & 1) << 15;
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const v4i s4 = *reinterpret_cast<const v4i *>(&shift_l[4 * NT * quad + 4 * t]);
                    const v4i c01 = *reinterpret_cast<const v4i *>(&fast_l[4 * NT * quad + 4 * t]);
                    const v4i c23 = *reinterpret_cast<const v4i *>(&fast_l[4 * NT * quad + 4 * t + 2]);
                    int q[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int fh = r < 2 ? c01[2 * r] : c23[2 * (r - 2)], fl = r < 2 ? c01[2 * r + 1] : c23[2 * (r - 2) + 1];
                        const int l = fl + pl, mid = acc[FIN][2 * t + 1][r] + (l >> 8);
                        const int x = acc[FIN][2 * t][r] + fh + ph + (mid >> 8);
                        if constexpr (LOW) {
                            const int top = min(max(x, -32768), 32767);
                            const int v = (top << 16) | ((mid & 255) << 8) | (l & 255);
                            q[r] = s4[r] < 16 ? v >> s4[r] : x >> (s4[r] - 16);
                        } else {
                            q[r] = x >> (s4[r] - 16);
                        }
                    }
                    words[2 * t] = __builtin_bit_cast(int, __builtin_elementwise_max(__builtin_amdgcn_cvt_pk_i16(q[0], q[1]), floor2));
                    words[2 * t + 1] = __builtin_bit_cast(int, __builtin_elementwise_max(__builtin_amdgcn_cvt_pk_i16(q[2], q[3]), floor2));
                }
            };
            if (!fast) {
                const bool relu = a.relu != 0, half_even = a.half_even != 0;
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    int q[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int f = 4 * NT * quad + 4 * t + r;
                        const long long v = bias_l[f] + 32768ll * total + ((long long)acc[FIN][2 * t][r] << 16) + ((long long)acc[FIN][2 * t + 1][r] << 8);
                        q[r] = requant_s16(v, shift_l[f], relu, half_even);
                    }
                    words[2 * t] = (q[0] & 0xffff) | (q[1] << 16);
                    words[2 * t + 1] = (q[2] & 0xffff) | (q[3] << 16);
                }
            } else if (any_low) {
                finish(std::true_type{});
            } else {
                finish(std::false_type{});
            }
            if (a.table != nullptr) {
#pragma unroll
                for (int i = 0; i < 2 * NT; i++) {
                    const int lo = nearest(words[i], a.table_shift, a.half_even != 0), hi = nearest(words[i] >> 16, a.table_shift, a.half_even != 0);
                    const v2s entries = {table_l[lo], table_l[hi]};
                    words[i] = __builtin_bit_cast(int, entries);
                }
            }
            const __amdgpu_buffer_rsrc_t rs = rsrc_of(reinterpret_cast<const int8_t *>(a.out) + c_soff, a.out_bytes - c_soff);
            if constexpr (NT == 2)
                __builtin_amdgcn_raw_buffer_store_b128(v4u{(unsigned)words[0], (unsigned)words[1], (unsigned)words[2], (unsigned)words[3]}, rs, vout, 0, 0);
            else
                __builtin_amdgcn_raw_buffer_store_b64(v2u{(unsigned)words[0], (unsigned)words[1]}, rs, vout, 0, 0);
        } else {
            no_stores();
        }
        c_y++;
        c_soff += a.out_row;
    };
    while (left > 0) { // the accumulators' roles rotate with the steps
        step(std::integral_constant<int, 0>{});
        if (--left == 0)
            break;
        step(std::integral_constant<int, 1>{});
        if (--left == 0)
            break;
        step(std::integral_constant<int, 2>{});
        left--;
    }
}

struct X8WalkPlan {
    bool ok;
    int cu, nt;
    X8WalkArgs a;
};

X8WalkPlan x8_walk_plan(const ConvGeom &g, const void *in, const void *out, int table_size, int cus)
{
    X8WalkPlan plan = {};
    plan.cu = g.in_c / 16;
    plan.nt = plan.cu <= 4 ? 2 : 1;
    if (g.k_h != 3 || g.k_w != 3 || g.stride_h != 1 || g.stride_w != 1 || g.dil_h != 1 || g.dil_w != 1 || !conv_is_dense(g) || g.in_c % 16 != 0 ||
        plan.cu < 1 || plan.cu > 8 || plan.cu == 5 || plan.cu == 7 || g.out_c % (4 * plan.nt) != 0 || table_size > kTable || g.batch <= 0 ||
        g.out_h <= 0 || g.out_w <= 0 || (reinterpret_cast<uintptr_t>(in) & 15) != 0 || (reinterpret_cast<uintptr_t>(out) & 15) != 0)
        return plan;
    const long long most = (1ll << 31) - 65536;
    const long long in_bytes = (long long)g.batch * g.in_h * g.in_w * g.in_c, out_bytes = 2ll * g.batch * g.out_h * g.out_w * g.out_c;
    const long long over = (long long)(g.out_w - 1) + 2 - g.pad_left - (g.in_w - 1);
    const long long pitch = std::max<long long>(g.in_w + std::max<long long>({0, g.pad_left, over}), g.out_w);
    const long long cols = (g.batch - 1) * pitch + g.out_w, groups = (cols + 16 * kWaves - 1) / (16 * kWaves);
    if (in_bytes >= most || out_bytes >= most || g.batch * pitch + 4096 >= most || groups * g.out_h >= (1ll << 30))
        return plan;
    X8WalkArgs &a = plan.a;
    a.in_bytes = (int)in_bytes;
    a.in_h = g.in_h;
    a.in_w = g.in_w;
    a.in_c = g.in_c;
    a.in_row = g.in_w * g.in_c;
    a.in_img = a.in_row * g.in_h;
    a.out_h = g.out_h;
    a.out_w = g.out_w;
    a.out_c = g.out_c;
    a.out_row = 2 * g.out_w * g.out_c;
    a.out_img = a.out_row * g.out_h;
    a.out_bytes = (int)out_bytes;
    a.batch = g.batch;
    a.n_shift = g.n_shift;
    a.relu = g.relu;
    a.half_even = g.half_even;
    a.pad_top = g.pad_top;
    a.pad_left = g.pad_left;
    a.fd_p = make_fastdiv((unsigned)pitch);
    a.fd_oh = make_fastdiv((unsigned)g.out_h);
    // one workgroup per compute unit over the chunks of filters, each with the same number of rows of the column groups
    const int chunks = (g.out_c + 16 * plan.nt - 1) / (16 * plan.nt), want = std::max(8, cus / chunks / 8 * 8);
    a.rows_total = (int)(groups * g.out_h);
    a.rows_per_group = (a.rows_total + want - 1) / want;
    a.n_groups = ((a.rows_total + a.rows_per_group - 1) / a.rows_per_group + 7) / 8 * 8;
    plan.ok = true;
    return plan;
}

template <int CU, int NT>
hipError_t launch_one(const X8WalkPlan &plan, hipStream_t stream)
{
    const dim3 grid((unsigned)plan.a.n_groups, (unsigned)((plan.a.out_c + 16 * NT - 1) / (16 * NT)));
    hipLaunchKernelGGL((conv2d_s16_x8_walk_kernel<CU, NT>), grid, dim3(kThreads), 0, stream, plan.a);
    return hipGetLastError();
}

} // namespace

// Set-up and one workgroup's steps (fifteen layers of 1 to 64 images, within 20 %).
float conv2d_s16_x8_walk_us(const ConvGeom &g, const void *in, const void *out, int table_size, int cu_count)
{
    const X8WalkPlan plan = x8_walk_plan(g, in, out, table_size, cu_count > 0 ? cu_count : 256);
    if (!plan.ok)
        return 1e30f;
    const X8WalkArgs &a = plan.a;
    const float steps = (float)a.rows_per_group + 2.f * (1.f + (float)(a.rows_per_group - 1) / (float)a.out_h);
    const float products = (float)(6 * ((3 * plan.cu + 3) / 4) * plan.nt);
    return 6.f + steps * (0.2f + 0.0155f * products + (float)plan.nt * (table_size > 0 ? 0.38f : 0.2f));
}

hipError_t launch_conv2d_s16_x8_walk(const ConvGeom &g, const int8_t *in, const int16_t *filter, const int64_t *bias, const int32_t *shift,
                                     const int16_t *table, int table_size, int table_shift, int16_t *out, int cu_count, hipStream_t stream)
{
    X8WalkPlan plan = x8_walk_plan(g, in, out, table_size, cu_count > 0 ? cu_count : 256);
    if (!plan.ok)
        return hipErrorInvalidValue;
    X8WalkArgs &a = plan.a;
    a.in = in;
    a.w = filter;
    a.bias = bias;
    a.shift = shift;
    a.table = table;
    a.table_size = table_size;
    a.table_shift = table_shift;
    a.out = out;
    switch (plan.cu) {
    case 1:
        return launch_one<1, 2>(plan, stream);
    case 2:
        return launch_one<2, 2>(plan, stream);
    case 3:
        return launch_one<3, 2>(plan, stream);
    case 4:
        return launch_one<4, 2>(plan, stream);
    case 6:
        return launch_one<6, 1>(plan, stream);
    default:
        return launch_one<8, 1>(plan, stream);
    }
}

} // namespace espdl
