// The core of a quantized attention block as one kernel for gfx950: q^T x k -> [x constant] -> Softmax -> quantize to
// int8 -> v x attn^T, for every head of every image, read straight from the [batch][positions][channels] tensor the
// 1x1 convolution in front leaves and written as [batch][positions][heads * head_dim].
//
// Operator by operator this is two layout changes of the convolution's output, a Split, MatMul, Mul, Softmax (with a
// float32 tensor four times the size of the scores), QuantizeLinear, three more layout changes and MatMul
// (esp-dl/dl/module/include/dl_module_matmul.hpp, dl_module_mul.hpp, dl_module_softmax.hpp:148-217,
// esp-dl/dl/tensor/src/dl_tensor_base.cpp:251-268): thirteen launches and a dozen passes over positions^2 scores.
// Every value is formed here exactly as those operators form it:
//   score  = clamp(act(shift_round(sum_d q[i][d] * k[j][d], qk_shift)))
//   T[x]   = expf(2^e * x), with the multiplication by a constant folded into the index of the table: T[requant(x * c)]
//   prob   = saturate(round_half_up((T / sum_j T) * 2^-prob_exp)), the sum in float32 in index order
//   out    = clamp(act(shift_round(sum_j prob[i][j] * v[j][d], av_shift)))
//
// A workgroup of eight wavefronts owns 64 query positions of one head; neither scores nor probabilities leave it.
//   1. Per chunk of 64 keys a pair of wavefronts (half of the keys each) multiplies k (operand A, rows = keys) by q
//      (operand B, columns = 16 queries): a lane then holds four neighbouring keys of one query, requantizes them and
//      looks them up in the table.  The table values stay in registers for step 2 and go to LDS as float32, where one
//      wavefront in turn adds a chunk in index order, a query per lane, while the others work on the next chunk.
//   2. The registers become probabilities.  The exact result is an IEEE division, but only its rounding to int8 is
//      kept: a product with the reciprocal decides it unless it lies within 2^-18 of a rounding boundary; there the lane
//      divides.
//   3. v is brought in by the whole workgroup, as many positions as fit where the table values lay (512 of them at 64 channels),
//      transposed in registers on its way into LDS, and multiplied by the probabilities, a half of the head's channels per
//      wavefront of a pair.  A tile's operand-A row m is channel (m / 4) * 4 HT + 4 t + m % 4 of the head, so a lane ends with
//      neighbouring channels of one position.
// Not bound by memory or the matrix pipe; two workgroups fit on a compute unit.  Of 9.6 us with 400 positions and one image (two heads
// of 32 + 32 + 64 channels) the scores take 4.2, in which one wavefront's additions and its next scores follow each other seven
// times (without additions 3.1, without lookups either 2.5), the probabilities 1.1, v and its product 1.2; 64 heads 13.5 (launch to
// launch one image takes 10.4, eight 11.2, 64 heads 14.9, 15.3 on inputs that change), the operators one by one 117 us.  With v a chunk of 64 and a barrier at a time, the epilogue's form chosen at run time and divisions out of line
// one image took 10.7 us, eight 11.3 (10.6 now), 64 heads 14.3.  Tried: a wavefront that owns 16 queries and all keys, sums passed from
// row to row by v_permlane swaps, k and v in LDS, no barriers (9.5 us for one image, 15 for 64 heads: four times the additions); three
// chunks of k on their way (14.0); four wavefronts that each owned 16 queries and re-read their scores from LDS (18.3), a ninth
// wavefront that only adds (17.7).
#include "conv_window.h"

namespace espdl {
namespace {

constexpr int kThreads = 512, kQueries = 64;
constexpr int kSumStride = 68; // floats per query row of the table values: 4 mod 64 banks, rows apart

struct Args {
    AttentionParams p;
    int prob_stride;  // bytes per row of probabilities: positions rounded up to 64, + 16 so that rows start in different banks
    int chunks;       // of 64 positions
    int v_chunks;     // of v in LDS at a time
    int v_stride;     // bytes per channel row of transposed v: 64 v_chunks + 16, 16 rows of 16 bytes hit distinct banks
    int av_mode;      // of the second product's epilogue, see requant4
    FastDiv fd_n16;   // 16-byte pieces of a head's values
    float inv_scale;
    float table[256];
};

// Four accumulators requantized and packed.  MODE 0: short epilogue, half up; 1: short, half even; both hold 2^(s-1) (- 1) already;
// 2: general.
template <int MODE>
__device__ __forceinline__ int requant4(const v4i &acc, int shift, int relu, int half_even)
{
    if constexpr (MODE == 2) {
        int q[4];
#pragma unroll
        for (int e = 0; e < 4; e++)
            q[e] = requant_s8(acc[e], shift, relu != 0, half_even != 0);
        return pack4_s8(q[0], q[1], q[2], q[3]);
    } else {
        const int l = max(0, 8 - shift), r = shift - 8 + l;
        return pack_fast4<MODE == 0 ? 1 : 5>(acc, v4i{l, l, l, l}, v4i{r, r, r, r}, relu ? 0 : (int)0x80008000u);
    }
}
__device__ __forceinline__ v4i start4(int mode, int shift)
{
    const int v = mode == 2 ? 0 : (1 << (shift - 1)) - (mode == 1 ? 1 : 0);
    return v4i{v, v, v, v};
}

// QuantizeLinear of four elements of Softmax.
__device__ __forceinline__ unsigned divide4(const float4 &e, float sum, float inv_scale)
{
    const float v[4] = {e.x, e.y, e.z, e.w};
    int q[4];
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const float quotient = v[b] / sum;
        q[b] = min(max(round_half_up_f32(quotient * inv_scale), -128), 127);
    }
    return (unsigned)pack4_s8(q[0], q[1], q[2], q[3]);
}

// HT: 16-channel tiles of a head's values (head_dim <= 16 HT, even).
// CH: chunks whose table values a lane keeps in registers (positions <= 64 CH).
template <int HT, int CH, int MODE>
__global__ __launch_bounds__(kThreads) void attention_s8_kernel(const Args a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    float *table = reinterpret_cast<float *>(smem);
    float *sums = table + 256;
    unsigned char *probs = smem + (256 + kQueries) * sizeof(float);
    unsigned char *scratch = probs + kQueries * a.prob_stride; // table values of two chunks, later transposed v
    const AttentionParams &p = a.p;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int pair = wave & 3, half = wave >> 2; // 16 queries, half of the keys of a chunk
    const int L = p.positions, C = p.channels;
    const int image = blockIdx.y / p.heads, head = blockIdx.y - image * p.heads;
    const __amdgpu_buffer_rsrc_t qkv = window::tensor_rsrc(p.qkv + (long long)image * L * C, L * C);
    const int ch0 = head * p.head_pitch;
    const int i0 = blockIdx.x * kQueries + pair * 16; // the wavefront's first query
    unsigned char *prob_row = probs + (pair * 16 + r) * a.prob_stride;

    if (tid < 256) {
        int q = tid - 128;
        if (p.mul_constant)
            q = requant_s8(q * (int)*p.mul_constant, p.mul_shift, false, p.half_even != 0);
        table[tid] = a.table[q + 128];
    }
    // v alone, for whoever reads it besides the product
    if (p.v_out) {
        const int n16 = p.head_dim >> 4;
        for (int e = tid; e < kQueries * n16; e += kThreads) {
            const int row = (int)fastdiv((unsigned)e, a.fd_n16), at = e - row * n16, pos = blockIdx.x * kQueries + row;
            if (pos < L)
                *reinterpret_cast<v4i *>(p.v_out + ((long long)image * L + pos) * (p.heads * p.head_dim) + head * p.head_dim + 16 * at) =
                    __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(qkv, pos * C + ch0 + p.v_offset + 16 * at, 0, 0));
        }
    }

    // positions past the end of the image lie past the descriptor's end and read as zeros
    const bool has_channels = 16 * g < p.key_dim;
    const auto load = [&](int pos, int offset) {
        return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                           qkv, has_channels ? pos * C + ch0 + offset + 16 * g : window::kParked, 0, 0));
    };
    const v4i qf = load(i0 + r, p.q_offset);
    v4i kf[2];
    kf[0] = load(32 * half + r, p.k_offset);
    kf[1] = load(32 * half + 16 + r, p.k_offset);
    const v4i qk_start = start4(MODE, p.qk_shift);
    float4 kept[CH][2]; // table values of the lane's keys 64 c + 32 half + 16 t + 4 g + (0 .. 3), query r
    __syncthreads();    // the table is there
#pragma unroll
    for (int c = 0; c < CH; c++) {
        if (c < a.chunks) {
            v4i acc[2];
#pragma unroll
            for (int t = 0; t < 2; t++)
                acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf[t], qf, qk_start, 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 2; t++) // (past the last chunk: zeros nobody reads)
                kf[t] = load(64 * (c + 1) + 32 * half + 16 * t + r, p.k_offset);
            int s[2];
#pragma unroll
            for (int t = 0; t < 2; t++)
                s[t] = requant4<MODE>(acc[t], p.qk_shift, p.qk_relu, p.half_even);
            const int n0 = L - (64 * c + 32 * half + 4 * g); // keys of the image from the lane's first on
            float *to = reinterpret_cast<float *>(scratch) + ((c & 1) * kQueries + pair * 16 + r) * kSumStride + 32 * half + 4 * g;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const unsigned index = (unsigned)s[t] ^ 0x80808080u; // q + 128
                float4 e;
                e.x = table[index & 255];
                e.y = table[(index >> 8) & 255];
                e.z = table[(index >> 16) & 255];
                e.w = table[index >> 24];
                if (64 * c + 64 > L) { // keys that do not exist add +0, which changes no sum, and weigh nothing
                    const int n = n0 - 16 * t;
                    e.x = n > 0 ? e.x : 0.f;
                    e.y = n > 1 ? e.y : 0.f;
                    e.z = n > 2 ? e.z : 0.f;
                    e.w = n > 3 ? e.w : 0.f;
                }
                kept[c][t] = e;
                *reinterpret_cast<float4 *>(to + 16 * t) = e;
            }
            __syncthreads();
            // One wavefront in turn adds the chunk, a query per lane, while the others go on: the half of the scratch it
            // reads is written again behind the next barrier, which also orders the sum's way to the next wavefront.
            if (wave == (c & 7)) {
                const float *from = reinterpret_cast<const float *>(scratch) + ((c & 1) * kQueries + lane) * kSumStride;
                float sum = c == 0 ? 0.f : sums[lane];
#pragma unroll
                for (int j = 0; j < 16; j++) {
                    const float4 e = *reinterpret_cast<const float4 *>(from + 4 * j);
                    sum += e.x;
                    sum += e.y;
                    sum += e.z;
                    sum += e.w;
                }
                sums[lane] = sum;
            }
        }
    }

    // v, as much of it as fits where the table values lay: a piece is eight channels of four positions, transposed in registers on
    // its way, two pieces a thread at a time.  The first ones arrive while the last chunk is added and the probabilities are formed.
    constexpr int kPerChunk = 2 * HT * 16; // pieces of a chunk of 64 positions
    const int v_at = tid % (2 * HT);       // the thread's eight channels
    v2i vr[2][4];
    const auto load_values = [&](int first, int end) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int piece = first + j * kThreads;
            const int off = 8 * v_at < p.head_dim && piece < end ? 4 * (piece / (2 * HT)) * C + ch0 + p.v_offset + 8 * v_at : window::kParked;
#pragma unroll
            for (int e = 0; e < 4; e++)
                vr[j][e] = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(qkv, off + e * C, 0, 0));
        }
    };
    const auto place_values = [&](int first, int end, int first_chunk) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int piece = first + j * kThreads;
#pragma unroll
            for (int d = 0; d < 2; d++) {
                if (piece >= end)
                    continue;
                // channel 4 db + e of the head is row (db % HT) * 16 + (db / HT) * 4 + e
                const int db = 2 * v_at + d;
                unsigned char *const dst = scratch + ((db % HT) * 16 + (db / HT) * 4) * a.v_stride + 4 * (piece / (2 * HT)) - 64 * first_chunk;
                const unsigned t0 = __builtin_amdgcn_perm((unsigned)vr[j][1][d], (unsigned)vr[j][0][d], 0x05010400u);
                const unsigned t1 = __builtin_amdgcn_perm((unsigned)vr[j][1][d], (unsigned)vr[j][0][d], 0x07030602u);
                const unsigned u0 = __builtin_amdgcn_perm((unsigned)vr[j][3][d], (unsigned)vr[j][2][d], 0x05010400u);
                const unsigned u1 = __builtin_amdgcn_perm((unsigned)vr[j][3][d], (unsigned)vr[j][2][d], 0x07030602u);
                *reinterpret_cast<unsigned *>(dst) = __builtin_amdgcn_perm(u0, t0, 0x05040100u);
                *reinterpret_cast<unsigned *>(dst + a.v_stride) = __builtin_amdgcn_perm(u0, t0, 0x07060302u);
                *reinterpret_cast<unsigned *>(dst + 2 * a.v_stride) = __builtin_amdgcn_perm(u1, t1, 0x05040100u);
                *reinterpret_cast<unsigned *>(dst + 3 * a.v_stride) = __builtin_amdgcn_perm(u1, t1, 0x07060302u);
            }
        }
    };
    load_values(tid, min(a.v_chunks, a.chunks) * kPerChunk);
    __syncthreads(); // the sums are there, the table values are done with

    // Probabilities.  v_cvt_pk_u8_f32 rounds to nearest and saturates at 255; the two factors bracket the exact one by
    // 2^-18, so a byte both agree on is the exact quotient's rounding (a tie, where half up and to nearest part, lies
    // between them), and one they do not agree on is divided out.
    const float sum = sums[pair * 16 + r];
    const bool short_sum = sum >= 0x1p-60f && sum <= 0x1p60f;
    const float factor = short_sum ? __builtin_amdgcn_rcpf(sum) * a.inv_scale : 0.f;
    const float factor_lo = factor * (1.f - 0x1p-18f), factor_hi = factor * (1.f + 0x1p-18f);
#pragma unroll
    for (int c = 0; c < CH; c++) {
        if (c < a.chunks) {
            unsigned w[2], differ = 0;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const float e[4] = {kept[c][t].x, kept[c][t].y, kept[c][t].z, kept[c][t].w};
                unsigned lo = 0, hi = 0;
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    lo = __builtin_amdgcn_cvt_pk_u8_f32(e[b] * factor_lo, b, lo);
                    hi = __builtin_amdgcn_cvt_pk_u8_f32(e[b] * factor_hi, b, hi);
                }
                const unsigned over = lo & 0x80808080u; // 128 .. 255 become 127
                w[t] = (lo | (over - (over >> 7))) & 0x7f7f7f7fu;
                differ |= lo ^ hi;
            }
            if (differ != 0 || !short_sum)
#pragma unroll
                for (int t = 0; t < 2; t++)
                    w[t] = divide4(kept[c][t], sum, a.inv_scale);
#pragma unroll
            for (int t = 0; t < 2; t++)
                *reinterpret_cast<unsigned *>(prob_row + 64 * c + 32 * half + 16 * t + 4 * g) = w[t];
        }
    }

    const v4i av_start = start4(a.av_mode, p.av_shift);
    v4i acc[HT / 2];
#pragma unroll
    for (int t = 0; t < HT / 2; t++)
        acc[t] = av_start;
    for (int c0 = 0; c0 < a.chunks; c0 += a.v_chunks) {
        const int c1 = min(c0 + a.v_chunks, a.chunks), end = c1 * kPerChunk;
        if (c0 != 0) {
            __syncthreads(); // the chunks before have been read
            load_values(c0 * kPerChunk + tid, end);
        }
        for (int piece = c0 * kPerChunk + tid; piece - tid < end; piece += 2 * kThreads) {
            place_values(piece, end, c0);
            if (piece - tid + 2 * kThreads < end) // uniform
                load_values(piece + 2 * kThreads, end);
        }
        __syncthreads();
        const unsigned char *const row = scratch + (16 * half * (HT / 2) + r) * a.v_stride + 16 * g;
        for (int c = c0; c < c1; c++) {
            const v4i pf = *reinterpret_cast<const v4i *>(prob_row + 64 * c + 16 * g);
#pragma unroll
            for (int t = 0; t < HT / 2; t++) {
                const v4i vf = *reinterpret_cast<const v4i *>(row + 16 * t * a.v_stride + 64 * (c - c0));
                acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(vf, pf, acc[t], 0, 0, 0);
            }
        }
    }
    const int i = i0 + r;
    if (i < L) {
        const int d0 = g * 4 * HT + half * 2 * HT;
        int8_t *dst = p.out + ((long long)image * L + i) * (p.heads * p.head_dim) + head * p.head_dim + d0;
        int word[HT / 2];
#pragma unroll
        for (int t = 0; t < HT / 2; t++)
            word[t] = a.av_mode == 0 ? requant4<0>(acc[t], p.av_shift, p.av_relu, 0) // (uniform)
                : a.av_mode == 1     ? requant4<1>(acc[t], p.av_shift, p.av_relu, 1)
                                     : requant4<2>(acc[t], p.av_shift, p.av_relu, p.half_even);
#pragma unroll
        for (int t = 0; t < HT / 2; t++)
            if (d0 + 4 * t < p.head_dim)
                *reinterpret_cast<int *>(dst + 4 * t) = word[t];
    }
}

// Bytes where the table values of two chunks lie, then v: more than that only where a single chunk of v needs it.
size_t scratch_bytes(int ht)
{
    return std::max((size_t)16 * ht * (64 + 16), sizeof(float) * 2 * kQueries * kSumStride);
}
int value_tiles(int head_dim)
{
    return head_dim <= 32 ? 2 : head_dim <= 64 ? 4 : 8;
}

// The short epilogue: shifts of 1..31 whose start value and left-shifted sum stay inside int32.
int epilogue_mode(int shift, int half_even, long long mac_bound)
{
    if (shift < 1 || shift > 31 || mac_bound + (1ll << (shift - 1)) >= 1ll << (31 - std::max(0, 8 - shift)))
        return 2;
    return half_even ? 1 : 0;
}

template <int HT>
auto pick_kernel(int chunks, int mode)
{
    if (chunks <= 8)
        return mode == 0 ? attention_s8_kernel<HT, 8, 0> : mode == 1 ? attention_s8_kernel<HT, 8, 1> : attention_s8_kernel<HT, 8, 2>;
    return mode == 0 ? attention_s8_kernel<HT, 16, 0> : mode == 1 ? attention_s8_kernel<HT, 16, 1> : attention_s8_kernel<HT, 16, 2>;
}

} // namespace

// Whole 16-byte pieces of every operand (key_dim one MFMA step, head_dim up to 128 accumulator registers' worth), and
// table values that fit the registers (64 VGPRs to 512 positions, 128 to 1024).
bool attention_s8_supports(const AttentionParams &p)
{
    return p.key_dim > 0 && p.key_dim <= 64 && p.head_dim > 0 && p.head_dim <= 128 && p.positions > 0 && p.heads > 0 &&
        ((p.key_dim | p.head_dim | p.channels | p.head_pitch | p.q_offset | p.k_offset | p.v_offset) & 15) == 0 &&
        (long long)p.heads * p.head_pitch <= p.channels && p.heads <= 65535 && p.q_offset + p.key_dim <= p.head_pitch &&
        p.k_offset + p.key_dim <= p.head_pitch && p.v_offset + p.head_dim <= p.head_pitch &&
        ((long long)p.positions + 128) * p.channels < 0x7fffffffll && p.positions <= 1024;
}

hipError_t launch_attention_s8(const AttentionParams &params, hipStream_t stream)
{
    Args a = {};
    a.p = params;
    a.prob_stride = (params.positions + 63) / 64 * 64 + 16;
    a.chunks = (params.positions + 63) / 64;
    const int qk_mode = epilogue_mode(params.qk_shift, params.half_even, 128ll * 128 * params.key_dim);
    a.av_mode = epilogue_mode(params.av_shift, params.half_even, 128ll * 128 * params.positions);
    a.fd_n16 = make_fastdiv((unsigned)(params.head_dim >> 4));
    a.inv_scale = dl_rescale(params.prob_exp);
    const float scale = dl_scale(params.softmax_exp);
    for (int i = 0; i < 256; i++)
        a.table[i] = expf(scale * (float)(i - 128));
    const int ht = value_tiles(params.head_dim);
    a.v_chunks = std::min(a.chunks, (int)((scratch_bytes(ht) / (16 * ht) - 16) / 64));
    a.v_stride = 64 * a.v_chunks + 16;
    const size_t lds = (256 + kQueries) * sizeof(float) + (size_t)kQueries * a.prob_stride + scratch_bytes(ht);
    const auto kernel = ht == 2 ? pick_kernel<2>(a.chunks, qk_mode) : ht == 4 ? pick_kernel<4>(a.chunks, qk_mode) : pick_kernel<8>(a.chunks, qk_mode);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    const int images = 65535 / params.heads; // per launch: grid.y is 16 bits wide
    const long long in_image = (long long)params.positions * params.channels;
    const long long out_image = (long long)params.positions * params.heads * params.head_dim;
    for (int n0 = 0; n0 < params.batch && e == hipSuccess; n0 += images) {
        const int n = std::min(images, params.batch - n0);
        a.p.qkv = params.qkv + n0 * in_image;
        a.p.out = params.out + n0 * out_image;
        a.p.v_out = params.v_out ? params.v_out + n0 * out_image : nullptr;
        kernel<<<dim3((unsigned)((params.positions + kQueries - 1) / kQueries), (unsigned)(n * params.heads)), dim3(kThreads), lds,
                 stream>>>(a);
        e = hipGetLastError();
    }
    return e;
}

} // namespace espdl
