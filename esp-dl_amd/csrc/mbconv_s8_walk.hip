// Planner and launches of the inverted residual block as a walk down the image (mbconv_s8_walk_kernel.h).
#include "mbconv_s8_walk_kernel.h"

namespace espdl {
namespace {
using namespace mbwalk;

struct MbWalkPlan {
    bool ok;
    int ce, rt; // of the build
    MbWalkArgs a;
};

MbWalkPlan walk_plan(const MbconvParams &p, int cus)
{
    MbWalkPlan plan = {};
    const int s = p.stride_h;
    if (p.w_expand == nullptr || !mbconv_expand_is_pointwise(p) || p.k_h != 3 || p.k_w != 3 || p.dil_h != 1 || p.dil_w != 1 ||
        p.stride_w != s || (s != 1 && s != 2) || p.batch <= 0)
        return plan;
    // a lane holds 4 RT output channels and stores them at once
    plan.rt = p.out_c % 8 == 0 && p.out_c <= 32 ? 2 : (p.out_c % 16 == 0 && p.out_c <= 64 ? 4 : 0);
    plan.ce = (p.exp_c + 47) / 48 * 3;
    if (plan.rt == 0 || p.exp_c % 16 != 0 || plan.ce > 9 || p.in_c % 4 != 0 || p.in_c < 16 || p.in_c > 16 * kUnits)
        return plan;
    if (p.residual != nullptr && (s != 1 || plan.rt != 2))
        return plan;
    MbWalkArgs &a = plan.a;
    a.p = p;
    // columns from image to image: the padding between them at least once
    const long long over = (long long)(p.out_w - 1) * s + 2 - p.pad_left - (p.in_w - 1);
    long long pitch = std::max<long long>(p.in_w + std::max<long long>({0, p.pad_left, over}), (long long)p.out_w * s);
    pitch = (pitch + s - 1) / s * s;
    const long long cols = (p.batch - 1) * (pitch / s) + p.out_w;
    const long long in_bytes = (long long)p.batch * p.in_h * p.in_w * p.in_c, out_bytes = (long long)p.batch * p.out_h * p.out_w * p.out_c;
    const long long seg_rows = s == 1 ? (p.out_h + 1) / 2 : p.out_h;
    const int width = (s == 1 ? 14 : 15) * MbShape<3, 2, 1, false>::W;
    const long long strips = (cols + width - 1) / width;
    if (in_bytes > 0x7fff0000ll || out_bytes > 0x7fff0000ll || pitch * (p.batch + 1) > (1ll << 30) || strips * seg_rows > (1ll << 30))
        return plan;
    a.in_row = p.in_w * p.in_c;
    a.in_img = a.in_row * p.in_h;
    a.in_bytes = (int)in_bytes;
    a.out_row = p.out_w * p.out_c;
    a.out_img = a.out_row * p.out_h;
    a.out_bytes = (int)out_bytes;
    a.bound_e = (long long)p.in_c * 16384;
    a.bound_d = 9ll * 16384;
    a.bound_p = (long long)p.exp_c * 16384;
    a.fd_p = make_fastdiv((unsigned)pitch);
    a.fd_po = make_fastdiv((unsigned)(pitch / s));
    // one workgroup per compute unit, each with the same number of row pairs of the strips laid end to end
    a.seg_rows = (int)seg_rows;
    a.rows_total = (int)(strips * seg_rows);
    const int want = std::max(8, cus / 8 * 8);
    a.rows_per_group = (a.rows_total + want - 1) / want;
    a.n_groups = ((a.rows_total + a.rows_per_group - 1) / a.rows_per_group + 7) / 8 * 8;
    a.fd_seg = make_fastdiv((unsigned)a.seg_rows);
    plan.ok = true;
    return plan;
}

template <int CE, int RT, int S, bool HE, bool RES>
hipError_t launch_one(const MbWalkPlan &plan, hipStream_t stream)
{
    hipLaunchKernelGGL((mbconv_s8_walk_kernel<CE, RT, S, HE, RES>), dim3((unsigned)plan.a.n_groups), dim3(64 * MbShape<CE, RT, S, RES>::W), 0,
                       stream, plan.a);
    return hipGetLastError();
}

template <int CE, bool HE>
hipError_t launch_ce(const MbWalkPlan &plan, hipStream_t stream)
{
    if (plan.a.p.stride_h == 2)
        return plan.rt == 2 ? launch_one<CE, 2, 2, HE, false>(plan, stream) : launch_one<CE, 4, 2, HE, false>(plan, stream);
    if (plan.a.p.residual != nullptr)
        return launch_one<CE, 2, 1, HE, true>(plan, stream);
    return plan.rt == 2 ? launch_one<CE, 2, 1, HE, false>(plan, stream) : launch_one<CE, 4, 1, HE, false>(plan, stream);
}

template <bool HE>
hipError_t launch_he(const MbWalkPlan &plan, hipStream_t stream)
{
    return plan.ce == 3 ? launch_ce<3, HE>(plan, stream) : (plan.ce == 6 ? launch_ce<6, HE>(plan, stream) : launch_ce<9, HE>(plan, stream));
}

} // namespace

// Set-up and one workgroup's steps (160 random blocks of batch 1 to 256: 5 % rms, 15 % at most).
float mbconv_s8_walk_us(const MbconvParams &p, int cu_count)
{
    const MbWalkPlan plan = walk_plan(p, cu_count > 0 ? cu_count : 256);
    if (!plan.ok)
        return 1e30f;
    const MbWalkArgs &a = plan.a;
    const int segments = std::min(a.rows_total / a.seg_rows, (a.rows_per_group + a.seg_rows - 2) / a.seg_rows + 1);
    const bool s1 = p.stride_h == 1;
    const float steps = ((float)a.rows_per_group + (s1 ? 0.6f : 0.9f) * (float)segments) * (p.half_even ? (s1 ? 1.36f : 1.46f) : 1.f);
    const float ce = (float)plan.ce, rt = (float)(plan.rt + (p.residual != nullptr ? 4 : 0));
    return s1 ? 4.6f + 0.28f * ce + steps * (0.42f + 0.255f * ce + 0.18f * rt)
              : 4.3f + 0.24f * ce + steps * (0.34f + 0.27f * ce + 0.15f * rt);
}

hipError_t launch_mbconv_s8_walk(const MbconvParams &p, int cu_count, hipStream_t stream)
{
    const MbWalkPlan plan = walk_plan(p, cu_count > 0 ? cu_count : 256);
    if (!plan.ok)
        return hipErrorInvalidValue;
    return p.half_even ? launch_he<true>(plan, stream) : launch_he<false>(plan, stream);
}

} // namespace espdl
