// The walking convolution kernel's builds for 3 x 3 filters at stride 2.
#include "conv2d_s8_walk_kernel.h"

namespace espdl {
namespace walk {

hipError_t launch_3x3_s2(int cu, int nt, WalkArgs &a, const WalkLaunch &l)
{
    switch (cu) {
    case 1:
        return launch_cu<3, 2, 1>(nt, a, l);
    case 2:
        return launch_cu<3, 2, 2>(nt, a, l);
    case 3:
        return launch_cu<3, 2, 3>(nt, a, l);
    case 4:
        return launch_cu<3, 2, 4>(nt, a, l);
    case 5:
        return launch_cu<3, 2, 5>(nt, a, l);
    case 6:
        return launch_cu<3, 2, 6>(nt, a, l);
    case 7:
        return launch_cu<3, 2, 7>(nt, a, l);
    case 8:
        return launch_cu<3, 2, 8>(nt, a, l);
    default:
        return hipErrorInvalidValue;
    }
}

} // namespace walk
} // namespace espdl
