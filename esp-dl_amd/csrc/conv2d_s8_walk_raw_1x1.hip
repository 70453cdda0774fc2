// The walking convolution kernel's builds for channels that are no multiple of 4, 1 x 1 filters.
#include "conv2d_s8_walk_kernel.h"

namespace espdl {
namespace walk {

hipError_t launch_raw_1x1(int cu, int nt, WalkArgs &a, const WalkLaunch &l)
{
    switch (cu) {
    case 2:
        return launch_raw<1, 1, 2>(nt, a, l);
    case 3:
        return launch_raw<1, 1, 3>(nt, a, l);
    case 4:
        return launch_raw<1, 1, 4>(nt, a, l);
    case 5:
        return launch_raw<1, 1, 5>(nt, a, l);
    case 6:
        return launch_raw<1, 1, 6>(nt, a, l);
    case 7:
        return launch_raw<1, 1, 7>(nt, a, l);
    case 8:
        return launch_raw<1, 1, 8>(nt, a, l);
    case 9:
        return launch_raw<1, 1, 9>(nt, a, l);
    case 10:
        return launch_raw<1, 1, 10>(nt, a, l);
    case 11:
        return launch_raw<1, 1, 11>(nt, a, l);
    case 12:
        return launch_raw<1, 1, 12>(nt, a, l);
    case 13:
        return launch_raw<1, 1, 13>(nt, a, l);
    case 14:
        return launch_raw<1, 1, 14>(nt, a, l);
    case 15:
        return launch_raw<1, 1, 15>(nt, a, l);
    case 16:
        return launch_raw<1, 1, 16>(nt, a, l);
    default:
        return hipErrorInvalidValue;
    }
}

} // namespace walk
} // namespace espdl
