// The walking convolution kernel's builds for channels that are no multiple of 4, 3 x 3 filters at stride 1.  (At stride 2
// most layers lost to the other kernels: 32 x 20 x 80 x 30 -> 139 took 10.2 us where those take 8.6.)
#include "conv2d_s8_walk_kernel.h"

namespace espdl {
namespace walk {

hipError_t launch_raw_3x3(int cu, int nt, WalkArgs &a, const WalkLaunch &l)
{
    switch (cu) {
    case 2:
        return launch_raw<3, 1, 2>(nt, a, l);
    case 3:
        return launch_raw<3, 1, 3>(nt, a, l);
    case 4:
        return launch_raw<3, 1, 4>(nt, a, l);
    case 5:
        return launch_raw<3, 1, 5>(nt, a, l);
    case 6:
        return launch_raw<3, 1, 6>(nt, a, l);
    case 7:
        return launch_raw<3, 1, 7>(nt, a, l);
    case 8:
        return launch_raw<3, 1, 8>(nt, a, l);
    case 9:
        return launch_raw<3, 1, 9>(nt, a, l);
    case 10:
        return launch_raw<3, 1, 10>(nt, a, l);
    case 11:
        return launch_raw<3, 1, 11>(nt, a, l);
    case 12:
        return launch_raw<3, 1, 12>(nt, a, l);
    default:
        return hipErrorInvalidValue;
    }
}

} // namespace walk
} // namespace espdl
