// The walking convolution kernel's builds for 5 x 5 filters.
#include "conv2d_s8_walk_kernel.h"

namespace espdl {
namespace walk {

hipError_t launch_5x5(int cu, int stride, int nt, WalkArgs &a, const WalkLaunch &l)
{
    if (stride == 1) {
        switch (cu) {
        case 1:
            return launch_cu<5, 1, 1>(nt, a, l);
        case 2:
            return launch_cu<5, 1, 2>(nt, a, l);
        case 3:
            return launch_cu<5, 1, 3>(nt, a, l);
        case 4:
            return launch_cu<5, 1, 4>(nt, a, l);
        case 5:
            return launch_cu<5, 1, 5>(nt, a, l);
        default:
            return hipErrorInvalidValue;
        }
    }
    switch (cu) {
    case 1:
        return launch_cu<5, 2, 1>(nt, a, l);
    case 2:
        return launch_cu<5, 2, 2>(nt, a, l);
    case 3:
        return launch_cu<5, 2, 3>(nt, a, l);
    case 4:
        return launch_cu<5, 2, 4>(nt, a, l);
    case 5:
        return launch_cu<5, 2, 5>(nt, a, l);
    default:
        return hipErrorInvalidValue;
    }
}

} // namespace walk
} // namespace espdl
