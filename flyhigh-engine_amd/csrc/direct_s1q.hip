// Generated by gen_direct.py: direct conv kernel instantiations, group s1q. Do not edit.
#include "direct_impl.h"

namespace fhc {

LaunchFn direct_launcher_s1q(int index, const void** kernel, bool residual) {
    switch (index) {
        case 132:
            if (kernel) *kernel = direct_kernel<3, 1, 96, 4, 1, 2, 1, 1, true>(residual);
            return launch_direct<3, 1, 96, 4, 1, 2, 1, 1, true>;
        case 133:
            if (kernel) *kernel = direct_kernel<3, 1, 96, 4, 1, 3, 1, 1, true>(residual);
            return launch_direct<3, 1, 96, 4, 1, 3, 1, 1, true>;
        case 134:
            if (kernel) *kernel = direct_kernel<3, 1, 96, 4, 1, 4, 1, 1, true>(residual);
            return launch_direct<3, 1, 96, 4, 1, 4, 1, 1, true>;
        case 135:
            if (kernel) *kernel = direct_kernel<3, 1, 96, 4, 1, 6, 1, 1, true>(residual);
            return launch_direct<3, 1, 96, 4, 1, 6, 1, 1, true>;
        case 136:
            if (kernel) *kernel = direct_kernel<3, 1, 96, 4, 1, 8, 1, 1, true>(residual);
            return launch_direct<3, 1, 96, 4, 1, 8, 1, 1, true>;
        case 137:
            if (kernel) *kernel = direct_kernel<3, 1, 128, 4, 1, 2, 1, 1, true>(residual);
            return launch_direct<3, 1, 128, 4, 1, 2, 1, 1, true>;
        case 138:
            if (kernel) *kernel = direct_kernel<3, 1, 128, 4, 1, 3, 1, 1, true>(residual);
            return launch_direct<3, 1, 128, 4, 1, 3, 1, 1, true>;
        case 139:
            if (kernel) *kernel = direct_kernel<3, 1, 128, 4, 1, 4, 1, 1, true>(residual);
            return launch_direct<3, 1, 128, 4, 1, 4, 1, 1, true>;
        case 140:
            if (kernel) *kernel = direct_kernel<3, 1, 128, 4, 1, 6, 1, 1, true>(residual);
            return launch_direct<3, 1, 128, 4, 1, 6, 1, 1, true>;
        case 141:
            if (kernel) *kernel = direct_kernel<3, 1, 128, 4, 1, 8, 1, 1, true>(residual);
            return launch_direct<3, 1, 128, 4, 1, 8, 1, 1, true>;
        default: return nullptr;
    }
}

}  // namespace fhc
