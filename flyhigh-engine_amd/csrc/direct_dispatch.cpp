// Generated by gen_direct.py: index -> launcher of the direct conv kernel. Do not edit.
#include "conv_kernels.h"
#include "direct_table.h"

namespace fhc {

LaunchFn direct_launcher_s1a(int index, const void** kernel, bool residual);
LaunchFn direct_launcher_s1b(int index, const void** kernel, bool residual);
LaunchFn direct_launcher_s1c(int index, const void** kernel, bool residual);
LaunchFn direct_launcher_s1d(int index, const void** kernel, bool residual);
LaunchFn direct_launcher_s1p(int index, const void** kernel, bool residual);
LaunchFn direct_launcher_s2(int index, const void** kernel, bool residual);
LaunchFn direct_launcher_k1(int index, const void** kernel, bool residual);
LaunchFn direct_launcher_w(int index, const void** kernel, bool residual);
LaunchFn direct_launcher_s1q(int index, const void** kernel, bool residual);

LaunchFn direct_launcher(int index, const void** kernel, bool residual) {
    if (index < 0 || index >= kNumDirect) return nullptr;
    if (index >= 0 && index <= 29) return direct_launcher_s1a(index, kernel, residual);
    if (index >= 30 && index <= 46) return direct_launcher_s1b(index, kernel, residual);
    if (index >= 47 && index <= 51) return direct_launcher_s1c(index, kernel, residual);
    if (index >= 52 && index <= 60) return direct_launcher_s1d(index, kernel, residual);
    if (index >= 61 && index <= 76) return direct_launcher_s1p(index, kernel, residual);
    if (index >= 77 && index <= 107) return direct_launcher_s2(index, kernel, residual);
    if (index >= 108 && index <= 123) return direct_launcher_k1(index, kernel, residual);
    if (index >= 124 && index <= 131) return direct_launcher_w(index, kernel, residual);
    if (index >= 132 && index <= 141) return direct_launcher_s1q(index, kernel, residual);
    return nullptr;
}

}  // namespace fhc
