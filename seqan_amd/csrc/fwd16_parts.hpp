// fwd16_parts.hpp -- the packed trace kernels are compiled in two units
// (fwd16.hip built with SQMI_FWD_DNA = 0 / 1); each exports its kernels
// through one of these tables.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace sqmi {

struct Fwd16Part {
    hipError_t (*launchTrace)(uint32_t track, const FwdArgs &args, int gridBlocks, hipStream_t stream);
    const void *(*traceKernel)();
    int (*traceSteps)(int maxN);
};

extern const Fwd16Part kFwdPartDna, kFwdPartTab;

}  // namespace sqmi
