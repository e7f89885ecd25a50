// fwd16.hip -- one instantiation unit of the packed trace kernels
// (fwd16.hpp) with the DNA profile (SQMI_FWD_DNA = 1) or the substitution
// table (0).  Built twice, exporting SQMI_FWD_PART.
#include "fwd16.hpp"
#include "fwd16_parts.hpp"

#if !defined(SQMI_FWD_DNA) || !defined(SQMI_FWD_PART)
#error "fwd16.hip is built with SQMI_FWD_DNA and SQMI_FWD_PART defined"
#endif

namespace sqmi {
namespace {

constexpr bool kDna = SQMI_FWD_DNA != 0;

hipError_t launchTraceOf(uint32_t track, const FwdArgs &args, int gridBlocks, hipStream_t stream)
{
    const dim3 grid(gridBlocks), block(256);
    switch (track) {
        case kTrackEnd: hipLaunchKernelGGL((kFwdTrace16<kDna, kTrackEnd>), grid, block, 0, stream, args); break;
        case kTrackBottom: hipLaunchKernelGGL((kFwdTrace16<kDna, kTrackBottom>), grid, block, 0, stream, args); break;
        case kTrackRight: hipLaunchKernelGGL((kFwdTrace16<kDna, kTrackRight>), grid, block, 0, stream, args); break;
        case kTrackBottom | kTrackRight:
            hipLaunchKernelGGL((kFwdTrace16<kDna, kTrackBottom | kTrackRight>), grid, block, 0, stream, args);
            break;
        case kTrackLocal: hipLaunchKernelGGL((kFwdTrace16<kDna, kTrackLocal>), grid, block, 0, stream, args); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

const void *traceKernelOf() { return (const void *)&kFwdTrace16<kDna, kTrackEnd>; }

int traceStepsOf(int maxN) { return Fwd16<16, 16, kDna, kTrackEnd, true>::stepsFor(maxN); }

}  // namespace

// The table holds host function pointers: host pass only (the device pass
// instantiates the kernels through the functions above).
#ifndef __HIP_DEVICE_COMPILE__
extern const Fwd16Part SQMI_FWD_PART = {launchTraceOf, traceKernelOf, traceStepsOf};
#endif

}  // namespace sqmi
