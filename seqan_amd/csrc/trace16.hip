// trace16.hip -- one instantiation unit of the packed trace kernels
// (trace16.hpp) with the DNA profile (SQMI_TRACE_DNA = 1) or the substitution
// table (0).  Built twice, exporting SQMI_TRACE_PART.
#include "score16_parts.hpp"
#include "trace16.hpp"

#if !defined(SQMI_TRACE_DNA) || !defined(SQMI_TRACE_PART)
#error "trace16.hip is built with SQMI_TRACE_DNA and SQMI_TRACE_PART defined"
#endif

namespace sqmi {

const void *SQMI_TRACE_PART(uint32_t track)
{
    constexpr bool dna = SQMI_TRACE_DNA != 0;
    switch (track) {
        case kTrackEnd: return (const void *)&kTrace16<dna, kTrackEnd>;
        case kTrackBottom: return (const void *)&kTrace16<dna, kTrackBottom>;
        case kTrackRight: return (const void *)&kTrace16<dna, kTrackRight>;
        case kTrackBottom | kTrackRight: return (const void *)&kTrace16<dna, kTrackBottom | kTrackRight>;
        case kTrackLocal: return (const void *)&kTrace16<dna, kTrackLocal>;
        default: return nullptr;
    }
}

}  // namespace sqmi
