// band16.hip -- one instantiation unit of the packed banded kernels
// (band16.hpp): DNA profile (SQMI_BAND_DNA = 1) or substitution table (0), and
// a kind (SQMI_BAND_KIND, BandKind).  Built six times, exporting
// SQMI_BAND_PART.
#include "band16.hpp"
#include "band16_parts.hpp"

#if !defined(SQMI_BAND_DNA) || !defined(SQMI_BAND_KIND) || !defined(SQMI_BAND_PART)
#error "band16.hip is built with SQMI_BAND_DNA, SQMI_BAND_KIND and SQMI_BAND_PART defined"
#endif

namespace sqmi {

// Rows per block: 8 and 12 with LDS rings, 16 with either.
template <bool WIDE>
static const void *part(int R, bool lds)
{
    constexpr bool dna = SQMI_BAND_DNA != 0;
    constexpr int kind = SQMI_BAND_KIND;
    if (R == 16)
        return lds ? (const void *)&kBand16<16, dna, kind, WIDE, true> : (const void *)&kBand16<16, dna, kind, WIDE, false>;
    if (!lds)
        return nullptr;
    return R == 12 ? (const void *)&kBand16<12, dna, kind, WIDE, true>
                   : R == 8 ? (const void *)&kBand16<8, dna, kind, WIDE, true> : nullptr;
}

const void *SQMI_BAND_PART(int R, bool wide, bool lds) { return wide ? part<true>(R, lds) : part<false>(R, lds); }

}  // namespace sqmi
