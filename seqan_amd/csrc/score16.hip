// score16.hip -- one instantiation unit of the packed score kernels
// (score16.hpp): DNA profile (SQMI_SCORE_DNA = 1) or substitution table (0),
// and a kind (SQMI_SCORE_KIND, ScoreKind).  Built six times, exporting
// SQMI_SCORE_PART.
#include "score16.hpp"
#include "score16_parts.hpp"

#if !defined(SQMI_SCORE_DNA) || !defined(SQMI_SCORE_KIND) || !defined(SQMI_SCORE_PART)
#error "score16.hip is built with SQMI_SCORE_DNA, SQMI_SCORE_KIND and SQMI_SCORE_PART defined"
#endif

namespace sqmi {

const void *SQMI_SCORE_PART() { return (const void *)&kScore16<SQMI_SCORE_DNA != 0, SQMI_SCORE_KIND>; }

}  // namespace sqmi
