// score16_parts.hpp -- the packed score kernels are compiled in six units
// (score16.hip built per DNA profile / table and kind), the trace kernels in
// two (trace16.hip per DNA profile / table); each exports its kernels.
#pragma once

#include <cstdint>

namespace sqmi {

const void *scoreDnaGlobal();
const void *scoreDnaRight();
const void *scoreDnaLocal();
const void *scoreTabGlobal();
const void *scoreTabRight();
const void *scoreTabLocal();
// By tracking kind (Track).
const void *traceDna(uint32_t track);
const void *traceTab(uint32_t track);

}  // namespace sqmi
