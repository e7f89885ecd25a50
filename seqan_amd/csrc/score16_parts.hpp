// score16_parts.hpp -- the packed score kernels are compiled in six units
// (score16.hip built per DNA profile / table and kind); each exports its
// kernel.
#pragma once

namespace sqmi {

const void *scoreDnaGlobal();
const void *scoreDnaRight();
const void *scoreDnaLocal();
const void *scoreTabGlobal();
const void *scoreTabRight();
const void *scoreTabLocal();

}  // namespace sqmi
