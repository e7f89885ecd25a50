// band16_parts.hpp -- the instantiation units of the packed banded kernels
// (band16.hip, one per profile / table and kind).
#pragma once

namespace sqmi {

const void *bandTabEnd(int R, bool wide, bool lds);
const void *bandTabFree(int R, bool wide, bool lds);
const void *bandTabLocal(int R, bool wide, bool lds);
const void *bandDnaEnd(int R, bool wide, bool lds);
const void *bandDnaFree(int R, bool wide, bool lds);
const void *bandDnaLocal(int R, bool wide, bool lds);

}  // namespace sqmi
