// resident_team.cpp with the assembly that leaves sums per row of a tile: the
// full team reads them at its start, a partial team combines them first.
#include "oc_internal.hpp"

#define oc_cloth_set_dv(c, dv) (const_cast<oc::DevCloth&>(oc::cloth_view(c)).asm_rows = 1, oc_cloth_set_dv(c, dv))
#include "resident_team.cpp"
