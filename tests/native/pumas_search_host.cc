// Host build of noa_amd/csrc/pumas_search.hh for its test.
#include "../../noa_amd/csrc/pumas_search.hh"

extern "C" int pumas_cell(const float* t, int n, float x, int in) { return noa_hip::pumas::cell(t, n, x, in != 0); }

// (a constant expression: a shift beyond the type's width does not compile)
static_assert(noa_hip::pumas::tree_levels(6) == 0x7fffffffu, "depth 5, a level more");

extern "C" uint32_t pumas_tree_levels(int levels) { return noa_hip::pumas::tree_levels(levels); }
