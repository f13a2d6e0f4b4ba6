// Host build of noa_amd/csrc/pumas_search.hh for its test.
#include "../../noa_amd/csrc/pumas_search.hh"

extern "C" int pumas_cell(const float* t, int n, float x, int in) { return noa_hip::pumas::cell(t, n, x, in != 0); }
