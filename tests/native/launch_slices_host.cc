// Host build of noa_amd/csrc/launch_slices.hh for its test: the ranges of a
// launch into first[] and count[], at most `room`; their number, or the
// callback's value at range number `fail_at`.
#include "../../noa_amd/csrc/launch_slices.hh"

extern "C" int slices(int64_t workgroups, int lanes, int64_t* first, uint32_t* count, int room, int fail_at) {
    int n = 0;
    const int rc = noa_hip::launch_slices(workgroups, lanes, [&](int64_t f, uint32_t c) {
        if (n == fail_at) return -7;
        if (n < room) {
            first[n] = f;
            count[n] = c;
        }
        n++;
        return 0;
    });
    return rc ? rc : n;
}
