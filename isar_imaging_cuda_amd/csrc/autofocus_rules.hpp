// autofocus_rules.hpp — what the host decides about the resident autofocus (k_af_resident) from sizes alone.
// Plain C++.
#pragma once

#include <algorithm>

namespace isar {

// Bound of a resident wait in the default form, in polls of about 0.25 us (0.57 with four waiting workgroups
// on every CU); a frame that reaches it is done over by one workgroup. A frame that is placed in part
// waits for the frames ahead of it, so for as long as those run: 4 to 22 us an iteration (22: 1024 pulses,
// all 512 bins, two workgroups a CU). So the bound goes with the iterations, 256 polls each, three
// times the slowest; a wait that nobody ends costs 12 ms of a run of 120.
constexpr int af_guarded_polls(int iterations) {
    return static_cast<int>(std::min<long long>(256ll * (iterations + 64ll), 0x7fffffff));
}

}  // namespace isar
