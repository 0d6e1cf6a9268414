// autofocus_rules.hpp — what the host decides about the resident autofocus (k_af_resident) from sizes alone.
// Plain C++.
#pragma once

#include <stddef.h>

#include <algorithm>

namespace isar {

constexpr int kComputeUnits = 256;         // of the GPU, in 8 XCDs
constexpr size_t kLdsBytes = 160 * 1024;   // of a compute unit

// Bound of a resident wait in the default form, in polls of about 0.25 us (0.57 with four waiting workgroups
// on every CU); a frame that reaches it is done over by one workgroup. A frame that is placed in part
// waits for the frames ahead of it, so for as long as those run: 4 to 22 us an iteration (22: 1024 pulses,
// all 512 bins, two workgroups a CU). So the bound goes with the iterations, 256 polls each, three
// times the slowest; a wait that nobody ends costs 12 ms of a run of 120.
constexpr int af_guarded_polls(int iterations) {
    return static_cast<int>(std::min<long long>(256ll * (iterations + 64ll), 0x7fffffff));
}

// How a batch's resident workgroups are placed. The dispatcher fills a CU that has the LDS for another
// workgroup while other CUs are idle, and the fullest CU sets the pace of every iteration. So a
// workgroup asks for so much LDS that a CU takes only its share of them.
struct AfResidentShape {
    size_t lds;        // bytes a workgroup asks for
    int places;        // workgroups that the GPU holds at once
    int sub_chunks;    // takes the frames of up to this many sub-chunks
};

// The LDS with which a CU takes `share` workgroups that need `need` bytes and of which it can hold `fit`.
// Allocations are multiples of 1280 bytes, so shares above 8 cannot be told apart from fit.
constexpr AfResidentShape af_shape(int share, size_t need, int fit) {
    if (share >= fit || share > 8) return {need, fit * kComputeUnits, 0};
    return {std::max(need, kLdsBytes / (static_cast<size_t>(share) + 1) + 1024), share * kComputeUnits, 0};
}

// How many bins a frame has selected (up to 512) only the device knows. A frame commonly has up to 64:
// shape[0] is the share of such a batch, with a quarter of the places to spare. It takes the frames that
// find a place at once with it if all of the batch are like them. Frames of more sub-chunks go to a launch of their
// own with shape[1], the share of a batch whose frames all have 512 bins; n = 1 where no frame
// can need it. At 512
// bins, in ms with one shape for all and with two: 32 frames of 256 pulses 3.31 and 1.33 (split 1.98), 16 of 64 1.55 and
// 0.83, 128 of 64 4.77 and 1.41 (one workgroup a frame 2.84), 40 of 512 5.6 and 3.9, 8 of 1024 4.9 and 2.9.
// With the LDS needed for all, 40 frames of 256 pulses with 64 bins take 0.78 instead of 0.51, 128 of
// them 0.86 instead of 0.75, 40 of 512 1.10 instead of 0.72. The launch that has no frames takes 3 us.
struct AfResidentShapes {
    AfResidentShape shape[2];
    int n;
};
constexpr AfResidentShapes af_resident_shapes(int frames, int sub, size_t need, int fit) {
    const int most = 512 / sub, common = 64 / sub;
    auto share = [](long long groups, long long places) { return static_cast<int>((groups + places - 1) / places); };
    AfResidentShapes r{};
    r.shape[0] = af_shape(share(4ll * frames * common, 3 * kComputeUnits), need, fit);
    r.shape[1] = af_shape(share(1ll * frames * most, kComputeUnits), need, fit);
    r.shape[0].sub_chunks = r.shape[0].places / frames;
    r.shape[1].sub_chunks = most;
    r.n = r.shape[0].sub_chunks >= most || r.shape[0].lds == r.shape[1].lds ? 1 : 2;
    if (r.n == 1) r.shape[0].sub_chunks = most;
    return r;
}

}  // namespace isar
