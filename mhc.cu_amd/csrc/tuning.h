// Launch-heuristic overrides for experiments and for tests that must reach a path the heuristics
// would not pick at the test's shape (host side only).  They exist only in a build with -DMHC_TUNING
// (libmhc_hip_tuning.so, `build.py --tuning`): there, mhc_tuning_set changes a knob for the whole
// process, unsynchronised.  In the product library tuning_get() is the constant 0 = "use the built-in
// heuristic", no knob and no setter exist, and the dispatch code reads no global state.
#pragma once

namespace mhc {

enum TuneKey {
    kTuneOnepassOff = 0,    // one-pass forwards: 0 = by size, 1 = neither, 2 = the one-launch forward, 3 = the held one, whenever the shape allows
    kTuneOnepassG = 1,      // samples per workgroup of the one-launch forward
    kTuneGramFused = 2,     // n <= 8 channel sums and coefficient backward: 1 = two launches, 2 = one launch (n <= 4: four samples per workgroup, n = 5 .. 8: one per wave), 3 = VALU sums of n <= 4: one sample per wave
    kTuneSlabSplits = 3,    // batch splits of the slab backward (n <= 8) and of the projection backward (n = 5 .. 18)
    kTuneSeparateFinalize = 4,  // 1 = batch sums always as a launch of their own, never inside the dphi launch
    kTuneProjApart = 5,     // n <= 18 projection backward: 1 = both products in one launch, 2 = two launches
    kTuneStaticSpg = 6,     // static backward (n <= 8): samples per workgroup (bf16: 1 = the sample-resident kernel)
    kTuneResident = 7,      // n <= 8 sample-resident backward: 0 = by heuristic, 1 = never, 2 = whenever the shape allows
    kTuneWideDxBeside = 8,  // wide projections (n > 18): dx workgroups beside the coefficient launch: 1 = never, 2 = always
    kTuneSpareB = 9,        // projection forward (matrix-core kernels): K splits, 0 = by heuristic
    kTuneGather = 10,       // the caller's fp32 parameters read by the kernels of the forward themselves: 1 = never, 2 = whenever the shape allows
    kTuneSlabWidth = 11,    // slab backward (n <= 4, bf16): channels per workgroup, 1 = 64, 2 = 128, 0 = by size
    kTuneSlab8 = 12,        // slab backward of n = 5 .. 8 behind the channel sums: 1 = never (general kernels), 2 = always
    kTuneCount = 13
};

// What mhc_tuning_route() of the same build tells about the built-in heuristic, for tests of its lines.
enum RouteKey {
    kRouteBackward = 0,     // n <= 8, bf16 arithmetic: 0 = sample-resident, 1 = tiled
    kRouteForward = 1,      // dynamic forward from the caller's fp32 parameters: 0 = two launches, 1 = one launch from packed phi, 2 = one that reads them itself, 3 = held
    kRouteSums = 2,         // channel sums of the fp32 tier, n <= 8: 0 = two launches, 1 = one, 2 = one with a wave per sample
};

#ifdef MHC_TUNING
extern int g_tuning[kTuneCount];
inline int tuning_get(int key) { return g_tuning[key]; }
#else
constexpr int tuning_get(int) { return 0; }
#endif

}  // namespace mhc
