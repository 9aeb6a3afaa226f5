// Process-wide tuning of the FP32 pair kernels (written by halma_tune_set).
#pragma once

namespace halma {

// Defaults: the autotuner's choice on the 2.1M-particle clump workload (first unbinding
// pass 4.34 ms against 4.99 ms for R=2, SUB=8, 16 waves/CU, 4 items/wave).
struct Tuning {
    int tests_per_lane = 2;   // R: test particles held in registers per lane
    int subtile = 4;          // sources summed in plain FP32 before each FP64 add
    int min_chunk = 512;      // smallest source chunk when a source range is split
    int items_per_wave = 8;   // queue items targeted per resident wave
    int waves_per_cu = 32;    // persistent waves per compute unit
    int sym_max = 65536;      // largest halo on the symmetric kernel in the unbinding
};

extern Tuning g_tuning;

// Rigorous relative error bound of the FP32 sums with sub-tiles of SUB terms, u = 2^-24:
// per term 5.5u (FP32 differences and squares 2.5u after the square root, v_rsq_f32
// <= 1 ulp = 2u, the mass product u), the plain sub-tile sum (SUB-1)u, and 0.5u + 1e-11 for
// the FP64 sums of the sub-tiles, the float pair they are kept in, the merge and the
// higher-order terms.
inline double pot_error_bound(int sub) {
    const double u = 5.9604644775390625e-08;  // 2^-24
    return (sub + 5.0) * u + 1e-11;
}

// The symmetric self-potential kernel: test side as above with sub-tiles of 8 terms;
// source side per term 4.5u (differences, squares, v_rsq_f32), a lane's chain over four
// tests 4u (the products included), the two chains' sum u, the tree's three FP32 levels 3u,
// its FP64 levels and the merge 0.5u: 13u either way.
inline double pot_sym_error_bound() { return pot_error_bound(8); }

}  // namespace halma
