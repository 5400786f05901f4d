// fdns_sweep.h -- how the wavefronts of a workgroup share the column-block
// sweeps of the LU-mode solves (plain C++, so that the host can go over it).
#pragma once

#ifdef __HIPCC__
#define SWEEP_FN __host__ __device__ constexpr
#else
#define SWEEP_FN constexpr
#endif

namespace fdns {

constexpr int LUX_NB = 8;      // columns per block
constexpr int LUX_ROWS = 128;  // rows per wavefront
constexpr int LUX_WB = LUX_ROWS / LUX_NB;   // blocks per wavefront
SWEEP_FN int lux_waves(int n) { return (n + LUX_ROWS - 1) / LUX_ROWS; }
SWEEP_FN int lux_blocks(int n) { return (n + LUX_NB - 1) / LUX_NB; }

// A sweep goes in pairs of blocks, two barriers a pair.  Wavefront wv (rows
// LUX_ROWS wv ..) takes part in the first `mine` pairs and keeps the barriers
// of the others, so every wavefront of the launch must have 0 <= mine <= pairs
// -- those past the matrix too (the m = 0 system has n = N rows in a launch
// with the wavefronts of 2 N).
struct LuxShare {
    int pairs, mine;
};
// forward from block b0 (b0 = nblk: nothing to do)
SWEEP_FN LuxShare lux_forward(int nblk, int b0, int wv)
{
    const int pairs = (nblk - b0 + 1) / 2, last = (LUX_WB * wv + LUX_WB - b0 + 1) / 2;
    return {pairs, last < 0 ? 0 : (last < pairs ? last : pairs)};
}
// backward from block nblk - 1
SWEEP_FN LuxShare lux_backward(int nblk, int wv)
{
    const int mine = (nblk - LUX_WB * wv + 1) / 2;
    return {(nblk + 1) / 2, mine < 0 ? 0 : mine};
}

}  // namespace fdns
