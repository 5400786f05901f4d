// fdns_sweep.h -- how the wavefronts of a workgroup share the column-block
// sweeps of the LU-mode solves, and the sweeps' division (plain C++, so that
// the host can go over them).
#pragma once

#ifdef __HIPCC__
#define SWEEP_DEV __host__ __device__
#define SWEEP_FN __host__ __device__ constexpr
#else
#define SWEEP_DEV
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

// x / d by the reciprocal rcp = 1 / d (rounded): quotient, remainder,
// correction (Markstein), which gives the correctly rounded quotient where
// neither the reciprocal (rcp_safe) nor the quotient or the remainder (usual)
// leaves the normal range: |x| >= 2^-900 keeps the remainder's 106 bits above
// 2^-1022, and runs that decay go a long way before they leave it (1e-241).
// Beyond it an infinity, and a quotient next to the
// largest number, give NaN.
SWEEP_DEV inline double div_by(double x, double d, double rcp)
{
    const double q = x * rcp;
    return __builtin_fma(__builtin_fma(-q, d, x), rcp, q);
}
// the quotient that stays in the solution: where it is zero the number itself,
// zero or not usual
SWEEP_DEV inline double div_last(double x, double d, double rcp)
{
    const double q = div_by(x, d, rcp);
    return q == 0.0 ? x : q;
}
SWEEP_DEV inline bool rcp_safe(double d) { return __builtin_fabs(d) > 0x1p-100 && __builtin_fabs(d) < 0x1p100; }
SWEEP_DEV inline bool usual(double q) { return q == 0.0 || (__builtin_fabs(q) > 0x1p-800 && __builtin_fabs(q) < 0x1p900); }

}  // namespace fdns
