// The choice between tiles of 128 and of 64 columns for up to 16 rows: plain host arithmetic of the dispatcher (fp6m_gemm.hip).
#pragma once
#include "mb_plan.h"

namespace fp6m {

// How a launch of gemm_m16_kernel (steps of 32 rows of k) or gemm_m16h_kernel (steps of 64) is cut, in steps.
struct M16Cut {
    int wk;                   // waves per workgroup
    long long ks, wgs;        // parts per INT4 tile, workgroups
    double longest, younger;  // INT4 slices of waves 0-3, and of 4-7
    double longest6;          // FP6 slices
    double mean;              // all steps of a tile over its slices
};

// The time of one launch, us, to choose by.
//
// Tiles of 64 columns need half as many parts to occupy the chip, and what parts cost (publish, count, gather: three round
// trips) is a fifth of a launch of 10 us; but a tile's workgroup reads all rows of A for half as many columns, so with many
// rows, a long k or enough tiles for every CU the wide tiles win.  Where the line lies depends on how k divides, so both
// are estimated: least squares without negative terms over 7000 points, all splits of 650 random shapes (2 to 16 rows, k = 1152
// .. 28672, n = 2048 .. 46080, both scale modes, none to 1024 FP6 columns, row mixes), which they reproduce to 2-5 %.
// 64-column tiles are taken on 55 % of those shapes; the choice is 1 % behind the best of all measured splits, 9.5 % faster than 128-column
// tiles alone, and three of 650 lost (the worst 3 %).  us: 16 x 4096 x 4096 8.5 -> 7.1, 5 x 5120 x 15360 12.7 -> 10.6,
// 8 x 11008 x 4096 11.2 -> 9.9, 16 x 2816 x 2304 9.3 -> 6.4; 16 x 8192 x 8192 keeps 128 columns (12.3, 13.1 with 64).
// Fitted before either kernel stopped fetching past the end of a slice, which took 1 to 9 % off both, and over INT4 tiles with up to
// 1024 FP6 columns.  Hence the margins by which 64-column tiles have to be ahead: over 2013 calls at other random shapes they are
// taken 1314 times and 16 % faster on average, twice more than 2 % slower (with 2 % instead of 4 eleven times, 9 x 18560 x 4352 14.6 us against
// 13.5); over 2279 of FP6 columns alone, whose times the estimates miss by 4-10 %, 1539 times and 16 %, twice (with 2 % instead of 8
// 35 times, 14 x 19328 x 4608 19.5 against 17.5).  Row mixes: with 4 % five of 2342 calls were 5 to 12 % slower (1 x 1792 x 20224 with 512
// FP6 rows 9.2 against 8.2), with 8 % one of 2150, by 3 %.  (Words in gfx950 order gain less -- of 714 such calls six are 4 to 8 % slower
// -- but take what the reference's order takes, for the same bits.)
inline double half_margin(bool all_fp6, bool row_mix) { return all_fp6 || row_mix ? 0.92 : 0.96; }
struct M16Time {
    // us once; once with a split, per part, and per part and row; per step of the longest slice, of the mean one, of the mean one
    // at full occupation, per row that A is fetched in, and with group scales; per step by which 1.7 FP6 steps exceed an INT4
    // slice; per MB of weights; per step of the younger waves' slices.  Beyond one workgroup per CU `rows` goes with their number.
    double start, split, part, part_rows, longest, mean, mean_busy, rows, group, fp6, mbytes, younger;
};
// [64 columns][more than one workgroup per CU, or eight waves][more than four rows]
constexpr M16Time kM16TimeFour[2][2][2] = {
    {{{3.867, 0.855, 0.0, 0.0219, 0.079, 0.167, 0.0, 0.0, 0.023, 0.135, 0.044, 0.036},
      {4.556, 0.334, 0.248, 0.001, 0.1245, 0.1207, 0.0942, 0.0007, 0.0158, 0.21, 0.0, 0.02}},
     {{5.111, 0.376, 0.0, 0.0228, 0.2076, 0.0, 0.0, 0.0, 0.0252, 0.019, 0.1044, 0.0},
      {4.932, 0.565, 0.186, 0.005, 0.2604, 0.0, 0.0, 0.0009, 0.006, 0.111, 0.0944, 0.0}}},
    {{{3.281, 0.822, 0.0, 0.015, 0.231, 0.0475, 0.0, 0.0, 0.044, 0.066, 0.0336, 0.02},
      {3.544, 0.767, 0.166, 0.0002, 0.1213, 0.1008, 0.0, 0.0024, 0.0445, 0.0743, 0.0437, 0.031}},
     {{3.937, 0.906, 0.0, 0.0037, 0.2598, 0.0, 0.0, 0.0, 0.0467, 0.0394, 0.0992, 0.0},
      {4.444, 0.427, 0.0777, 0.0046, 0.261, 0.0, 0.0, 0.0063, 0.0318, 0.089, 0.0797, 0.0}}}};
constexpr M16Time kM16TimeEight[2][2] = {
    {{4.316, 0.764, 0.0, 0.025, 0.09, 0.008, 0.0, 0.0, 0.0214, 0.071, 0.0786, 0.191},
     {4.984, 0.951, 0.13, 0.0037, 0.0552, 0.0332, 0.0808, 0.0031, 0.0325, 0.059, 0.0546, 0.182}},
    {{3.779, 0.67, 0.0, 0.0155, 0.0974, 0.0, 0.0, 0.0, 0.0395, 0.0403, 0.0698, 0.2547},
     {4.132, 1.115, 0.0, 0.0121, 0.0, 0.0623, 0.0364, 0.0117, 0.0245, 0.015, 0.0565, 0.2277}}};

// 0: no estimate (more workgroups than the CUs hold at once).
inline double m16_time(bool half, const M16Cut& c, int m, bool g128, double mbytes, int cus)
{
    const double load = (double)c.wgs / cus;
    if (load > (c.wk == 8 ? 1.0 : 2.0)) return 0.0;
    const bool many = load > 1.0;
    const int rows = m <= 4 ? 4 : (m <= 8 ? 8 : 16);
    const M16Time& t = c.wk == 8 ? kM16TimeEight[half][m > 4] : kM16TimeFour[half][many][m > 4];
    double us = t.start + t.longest * c.longest + t.younger * c.younger + t.mean * c.mean + t.mean_busy * c.mean * load +
                t.rows * rows * c.longest * (many ? load : 1.0) + (g128 ? t.group * c.longest : 0.0) + t.mbytes * mbytes;
    const double over6 = 1.7 * c.longest6 - c.longest;
    if (over6 > 0.0) us += t.fp6 * over6;
    if (c.ks > 1) us += t.split + t.part * c.ks + t.part_rows * c.ks * m;
    // (a grid of exactly, or all but, as many workgroups as fit one or two to a CU: 3 and 6 % over the estimate on average)
    const long long room = many ? 2LL * cus : cus;
    if (c.wgs > room - room / 32) us *= many ? 1.06 : 1.03;
    return us;
}

}  // namespace fp6m
