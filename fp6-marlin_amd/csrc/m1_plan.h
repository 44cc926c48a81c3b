// One row: which kernel, and how gemm_m1_kernel's launch is cut.  Plain host arithmetic of the dispatcher (fp6m_gemm.hip).
#pragma once
#include "mb_plan.h"

namespace fp6m {

constexpr int kM1Steps = 16;                              // of 64 rows: longest slice of a wave that gemm_m1_kernel takes

struct M1Plan {
    int depth, wk;            // ring slots of an INT4 step, waves per workgroup
    long long ks4, ks6, wgs;  // k parts per 64-column tile, workgroups
    double us;                // estimate; 0: no plan
};
// A wave's longest slices, in units of 128 rows, and whether they fit the kernel's slabs.
struct M1Slices {
    int longest4, younger4, longest6, younger6;
    bool fit;
};
inline M1Slices m1_slices(int units, int wk, long long ks4, long long ks6, bool has4, bool has6, int young_pct)
{
    const WaveRule r4 = make_wave_rule(units, ks4, wk, young_pct), r6 = make_wave_rule(units, ks6, wk, young_pct);
    M1Slices s{0, 0, 0, 0, true};
    if (has4) {
        s.longest4 = longest_older(r4);
        s.younger4 = longest_younger(r4, wk);
    }
    if (has6) {
        s.longest6 = longest_older(r6);
        s.younger6 = longest_younger(r6, wk);
    }
    const int most = kM1Steps / 2;
    s.fit = s.longest4 <= most && s.younger4 <= most && s.longest6 <= most && s.younger6 <= most;
    return s;
}

// The time of one launch, us: least squares without negative terms over 18000 launches, every cut that is resident at once of 789
// random shapes (k = 1024 .. 28672, n = 1024 .. 51200, no to 1024 FP6 columns, both scale modes), which they reproduce to 2-4 %.
// Terms: once; with a split; per part; per unit of 128 rows of the longest older and younger slices and of the mean one; per
// unit by which 1.7 FP6 units exceed the longest slice; per MB of weights; per unit with group scales; per CU beyond `edge`
// workgroups (shares of all CUs).  [ring of four steps][up to one, up to two workgroups per CU, eight waves].
struct M1Time {
    double start, split, part, longest, younger, mean, fp6, mbytes, group, edge;
};
constexpr M1Time kM1Time[2][3] = {
    {{2.591, 0.534, 0.0131, 0.490, 0.0, 0.221, 0.125, 0.0457, 0.0380, 0.0},
     {2.850, 0.765, 0.0049, 0.398, 0.0, 0.174, 0.220, 0.0892, 0.0601, 1.137},
     {2.975, 0.522, 0.0219, 0.178, 0.067, 0.542, 0.253, 0.0523, 0.0441, 4.187}},
    {{2.730, 0.484, 0.0148, 0.309, 0.0, 0.233, 0.331, 0.0438, 0.0424, 0.0},
     {3.074, 0.738, 0.0032, 0.275, 0.0, 0.168, 0.233, 0.1046, 0.0640, 0.341},
     {3.103, 0.489, 0.0182, 0.041, 0.188, 0.472, 0.368, 0.0595, 0.0487, 5.588}}};
// The same for FP6 columns alone, which have one ring; [.. up to three workgroups per CU, eight waves] (7900 launches, every cut of 1016 shapes, k = 1024 .. 28672, n = 1024 ..
// 48000: 2-4 %).  By the entries above, which charge parts and slices of INT4 tiles, 116 of those shapes were more than 2 % slower
// than with the one-wave kernel (3712 x 9216 10.5 us against 9.2); by these none is, nor any of 1208 calls at other random shapes.
constexpr M1Time kM1TimeFp6[4] = {{2.808, 0.528, 0.0105, 0.667, 0.0, 0.161, 0.0, 0.0469, 0.0, 0.0},
                                  {3.344, 0.742, 0.0, 0.650, 0.0, 0.172, 0.0, 0.0852, 0.0, 3.719},
                                  {2.980, 1.126, 0.0072, 0.739, 0.0, 1.114, 0.0, 0.0606, 0.0, 0.286},
                                  {3.248, 0.518, 0.0146, 0.349, 0.304, 0.392, 0.0, 0.0559, 0.0, 9.641}};

inline double m1_time(const M1Time& t, long long ks, int longest, int younger, double mean, double over6, double mbytes, bool g128, double edge)
{
    return t.start + (ks > 1 ? t.split : 0.0) + t.part * ks + t.longest * longest + t.younger * younger + t.mean * mean +
           t.fp6 * (over6 > 0.0 ? over6 : 0.0) + t.mbytes * mbytes + (g128 ? t.group * longest : 0.0) + t.edge * (edge > 0.0 ? edge : 0.0);
}

// The best cut of one row over k = 128 * units, n4 INT4 and qc FP6 columns that is resident at once: one workgroup of eight waves
// or two of four per CU.  (A third fits, but with INT4 tiles 24 of the 104 shapes that took it were more than 2 % slower than one-wave
// workgroups, 21632 x 5888 15.6 us against 14.4, and the others no more than 2 % faster on average.)
inline M1Plan m1_plan(int units, long long n4, long long qc, bool g128, int cus, int young_pct)
{
    M1Plan best{0, 0, 0, 0, 0, 0.0};
    const double mbytes = 128.0 * units * (n4 * 0.5 + qc * 0.75) * 1e-6;
    for (int wk = 4; wk <= 8; wk += 4)
        for (long long ks = 1; ks <= (n4 ? 16 : 24) && ks * wk <= units; ks++)
            for (int fine = 1; fine <= (n4 && qc ? 2 : 1); fine++) {
                const long long ks6 = fine * ks, wgs = n4 / 64 * ks + qc / 64 * ks6;
                if (ks6 * wk > units || wgs > (wk == 8 ? 1LL : (n4 ? 2LL : 3LL)) * cus) continue;
                const M1Slices s = m1_slices(units, wk, ks, ks6, n4 > 0, qc > 0, young_pct);
                if (!s.fit) continue;
                const double edge = (wgs - ((wk == 8 ? cus : 2LL * cus) - cus / 16)) / (double)cus, mean = units / (double)(ks * wk);
                const int where = wk == 8 ? (n4 ? 2 : 3) : (int)((wgs - 1) / cus);
                for (int four = 0; four < (n4 ? 2 : 1); four++) {
                    const double us = n4 ? m1_time(kM1Time[four][where], ks, s.longest4, s.younger4, mean, 1.7 * s.longest6 - s.longest4, mbytes, g128, edge)
                                         : m1_time(kM1TimeFp6[where], ks, s.longest6, s.younger6, mean, 0.0, mbytes, false, edge);
                    if (best.us == 0.0 || us < best.us) best = M1Plan{3 + four, wk, ks, ks6, wgs, us};
                }
            }
    return best;
}

// The same of gemm_sk_kernel's launch, to 4-5 %.  With INT4 tiles it is the fit over the 789 shapes; that kernel has become 3 % faster since.
inline double sk_time(int units, long long n4, long long qc, bool g128)
{
    const double mbytes = 128.0 * units * (n4 * 0.5 + qc * 0.75) * 1e-6, tiles = (n4 + qc) / 128.0;
    if (n4 == 0) return 4.352 + 0.1634 * mbytes + 0.0051 * units + 0.00224 * tiles + 0.1331 * units / tiles;
    return 4.137 + (g128 ? 0.1656 : 0.1511) * mbytes + 0.0061 * units + 0.00116 * tiles + 0.1546 * units / tiles + 0.0261 * qc / 256.0;
}

// The plan that is taken in place of gemm_sk_kernel; us = 0: none.  The margin covers what that kernel gained since its fit and 2 % of
// what the estimates miss: of 5250 calls at other random shapes (no to 1024 FP6 columns, both scale modes) 3400 take 64-column tiles
// by it, 14 % faster on average; 25 of those are more than 2 % slower, the worst 8 %.  With 6 % instead of 5 it would be fewer, but square
// shapes in whole parts, 8192 x 8192 9.4 us against 10.3, would go back.  Fewer than twelve units with a fifth or more of the columns in FP6,
// whose few waves then end last, were 2 % slower on average (1280 x 3968, 1024 of them FP6, 4.9 us against 4.5).
// Words in gfx950 order, of which a 64-column tile reads half of every tile's lines, gain 4 % less: 15 of 1096 such calls are more than
// 4 % slower than one-wave workgroups (20224 x 6272 17.5 us against 15.7).  They take what the reference's order takes, for the same bits.
inline M1Plan m1_choice(int units, long long n4, long long qc, bool g128, int cus, int young_pct)
{
    M1Plan plan = m1_plan(units, n4, qc, g128, cus, young_pct);
    if (plan.us > 0.95 * sk_time(units, n4, qc, g128) || (n4 > 0 && units < 12 && 5 * qc >= n4 + qc)) plan.us = 0.0;
    return plan;
}

}  // namespace fp6m
