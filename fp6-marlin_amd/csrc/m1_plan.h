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
// workgroups (shares of all CUs).  [ring of four steps][workgroups beyond one, two per CU, or eight waves].
struct M1Time {
    double start, split, part, longest, younger, mean, fp6, mbytes, group, edge;
};
constexpr M1Time kM1Time[2][4] = {
    {{2.591, 0.534, 0.0131, 0.490, 0.0, 0.221, 0.125, 0.0457, 0.0380, 0.0},
     {2.850, 0.765, 0.0049, 0.398, 0.0, 0.174, 0.220, 0.0892, 0.0601, 1.137},
     {2.770, 0.889, 0.0256, 0.372, 0.0, 0.238, 0.343, 0.1144, 0.0929, 0.0},
     {2.975, 0.522, 0.0219, 0.178, 0.067, 0.542, 0.253, 0.0523, 0.0441, 4.187}},
    {{2.730, 0.484, 0.0148, 0.309, 0.0, 0.233, 0.331, 0.0438, 0.0424, 0.0},
     {3.074, 0.738, 0.0032, 0.275, 0.0, 0.168, 0.233, 0.1046, 0.0640, 0.341},
     {2.819, 0.868, 0.0210, 0.341, 0.0, 0.547, 0.298, 0.0968, 0.0917, 0.0},
     {3.103, 0.489, 0.0182, 0.041, 0.188, 0.472, 0.368, 0.0595, 0.0487, 5.588}}};

// The best cut of one row over k = 128 * units, n4 INT4 and qc FP6 columns that is resident at once: one workgroup of eight waves
// or three of four per CU.
inline M1Plan m1_plan(int units, long long n4, long long qc, bool g128, int cus, int young_pct)
{
    M1Plan best{0, 0, 0, 0, 0, 0.0};
    const double mbytes = 128.0 * units * (n4 * 0.5 + qc * 0.75) * 1e-6;
    for (int wk = 4; wk <= 8; wk += 4)
        for (long long ks4 = 1; ks4 <= 16 && ks4 * wk <= units; ks4++)
            for (int fine = 1; fine <= (qc ? 2 : 1); fine++) {
                const long long ks6 = fine * ks4, wgs = n4 / 64 * ks4 + qc / 64 * ks6;
                if (ks6 * wk > units || wgs > (wk == 8 ? 1LL : 3LL) * cus) continue;
                const M1Slices s = m1_slices(units, wk, ks4, ks6, n4 > 0, qc > 0, young_pct);
                if (!s.fit) continue;
                const long long edge = (wk == 8 ? cus : 2LL * cus) - cus / 16;
                for (int four = 0; four < 2; four++) {
                    const M1Time& t = kM1Time[four][wk == 8 ? 3 : (int)((wgs - 1) / cus)];
                    double us = t.start + t.part * ks4 + t.longest * s.longest4 + t.younger * s.younger4 +
                                t.mean * units / (double)(ks4 * wk) + t.mbytes * mbytes;
                    if (ks4 > 1) us += t.split;
                    if (g128) us += t.group * s.longest4;
                    if (1.7 * s.longest6 > s.longest4) us += t.fp6 * (1.7 * s.longest6 - s.longest4);
                    if (wgs > edge) us += t.edge * (wgs - edge) / (double)cus;
                    if (best.us == 0.0 || us < best.us) best = M1Plan{3 + four, wk, ks4, ks6, wgs, us};
                }
            }
    return best;
}

// The same of gemm_sk_kernel's launch (the same shapes, to 4 %).
inline double sk_time(int units, long long n4, long long qc, bool g128)
{
    const double mbytes = 128.0 * units * (n4 * 0.5 + qc * 0.75) * 1e-6, tiles = (n4 + qc) / 128.0;
    return 4.137 + (g128 ? 0.1656 : 0.1511) * mbytes + 0.0061 * units + 0.00116 * tiles + 0.1546 * units / tiles + 0.0261 * qc / 256.0;
}

}  // namespace fp6m
