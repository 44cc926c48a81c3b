// How a launch of more than 16 rows is cut: plain host arithmetic of the dispatcher (fp6m_gemm.hip).
#pragma once
#include <cstddef>

namespace fp6m {

constexpr int kWaves = 4;
constexpr int kTileN = 128;          // columns per tile

// Partial tiles that a launch may write to: the highest slot in use, plus one.  Slots are numbered row tile by row tile, FP6 tiles
// first, over all (tile, part), those of tiles in one part included, which are stored directly.
inline size_t slots_used(long long parts4, long long parts6, long long tiles4, long long tiles6, long long mtiles)
{
    const long long slots4 = tiles4 * parts4, slots6 = tiles6 * parts6;
    const long long last = parts4 > 1 && tiles4 ? slots6 + slots4 : (parts6 > 1 ? slots6 : 0);
    return last ? (size_t)((mtiles - 1) * (slots6 + slots4) + last) : 0;
}

// The k slices of a tile by wave, in units.  A workgroup of eight waves puts two on every SIMD, and the SIMD serves
// the one that arrived first (waves 0-3) ahead of the other (waves 4-7): with equal slices the second wave of every
// SIMD leaves its loop a third later than the first (8192 x 8192 at 128 rows: 14.3 against 19.6 us), and the
// workgroup's reduction waits for it.  So a part (workgroup) of a tile gives its first four waves `lo` units each and
// the others `ly` <= lo; what does not divide goes, a unit each, to the first `eo` older waves in (part, wave) order,
// then to the first `ey` younger ones.  Four-wave workgroups have older waves only.  Slices follow each other along
// k in (part, wave) order.
struct WaveRule {
    int lo, ly, eo, ey;
};
// k slices of the `ks` parts x `wk` waves of a tile.  With eight waves per workgroup and at least two units for every
// wave, the second wave of every SIMD (waves 4-7) gets `young_pct` per cent of what the first gets; otherwise all waves
// get the same.  What does not divide goes to the older waves first.
inline WaveRule make_wave_rule(long long units, long long ks, int wk, int young_pct)
{
    WaveRule r;
    if (ks < 1) ks = 1;
    const long long per_part = units / ks;
    long long lo = per_part / wk, ly = lo;
    if (wk == 8 && per_part >= 16 && young_pct > 0 && young_pct < 100) {
        lo = (per_part * 100 + 2 * (100 + young_pct)) / (4 * (100 + young_pct));     // per_part / (4 (1 + share)), rounded
        if (4 * lo > per_part) lo = per_part / 4;
        ly = (per_part - 4 * lo) / 4;
        if (ly > lo) ly = lo;
    }
    const long long rem = units - ks * (4 * lo + (wk - 4) * ly);
    r.lo = (int)lo;
    r.ly = (int)ly;
    r.eo = (int)(rem < 4 * ks ? rem : 4 * ks);
    r.ey = (int)(rem - r.eo);
    return r;
}
// Units of the longest slice among the older and among the younger waves.
inline int longest_older(const WaveRule& r) { return r.lo + (r.eo > 0); }
inline int longest_younger(const WaveRule& r, int wk) { return wk > 4 ? r.ly + (r.ey > 0) : 0; }

// How a launch of gemm_mb_kernel cuts the k range: parts per INT4 and FP6 tile, k slices (waves) per workgroup.
struct MbSplit {
    long long ks, ks6;
    int wk;
    bool too_large;           // more partial tiles than a scratch of fixed size holds
};
struct MbLaunch {
    long long tiles, tiles6;  // column tiles, and FP6 ones among them
    int mtiles, k, units;     // row tiles; rows of the weight, and in units that slices are made of (128 rows with group scales, else 64)
    int cus, sms;             // compute units; the caller's limit on parts per tile (<= 0: none)
    long long forced_parts;   // tuning hook: parts per tile (< 1: not forced), waves per workgroup (0: not forced)
    int forced_waves;
    bool row_mix, fixed_scratch;
    size_t scratch_bytes;
    int young_pct = 72;       // make_wave_rule
};

// The split of one launch of gemm_mb_kernel with tiles of 16 * mb rows (16 rows and more).
inline MbSplit mb_split(int mb, const MbLaunch& l)
{
    // m > 16: a task is one workgroup (one tile x four k slices) on one row tile and k part.
    // Split k only as far as needed to give every CU a workgroup; partial tiles are 16*MB rows
    // of fp32, so the split is also capped by their traffic relative to the weight stream.
    const int rows_per_tile = 16 * mb, units = l.units;
    const long long base = l.tiles * l.mtiles;
    const size_t tile_bytes = (size_t)rows_per_tile * kTileN * sizeof(float);
    MbSplit sp;
    long long ks = l.cus / base;
    // (two k units per wave at least, one on a short k up to four parts; a grid that leaves half of the CUs idle even
    // so may split twice as far as the partial tiles' traffic would otherwise allow: 2048 x 2560 .. 7680 at 32 and
    // 64 rows 10.4 -> 9.2-9.8 us and 13.8 -> 12.7-13.0; eight parts instead of four on k = 4096 cost 6-12 %)
    long long ks_k = units / (kWaves * 2);
    if (ks_k < 4) ks_k = units / kWaves < 4 ? units / kWaves : 4;
    if (ks_k < 1) ks_k = 1;
    long long cap = (long long)l.k / (16LL * rows_per_tile) > 0 ? (long long)l.k / (16LL * rows_per_tile) : 1;
    if (base * 2 * cap <= l.cus) cap *= 2;
    if (ks > ks_k) ks = ks_k;
    if (ks > cap) ks = cap;
    if (l.sms > 0 && ks > l.sms) ks = l.sms;
    if (l.forced_parts >= 1) ks = l.forced_parts;
    if (ks < 1) ks = 1;
    sp.too_large = l.fixed_scratch && ks > 1 && (size_t)(l.tiles + l.tiles6) * l.mtiles * ks * tile_bytes > l.scratch_bytes;
    while (ks > 1 && (size_t)(l.tiles + l.tiles6) * l.mtiles * ks * tile_bytes > l.scratch_bytes) ks--;   // (FP6 tiles: 2 ks)
    // A grid of at most one workgroup per CU would leave every SIMD a single wave: give the workgroup eight
    // k slices instead of four (same partial-sum traffic, two waves per SIMD) when k is long enough.
    // (Two waves on a SIMD take turns at its one VALU/MFMA port: eight half-length slices last as long as four
    // whole ones, so eight (which hide latency better: 13824 x 5120 at 256 rows 60.6 vs 67.8 us) only pay while
    // their longest slice, in whole k units, is no more than 0.58 of the longest of four: 5120 x 13824 at 64
    // rows, 40 units over 16 slices of up to 3: 24.1 us, over 8 slices of 5: 21.7.)
    // From forced tables (4 or 8 slices x 1 .. 8 parts, 32 / 64 / 128 rows): a split is no finer than its longest
    // slice needs (8192 x 6144 at 32 rows: 64 units in 5 parts = 20 slices of up to 4, 16.7 us; in 4 parts = 16
    // slices of 4, 16.0; as eight-wave workgroups 14.3); one unit per wave is enough for eight (8192 x 2048 at
    // 32 rows 12.8 -> 12.0); 0.58 rather than 0.55 (14336 x 8192 at 32 rows, 4 against 7 units, 23.0 -> 20.5);
    // and beyond eight parts the partners' partial tiles cost more than shorter slices gain (14336 x 2048 at
    // 32 rows: 14 parts of four slices 16.7 us, 8 parts of eight 14.8; at 64 rows 24.0 -> 21.0).
    auto longest = [&](long long slices) { return (units + slices - 1) / slices; };
    const bool free_split = l.forced_parts < 1 && l.sms <= 0 && !l.row_mix && mb != 8;
    if (free_split)
        while (ks > 1 && longest(4 * (ks - 1)) == longest(4 * ks)) ks--;
    // (32-row tiles are not issue-bound: two waves per SIMD pay up to two thirds, 11008 x 2560 at 32 rows 14.9 -> 13.2)
    const bool eight_pays = mb == 2 ? 3 * longest(8 * ks) <= 2 * longest(4 * ks) : 50 * longest(8 * ks) <= 29 * longest(4 * ks);
    int wk = base * ks <= l.cus && units / 8 >= ks && eight_pays ? 8 : kWaves;
    if (free_split && !l.forced_waves && ks > 8 && base * 8 <= l.cus && units / 8 >= 8) {
        wk = 8;
        ks = 8;
    }
    if (l.forced_waves) wk = l.forced_waves;
    if (mb == 8) wk = kWaves;                                  // (512 registers per wave: one wave per SIMD)
    // An FP6 step costs more issue slots than an INT4 one, and in a grid that is resident all at once the few
    // FP6 tiles' workgroups set the length of the launch (8192 x 8192 at m = 128: 33 us against 29 us with INT4
    // only).  Their k range is cut twice as finely where every slice still gets two units and the grid still
    // fits the CUs in one go (5120 x 13824 at m = 128: 40 -> 31 us; a grid whose last workgroups must wait for
    // a free CU loses far more than that).  A forced split applies to both kinds.
    sp.ks = sp.ks6 = ks;
    sp.wk = wk;
    // (a grid that fits one workgroup per CU must still do so afterwards: a CU with two runs both at little
    // more than half speed, 11008 x 4096 at 256 rows 34 -> 52 us with 272 workgroups)
    const long long resident = (long long)l.cus * (wk == 8 || mb == 8 || base * ks <= l.cus ? 1 : 2);
    // (Not for 128-row tiles, whose FP6 workgroups are only a few per cent behind: there the second partner's
    // partial tiles cost more than the shorter loop gains, 8192 x 8192 at m = 384 61.8 vs 58.4 us.)
    // Re-measured with every tile on the paired loop (ten shapes x 32 .. 256 rows, alternating): still 5-13 % on
    // wide weights up to two row tiles (4096 x 11008 at 128 rows 25.3 -> 22.2 us, 8192 x 28672 at 32 rows
    // 38.2 -> 34.5), but 3-8 % slower from three row tiles on (5120 x 5120 at 256 rows 27.4 -> 29.7): up to two.
    // Where twice does not fit, as finely as does (13824 x 5120 with 512 FP6 columns, per-column scales, 64 rows: 6 parts for
    // all tiles 22.1 us, 10 for the FP6 tiles 21.4).  In four-wave workgroups and beyond eight parts only if that shortens the
    // loop by 128 rows of k at least, for a wave served first or for a SIMD: with less, the additional partial tiles cost more
    // than the loop gains (3840 x 2048 at 86 rows 15.4 -> 17.4 us).
    // Two row tiles whose workgroups are a multiple of eight apart must stay so: the same part of both is then on one XCD,
    // whose L2 reads the words once (16384 x 2560 at 110 rows: 120 workgroups per row tile 23.6 us, 122 25.5).  A cut that
    // makes it a multiple is taken.
    // Random shapes from k = 2048 against no finer cut: what is cut takes 4.9 % less on 84 of 17 to 32 rows and on 35 of 49 to
    // 128 (the worst 8 % more); what is not would take 3.9 % more on 6 and 5.8 % on 21 for want of 128 rows, and 6.2 % on the 14
    // whose row tiles would come apart.
    if (l.forced_parts < 1 && !l.row_mix && l.tiles6 > 0 && mb != 8 && l.mtiles <= 2) {
        long long c6 = units / (2 * wk) < 2 * ks ? units / (2 * wk) : 2 * ks;
        const long long room = (resident - (base - l.tiles6 * l.mtiles) * ks) / (l.tiles6 * l.mtiles);
        if (c6 > room) c6 = room;
        while (c6 > ks && slots_used(ks, c6, l.tiles - l.tiles6, l.tiles6, l.mtiles) * tile_bytes > l.scratch_bytes) c6--;
        auto shared_l2 = [&](long long parts6) { return l.mtiles == 1 || ((l.tiles - l.tiles6) * ks + l.tiles6 * parts6) % 8 == 0; };
        auto pays = [&](long long parts6) {
            if (parts6 == 2 * ks) return true;
            if (shared_l2(ks) != shared_l2(parts6)) return shared_l2(parts6);
            if (wk == 8 && parts6 <= 8) return true;
            const WaveRule now = make_wave_rule(units, ks, wk, l.young_pct), cut = make_wave_rule(units, parts6, wk, l.young_pct);
            const int older = longest_older(now) - longest_older(cut), both = older + longest_younger(now, wk) - longest_younger(cut, wk);
            return (older > both ? older : both) * (long long)(l.k / units) >= 128;
        };
        while (c6 > ks && !pays(c6)) c6--;
        if (c6 > ks) sp.ks6 = c6;
    }
    return sp;
}

// The time of one launch of gemm_mb_kernel, us, for the choice among its tiles of 32, 48 and 64 rows.
//
// None of them wins everywhere: a taller tile dequantises less often and reads fewer words, a shorter one fills its rows and
// the CUs better and reduces less per workgroup.  Which of them does follows from how many workgroups there are and how long
// their slices get, so the launch is estimated from its split (least squares without negative terms, over 882 points: 28
// shapes and 130 random ones of k = 2048 .. 20480 by n = 2048 .. 40960 at 33 to 400 rows, both scale modes, none to 1024 FP6
// columns; they reproduce the times to 3-6 %).  The entry of 32-row tiles in four-wave workgroups, which only short k takes, is
// from 110 shapes of its own up to k = 3840 (3.6 %, the worst 11 %): the 882 held too few, and gave it no start (64 x 2048 x 2560
// without FP6 columns 5.4 us, measured 9.2; now 8.9).  No choice in 30000 random shapes depends on that.
// Fitted to plain calls; against the rule before, 500 random calls with bias and residual and 200 in the gfx950 word order are
// 14 % and 8 % faster on average, none more than 1.5 % slower.
// Against the one tile height that the rows suggested (64 from 49 on, or 128, or the many-rows kernel where those were
// estimated faster) the choice takes 6.4 % off over all 882 and is within 0.7 % of the best of all of them on average, where that rule
// was 7.6 % off; fitted to one half of the points it does the same on the other.  A challenger must be 5 % faster by the
// estimate.  Together with the 48-row tiles for 33 to 48 rows and the finer cut of the FP6 tiles (mb_split) it changes 326 of
// 700 other random shapes (17 to 900 rows, k to 28672, n to 57344): -12.8 % on average, 319 of them more than 1.5 % faster,
// none that much slower; and 63 of 138 with at most 28 column tiles on k from 9216 on: -13.9 %, none that much slower.
// 32-row tiles: 64 x 4096 x 4096 14.4 -> 10.9 us, 96 x 5120 x 5120 18.5 -> 14.7, 80 x 8192 x 10240 36.4 -> 28.7; 48-row
// tiles: 96 x 8192 x 8192 26.7 -> 24.1, 96 x 13824 x 5120 29.9 -> 26.7, 144 x 4096 x 12288 33.1 -> 29.3.
struct MbTime {
    // At most one workgroup per CU: us once; per k step (32 rows) of the mean and of the longest slice, and what group scales
    // and full occupation add per step; per step by which an FP6 slice exceeds 0.7 of an INT4 slice; with a split: us once,
    // per part, and for full occupation.
    double start, mean, longest, group, busy, fp6, split, part, split_busy;
};
struct MbTimeMany {
    // More: per CU two workgroups of four waves at a time.  us once; per step of a full round, and with group scales; the last
    // round up to one workgroup per CU, by occupation and once, and beyond one, once and by occupation; us per round; group
    // scales in the last round.
    double start, full, full_group, low_busy, low, high, high_busy, round, last_group;
};
constexpr MbTime kMbTimeEight[] = {{5.479, 0.322, 0.224, 0.046, 0.125, 0.181, 1.422, 0.099, 0.427},    // 32, 48, 64 rows, eight waves
                                   {6.556, 0.302, 0.268, 0.043, 0.237, 0.249, 0.924, 0.311, 0.588},
                                   {7.479, 0.488, 0.107, 0.054, 0.358, 0.284, 0.0, 0.509, 1.348}};
constexpr MbTime kMbTimeFour[] = {{6.637, 0.0, 0.427, 0.0, 0.0, 0.293, 0.0, 0.0, 0.893},               // ... four waves
                                  {6.091, 0.0, 0.429, 0.025, 0.0, 0.143, 0.312, 0.618, 0.841},
                                  {7.553, 0.032, 0.375, 0.0, 0.079, 0.102, 0.372, 0.676, 1.243}};
constexpr MbTime kMbTimeTall = {9.971, 0.0, 0.533, 0.01, 0.191, 0.224, 2.606, 0.959, 0.0};             // 128 rows
constexpr MbTimeMany kMbTimeMany[] = {{1.919, 0.91, 0.034, 0.24, 0.207, 0.749, 0.179, 1.99, 0.018},
                                      {3.003, 0.932, 0.037, 0.241, 0.172, 0.679, 0.24, 2.954, 0.066},
                                      {4.016, 1.055, 0.06, 0.289, 0.208, 0.804, 0.246, 3.459, 0.052}};
// tiles: all, tiles6 of them FP6.  No estimate for 128-row tiles beyond one workgroup per CU (0).
inline double mb_time(int mb, const MbSplit& sp, long long tiles, long long tiles6, long long mtiles, int k, int units, bool g128, int cus)
{
    const double per_unit = k / (32.0 * units), g = g128 ? 1.0 : 0.0;
    auto longest = [&](long long slices) { return (double)((units + slices - 1) / slices) * per_unit; };
    const double s = longest(sp.ks * sp.wk), mean = k / (32.0 * sp.ks * sp.wk);
    const long long base = tiles * mtiles;
    if (base * sp.ks <= cus) {
        const MbTime& c = mb == 8 ? kMbTimeTall : (sp.wk == 8 ? kMbTimeEight : kMbTimeFour)[mb - 2];
        const double busy = (double)((tiles - tiles6) * sp.ks + tiles6 * sp.ks6) * mtiles / cus;
        const double mean6 = tiles6 ? k / (32.0 * sp.ks6 * sp.wk) : 0.0, over6 = mean6 - 0.7 * mean;
        return c.start + c.mean * mean + c.longest * s + c.group * mean * g + c.busy * mean * busy + (over6 > 0 ? c.fp6 * over6 : 0.0) +
               (sp.ks > 1 ? c.split + c.part * sp.ks + c.split_busy * busy : 0.0);
    }
    if (mb == 8) return 0.0;
    const MbTimeMany& c = kMbTimeMany[mb - 2];
    const long long wgs = base * sp.ks, full = wgs / (2 * cus), rem = wgs % (2 * cus);
    double t = c.start + full * s * (c.full + c.full_group * g) + c.round * (full + (rem ? 1 : 0));
    if (rem) t += s * (c.last_group * g + (rem <= cus ? c.low + c.low_busy * rem / cus : c.high + c.high_busy * (rem - cus) / cus));
    return t;
}

}  // namespace fp6m
