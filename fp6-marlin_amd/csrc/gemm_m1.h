// gemm_m1_kernel: one row on tiles of 64 columns, a workgroup per tile and k part (fp6m_gemm.hip).
#pragma once
#include "gemm_m16h.h"
#include "m1_plan.h"

namespace fp6m {

// ------------------------------------------------------------------------------------------------ one row, 64-column tiles
//
// A workgroup of four or eight waves is one tile of 64 columns x consecutive k slices; the slices meet through LDS, and where a
// tile has several k parts these meet in its cells, one atomic per column and workgroup.  gemm_sk_kernel cuts a tile of 128
// columns into one-wave workgroups and pays a returning atomic per column and wave, eight to thirty times as many, and a
// thousand workgroups to dispatch; it keeps the problems that are not resident here at once (m1_plan.h).
// us in a graph, one-wave workgroups -> this: 4096 x 4096 5.8 -> 5.2, 4096 x 12288 8.7 -> 7.4,
// 11008 x 4096 8.3 -> 7.8, 8192 x 8192 10.5 -> 9.5, 24192 x 2048 12.6 -> 7.5; 789 random shapes 12 % on average.
//
// What bounds it is the launch (3 us), then requests in flight -- where more is worse: a CU with eight waves wants two or three
// steps of 2 KiB each.  A ring of eight steps, whole slices in flight, was 5 % (4096 x 4096) to 16 % (4096 x 12288) slower
// than one of three or four: queued deeper, the memory system serves some waves to their end before others begin, and the
// last ones' dequantisation is left over.
//
// All of a slice that is not packed words is fetched in front: its activations (128 bytes a step), and up to eight groups' scales
// with one load.  The loop's waits then count words alone, and know how many steps are left: nothing is fetched twice.  Step,
// lanes and columns as in stream_half (gemm_m16h.h); every MFMA column holds the same row.
struct M1Args {
    const uint16_t* A;
    const uint32_t* b_int4;
    const uint32_t* b_fp6_2;
    const uint32_t* b_fp6_4;
    const uint16_t* s_int4;   // per column (permuted order) or [k/128][n4] group scales
    const uint16_t* s_fp6;
    uint16_t* C;
    unsigned long long* cells;
    int n4, qc;
    int groups6, groups4;     // 64-column tiles per region; FP6 first in the grid and among the cells
    int ks6, ks4;             // k parts per tile
    WaveRule rule6, rule4;    // units of 128 rows
    FastDiv div6, div4;       // by groups6 / groups4
    // fp6m_mul_fused (the build with EXTRAS)
    const int32_t* c_cols;
    const uint16_t* bias;
    const uint16_t* residual;
    int n, native;            // (words in gfx950 order: EXTRAS as well)
    const int32_t* a_cols;    // (a row of `lda` activations, of which the weight's rows take these)
    int lda;
    size_t tile4, tile2;      // bytes of a tile of 128 columns in that order, per k-block of 1024 (512)
#ifdef FP6M_TIMELINE
    unsigned long long* timeline;   // performance debugging builds only
#endif
};

constexpr int kM1ABytes = kM1Steps * 128;
constexpr int kM1ScaleBytes = kM1Steps / 2 * 128;         // group scales of a slice; or the tile's column scales
constexpr int m1_wave_lds(int d4, int d6) { return max3(d4 * 2048, d6 * 3072, 0) + kM1ABytes + kM1ScaleBytes; }

// One wave's slice: `steps` (even, 2 .. kM1Steps) steps of 64 rows of a 64-column tile.  base4 / base2: the slice's first k-block
// of the planes, row4 / row2: bytes between k-blocks; base_gs: the slice's first group's scales, gs_row bytes apart.  `native`:
// gfx950 order (see stream_half).
// STAGED: with the gather, from a row that the workgroup has fetched to LDS whole with a few wide loads.  (From memory it costs a
// cycle of the CU's address unit per element, 11008 x 4096 2.6 us on 7.7; from LDS next to nothing.)
constexpr int kM1RowBytes = 28 * 1024;                    // two workgroups of four waves still share a CU
struct M1Gather {
    const int32_t* map;       // of the slice's rows of k
    int lda;
    uint32_t row_lds;         // the staged row
};
template <bool FP6, bool GROUP, int DEPTH, bool STAGED>
__device__ __forceinline__ void stream_m1(const M1Args& p, const unsigned char* base4, uint32_t row4, const unsigned char* base2, uint32_t row2,
                                          const unsigned char* base_a, const unsigned char* base_gs, uint32_t gs_row,
                                          unsigned char* ring, unsigned char* a_lds, unsigned char* gs_lds, int steps, bool native, const M1Gather& gather, f4 (&acc)[4])
{
    constexpr int kSlot = FP6 ? 3072 : 2048;
    constexpr int kOps = FP6 ? 3 : 2;
    constexpr int kReads = FP6 ? 12 : 8;                  // LDS reads per step
    const int lane = threadIdx.x & 63;
    const int i = lane >> 4, c = lane & 15, b = c >> 3, l = c & 7;

    DequantConsts kc;
    kc.lo = vgpr_const(0x000f000fu);
    kc.hi = vgpr_const(0x00f000f0u);
    kc.ex = vgpr_const(0x64006400u);
    kc.top2 = vgpr_const(0xc0c0c0c0u);
    kc.exp_man = vgpr_const(0x9f009f00u);

    // ---- fetch side
    const int lg = lane & 31;
    const int o4 = lg ^ ((lg >> 3) & 3);
    const uint32_t v4 = (uint32_t)(lane >> 5) * row4 + (native ? 16 * (o4 & 3) + (o4 >> 2) : o4) * 16;
    const uint32_t v2 = (uint32_t)(lane >> 4) * row2 + (native ? 128 * ((lane >> 2) & 3) + 16 * (lane & 3) : 16 * (lane & 15));
    int issued = 0, slot_in = 0;
    auto issue = [&]() {
        unsigned char* dst = ring + slot_in * kSlot;
        dma16_stream(base4 + v4, dst);
        dma16_stream(base4 + 2 * (size_t)row4 + v4, dst + 1024);
        if (FP6) dma16_stream(base2 + v2, dst + 2048);
        issued++;
        slot_in = slot_in + 1 == DEPTH ? 0 : slot_in + 1;
        base4 += 4 * (size_t)row4;
        base2 += 4 * (size_t)row2;
    };
    // The gather: the map's entries in front of the first words, the values behind them, so that the one latency more than a
    // slice's own activations need begins while the words are under way.  (Lane `lane` fetches row 64 t + lane of the slice.)
    uint32_t entry[kM1Steps];
    auto some = [&](auto&& f) {                           // steps in fours (a slice has two at least)
#pragma unroll
        for (int t0 = 0; t0 < kM1Steps; t0 += 4)
            if (t0 < steps) {
#pragma unroll
                for (int t = t0; t < t0 + 4; t++) f(t);
            }
    };
    if constexpr (STAGED) {
        const uint32_t last = 64u * steps - 1;            // (past the slice's end: its last row again)
        some([&](int t) {
            const uint32_t row = 64u * t + lane;
            asm volatile("global_load_dword %0, %1, %2" : "=&v"(entry[t]) : "v"(4 * (row < last ? row : last)), "s"(gather.map) : "memory");
        });
    } else {
        const uint32_t last = 128u * steps - 16, at = 16u * lane;
        dma16(base_a + (at < last ? at : last), a_lds);
        if (steps > 8) dma16(base_a + (1024 + at < last ? 1024 + at : last), a_lds + 1024);
    }
    if (GROUP) {
        const int g = lane >> 3, gl = steps / 2 - 1;
        dma16(base_gs + (size_t)(g < gl ? g : gl) * gs_row + 16 * (lane & 7), gs_lds);
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; d++)
        if (d < steps) issue();
    if constexpr (STAGED) {
        wait_steps<kOps, false, false, DEPTH - 1>(issued);              // (and this wave's piece of the staged row)
        __builtin_amdgcn_s_barrier();                     // (every wave of the workgroup passes one: see the kernel)
        some([&](int t) {
            asm volatile("" : "+v"(entry[t]));
            int col = (int)entry[t];
            col = col < 0 ? 0 : (col >= gather.lda ? gather.lda - 1 : col);
            asm volatile("ds_read_u16 %0, %1" : "=&v"(entry[t]) : "v"(gather.row_lds + 2u * (uint32_t)col) : "memory");
        });
        __builtin_amdgcn_s_waitcnt(lgkmcnt_only(0));
        some([&](int t) {
            asm volatile("" : "+v"(entry[t]));
            asm volatile("ds_write_b16 %0, %1" : : "v"(lds_addr(a_lds) + 128 * t + 2 * lane), "v"(entry[t]) : "memory");
        });
    }

    // ---- read side
    const int owner = 4 * l + i;
    const uint32_t ring_lds = lds_addr(ring);
    const uint32_t rd4 = ring_lds + (owner ^ ((owner >> 3) & 3)) * 16 + 8 * b;
    const uint32_t rd2 = ring_lds + 2048 + (native ? 8 * i + l : owner) * 8 + 4 * b;
    uint32_t rda = lds_addr(a_lds) + 4 * i;
    const int q = i;
    uint32_t rdgs = lds_addr(gs_lds) + (32 * (q >> 1) + 4 * (q & 1)) * 2;

    struct Regs {
        u2 q[4];
        uint32_t t[4];
        u2 a[4];
    };
    int slot_rd = 0;
    auto fetch = [&](Regs& r) {
        const uint32_t so = slot_rd * kSlot;
        asm volatile(
            "ds_read_b64 %0, %4\n\tds_read_b64 %1, %4 offset:512\n\tds_read_b64 %2, %4 offset:1024\n\tds_read_b64 %3, %4 offset:1536"
            : "=&v"(r.q[0]), "=&v"(r.q[1]), "=&v"(r.q[2]), "=&v"(r.q[3]) : "v"(rd4 + so) : "memory");
        if (FP6)
            asm volatile(
                "ds_read_b32 %0, %4\n\tds_read_b32 %1, %4 offset:256\n\tds_read_b32 %2, %4 offset:512\n\tds_read_b32 %3, %4 offset:768"
                : "=&v"(r.t[0]), "=&v"(r.t[1]), "=&v"(r.t[2]), "=&v"(r.t[3]) : "v"(rd2 + so) : "memory");
        asm volatile("ds_read2_b32 %0, %4 offset1:4\n\tds_read2_b32 %1, %4 offset0:8 offset1:12\n\t"
                     "ds_read2_b32 %2, %4 offset0:16 offset1:20\n\tds_read2_b32 %3, %4 offset0:24 offset1:28"
                     : "=&v"(r.a[0]), "=&v"(r.a[1]), "=&v"(r.a[2]), "=&v"(r.a[3]) : "v"(rda) : "memory");
        rda += 128;
        slot_rd = slot_rd + 1 == DEPTH ? 0 : slot_rd + 1;
    };
    auto settle = [&](Regs& r) {
        asm volatile("" : "+v"(r.q[0]), "+v"(r.q[1]), "+v"(r.q[2]), "+v"(r.q[3]));
        if (FP6) asm volatile("" : "+v"(r.t[0]), "+v"(r.t[1]), "+v"(r.t[2]), "+v"(r.t[3]));
        asm volatile("" : "+v"(r.a[0]), "+v"(r.a[1]), "+v"(r.a[2]), "+v"(r.a[3]));
    };
    auto compute = [&](const Regs& r, f4 (&dst)[4], bool fresh) {
        const f4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const h8 av = __builtin_bit_cast(h8, u4{r.a[2 * h][0], r.a[2 * h][1], r.a[2 * h + 1][0], r.a[2 * h + 1][1]});
            const bool first = fresh && h == 0;
#pragma unroll
            for (int jp = 0; jp < 2; jp++) {
                h2 r0[4], r1[4];
                if (FP6) {
                    dequant_fp6_fast(r.t[2 * h] << (4 * jp), r.q[2 * h][jp], kc, r0);
                    dequant_fp6_fast(r.t[2 * h + 1] << (4 * jp), r.q[2 * h + 1][jp], kc, r1);
                } else {
                    dequant_int4_fast(r.q[2 * h][jp], kc, r0);
                    dequant_int4_fast(r.q[2 * h + 1][jp], kc, r1);
                }
                const h8 w_lo = join(r0[0], r0[1], r1[0], r1[1]);  // columns 32b + 16jp + l
                const h8 w_hi = join(r0[2], r0[3], r1[2], r1[3]);  // ... + 8
                dst[2 * jp + 0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w_lo, av, first ? zero : dst[2 * jp + 0], 0, 0, 0);
                dst[2 * jp + 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w_hi, av, first ? zero : dst[2 * jp + 1], 0, 0, 0);
            }
        }
    };

    Regs regs[2];
    wait_steps<kOps, false, false, DEPTH - 2>(issued - 1);
    FP6M_MARK(p, 1);
    fetch(regs[0]);
    f4 grp[4];
#pragma unroll 1
    for (int s = 0; s < steps; s += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (issued < steps) issue();                          // step s+u+DEPTH-1, to the slot that step s+u-1 was read from
            wait_steps<kOps, false, false, DEPTH - 2>(issued - (s + u + 2));    // step s+u+1 has landed (past the end: all has)
            fetch(regs[(u + 1) & 1]);                             // (past the end: bytes that nobody uses)
            __builtin_amdgcn_s_waitcnt(lgkmcnt_only(kReads));     // reads of step s+u (older) are done
            settle(regs[u & 1]);
            if (GROUP)
                compute(regs[u & 1], grp, u == 0);
            else
                compute(regs[u & 1], acc, false);
        }
        if (GROUP) {
            u2 sv[4];
            asm volatile(
                "ds_read_b64 %0, %4\n\tds_read_b64 %1, %4 offset:16\n\tds_read_b64 %2, %4 offset:32\n\t"
                "ds_read_b64 %3, %4 offset:48\n\ts_waitcnt lgkmcnt(0)"
                : "=&v"(sv[0]), "=&v"(sv[1]), "=&v"(sv[2]), "=&v"(sv[3]) : "v"(rdgs) : "memory");
            rdgs += 128;
            settle(regs[0]);                                      // lgkmcnt(0) also completed the look-ahead reads
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const h2 lo = as_h2(sv[t][0]), hi = as_h2(sv[t][1]);
                acc[t][0] += (float)lo[0] * grp[t][0];
                acc[t][1] += (float)lo[1] * grp[t][1];
                acc[t][2] += (float)hi[0] * grp[t][2];
                acc[t][3] += (float)hi[1] * grp[t][3];
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0) & lgkmcnt_only(0));  // (the epilogue reuses the ring)
    settle(regs[0]);
    if (FP6) {
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t] *= 4096.0f;            // the deferred e3m2 exponent re-bias
    }
}

// EXTRAS: the build with map, bias, residual and gfx950 order.  STAGED: with the gather as well.
template <bool G128, int WK, int D4, int D6, bool EXTRAS, bool STAGED>
__global__ __launch_bounds__(64 * WK, 2) void gemm_m1_kernel(const M1Args p)
{
    constexpr int kWaveLds = m1_wave_lds(D4, D6), kRing = kWaveLds - kM1ABytes - kM1ScaleBytes;
    constexpr int kRow = STAGED ? kM1RowBytes : 0;
    static_assert((8 / WK) * (WK * kWaveLds + kRow) <= 160 * 1024, "LDS of one CU");
    __shared__ __attribute__((aligned(16))) unsigned char smem[WK * kWaveLds + kRow];

    asm volatile("" : : "s"(p.A), "s"(p.b_int4), "s"(p.b_fp6_2), "s"(p.b_fp6_4), "s"(p.s_int4), "s"(p.s_fp6), "s"(p.C), "s"(p.cells),
                        "s"(p.n4), "s"(p.qc), "s"(p.groups6), "s"(p.groups4), "s"(p.ks6), "s"(p.ks4), "s"(gridDim.x));
    asm volatile("" : : "s"(p.rule6.lo), "s"(p.rule6.ly), "s"(p.rule6.eo), "s"(p.rule6.ey), "s"(p.rule4.lo), "s"(p.rule4.ly),
                        "s"(p.rule4.eo), "s"(p.rule4.ey), "s"(p.div6.d), "s"(p.div6.magic), "s"(p.div4.d), "s"(p.div4.magic));
    if constexpr (EXTRAS)
        asm volatile("" : : "s"(p.native), "s"(p.tile4), "s"(p.tile2), "s"(p.n), "s"(p.c_cols), "s"(p.bias), "s"(p.residual));
    if constexpr (STAGED) asm volatile("" : : "s"(p.a_cols), "s"(p.lda));
    FP6M_MARK(p, 0);
#ifdef FP6M_TIMELINE
    if (p.timeline && threadIdx.x < 64) {                         // waves per workgroup, and where this one runs: XCC_ID and HW_ID
        const uint32_t hw = __builtin_amdgcn_s_getreg((4 << 0) | (0 << 6) | (31 << 11));
        const uint32_t xcc = __builtin_amdgcn_s_getreg((20 << 0) | (0 << 6) | (3 << 11));
        p.timeline[(size_t)blockIdx.x * 8 + 5] = ((unsigned long long)WK << 40) | ((unsigned long long)xcc << 32) | hw;
    }
#endif
    const int lane = threadIdx.x & 63;
    const int wk = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int logical = xcd_contiguous_id(blockIdx.x, gridDim.x);
    const int wgs6 = p.groups6 * p.ks6;
    const bool fp6 = logical < wgs6;
    const int local = fp6 ? logical : logical - wgs6;
    const int groups = fp6 ? p.groups6 : p.groups4, ks = fp6 ? p.ks6 : p.ks4;
    const FastDiv div = {fp6 ? p.div6.d : p.div4.d, fp6 ? p.div6.magic : p.div4.magic};
    const int part = fast_div(div, local);                        // part-major: neighbours share k, adjoin in n
    const int group = local - part * groups;
    const WaveRule rule = {fp6 ? p.rule6.lo : p.rule4.lo, fp6 ? p.rule6.ly : p.rule4.ly, fp6 ? p.rule6.eo : p.rule4.eo,
                           fp6 ? p.rule6.ey : p.rule4.ey};
    const int unit = __builtin_amdgcn_readfirstlane(wave_rule_begin(rule, WK, part, wk));
    const int steps = 2 * (__builtin_amdgcn_readfirstlane(wave_rule_begin(rule, WK, part, wk + 1)) - unit);
    const bool column_scales = fp6 || !G128;
    unsigned char* ring = smem + wk * kWaveLds;
    unsigned char* a_lds = ring + kRing;
    unsigned char* gs_lds = a_lds + kM1ABytes;

    if (column_scales && wk == 0)                                 // (128 bytes, twice: the region may end with them)
        dma4(reinterpret_cast<const unsigned char*>(fp6 ? p.s_fp6 : p.s_int4) + 128 * (size_t)group + 4 * (lane & 31), gs_lds);
    if constexpr (STAGED) {
        const uint32_t bytes = 2u * (uint32_t)p.lda;              // (a multiple of 16)
        for (uint32_t o = 1024u * wk; o < bytes; o += 1024u * WK) {
            const uint32_t at = o + 16 * lane;
            dma16(reinterpret_cast<const unsigned char*>(p.A) + (at < bytes ? at : bytes - 16), smem + WK * kWaveLds + o);
        }
    }
    f4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; t++) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    if (steps > 0) {
        const unsigned char* base_a = reinterpret_cast<const unsigned char*>(p.A) + 256 * (size_t)unit;
        const bool native = EXTRAS && p.native != 0;
        const M1Gather gather = {STAGED ? p.a_cols + 128 * (size_t)unit : nullptr, STAGED ? p.lda : 0, lds_addr(smem + WK * kWaveLds)};
        const size_t at4 = native ? (group >> 1) * p.tile4 + 128 * (group & 1) : 512 * (size_t)group;
        const size_t at2 = native ? (group >> 1) * p.tile2 + 64 * (group & 1) : 256 * (size_t)group;
        if (fp6) {
            const uint32_t row4 = native ? 1024 : 8 * (uint32_t)p.qc, row2 = native ? 512 : 4 * (uint32_t)p.qc;
            stream_m1<true, false, D6, STAGED>(p, reinterpret_cast<const unsigned char*>(p.b_fp6_4) + at4 + 8 * (size_t)unit * row4, row4,
                                       reinterpret_cast<const unsigned char*>(p.b_fp6_2) + at2 + 8 * (size_t)unit * row2, row2,
                                       base_a, nullptr, 0, ring, a_lds, gs_lds, steps, native, gather, acc);
        } else {
            const uint32_t row4 = native ? 1024 : 8 * (uint32_t)p.n4, gs_row = 2 * (uint32_t)p.n4;
            stream_m1<false, G128, D4, STAGED>(p, reinterpret_cast<const unsigned char*>(p.b_int4) + at4 + 8 * (size_t)unit * row4, row4,
                                       nullptr, 0, base_a,
                                       reinterpret_cast<const unsigned char*>(p.s_int4) + 128 * (size_t)group + (size_t)unit * gs_row, gs_row,
                                       ring, a_lds, gs_lds, steps, native, gather, acc);
        }
    } else if constexpr (STAGED) {
        __builtin_amdgcn_s_waitcnt(vmcnt_only(0));                // (its piece of the row, for the others)
        __builtin_amdgcn_s_barrier();
    }
    FP6M_MARK(p, 2);
    // Every lane column c holds the one row; the slab of a wave's 64 sums lies in its drained ring.
    const int q = lane >> 4;
    if ((lane & 15) == 0) {
        float* mine = reinterpret_cast<float*>(ring) + 32 * (q >> 1) + 4 * (q & 1);
#pragma unroll
        for (int t = 0; t < 4; t++) *reinterpret_cast<f4*>(mine + 16 * (t >> 1) + 8 * (t & 1)) = acc[t];
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));                    // (wave 0 without a slice: its column scales)
    __syncthreads();
    if (wk) return;
    float v = 0.f;
#pragma unroll
    for (int j = 0; j < WK; j++) v += *reinterpret_cast<const float*>(smem + j * kWaveLds + 4 * lane);
    FP6M_MARK(p, 3);
    if (column_scales) v *= (float)reinterpret_cast<const _Float16*>(gs_lds)[(lane & 32) + scale_slot(lane & 31)];
    int col = (fp6 ? p.n4 : 0) + 64 * group + lane;
    if (ks > 1) {                                                 // (the protocol, and why it holds: gemm_sk.h)
        unsigned long long* cell = p.cells + 64 * (size_t)(fp6 ? group : p.groups6 + group) + lane;
        const unsigned long long mine = cell_contribution(v);
        const unsigned long long old = __hip_atomic_fetch_add(cell, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        FP6M_MARK(p, 4);
        if ((int)(old >> 56) != ks - 1) {
            FP6M_MARK(p, 7);
            return;
        }
        v = cell_total(old, mine, ks);
        __hip_atomic_store(cell, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if constexpr (EXTRAS) {
        if (p.c_cols) {
            col = p.c_cols[col];
            col = col < 0 ? 0 : (col >= p.n ? p.n - 1 : col);
        }
        if (p.bias) v += (float)__builtin_bit_cast(_Float16, p.bias[col]);
        if (p.residual) v += (float)__builtin_bit_cast(_Float16, p.residual[col]);
    }
    p.C[col] = __builtin_bit_cast(uint16_t, (_Float16)v);
    FP6M_MARK(p, 6);
    FP6M_MARK(p, 7);
}

}  // namespace fp6m
