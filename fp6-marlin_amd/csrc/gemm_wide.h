// gemm_wide_kernel: the kernel of fp6m_gemm.hip for many rows (waves side by side in n that share their rows of A).
#pragma once
#include "gemm_mb.h"

namespace fp6m {

// ------------------------------------------------------------------------------------------------ many rows
//
// What bounds many rows is the SIMD's one issue port for MFMAs and other vector instructions, and whether there is a
// second wave to issue while the first waits.  A wave of gemm_mb_kernel multiplies 128 columns: with 128 rows its
// accumulators are 256 registers, so it has its SIMD to itself, and every wait stops the SIMD (the MFMA pipe was busy
// 41-45 % of the time).  Here a wave multiplies 16 * MB rows x 64 columns of a k slice: a weight is still
// dequantised once per 128 rows, the accumulators are 128 registers, and two waves share a SIMD.  What the narrower wave
// would pay in activation traffic it does not, because WN waves side by side in n read one copy of A: a workgroup is
// WN column groups x WK k slices, and a slice's waves load the slice's stages of A (64 rows of k each) together into
// one ring of NS slots, with one barrier per stage.
//
// Lanes.  The packed layout's fragment owner t = 4 l + i holds 64-column group columns 16 j + l + 8 half (j = 0 .. 3) at
// k = 16 kb + {2i, 2i+1, 2i+8, 2i+9}.  Lane 16 i + 8 b + l takes words j = 2b and 2b + 1 of owner 4 l + i -- eight
// bytes per k-block, nothing loaded twice -- so that fragment (jp, half) of a step (two k-blocks) is columns
// 32 b + 16 jp + 8 half + l of the group, and dequant_entry (gemm_mb.h) applies as it is.  The words go straight to
// registers, four steps ahead (four register sets); A is read from LDS as in gemm_mb.h.
//
// One trip of the loop is 128 rows of k: two stages, four steps.  Order of a wave's loads within a trip (u = step):
//     u = 0: group scales of the next trip, words of the step four on      u = 2: words
//     u = 1: words, then at the stage's end A of NS stages on              u = 3: words, then A
// and a wait names how many of the newer ones may be outstanding.  Loads past a slice's end are repeated, so
// the counts never change.  At a stage's end, in front of its last two row blocks, a wave waits for its own part of
// the next stage's A and for its own reads of this one, meets the others at the barrier, refills the slot that
// everybody has read, and reads the next stage's first blocks behind the MFMAs of those two.
constexpr int kWideHalf = 1024;                           // from a block's first load of a stage to its second
constexpr int kWideBlock = 2 * kWideHalf;
constexpr int wide_slot_bytes(int mb) { return mb * kWideBlock; }
constexpr int wide_a_loads(int mb, int wn) { return ((2 * mb + wn - 1) / wn + 1) / 2 * 2; }

// Epilogue of the WK slices: fragments are exchanged through LDS in the lanes' own layout (each wave finishes every WK-th
// row block), as many blocks at a time as fit the ring's memory beside a slab of 16 rows x 64 fp16 per wave.
constexpr int kWideSlabRow = 64 * 2 + 16;                 // bytes of one row of the slab
constexpr int wide_round_bytes(int wn, int wk) { return wk == 1 ? 0 : wn * wk * wk * 4096; }
constexpr int wide_slab_bytes(int wn, int wk) { return wn * wk * 16 * kWideSlabRow; }
constexpr int wide_lds_bytes(int mb, int wn, int wk)
{
    return max3(wk * 3 * wide_slot_bytes(mb), wide_round_bytes(wn, wk) + wide_slab_bytes(wn, wk), 0);
}

template <bool FP6, bool G128, int MB, int WN, typename Args>
__device__ __forceinline__ void wide_stream(const Args& p, const TileInfo& ti, int sigma, int wn, uint32_t ring, int trip_begin,
                                            int trips, int most_trips, f4 (&acc)[MB][4])
{
    constexpr bool kGroup = G128 && !FP6;
    constexpr int kEPP = dequant_entries_per_pair<FP6, kGroup>();
    constexpr int kEntries = 4 * kEPP;
    constexpr int nA = wide_a_loads(MB, WN), nW = FP6 ? 4 : 2, nS = kGroup ? 4 : 0;
    constexpr int kSlot = wide_slot_bytes(MB);
    constexpr int kAhead = MB > 3 ? 3 : MB - 1;           // row blocks of A read ahead of the one being multiplied
    static_assert(MB >= 2 && nA % 2 == 0, "A's loads are dealt to the two steps of a stage");
    // newer loads that may be outstanding when the words of step u + 1 must have landed
    constexpr int kWordWait = 3 * nW + 3 * (nA / 2);      // (+ nS, but in the step after the scales went out with those words)
    // ... when the next stage's A must have: what this stage issued
    constexpr int kStageWait = 2 * nW + nA;               // (+ nS in a trip's first stage)
    static_assert(kWordWait + nS <= 63, "vmcnt is a 6-bit counter");
    const int lane = threadIdx.x & 63;
    const int i = lane >> 4, c = lane & 15, b = c >> 3, l = c & 7;
    const uint32_t ex = vgpr_const(0x64006400u), b72 = vgpr_const(0xd480d480u);

    // ---- fetch side: uniform bases on the scalar unit, constant lane offsets
    const PlaneGeometry geo = plane_geometry(p, ti);
    const size_t row4 = geo.row4, row2 = geo.row2;
    const int owner = p.native ? 16 * i + 8 * sigma + l : 32 * sigma + 4 * l + i;
    const uint32_t v4 = (uint32_t)owner * 16 + 8 * b, v4b = v4 + (uint32_t)row4;
    const uint32_t v2 = (uint32_t)owner * 8 + 4 * b, v2b = v2 + (uint32_t)row2;
    const unsigned char* base4 = uniform_ptr(reinterpret_cast<const unsigned char*>(FP6 ? p.b_fp6_4 : p.b_int4) + geo.tile4 +
                                             (size_t)(8 * trip_begin) * row4);
    const unsigned char* base2 = uniform_ptr(reinterpret_cast<const unsigned char*>(p.b_fp6_2) + geo.tile2 +
                                             (size_t)(8 * trip_begin) * row2);
    u2 wq[4][2];                                          // [register set][k-block]
    uint32_t tq[4][2];
    int words_left = 4 * trips - 1;                       // steps beyond the one fetched next
    auto issue_w = [&](u2 (&q)[2], uint32_t (&t)[2]) {
        asm volatile("global_load_dwordx2 %0, %2, %4\n\tglobal_load_dwordx2 %1, %3, %4"
                     : "=&v"(q[0]), "=&v"(q[1]) : "v"(v4), "v"(v4b), "s"(base4) : "memory");
        if (FP6)
            asm volatile("global_load_dword %0, %2, %4\n\tglobal_load_dword %1, %3, %4"
                         : "=&v"(t[0]), "=&v"(t[1]) : "v"(v2), "v"(v2b), "s"(base2) : "memory");
        if (words_left > 0) {                             // (uniform; past the end the last step is fetched again)
            words_left--;
            base4 += 2 * row4;
            base2 += 2 * row2;
        }
    };
    // A: load q of a stage brings rows 8q .. 8q+7, eight lanes (128 bytes) per row, as in gemm_mb.h; wave wn issues loads
    // wn, wn + WN, ..  (beyond the last: the last again, to the same place).
    const int tile_row0 = ti.mtile * 16 * MB;
    const int prow = lane >> 3, pch = lane & 7;
    uint32_t va[nA];
#pragma unroll
    for (int x = 0; x < nA; x++) {
        int q = wn + WN * x;
        q = q < 2 * MB ? q : 2 * MB - 1;
        int row = tile_row0 + 8 * q + prow;
        row = row < p.m ? row : p.m - 1;
        va[x] = (uint32_t)(row - tile_row0) * (uint32_t)p.k * 2 + 16 * (pch ^ prow);
    }
    const unsigned char* base_a = uniform_ptr(reinterpret_cast<const unsigned char*>(p.A + (size_t)tile_row0 * p.k) + (size_t)trip_begin * 256);
    int stages_left = 2 * trips - 1;
    uint32_t fill = ring;                                 // slot that the next stage of A goes to
    auto issue_a = [&](auto xx) {                         // one load of the stage; the last one moves on
        constexpr int x = decltype(xx)::value;
        int q = wn + WN * x;
        q = q < 2 * MB ? q : 2 * MB - 1;
        set_m0(fill + (q >> 1) * kWideBlock + (q & 1) * kWideHalf);
        dma16_m0<0, false>(base_a, va[x]);
        if constexpr (x == nA - 1) {
            fill = fill == ring + 2 * kSlot ? ring : fill + kSlot;
            if (stages_left > 0) {
                stages_left--;
                base_a += 128;
            }
        }
    };
    const unsigned char* base_gs = uniform_ptr(reinterpret_cast<const unsigned char*>(p.s_int4 + (size_t)ti.tcol * kTileN + 64 * sigma) +
                                               (size_t)trip_begin * (size_t)uniform32(p.n4) * 2);
    const uint32_t vgs = (32 * b + l) * 2;
    uint32_t gs[4], gs_next[4];                           // group scale of fragment 2 jp + half
    int groups_left = trips - 1;
    auto issue_scales = [&]() {
        asm volatile(
            "global_load_ushort %0, %4, %5\n\tglobal_load_ushort %1, %4, %5 offset:16\n\t"
            "global_load_ushort %2, %4, %5 offset:32\n\tglobal_load_ushort %3, %4, %5 offset:48"
            : "=&v"(gs_next[0]), "=&v"(gs_next[1]), "=&v"(gs_next[2]), "=&v"(gs_next[3]) : "v"(vgs), "s"(base_gs) : "memory");
        if (groups_left > 0) {
            groups_left--;
            base_gs += (size_t)uniform32(p.n4) * 2;
        }
    };
    auto settle_scales = [&]() {
#pragma unroll
        for (int f = 0; f < 4; f++) {
            asm volatile("" : "+v"(gs_next[f]));
            gs[f] = gs_next[f] | (gs_next[f] << 16);
        }
    };

    // ---- read side
    uint32_t rd[4], abuf[4][4];
    uint32_t slot = ring;                                 // of the stage being multiplied
#pragma unroll
    for (int d = 0; d < 4; d++) rd[d] = ring + (c >> 3) * kWideHalf + (8 * (c & 7) + (d ^ (c & 7))) * 16 + 4 * i;

    DequantRegs dq = {};
    h8 frag[2][8];                                        // (four used: 2 jp + half)
    auto entries = [&](auto first, auto last, u2 (&q)[2], uint32_t (&t)[2], h8 (&out)[8]) {
        constexpr int e0 = decltype(first)::value, e1 = decltype(last)::value;
        static_for<e0, e1>([&](auto e) {
            constexpr int E = decltype(e)::value, pr = E / kEPP, jp = pr >> 1;
            dequant_entry<FP6, kGroup, E>(dq, q[0][jp], q[1][jp], FP6 ? t[0] : 0u, FP6 ? t[1] : 0u, kGroup ? as_h2(gs[pr]) : h2{}, ex, b72, out);
        });
    };

    // Prologue: two stages of A and four steps of words in the order in which the loop would have issued them, which is
    // what its waits count on; the first trip's scales; then the first step's fragments.
    if (kGroup) issue_scales();
    issue_w(wq[0], tq[0]);
    static_for<0, nA / 2>(issue_a);
    issue_w(wq[1], tq[1]);
    static_for<nA / 2, nA>(issue_a);
    issue_w(wq[2], tq[2]);
    static_for<0, nA / 2>(issue_a);
    issue_w(wq[3], tq[3]);
    static_for<nA / 2, nA>(issue_a);
    __builtin_amdgcn_s_waitcnt(vmcnt_only(nA + 2 * nW));  // the first stage
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
    static_for<0, kAhead>([&](auto bb) { lds_read_a4<decltype(bb)::value * kWideBlock>(abuf[decltype(bb)::value], rd); });
    if (kGroup) settle_scales();
#pragma unroll
    for (int k = 0; k < 2; k++) {
        asm volatile("" : "+v"(wq[0][k]));
        if (FP6) asm volatile("" : "+v"(tq[0][k]));
    }
    entries(Int<0>{}, Int<kEntries>{}, wq[0], tq[0], frag[0]);

#pragma unroll 1
    for (int trip = 0; trip < trips; trip++) {
        static_for<0, 4>([&](auto uu) {
            constexpr int u = decltype(uu)::value;
            constexpr int phase = (u * MB) & 3;           // A buffer of the step's first block
            if (kGroup && u == 0) issue_scales();         // (in flight until this trip's last step)
            issue_w(wq[u], tq[u]);                        // step + 4: this set went into fragments during the step before
            __builtin_amdgcn_s_waitcnt(vmcnt_only(kWordWait + (u == 3 ? 0 : nS)));
            if (kGroup && u == 3) settle_scales();        // the next step starts a group
            u2 (&nq)[2] = wq[(u + 1) & 3];
            uint32_t (&nt)[2] = tq[(u + 1) & 3];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                asm volatile("" : "+v"(nq[k]));
                if (FP6) asm volatile("" : "+v"(nt[k]));
            }
            h8 (&cur)[8] = frag[u & 1];
            h8 (&nxt)[8] = frag[(u + 1) & 1];
            static_for<0, MB>([&](auto bb) {
                constexpr int blk = decltype(bb)::value, nb = blk + kAhead;
                // A of the stage after the next, a load at a time: into the slot that the barrier before this stage freed
                constexpr int x0 = blk * (nA / 2) / (MB - kAhead + 1), x1 = (blk + 1) * (nA / 2) / (MB - kAhead + 1);
                if constexpr (x0 < nA / 2) static_for<(u & 1) * (nA / 2) + x0, (u & 1) * (nA / 2) + (x1 < nA / 2 ? x1 : nA / 2)>(issue_a);
                if constexpr (nb == MB) {                 // on to the other half of the rows' lines
                    uint32_t step = 0;
                    if constexpr (u & 1) {                // the stage ends: see above
                        __builtin_amdgcn_s_waitcnt(vmcnt_only(kStageWait + (u == 1 ? nS : 0)) & lgkmcnt_only(0));
                        __builtin_amdgcn_s_barrier();
                        asm volatile("" : : : "memory");
                        step = slot == ring + 2 * kSlot ? 0u - 2 * kSlot : (uint32_t)kSlot;
                        slot += step;
                    }
#pragma unroll
                    for (int d = 0; d < 4; d++) rd[d] = (rd[d] ^ 64u) + step;
                }
                lds_read_a4<(nb < MB ? nb : nb - MB) * kWideBlock>(abuf[(phase + nb) & 3], rd);
                __builtin_amdgcn_s_waitcnt(lgkmcnt_only(4 * kAhead));   // (the reads of the blocks after this one)
                uint32_t (&src)[4] = abuf[(phase + blk) & 3];
                asm volatile("" : "+v"(src[0]), "+v"(src[1]), "+v"(src[2]), "+v"(src[3]));
                const h8 av = __builtin_bit_cast(h8, u4{src[0], src[1], src[2], src[3]});
                static_for<0, 4>([&](auto ff) {
                    constexpr int f = decltype(ff)::value, at = 4 * blk + f;
                    // (wait states in front of the blocks whose A was read in the trip before: those registers cross the
                    // loop's back edge, where the allocator may copy them; everywhere else nothing but loads and earlier
                    // entries write what an MFMA reads, and s_nops there cost 5 % of the time)
                    mfma_acc_a<f == 0 && u == 0 && blk < kAhead>(acc[blk][f], cur[f], av);
                    constexpr int e0 = at * kEntries / (4 * MB), e1 = (at + 1) * kEntries / (4 * MB);
                    entries(Int<e0>{}, Int<e1>{}, nq, nt, nxt);
                });
            });
        });
    }
    // (slices of one trip less than the longest: the others' barriers)
    for (int trip = trips; trip < most_trips; trip++) {
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_s_barrier();
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0) & lgkmcnt_only(0));
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7");        // MFMA results -> other readers (see stream_tile_mb)
#pragma unroll
    for (int blk = 0; blk < MB; blk++)
#pragma unroll
        for (int f = 0; f < 4; f++) asm volatile("" : "+a"(acc[blk][f]));
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
            asm volatile("" : "+v"(wq[s][k]));
            if (FP6) asm volatile("" : "+v"(tq[s][k]));
        }
#pragma unroll
    for (int f = 0; f < 4; f++) {
        asm volatile("" : "+v"(gs_next[f]));
#pragma unroll
        for (int d = 0; d < 4; d++) asm volatile("" : "+v"(abuf[f][d]));
    }
}

// What the kernel needs of a launch.  Names as in GemmArgs, so that the shared helpers take either.
struct WideArgs {
    const uint16_t* A;
    const uint32_t* b_int4;
    const uint32_t* b_fp6_2;
    const uint32_t* b_fp6_4;
    uint16_t* C;
    const uint16_t* s_int4;
    const uint16_t* s_fp6;
    int m, n, k;
    int n4, qc;
    int tiles6, tiles;        // 128-column tiles: FP6, all
    int native;
    const int32_t* c_cols;    // optional epilogue work (fp6m_mul_fused)
    const uint16_t* bias;
    const uint16_t* residual;
    int fused;
    static constexpr int k4 = 0;
};

// One workgroup: 64-column groups `group0` ..  of the tiles in launch order, FP6 first.
// FP6 / INT4: which regions its waves may lie in.  EXTRAS = false: without the fused epilogue and the gfx950 word order.
template <bool G128, int MB, int WN, int WK, bool EXTRAS, bool FP6, bool INT4>
__device__ __forceinline__ void wide_workgroup(const WideArgs& p, unsigned char* smem, int group0)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wn = wave % WN, wk = wave / WN;
    const int group = __builtin_amdgcn_readfirstlane(group0) + wn;
    TileInfo ti;
    ti.tile = group >> 1;
    const int sigma = group & 1;
    ti.fp6 = FP6 && (!INT4 || ti.tile < p.tiles6);
    ti.tcol = ti.fp6 ? ti.tile : ti.tile - p.tiles6;
    ti.region_n = ti.fp6 ? p.qc : p.n4;
    ti.mtile = blockIdx.y;
    ti.part = 0;
    ti.a_step0 = 0;
    ti.later = false;
    ti.col0 = (ti.fp6 ? p.n4 : 0) + ti.tcol * kTileN + 64 * sigma;
    const int trips_all = p.k >> 7;
    const int begin = trips_all * wk / WK, trips = trips_all * (wk + 1) / WK - begin, most = (trips_all + WK - 1) / WK;

    f4 acc[MB][4];
#pragma unroll
    for (int blk = 0; blk < MB; blk++)
#pragma unroll
        for (int f = 0; f < 4; f++) acc[blk][f] = f4{0.f, 0.f, 0.f, 0.f};
    const uint32_t ring = uniform32(lds_addr(smem)) + wk * (3 * wide_slot_bytes(MB));
    if (FP6 && (!INT4 || ti.fp6))
        wide_stream<FP6, G128, MB, WN>(p, ti, sigma, wn, ring, begin, trips, most, acc);
    else
        wide_stream<!INT4, G128, MB, WN>(p, ti, sigma, wn, ring, begin, trips, most, acc);

    // ---- epilogue: lane 16 q + c holds row c of a block, columns 32 (q >> 1) + 16 jp + 8 half + 4 (q & 1) + 0 .. 3
    const int q = lane >> 4, c = lane & 15;
    const int col_lane = 32 * (q >> 1) + 4 * (q & 1);
    const int row0 = ti.mtile * 16 * MB;
    constexpr bool kThroughSlab = EXTRAS && WK > 1;
    const bool fused = kThroughSlab && p.fused;
    f4 scale[4];
#pragma unroll
    for (int f = 0; f < 4; f++) scale[f] = f4{1.f, 1.f, 1.f, 1.f};
    if ((ti.fp6 || !G128) && !fused) {
        const uint16_t* sp = (ti.fp6 ? p.s_fp6 : p.s_int4) + ti.tcol * kTileN + 64 * sigma;
        const float re_bias = ti.fp6 ? 4096.0f : 1.0f;    // the deferred e3m2 exponent re-bias
#pragma unroll
        for (int f = 0; f < 4; f++)
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                const int col = col_lane + 16 * (f >> 1) + 8 * (f & 1) + e;
                const h2 sv = *reinterpret_cast<const h2*>(sp + (col & ~31) + scale_slot(col & 31));
                scale[f][e] = (float)sv[0] * re_bias;
                scale[f][e + 1] = (float)sv[1] * re_bias;
            }
    }
    unsigned char* slab = smem + wide_round_bytes(WN, WK) + wave * 16 * kWideSlabRow;
    // The fused epilogue (column map, bias, residual): a lane takes one column, and a block's rows, as fp32, change hands through
    // the wave's slab, eight at a time.  A row is then one load and one store of whole lines (of the mapped columns' lines, which
    // are mostly neighbours), and a block's residual is on its way while the slices are summed.  (Each lane adding to its own
    // fragments, two bytes of 64 lines at a time and in turn with the stores, as the residual may be C, cost a round of 48-row
    // tiles 10 us, more than these tiles gain over gemm_mb_kernel's: with bias and residual, us, 107 x 3328 x 19712 with that
    // kernel 36.2, here 40.0 -> 33.5; 300 x 4096 x 12288 52.0 -> 40.9, without additions 39.3; 2048 x 8192 x 10240 358 -> 308, 300.
    // 200 and 300 random calls: 18-28 % for every tile, none slower.)
    // Without slices there is no sum to wait for, and the accumulators of 128 rows leave no registers: there it is as it was.
    unsigned fcol = 0;                                    // bytes
    float fscale = 1.f, fbias = 0.f;
    uint16_t res[kThroughSlab ? 16 : 1] = {};
    if constexpr (kThroughSlab) {
        if (fused) {
            int col = ti.col0 + lane;
            if (p.c_cols) {
                col = p.c_cols[col];
                col = col < 0 ? 0 : (col >= p.n ? p.n - 1 : col);         // (a bad map cannot write outside C)
            }
            fcol = 2u * (unsigned)col;
            if (p.bias) fbias = (float)__builtin_bit_cast(_Float16, p.bias[col]);
            if (ti.fp6 || !G128)
                fscale = (float)reinterpret_cast<const _Float16*>(ti.fp6 ? p.s_fp6 : p.s_int4)[ti.tcol * kTileN + 64 * sigma + (lane & 32) + scale_slot(lane & 31)] *
                         (ti.fp6 ? 4096.0f : 1.0f);
        }
    }
    auto load_residual = [&](int blk) {
        if constexpr (kThroughSlab) {
            const int first = row0 + 16 * blk;
            if (!p.residual || first >= p.m) return;      // (uniform)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = first + r < p.m ? first + r : p.m - 1;
                res[r] = *reinterpret_cast<const uint16_t*>(reinterpret_cast<const unsigned char*>(p.residual + (size_t)row * p.n) + fcol);
            }
        }
    };
    auto store_fused_block = [&](int blk, const f4 (&v)[4]) {
        if constexpr (kThroughSlab) {
            const int first = row0 + 16 * blk;
            if (first >= p.m) return;                     // (uniform)
            constexpr int kRow = 64 + 4;                  // floats
            static_assert(8 * kRow * 4 <= 16 * kWideSlabRow, "eight rows of a block");
            float* rows = reinterpret_cast<float*>(slab);
#pragma unroll
            for (int half = 0; half < 2; half++) {
                __builtin_amdgcn_wave_barrier();
                if ((c >> 3) == half) {
#pragma unroll
                    for (int f = 0; f < 4; f++) *reinterpret_cast<f4*>(rows + (c & 7) * kRow + col_lane + 16 * (f >> 1) + 8 * (f & 1)) = v[f];
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int r = 0; r < 8; r++) {
                    const int row = first + 8 * half + r;
                    float o = rows[r * kRow + lane] * fscale + fbias;
                    if (p.residual) o += (float)__builtin_bit_cast(_Float16, res[8 * half + r]);
                    if (row < p.m) *reinterpret_cast<uint16_t*>(reinterpret_cast<unsigned char*>(p.C + (size_t)row * p.n) + fcol) = __builtin_bit_cast(uint16_t, (_Float16)o);
                }
            }
        }
    };
    FusedCols fc[EXTRAS && !kThroughSlab ? 4 : 1][2];
    if constexpr (EXTRAS && !kThroughSlab) {
#pragma unroll
        for (int f = 0; f < 4; f++)
#pragma unroll
            for (int e = 0; e < 2; e++) fc[f][e] = fused_cols(p, ti.col0 + col_lane + 16 * (f >> 1) + 8 * (f & 1) + 2 * e);
    }
    auto store_block = [&](int blk, const f4 (&v)[4]) {
        const int first = row0 + 16 * blk;
        if (first >= p.m) return;                         // (uniform)
        if constexpr (EXTRAS && !kThroughSlab) {
            if (p.fused) {
                if (first + c >= p.m) return;
#pragma unroll
                for (int f = 0; f < 4; f++)
#pragma unroll
                    for (int e = 0; e < 2; e++)
                        store_fused(p, fc[f][e], (size_t)(first + c), v[f][2 * e] * scale[f][2 * e], v[f][2 * e + 1] * scale[f][2 * e + 1]);
                return;
            }
        }
        // through the wave's slab, so that rows leave as whole 128-byte lines (LDS operations of a wave execute in order)
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int f = 0; f < 4; f++) {
            h4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = (_Float16)(v[f][e] * scale[f][e]);
            *reinterpret_cast<h4*>(slab + c * kWideSlabRow + 2 * (col_lane + 16 * (f >> 1) + 8 * (f & 1))) = o;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < 16; r += 8) {
            const int row = r + (lane >> 3);
            const u4 o = *reinterpret_cast<const u4*>(slab + row * kWideSlabRow + 16 * (lane & 7));
            if (first + row < p.m) *reinterpret_cast<u4*>(p.C + (size_t)(first + row) * p.n + ti.col0 + 8 * (lane & 7)) = o;
        }
        __builtin_amdgcn_wave_barrier();
    };
    if constexpr (WK == 1) {
        __builtin_amdgcn_s_barrier();                     // (the slab lies in the ring, which others may still be reading)
#pragma unroll
        for (int blk = 0; blk < MB; blk++) store_block(blk, acc[blk]);
    } else {
#pragma unroll
        for (int r = 0; r < (MB + WK - 1) / WK; r++) {
            if (fused && r * WK + wk < MB) load_residual(r * WK + wk);
            __syncthreads();
            f4* out = reinterpret_cast<f4*>(smem) + (size_t)(wn * WK * WK) * 256 + lane;   // [wn][owner][slice][fragment] 1 KiB each
#pragma unroll
            for (int o = 0; o < WK; o++)
                if (r * WK + o < MB) {
#pragma unroll
                    for (int f = 0; f < 4; f++) out[(o * WK + wk) * 256 + 64 * f] = acc[(r * WK + o) % MB][f];
                }
            __syncthreads();
            if (r * WK + wk < MB) {
                f4 sum[4];
#pragma unroll
                for (int f = 0; f < 4; f++) {
                    sum[f] = out[wk * WK * 256 + 64 * f];
#pragma unroll
                    for (int s = 1; s < WK; s++) sum[f] += out[(wk * WK + s) * 256 + 64 * f];
                }
                if (fused)
                    store_fused_block(r * WK + wk, sum);
                else
                    store_block(r * WK + wk, sum);
            }
        }
    }
}

// MB: 16-row blocks per tile; WN x WK waves: 64-column groups side by side x k slices.
// NARROW6: FP6 tiles (and the INT4 tile left over where the rest is an odd number of tiles) are workgroups of their own,
// 128 columns x four k slices instead of 256 x two.  An FP6 step dequantises for twice as long as an INT4 step, and where the
// whole launch is one round that workgroup is the one it waits for: with 256 FP6 columns 400 x 8192 x 10240 in 80-row tiles
// took 76.6 us with per-column scales and 76.9 with group scales, without any 60.4 and 70.4; like this 64.7 and 72.7.  (Four
// slices of tiles above 96 rows do not fit the LDS.)
template <bool G128, int MB, int WN, int WK, bool NARROW6, bool EXTRAS>
__global__ __launch_bounds__(64 * WN * WK, 2) void gemm_wide_kernel(const WideArgs args)
{
    static_assert(!NARROW6 || (WN == 4 && WK == 2), "eight waves either way");
    constexpr int kLds = max3(wide_lds_bytes(MB, WN, WK), NARROW6 ? wide_lds_bytes(MB, 2, 4) : 0, 0);
    static_assert(kLds <= 160 * 1024, "LDS of one CU");
    __shared__ __attribute__((aligned(16))) unsigned char smem[kLds];
    WideArgs p = args;
    if constexpr (!EXTRAS) {
        p.native = 0;
        p.fused = 0;
        p.c_cols = nullptr;
        p.bias = nullptr;
        p.residual = nullptr;
    }
    // Workgroups: x walks the columns (the FP6 region first), contiguous ranges per XCD; y the row tiles.
    const int x = __builtin_amdgcn_readfirstlane(xcd_contiguous_id(blockIdx.x, gridDim.x));
    if constexpr (NARROW6) {
        const int odd = (p.tiles - p.tiles6) & 1;         // (an INT4 tile that has no other to lie beside)
        if (x < p.tiles6)
            wide_workgroup<G128, MB, 2, 4, EXTRAS, true, false>(p, smem, 2 * x);
        else if (x < p.tiles6 + odd)
            wide_workgroup<G128, MB, 2, 4, EXTRAS, false, true>(p, smem, 2 * x);
        else
            wide_workgroup<G128, MB, WN, WK, EXTRAS, false, true>(p, smem, 2 * (p.tiles6 + odd) + 4 * (x - p.tiles6 - odd));
    } else {
        wide_workgroup<G128, MB, WN, WK, EXTRAS, true, true>(p, smem, x * WN);
    }
}

}  // namespace fp6m
