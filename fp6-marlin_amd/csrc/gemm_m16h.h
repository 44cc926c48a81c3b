// gemm_m16h_kernel: the m <= 16 kernel of fp6m_gemm.hip on tiles of 64 columns.
#pragma once
#include "gemm_m16.h"

namespace fp6m {

// ------------------------------------------------------------------------------------------------ m <= 16, 64-column tiles
//
// gemm_m16_kernel with half as many columns per workgroup.  The workgroups needed to keep the chip's requests in flight are
// the same, so a tile's k range is cut into half as many parts: where 128-column tiles meet in two parts, nothing is exchanged
// between workgroups at all, and what is exchanged is half as much per workgroup.  What it costs is A, which every workgroup
// reads for half as many columns.  us: 5 x 5120 x 15360 12.0 -> 10.1 (two parts -> one, eight waves), 8 x 11008 x 4096 with
// map, bias and residual 11.4 -> 10.1, 16 x 4096 x 4096 8.5 -> 7.1 (six parts -> three), the same as a row mix 9.0 -> 7.4.  A
// ring of eight rows for 5 to 8 rows of A instead of sixteen is 1-4 % of that.
//
// A step is 64 rows of k: four k-blocks of 512 bytes (FP6: + 4 x 256), as many bytes as 32 rows of 128 columns, and one whole
// 128-byte line of every row of A; slices are whole pairs of steps.  Lane 16 i + 8 b + l reads words 2b and 2b + 1 of fragment
// owner 4 l + i from the ring, so that fragment (jp, half) is columns 32 b + 16 jp + 8 half + l of the tile.  Order of a step's
// loads: A, words, group scales (every other step).  Nothing is fetched past a slice's end, the waits go by the steps that are
// still to land: repeating the last step instead, so that their counts never change, was three steps more on slices of four to
// eight (5 x 5120 x 15360 9.9 -> 9.1 us, 8 x 11008 x 4096 10.1 -> 9.7).  A ring of three steps, better for one row (gemm_m1.h), is
// up to 15 % slower here (16 x 4096 x 12288 9.5 -> 11.1).
struct HalfRegs {
    u2 q[4];            // words of the four k-blocks
    uint32_t t[4];      // FP6 2-bit plane
    uint32_t a[8];      // activations of the step's two halves in MFMA operand order
};
constexpr int kHalfStride = 64 + 4;                          // floats per row of the reduction slab
constexpr int kHalfScaleSlabs = 4;                           // groups of two steps, fetched up to three steps ahead

// At most `newer` steps of OPS loads each outstanding, with one load more (group scales) in the first, third, .. (EVEN) or the
// second, fourth, .. of them; MOST: the most there can be.
template <int OPS, bool GROUP, bool EVEN, int MOST>
__device__ __forceinline__ void wait_steps(int newer)
{
    if constexpr (MOST == 0) {
        __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    } else {
        if (newer >= MOST)
            __builtin_amdgcn_s_waitcnt(vmcnt_only(OPS * MOST + (GROUP ? (MOST + (EVEN ? 1 : 0)) / 2 : 0)));
        else
            wait_steps<OPS, GROUP, EVEN, MOST - 1>(newer);
    }
}

template <bool FP6, bool G128, int DEPTH, int AROWS, typename Args>
__device__ __forceinline__ void stream_half(const Args& p, const TileInfo& ti, int sigma, unsigned char* ring,
                                            int step_begin, int step_end, f4 (&acc)[4])
{
    static_assert(DEPTH >= 3, "needs two steps of look-ahead");
    constexpr bool kGroup = G128 && !FP6;                 // group scales apply to INT4 tiles only
    constexpr int kPair = pair_bytes(AROWS);
    constexpr int kSlot = FP6 ? 3072 : 2048;              // a step's packed words
    constexpr int kAOps = AROWS == 16 ? 2 : 1;
    constexpr int kOps = kAOps + (FP6 ? 3 : 2);           // direct-to-LDS loads per step
    constexpr int kReads = FP6 ? 16 : 12;                 // LDS reads per step
    const int lane = threadIdx.x & 63;
    const int i = lane >> 4, c = lane & 15, b = c >> 3, l = c & 7;

    DequantConsts kc;
    kc.lo = vgpr_const(0x000f000fu);
    kc.hi = vgpr_const(0x00f000f0u);
    kc.ex = vgpr_const(0x64006400u);
    kc.top2 = vgpr_const(0xc0c0c0c0u);
    kc.exp_man = vgpr_const(0x9f009f00u);

    // ---- fetch side (lane = position in the slot)
    const PlaneGeometry geo = plane_geometry(p, ti);
    const size_t row4 = geo.row4, row2 = geo.row2;
    const int lg = lane & 31;
    // (gfx950 order: owner 4 l + i lies at granule 16 i + 8 sigma + l of the 128-column tile, so this half is four whole lines
    // of every k-block; granules of the 2-bit plane are loaded in pairs, and so stay in that order in the ring)
    const int o4 = lg ^ ((lg >> 3) & 3);
    const uint32_t v4 = (uint32_t)((lane >> 5) * row4) + (p.native ? 16 * (o4 & 3) + (o4 >> 2) : o4) * 16;
    const unsigned char* base4 = reinterpret_cast<const unsigned char*>(FP6 ? p.b_fp6_4 : p.b_int4) + geo.tile4 +
                                 (p.native ? 128 : 512) * sigma + (size_t)(4 * step_begin) * row4;
    const uint32_t v2 = (uint32_t)((lane >> 4) * row2) + (p.native ? 128 * ((lane >> 2) & 3) + 16 * (lane & 3) : 16 * (lane & 15));
    const unsigned char* base2 = reinterpret_cast<const unsigned char*>(p.b_fp6_2) + geo.tile2 + (p.native ? 64 : 256) * sigma +
                                 (size_t)(4 * step_begin) * row2;
    // A: as in stream_tile, a slot per step
    const bool a_lane = AROWS >= 8 || lane < 32;
    uint32_t vap[kAOps];
#pragma unroll
    for (int o = 0; o < kAOps; o++) {
        const int prow = (lane >> 3) & (AROWS - 1) & 7, pch = lane & 7;
        int row = 8 * o + prow;
        row = row < p.m ? row : p.m - 1;
        vap[o] = (uint32_t)row * (uint32_t)p.k * 2 + 16 * ((pch & 4) | ((pch & 3) ^ ((prow >> 1) & 3)));
    }
    const unsigned char* base_a = reinterpret_cast<const unsigned char*>(p.A) + (size_t)ti.a_step0 * 64 + (size_t)step_begin * 128;
    unsigned char* a_ring = ring + DEPTH * kSlot;
    const unsigned char* base_gs = reinterpret_cast<const unsigned char*>(p.s_int4 + (size_t)ti.tcol * kTileN + 64 * sigma);
    const uint32_t vgs = 4 * lg;                          // (128 bytes, twice: a tile's scales end where the region may end)
    unsigned char* gs_ring = a_ring + DEPTH * kPair;

    int issued = step_begin;                              // next step to fetch
    auto issue = [&](int slot, bool even) {
        unsigned char* dst = ring + slot * kSlot;
        unsigned char* adst = a_ring + slot * kPair;
        if (a_lane) dma16(base_a + vap[0], adst);
        if (kAOps == 2) dma16(base_a + vap[kAOps - 1], adst + 1024);
        dma16_stream(base4 + v4, dst);
        dma16_stream(base4 + 2 * row4 + v4, dst + 1024);
        if (FP6) dma16_stream(base2 + v2, dst + 2048);
        if (kGroup && even)
            dma4(base_gs + (size_t)(issued >> 1) * p.n4 * 2 + vgs, gs_ring + ((issued >> 1) & (kHalfScaleSlabs - 1)) * 256);
        issued++;                                         // uniform: pointers move on the scalar unit
        base4 += 4 * row4;
        base2 += 4 * row2;
        base_a += 128;
    };

    // ---- read side (lane = MFMA identity)
    const int owner = 4 * l + i;
    const uint32_t ring_lds = lds_addr(ring);
    const uint32_t rd4 = ring_lds + (owner ^ ((owner >> 3) & 3)) * 16 + 8 * b;
    const uint32_t rd2 = ring_lds + 2048 + (p.native ? 8 * i + l : owner) * 8 + 4 * b;
    const int ar = c & (AROWS - 1);                       // rows beyond AROWS re-read a valid row; their sums are never stored
    uint32_t rda[4];
#pragma unroll
    for (int d = 0; d < 4; d++)
        rda[d] = lds_addr(a_ring) + (ar >> 3) * 1024 + (8 * (ar & 7) + (d ^ ((ar >> 1) & 3))) * 16 + 4 * i;
    const int q = i;                                      // result side: quarter of the column slots
    const uint32_t rdgs = lds_addr(gs_ring) + (32 * (q >> 1) + 4 * (q & 1)) * 2;

    auto fetch = [&](HalfRegs& r, int slot) {             // kReads LDS reads of one step, not waited for
        const uint32_t so = slot * kSlot, ao = slot * kPair;
        asm volatile(
            "ds_read_b64 %0, %4\n\tds_read_b64 %1, %4 offset:512\n\tds_read_b64 %2, %4 offset:1024\n\tds_read_b64 %3, %4 offset:1536"
            : "=&v"(r.q[0]), "=&v"(r.q[1]), "=&v"(r.q[2]), "=&v"(r.q[3]) : "v"(rd4 + so) : "memory");
        if (FP6)
            asm volatile(
                "ds_read_b32 %0, %4\n\tds_read_b32 %1, %4 offset:256\n\tds_read_b32 %2, %4 offset:512\n\tds_read_b32 %3, %4 offset:768"
                : "=&v"(r.t[0]), "=&v"(r.t[1]), "=&v"(r.t[2]), "=&v"(r.t[3]) : "v"(rd2 + so) : "memory");
        asm volatile("ds_read_b32 %0, %4\n\tds_read_b32 %1, %5\n\tds_read_b32 %2, %6\n\tds_read_b32 %3, %7"
                     : "=&v"(r.a[0]), "=&v"(r.a[1]), "=&v"(r.a[2]), "=&v"(r.a[3])
                     : "v"(rda[0] + ao), "v"(rda[1] + ao), "v"(rda[2] + ao), "v"(rda[3] + ao) : "memory");
        asm volatile("ds_read_b32 %0, %4 offset:64\n\tds_read_b32 %1, %5 offset:64\n\t"
                     "ds_read_b32 %2, %6 offset:64\n\tds_read_b32 %3, %7 offset:64"
                     : "=&v"(r.a[4]), "=&v"(r.a[5]), "=&v"(r.a[6]), "=&v"(r.a[7])
                     : "v"(rda[0] + ao), "v"(rda[1] + ao), "v"(rda[2] + ao), "v"(rda[3] + ao) : "memory");
    };
    auto settle = [&](HalfRegs& r) {
        asm volatile("" : "+v"(r.q[0]), "+v"(r.q[1]), "+v"(r.q[2]), "+v"(r.q[3]));
        if (FP6) asm volatile("" : "+v"(r.t[0]), "+v"(r.t[1]), "+v"(r.t[2]), "+v"(r.t[3]));
        asm volatile("" : "+v"(r.a[0]), "+v"(r.a[1]), "+v"(r.a[2]), "+v"(r.a[3]));
        asm volatile("" : "+v"(r.a[4]), "+v"(r.a[5]), "+v"(r.a[6]), "+v"(r.a[7]));
    };
    auto compute = [&](const HalfRegs& r, f4 (&dst)[4], bool fresh) {
        const f4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const h8 av = __builtin_bit_cast(h8, u4{r.a[4 * h], r.a[4 * h + 1], r.a[4 * h + 2], r.a[4 * h + 3]});
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

    int slot_in = 0;
#pragma unroll
    for (int d = 0; d < DEPTH - 1; d++)
        if (issued < step_end) {                          // (two steps at least)
            issue(slot_in, (d & 1) == 0);
            slot_in = slot_in + 1 == DEPTH ? 0 : slot_in + 1;
        }
    HalfRegs regs[2];
    wait_steps<kOps, kGroup, false, DEPTH - 2>(issued - step_begin - 1);
    FP6M_MARK(p, 1);
    fetch(regs[0], 0);
    int slot_rd = 1;                                      // slot of the step whose LDS reads come next
    f4 grp[4];
#pragma unroll 1
    for (int s = step_begin; s < step_end; s += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (issued < step_end) {
                issue(slot_in, ((u + DEPTH - 1) & 1) == 0);
                slot_in = slot_in + 1 == DEPTH ? 0 : slot_in + 1;
            }
            if (u == 0)                                                   // step s+u+1 has landed (past the end: all has)
                wait_steps<kOps, kGroup, true, DEPTH - 2>(issued - (s + 2));
            else
                wait_steps<kOps, kGroup, false, DEPTH - 2>(issued - (s + 3));
            fetch(regs[(u + 1) & 1], slot_rd);
            slot_rd = slot_rd + 1 == DEPTH ? 0 : slot_rd + 1;
            __builtin_amdgcn_s_waitcnt(lgkmcnt_only(kReads < 15 ? kReads : 15));   // reads of step s+u (older) are done
            settle(regs[u & 1]);
            if (kGroup)
                compute(regs[u & 1], grp, u == 0);
            else
                compute(regs[u & 1], acc, false);
        }
        if (kGroup) {
            // end of a 128-row group: fold it into the running sum with its scales (fp32)
            const uint32_t ga = rdgs + ((s >> 1) & (kHalfScaleSlabs - 1)) * 256;
            u2 sv[4];
            asm volatile(
                "ds_read_b64 %0, %4\n\tds_read_b64 %1, %4 offset:16\n\tds_read_b64 %2, %4 offset:32\n\t"
                "ds_read_b64 %3, %4 offset:48\n\ts_waitcnt lgkmcnt(0)"
                : "=&v"(sv[0]), "=&v"(sv[1]), "=&v"(sv[2]), "=&v"(sv[3]) : "v"(ga) : "memory");
            settle(regs[0]);                              // lgkmcnt(0) also completed the look-ahead reads
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
    // The look-ahead past the end reads bytes that nobody uses, and may still be in flight; the epilogue reuses the ring.
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0) & lgkmcnt_only(0));
    settle(regs[0]);
    if (FP6) {
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t] *= 4096.0f;    // the deferred e3m2 exponent re-bias
    }
}

constexpr int half_wave_lds_bytes(int d4, int d6, int arows)
{
    return max3(d4 * (2048 + pair_bytes(arows)) + kHalfScaleSlabs * 256, d6 * (3072 + pair_bytes(arows)), 16 * kHalfStride * 4);
}

// Epilogue: as wg_finish (gemm_m16.h), with a row of 64 columns to half a wave: lanes 32 h + x of wave wk own columns 2x, 2x + 1
// of rows 2 wk + h, 2 wk + h + 2 WK, ..  The protocols between workgroups, and why they hold, are the same.
template <int WK, bool CELLS, bool LOCAL>
__device__ __forceinline__ void wg_finish_half(const GemmArgs& p, const TileInfo& ti, int group, int sigma, int wk, int ks, int slot_base,
                                               int* counter, f4 (&acc)[4], bool per_column_scale, unsigned char* smem,
                                               int wave_lds, int* flag, int first_fp6)
{
    constexpr int RMAX = 8 / WK;                          // row pairs one wave finishes
    constexpr int PCHUNK = 16 / RMAX;                     // parts whose loads are in flight together
    typedef float f2 __attribute__((ext_vector_type(2)));
    static_assert(WK == 4 || WK == 8, "rows per wave");
    const int lane = threadIdx.x & 63;
    const int c = lane & 15, q = lane >> 4;
    {
        float* mine = reinterpret_cast<float*>(smem + wk * wave_lds) + c * kHalfStride + 32 * (q >> 1) + 4 * (q & 1);
#pragma unroll
        for (int t = 0; t < 4; t++) *reinterpret_cast<f4*>(mine + 16 * (t >> 1) + 8 * (t & 1)) = acc[t];
    }
    __syncthreads();
    FP6M_MARK(p, 3);

    const int nrows = p.m < 16 ? p.m : 16;
    const int x = lane & 31, row0 = 2 * wk + (lane >> 5);
    const int nr = ti.tcol * kTileN + 64 * sigma + 2 * x; // even column inside the region
    float s0 = 1.0f, s1 = 1.0f;
    if (per_column_scale) {
        const uint16_t* sp = ti.fp6 ? p.s_fp6 : p.s_int4;
        const h2 sv = *reinterpret_cast<const h2*>(sp + (nr & ~31) + scale_slot(nr & 31));
        s0 = (float)sv[0];
        s1 = (float)sv[1];
    }
    float x0 = 1.0f, x1 = 1.0f;                           // FP6 column scales of a row mix
    if (first_fp6 < WK) {
        const h2 sv = *reinterpret_cast<const h2*>(p.s_fp6 + (nr & ~31) + scale_slot(nr & 31));
        x0 = (float)sv[0];
        x1 = (float)sv[1];
    }
    uint16_t* c_out = p.C + ti.col0 + 2 * x;
    const FusedCols fcols = fused_cols(p, ti.col0 + 2 * x);
    auto store_row = [&](int m, float v0, float v1) {
        if (p.fused) {
            store_fused(p, fcols, (size_t)m, v0 * s0, v1 * s1);
            return;
        }
        h2 o = {(_Float16)(v0 * s0), (_Float16)(v1 * s1)};
        *reinterpret_cast<h2*>(c_out + (size_t)m * p.n) = o;
    };
    f2 tv[RMAX][WK];
#pragma unroll
    for (int r = 0; r < RMAX; r++)
#pragma unroll
        for (int j = 0; j < WK; j++)
            tv[r][j] = *reinterpret_cast<const f2*>(reinterpret_cast<const float*>(smem + j * wave_lds) + (row0 + 2 * WK * r) * kHalfStride + 2 * x);
    float v0[RMAX], v1[RMAX];
#pragma unroll
    for (int r = 0; r < RMAX; r++) {
        v0[r] = 0.f;
        v1[r] = 0.f;
        if (first_fp6 >= WK) {                            // (uniform) the usual case: plain sums
#pragma unroll
            for (int j = 0; j < WK; j++) {
                v0[r] += tv[r][j][0];
                v1[r] += tv[r][j][1];
            }
        } else {
#pragma unroll
            for (int j = 0; j < WK; j++) {
                v0[r] += j >= first_fp6 ? tv[r][j][0] * x0 : tv[r][j][0];
                v1[r] += j >= first_fp6 ? tv[r][j][1] * x1 : tv[r][j][1];
            }
        }
    }
    if (ks == 1) {
#pragma unroll
        for (int r = 0; r < RMAX; r++)
            if (row0 + 2 * WK * r < nrows) store_row(row0 + 2 * WK * r, v0[r], v1[r]);
        return;
    }

    if constexpr (CELLS) {
        unsigned long long* cell = p.cells + (size_t)group * (16 * 64) + x;   // [row][32 even | 32 odd columns]
        unsigned long long old[RMAX][2];
#pragma unroll
        for (int r = 0; r < RMAX; r++) {
            const int m = row0 + 2 * WK * r;
            v0[r] *= s0;
            v1[r] *= s1;
            if (m < nrows) {
                old[r][0] = __hip_atomic_fetch_add(cell + m * 64, cell_contribution(v0[r]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                old[r][1] = __hip_atomic_fetch_add(cell + m * 64 + 32, cell_contribution(v1[r]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
#pragma unroll
        for (int r = 0; r < RMAX; r++) {
            const int m = row0 + 2 * WK * r;
            if (m >= nrows) continue;
#pragma unroll
            for (int e = 0; e < 2; e++) {
                if ((int)(old[r][e] >> 56) != ks - 1) continue;               // somebody else arrives last at this element
                const float v = cell_total(old[r][e], cell_contribution(e ? v1[r] : v0[r]), ks);
                __hip_atomic_store(cell + m * 64 + 32 * e, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (p.fused)
                    store_fused_one(p, fcols, (size_t)m, e, v);
                else
                    c_out[(size_t)m * p.n + e] = __builtin_bit_cast(uint16_t, (_Float16)v);
            }
        }
        FP6M_MARK(p, 6);
        return;
    }

    // Publish.  A slot holds [16 rows][64 columns] fp32; this wave's rows 2 wk, 2 wk + 1 (+ 2 WK r) are 512 bytes, 8 per lane.
    constexpr int kSlotBytes = 16 * 64 * 4;
    const unsigned char* slot0 = reinterpret_cast<const unsigned char*>(p.scratch) + (size_t)slot_base * kSlotBytes;
    const unsigned char* my = uniform_ptr(slot0 + (size_t)ti.part * kSlotBytes);
    const uint32_t voff = 8 * lane + 512 * wk;
#pragma unroll
    for (int r = 0; r < RMAX; r++)
        if (row0 + 2 * WK * r < nrows) {
            const f2 v = {v0[r], v1[r]};
            st8_row<!LOCAL>(my, voff, voff + 4096, r * WK * 512, __builtin_bit_cast(unsigned long long, v));
        }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));            // (the stores are acknowledged: see wg_finish)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    FP6M_MARK(p, 4);
    if (threadIdx.x == 0) {
        if constexpr (LOCAL) {
            const unsigned mine = 1u << ti.part, all = (1u << ks) - 1;
            const unsigned seen = __hip_atomic_fetch_or(reinterpret_cast<unsigned*>(counter), mine, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
            if (seen & mine) {                            // this part has been here before
                __hip_atomic_fetch_or(reinterpret_cast<unsigned*>(counter), kPoisoned, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                *flag = 2;
            } else {
                *flag = ((seen | mine) & all) == all ? ((seen & kPoisoned) ? 2 : 1) : 0;
            }
        } else {
            const int seen = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *flag = seen == ks - 1;
        }
    }
    __syncthreads();
    FP6M_MARK(p, 5);
    const int finish = *flag;
    if (!finish) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
#pragma unroll
    for (int r = 0; r < RMAX; r++) {
        v0[r] = 0.f;
        v1[r] = 0.f;
    }
    // Gather: the loads of up to PCHUNK parts in flight together (rows past m are read too, they lie inside the slot,
    // and never stored), then the sums in part order.
    const unsigned char* part0 = uniform_ptr(slot0);
    for (int pp = 0; pp < ks; pp += PCHUNK) {
        unsigned long long t[PCHUNK][RMAX];
#pragma unroll
        for (int u = 0; u < PCHUNK; u++)
            if (pp + u < ks) {                            // (uniform)
                const unsigned char* src = part0 + (size_t)(pp + u) * kSlotBytes;
#pragma unroll
                for (int r = 0; r < RMAX; r++) t[u][r] = ld8_row<!LOCAL>(src, voff, voff + 4096, r * WK * 512);
            }
        __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
#pragma unroll
        for (int u = 0; u < PCHUNK; u++)
            if (pp + u < ks) {
#pragma unroll
                for (int r = 0; r < RMAX; r++) {
                    settle64(t[u][r]);
                    const f2 v = __builtin_bit_cast(f2, t[u][r]);
                    v0[r] += v[0];
                    v1[r] += v[1];
                }
            }
    }
    if (LOCAL && finish == 2) {                           // (see wg_finish)
        const float nan = __builtin_nanf("");
#pragma unroll
        for (int r = 0; r < RMAX; r++) v0[r] = v1[r] = nan;
    }
#pragma unroll
    for (int r = 0; r < RMAX; r++)
        if (row0 + 2 * WK * r < nrows) store_row(row0 + 2 * WK * r, v0[r], v1[r]);
    FP6M_MARK(p, 6);
    if (threadIdx.x == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Which builds there are with tiles placed per XCD (LOCAL): only they may be given the padded grid of such a launch.
constexpr bool m16h_has_local(int arows, int wk) { return arows > 4 && wk == 4; }

// Workgroups and their k slices as in gemm_m16_kernel; a group is a 64-column tile (groups6 / groups4 count those).
template <bool G128, int AROWS, int WK, int D4, int D6, bool CELLS, bool EXTRAS, bool LOCAL = false>
__global__ __launch_bounds__(64 * WK, WK == 8 || AROWS > 4 ? 2 : 3) void gemm_m16h_kernel(const GemmArgs args)
{
    static_assert(!LOCAL || !CELLS, "the cells are atomics, which have no XCD-local form");
    static_assert(!LOCAL || m16h_has_local(AROWS, WK), "a build that the dispatcher does not know of");
    constexpr int kWaveLds = half_wave_lds_bytes(D4, D6, AROWS);
    static_assert(WK * kWaveLds + 16 <= 160 * 1024, "LDS of one CU");
    __shared__ __attribute__((aligned(16))) unsigned char smem[WK * kWaveLds + 16];

    GemmArgs p = args;
    if constexpr (!EXTRAS) {
        p.k4 = 0;
        p.slices4 = 0;
        p.native = 0;
        p.fused = 0;
        p.c_cols = nullptr;
        p.bias = nullptr;
        p.residual = nullptr;
    }
    preload_args<false>(args);
    FP6M_MARK(p, 0);
    const int wk = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);     // scalar: addresses stay on the SALU
    TileInfo ti;
    int group;
    if constexpr (LOCAL) {
        const XcdPlace pl = xcd_place(p, blockIdx.x, p.groups6, p.groups4);
        if (!pl.valid) return;                                           // (the grid is padded to a multiple of eight)
        ti.fp6 = pl.fp6;
        ti.part = pl.part;
        group = pl.group;
    } else {
        const int logical = xcd_contiguous_id(blockIdx.x, gridDim.x);
        const int wgs6 = p.groups6 * p.ks6;                              // the FP6 region's workgroups come first
        ti.fp6 = logical < wgs6;
        const int local = ti.fp6 ? logical : logical - wgs6;
        const int groups = ti.fp6 ? p.groups6 : p.groups4;
        const FastDiv gdiv = {ti.fp6 ? p.div[1].d : p.div[0].d, ti.fp6 ? p.div[1].magic : p.div[0].magic};
        ti.part = fast_div(gdiv, local);                                 // part-major: neighbours share k, adjoin in n
        group = local - ti.part * groups;
    }
    const int ks = ti.fp6 ? p.ks6 : p.ks4;
    const WaveRule wrule = {ti.fp6 ? p.wrule[1].lo : p.wrule[0].lo, ti.fp6 ? p.wrule[1].ly : p.wrule[0].ly,
                            ti.fp6 ? p.wrule[1].eo : p.wrule[0].eo, ti.fp6 ? p.wrule[1].ey : p.wrule[0].ey};
    ti.tcol = group >> 1;
    const int sigma = group & 1;
    ti.region_n = ti.fp6 ? p.qc : p.n4;
    ti.tile = ti.fp6 ? ti.tcol : p.tiles6 + ti.tcol;
    ti.mtile = 0;
    ti.later = false;
    ti.col0 = (ti.fp6 ? p.n4 : 0) + group * 64;

    int step_begin = wave_rule_begin(wrule, WK, ti.part, wk) * 2;        // (units of 128 rows in either scale mode)
    int step_end = wave_rule_begin(wrule, WK, ti.part, wk + 1) * 2;
    ti.a_step0 = 0;
    const bool region6 = ti.fp6;                                         // the workgroup's column region
    if (p.k4) {                                                          // per wave: INT4 or FP6 rows of the tile (row_mix_slice)
        const int sl = ti.part * WK + wk;
        ti.fp6 = sl >= p.slices4;
        const SliceRule rule = {ti.fp6 ? p.rule[1].q : p.rule[0].q, ti.fp6 ? p.rule[1].first_long : p.rule[0].first_long};
        const int at = ti.fp6 ? sl - p.slices4 : sl;
        step_begin = slice_begin(rule, at) * 2;
        step_end = slice_begin(rule, at + 1) * 2;
        ti.a_step0 = ti.fp6 ? p.k4 / 32 : 0;
    }

    f4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; t++) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    unsigned char* ring = smem + wk * kWaveLds;
    if (step_begin < step_end) {
        if (ti.fp6)
            stream_half<true, G128, D6, AROWS>(p, ti, sigma, ring, step_begin, step_end, acc);
        else
            stream_half<false, G128, D4, AROWS>(p, ti, sigma, ring, step_begin, step_end, acc);
    }
    FP6M_MARK(p, 2);
    // scratch slots: FP6 tiles first (groups6 * ks6 slots), then INT4 tiles; counters likewise
    const int slot_base = region6 ? group * p.ks6 : p.groups6 * p.ks6 + group * p.ks4;
    const int cell_group = region6 ? group : p.groups6 + group;
    wg_finish_half<WK, CELLS, LOCAL>(p, ti, cell_group, sigma, wk, ks, slot_base, p.counters + cell_group, acc, !p.k4 && (ti.fp6 || !G128), smem,
                                     kWaveLds, reinterpret_cast<int*>(smem + WK * kWaveLds), p.k4 ? p.slices4 - ti.part * WK : WK);
    FP6M_MARK(p, 7);
}

}  // namespace fp6m
