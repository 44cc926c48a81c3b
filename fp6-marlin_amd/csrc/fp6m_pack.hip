// Weight preparation on the GPU: fp16 [k, n] -> the operands of fp6m_mul (B, s) and the dequantised
// check weight, bit for bit what the host path produces (INT4: reference test.py:85-121; FP6:
// test.py:13-58 + weight_quant.cpp:27-124 + weight_prepacking.cpp:123-177; scale order test.py:80-83;
// wire format test.py:123-152).
//
// What bounds it: memory (2 bytes in and 2.5 out per INT4 weight with the check weight) as long as the arithmetic stays
// near ten instructions per weight; a float division, a clamp and a conversion each way per weight, as the host path
// writes it, take 33 and are what used to bound it.  So: whole 16-byte row pieces go straight into registers in the
// order in which a thread needs them (four rows x two 8-column pieces are the 64 weights of eight fragment owners), the
// quotient is a product with the column's reciprocal and one correction (exact, see quotient()), rounding to an integer
// is one packed addition, and the packed words are an 8 x 8 nibble transpose in registers.  With group-128 scales a
// workgroup holds whole groups, so the weight is read once.
//
// Values are binary16; every operation is done in binary32 and rounded back to binary16 (what torch's CPU half kernels
// and the reference's __hmul do), with round-to-nearest-even conversions.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <thread>

#include "fp6m.h"
#include "fp6m_layout.h"

namespace fp6m {

int hip_fail(hipError_t e);            // fp6m_gemm.hip: records the HIP error, returns FP6M_ERR_HIP
bool capturing(hipStream_t stream);    // fp6m_gemm.hip

namespace {

// Makes `dev` the calling thread's current device for the lifetime of the object and puts the previous one back.
struct DeviceGuard {
    int prev = -1;
    hipError_t err;
    explicit DeviceGuard(int dev)
    {
        err = hipGetDevice(&prev);
        if (err == hipSuccess && prev != dev) err = hipSetDevice(dev);
        else if (err == hipSuccess) prev = -1;                          // nothing to restore
    }
    ~DeviceGuard()
    {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

__device__ __forceinline__ float h2f(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
__device__ __forceinline__ uint16_t f2h(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }

// Position of the per-column scale of column c in the reference's permuted order.
__device__ __forceinline__ size_t scale_pos(size_t c) { return (c & ~size_t(31)) + scale_slot((int)(c & 31)); }

// ---- INT4 region: columns [0, n4) of w

typedef unsigned short us2 __attribute__((ext_vector_type(2)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ us2 max2(us2 a, us2 b) { return __builtin_elementwise_max(a, b); }
__device__ __forceinline__ us2 magnitudes(uint32_t v) { return __builtin_bit_cast(us2, v & 0x7fff7fffu); }

// The magnitude maxima of up to kMaxChunks row ranges, column by column, for the scales that span all of k (per-column
// INT4 scales, FP6 scales): 256 columns x `rows` rows per workgroup, 16-byte loads, eight rows at a time.  The maximum
// is taken on the bit patterns of |x| (monotonic for binary16).  They go to `part` [chunk][cols], which is output
// memory that only later kernels on the stream fill: the call needs no scratch of its own.  (One thread per eight
// columns over all of k left all but a few CUs idle: 8192 x 8192 took 640 us; packing it with per-column scales takes 84 us
// in all like this.)
constexpr int kMaxChunks = 64;
__global__ __launch_bounds__(256) void column_maxima_kernel(const uint16_t* w, int k, int n, int cols, int rows, uint16_t* part)
{
    __shared__ us2 red[8][128];                                         // [row of eight][column pair]
    const int c = blockIdx.x * 256 + (threadIdx.x & 31) * 8, r0 = blockIdx.y * rows, r1 = r0 + rows < k ? r0 + rows : k;
    us2 m[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
    if (c < cols) {                                                     // cols is a multiple of 64
        const uint16_t* src = w + (size_t)(r0 + (threadIdx.x >> 5)) * n + c;
#pragma unroll 8
        for (int r = r0 + (threadIdx.x >> 5); r < r1; r += 8, src += (size_t)8 * n) {
            const uint4 v = *reinterpret_cast<const uint4*>(src);
            m[0] = max2(m[0], magnitudes(v.x));
            m[1] = max2(m[1], magnitudes(v.y));
            m[2] = max2(m[2], magnitudes(v.z));
            m[3] = max2(m[3], magnitudes(v.w));
        }
    }
#pragma unroll
    for (int t = 0; t < 4; t++) red[threadIdx.x >> 5][(threadIdx.x & 31) * 4 + t] = m[t];
    __syncthreads();
    const int pair = threadIdx.x, col = blockIdx.x * 256 + 2 * pair;
    if (pair < 128 && col < cols) {
        us2 v = red[0][pair];
#pragma unroll
        for (int r = 1; r < 8; r++) v = max2(v, red[r][pair]);
        *reinterpret_cast<us2*>(part + (size_t)blockIdx.y * cols + col) = v;
    }
}

// Scales from the chunks' maxima, of columns [first, first + cols) of w: INT4 (columns below n4) s = max|w| * 2/15
// (test.py:88-89), FP6 s = max|w| * 1/28 (test.py:19-23; the real-transpose layout replaces a zero scale by one), in the
// permuted order.  64 columns per workgroup, eight threads per column: all loads in flight at once.
// The range check of the true transpose's FP6 cast is settled here (`bad`): the quotients are clamped, so all that can go
// wrong is a NaN among them, and that takes an infinity or a NaN among the column's weights.  (A finite weight over its own
// column's scale stays below 43: the scale is the maximum / 28, off by at most a half of the smallest sub-normal, or one.)
__global__ __launch_bounds__(512) void column_scales_kernel(const uint16_t* part, int chunks, int first, int cols, int n4, int harness,
                                                            uint16_t* s4, uint16_t* s6, int* bad)
{
    __shared__ unsigned red[8][64];
    const int c = blockIdx.x * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6;   // (cols is a multiple of 64)
    unsigned m = 0;
#pragma unroll
    for (int i = 0; i < kMaxChunks / 8; i++) {
        const int chunk = q + 8 * i;
        const unsigned v = part[(size_t)(chunk < chunks ? chunk : q % chunks) * cols + c];
        m = v > m ? v : m;
    }
    red[q][threadIdx.x & 63] = m;
    __syncthreads();
    if (q) return;
#pragma unroll
    for (int i = 1; i < 8; i++) m = red[i][threadIdx.x] > m ? red[i][threadIdx.x] : m;
    const int at = first + c;
    // The product is rounded to binary32 first, as everywhere: a sub-normal scale can then lie half way (a maximum of 70 * 2^-24:
    // 2.5 units, to even 2), where one rounding of the exact product (v_fma_mixlo_f16, which the compiler takes) gives 3.
    float product = h2f((uint16_t)m) * (at < n4 ? (float)(2.0 / 15.0) : (float)(1.0 / 28.0));
    asm("" : "+v"(product));
    uint16_t sh = f2h(product);
    if (at < n4) {
        s4[scale_pos(at)] = sh;
    } else {
        if (bad && m >= 0x7c00u) __hip_atomic_store(bad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (!harness && (sh & 0x7fffu) == 0) sh = 0x3c00u;
        s6[scale_pos(at - n4)] = sh;
    }
}

// One thread per (group, 8 adjacent columns), 16-byte loads: scales of group sizes other than 128.
__global__ void int4_scales_kernel(const uint16_t* w, int k, int n, int n4, int g, uint16_t* s)
{
    const int c = (blockIdx.x * blockDim.x + threadIdx.x) * 8, gi = blockIdx.y;
    if (c >= n4) return;                                                // n4 is a multiple of 64
    us2 m[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
    const uint16_t* src = w + (size_t)gi * g * n + c;
#pragma unroll 4
    for (int r = 0; r < g; r++, src += n) {
        const uint4 v = *reinterpret_cast<const uint4*>(src);
        const uint32_t q[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int t = 0; t < 4; t++) m[t] = max2(m[t], magnitudes(q[t]));
    }
#pragma unroll
    for (int t = 0; t < 8; t++) s[(size_t)gi * n4 + c + t] = f2h(h2f(m[t >> 1][t & 1]) * (float)(2.0 / 15.0));
}

// w / s correctly rounded in binary32, from r = 1 / s correctly rounded: the product is off by at most one unit in the
// last place, the remainder w - q s is exact in the fused operation, and adding remainder * r rounds the quotient
// correctly (Markstein 1990).  For binary16 w and s nothing comes near the sub-normal range of binary32.
__device__ __forceinline__ float quotient(float w, float s, float r)
{
    const float q = w * r;
    return __builtin_fmaf(__builtin_fmaf(-q, s, w), r, q);
}
__device__ __forceinline__ h2 both(float v) { return h2{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ uint32_t bits(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// Nibble transpose: in[p] nibble m -> out[m] nibble p.
__device__ __forceinline__ void transpose_nibbles(const uint32_t (&in)[8], uint32_t (&out)[8])
{
    uint32_t x[4][2], y[2][2][2];
#pragma unroll
    for (int p = 0; p < 4; p++) {
        x[p][0] = __builtin_amdgcn_perm(in[p + 4], in[p], 0x05040100u);
        x[p][1] = __builtin_amdgcn_perm(in[p + 4], in[p], 0x07060302u);
    }
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int a = 0; a < 2; a++) {
            y[p][a][0] = __builtin_amdgcn_perm(x[p + 2][a], x[p][a], 0x06020400u);
            y[p][a][1] = __builtin_amdgcn_perm(x[p + 2][a], x[p][a], 0x07030501u);
        }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const uint32_t lo = y[0][a][b], hi = y[1][a][b];
            out[4 * a + 2 * b] = (lo & 0x0f0f0f0fu) | ((hi << 4) & 0xf0f0f0f0u);
            out[4 * a + 2 * b + 1] = ((lo >> 4) & 0x0f0f0f0fu) | (hi & 0xf0f0f0f0u);
        }
}

// Nibble m of a word of eight adjacent columns, built from pairs: nibbles 0 .. 3 the even columns, 4 .. 7 the odd ones.
constexpr int column_of(int m) { return m < 4 ? 2 * m : 2 * m - 7; }

// How a thread comes by the 64 weights it packs: four rows of 16 adjacent columns.  The lanes of a row (16, or 4) load
// adjacent 16-byte pieces, so that every load covers whole lines; of the first load's pieces every pair of lanes forms
// a 16-column block for its even lane, of the second load's one for its odd lane, and the lanes of a pair exchange the
// piece they do not keep.  The check weight leaves by the same way.  (Each lane moving its own two pieces, 16 bytes at a
// stride of 32, is right too: with those stores 4096 x 22016 took 107 us with the check weight, 39 without it.)
template <int LANES>
__device__ __forceinline__ int block_of(int jl) { return (jl >> 1) + (LANES / 2) * (jl & 1); }
__device__ __forceinline__ uint32_t from_neighbour(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, true);     // quad_perm [1, 0, 3, 2]
}
// in: a = the lane's piece of the first load, b = of the second; out: a, b = the low and the high half of its block
// (or the other way round: the exchange is its own inverse).  Even lanes keep a and take the neighbour's a for b; odd
// lanes keep b and take the neighbour's b for a.
__device__ __forceinline__ void exchange(uint4& a, uint4& b, bool odd)
{
    uint32_t* x = reinterpret_cast<uint32_t*>(&a);
    uint32_t* y = reinterpret_cast<uint32_t*>(&b);
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const uint32_t nx = from_neighbour(x[t]), ny = from_neighbour(y[t]);
        const uint32_t lo = odd ? ny : x[t], hi = odd ? y[t] : nx;
        x[t] = lo;
        y[t] = hi;
    }
}

// What pack_kernel tells a host that polls (0: nothing yet).
constexpr int kInRange = 1, kOutOfRange = 2;
struct PackArgs {
    const uint16_t* w;
    int k, n, n4, qc, g, per_column;
    uint16_t *s4, *s6;
    uint32_t *words, *plane2, *plane4;
    uint16_t* w_ref;
    // Host memory, for a caller that does not wait (null: not asked for): when the kernel starts, and the kernels before it are
    // done, it tells the host what they found about the range.
    const int* bad;
    int* verdict;
    int wgs6, blocks4;                // workgroups of the FP6 region (the first of the grid); INT4 workgroups per 128 rows
};

// A workgroup packs 128 rows x 256 columns: wave v k-block v, lane 16 i + jl its rows
// {2i, 2i+1, 2i+8, 2i+9} in the 16 columns of block_of(jl) -- word j = block & 3 of the eight owners
// t = 4l + i (l = 0 .. 7) of column group block / 4.
// GROUP128: the workgroup's rows are one scale group, whose scales it finds and writes itself.  Otherwise the scales are
// there: `g` rows per group, or one per column in the permuted order.
template <bool GROUP128>
struct Int4Smem {
    static constexpr int kScaleRows = GROUP128 ? 1 : 8;
    uint16_t max32[GROUP128 ? 32 : 1][256];                              // [wave, lane / 16][column]
    float r[kScaleRows][256], d[kScaleRows][256];                        // 1 / scale and scale, for quotient()
    uint16_t s[kScaleRows][256];
};
template <bool GROUP128>
__device__ __forceinline__ void int4_pack(const PackArgs& p, int col_block, int row_block, Int4Smem<GROUP128>& sm)
{
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i = lane >> 4, jl = lane & 15;
    const bool odd = jl & 1;
    const int col0 = col_block * 256, kb = row_block * 8 + wave;
    const int cols = p.n4 - col0 < 256 ? p.n4 - col0 : 256;              // a multiple of 64
    const int c = 16 * block_of<16>(jl);
    const bool first = 8 * jl < cols, second = 128 + 8 * jl < cols;      // (past the region's end: loads repeat its first
    const int at0 = first ? 8 * jl : 0, at1 = second ? 128 + 8 * jl : 0; // piece, nothing is stored)
    uint4 raw[4][2];                                                     // [row][8-column half]
    {
        const uint16_t* src = p.w + (size_t)(16 * kb < p.k ? 16 * kb : 0) * p.n + col0;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            raw[r][0] = *reinterpret_cast<const uint4*>(src + (size_t)k_off(i, r) * p.n + at0);
            raw[r][1] = *reinterpret_cast<const uint4*>(src + (size_t)k_off(i, r) * p.n + at1);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) exchange(raw[r][0], raw[r][1], odd);
    if constexpr (GROUP128) {
        uint32_t m[8];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            us2 v[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
#pragma unroll
            for (int r = 0; r < 4; r++) {
                v[0] = max2(v[0], magnitudes(raw[r][h].x));
                v[1] = max2(v[1], magnitudes(raw[r][h].y));
                v[2] = max2(v[2], magnitudes(raw[r][h].z));
                v[3] = max2(v[3], magnitudes(raw[r][h].w));
            }
#pragma unroll
            for (int t = 0; t < 4; t++) m[4 * h + t] = __builtin_bit_cast(uint32_t, v[t]);
        }
        uint4* dst = reinterpret_cast<uint4*>(&sm.max32[wave * 4 + i][c]);
        dst[0] = uint4{m[0], m[1], m[2], m[3]};
        dst[1] = uint4{m[4], m[5], m[6], m[7]};
        __syncthreads();
    }
    if (tid < cols) {
#pragma unroll
        for (int e = 0; e < Int4Smem<GROUP128>::kScaleRows; e++) {
            uint16_t sh;
            if constexpr (GROUP128) {
                unsigned m = 0;
#pragma unroll
                for (int q = 0; q < 32; q++) m = sm.max32[q][tid] > m ? sm.max32[q][tid] : m;
                sh = f2h(h2f((uint16_t)m) * (float)(2.0 / 15.0));
                p.s4[(size_t)row_block * p.n4 + col0 + tid] = sh;
            } else {
                int row = 16 * (row_block * 8 + e);
                row = row < p.k ? row : p.k - 1;
                sh = p.s4[p.per_column ? scale_pos(col0 + tid) : (size_t)(row / p.g) * p.n4 + col0 + tid];
            }
            // A zero scale (nothing in the group above 3 * 2^-24: codes 8) and an infinite one divide as "times zero"; what the
            // quotient of an infinity or a NaN becomes is settled where it is clamped.  (With an infinite scale the host path,
            // which packs the re-quantised check weight, has code 0 for the finite weights too; here they are 8.  Scale and check
            // weight are the same, and neither is a weight any more.)
            const bool none = (sh & 0x7fffu) == 0 || sh == 0x7c00u;
            sm.s[e][tid] = sh;
            sm.d[e][tid] = none ? 0.f : h2f(sh);
            sm.r[e][tid] = none ? 0.f : 1.0f / h2f(sh);
        }
    }
    __syncthreads();
    if (16 * kb >= p.k) return;                                          // (whole waves)
    const int e = GROUP128 ? 0 : wave;
    uint32_t v[8];
    uint16_t* back_to = p.w_ref + (size_t)(16 * kb) * p.n + col0 + 8 * jl;
#pragma unroll
    for (int r = 0; r < 4; r++) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t q[4] = {raw[r][h].x, raw[r][h].y, raw[r][h].z, raw[r][h].w};
            uint32_t word = 0, back[4];                                  // nibble t of `word`: column 2t, nibble 4 + t: column 2t + 1
#pragma unroll
            for (int t = 0; t < 4; t++) {
                // q = clamp(round(w / s) + 8, 0, 15) and the check weight (q - 8) * s (test.py:90-98).  |w / s| <= 11.25
                // (7.51 from normal scales on): adding 1544 = 1536 + 8, where binary16 counts in ones, rounds to the
                // nearest integer, ties to even, and leaves that + 8 in the low bits.  A NaN becomes code 0 in the
                // maximum.  (The harness packs the re-quantised check weight, test.py:99-101; that returns the same
                // q, as |q - 8| <= 8 and the product is rounded by at most 2^-11 relative, far from the next rounding
                // boundary, so it is not recomputed here.)
                const int at = c + 8 * h + 2 * t;
                const h2 wv = as_h2(q[t]);
                const h2 x = {(_Float16)quotient((float)wv[0], sm.d[e][at], sm.r[e][at]),
                              (_Float16)quotient((float)wv[1], sm.d[e][at + 1], sm.r[e][at + 1])};
                const h2 u = __builtin_elementwise_min(__builtin_elementwise_max(x + both(1544.0f), both(1536.0f)), both(1551.0f));
                word |= (bits(u) & 0x000f000fu) << (4 * t);
                back[t] = bits((u - both(1544.0f)) * *reinterpret_cast<const h2*>(&sm.s[e][at]));
            }
            v[4 * (r & 1) + (r >> 1) + 2 * h] = word;                    // the nibble of element x = r + 4 h
            raw[r][h] = uint4{back[0], back[1], back[2], back[3]};
        }
        if (p.w_ref) {
            exchange(raw[r][0], raw[r][1], odd);
            uint16_t* dst = back_to + (size_t)k_off(i, r) * p.n;
            if (first) *reinterpret_cast<uint4*>(dst) = raw[r][0];
            if (second) *reinterpret_cast<uint4*>(dst + 128) = raw[r][1];
        }
    }
    uint32_t o[8];
    transpose_nibbles(v, o);
    uint32_t* dst = p.words + (((size_t)kb * (p.n4 / 64) + (col0 + c) / 64) * 32 + i) * 4 + ((c >> 4) & 3);
    if (c < cols) {
#pragma unroll
        for (int m = 0; m < 8; m++) dst[16 * column_of(m)] = o[m];       // owner 4 l + i, word j
    }
}

// ---- FP6 region: columns [n4, n) of w

// e3m2 code of a binary16 value by truncation (weight_quant.cpp:27-96); 0xff when |x| is outside
// {0} u [0.0625, 28] or x is a NaN.
__device__ __forceinline__ uint32_t fp6_code(uint16_t h)
{
    const uint32_t sign = (h >> 15) << 5, e = (h >> 10) & 31u, m = h & 0x3ffu;
    if ((h & 0x7fffu) == 0) return sign;
    if (e >= 13 && e <= 19) {
        if (e == 19 && m > 0x300u) return 0xff;                      // above 28
        return sign | ((e - 12) << 2) | (m >> 8);
    }
    if (e == 12) return sign | ((0x400u | m) >> 9);                  // 0.125 .. 0.25: sub-normal codes 2, 3
    if (e == 11) return sign | 1;                                    // 0.0625 .. 0.125
    return 0xff;
}

// binary16 pattern of a code's value (exact).
__device__ __forceinline__ uint16_t fp6_value(uint32_t c)
{
    const uint32_t e = (c >> 2) & 7u, m = c & 3u;
    const float v = e == 0 ? (float)m * 0.0625f : (1.0f + 0.25f * (float)m) * __builtin_ldexpf(1.0f, (int)e - 3);
    return (uint16_t)(f2h(v) | ((c & 32u) ? 0x8000u : 0u));
}

// |x| < 0.0625 -> +0 (test.py:25; a NaN fails the test and stays), beyond +-28 -> +-28.
__device__ __forceinline__ uint16_t fp6_clamp(uint16_t v)
{
    if (h2f((uint16_t)(v & 0x7fffu)) < 0.0625f) return 0;
    if (h2f((uint16_t)(v & 0x7fffu)) > 28.0f) return (uint16_t)((v & 0x8000u) | 0x4f00u);
    return v;
}

// The FP6 planes of the true transpose, over threads like the INT4 words but 64 columns x 512 rows per workgroup (the
// region is narrow: 256 columns of a 4096 x 22016 weight would be 32 workgroups of the other shape too): lane
// 16 (k-block) + 4 i + jl.  4-bit plane: an 8 x 8 nibble transpose; 2-bit plane: another, whose nibbles' two bits are
// closed up, joined with those of the lane that holds the neighbouring tile of the pair.
struct Fp6Smem {
    float d[64], r[64];
};
__device__ __forceinline__ void fp6_pack(const PackArgs& p, int col_block, int row_block, Fp6Smem& sm)
{
    const int lane = threadIdx.x & 63, jl = lane & 3, i = (lane >> 2) & 3, j = block_of<4>(jl);
    const bool odd = jl & 1;
    const int kb = (row_block * 8 + (threadIdx.x >> 6)) * 4 + (lane >> 4);
    const bool here = 16 * kb < p.k;                                     // (whole waves: k is a multiple of 64)
    const uint16_t* src = p.w + (size_t)(here ? 16 * kb : 0) * p.n + p.n4 + col_block * 64 + 8 * jl;
    uint4 raw[4][2];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        raw[r][0] = *reinterpret_cast<const uint4*>(src + (size_t)k_off(i, r) * p.n);
        raw[r][1] = *reinterpret_cast<const uint4*>(src + (size_t)k_off(i, r) * p.n + 32);
    }
    if (threadIdx.x < 64) {
        // (never zero; an infinite or NaN scale comes from such a weight: the call fails)
        const float d = h2f(p.s6[scale_pos(col_block * 64 + threadIdx.x)]);
        sm.d[threadIdx.x] = d;
        sm.r[threadIdx.x] = 1.0f / d;
    }
    __syncthreads();
    if (!here) return;
    uint32_t lo[8], hi[8];                                               // [nibble of the word]: nibble t column 2t, 4 + t column 2t + 1
#pragma unroll
    for (int r = 0; r < 4; r++) {
        asm volatile("" : : : "memory");                                 // (reads the scales again: they do not fit the registers)
        exchange(raw[r][0], raw[r][1], odd);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t q[4] = {raw[r][h].x, raw[r][h].y, raw[r][h].z, raw[r][h].w};
            uint32_t low = 0, high = 0, back[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int at = 16 * j + 8 * h + 2 * t;
                const float d0 = sm.d[at], d1 = sm.d[at + 1];
                const h2 wv = as_h2(q[t]);
                h2 x = {(_Float16)quotient((float)wv[0], d0, sm.r[at]), (_Float16)quotient((float)wv[1], d1, sm.r[at + 1])};
                x = __builtin_elementwise_min(__builtin_elementwise_max(x, both(-28.0f)), both(28.0f));
                // Cut to two mantissa bits and scaled by 2^-12, exactly, the value has the code's five magnitude bits in
                // bits 8 .. 12, sub-normals included: e3m2's are binary16's.  (fp6_code is the same, case by case.)
                const uint32_t v = bits(as_h2(bits(x) & 0xff00ff00u) * both(1.0f / 4096));
                const uint32_t mag = v & 0x1f001f00u;
                // the sign, where the magnitude is not zero
                const uint32_t sign = v & 0x80008000u & __builtin_bit_cast(uint32_t, (us2)(__builtin_bit_cast(us2, mag) + (us2){0x7f00, 0x7f00}));
                low |= ((mag >> 8) & 0x000f000fu) << (4 * t);
                high |= (((mag >> 12) & 0x00010001u) | (sign >> 14)) << (4 * t);
                back[t] = bits(as_h2(mag | sign) * both(4096.0f) * (h2){(_Float16)d0, (_Float16)d1});
            }
            lo[7 - (2 * fp6_byte_of(r) + h)] = low;
            hi[7 - (2 * fp6_byte_of(r) + h)] = high;
            raw[r][h] = uint4{back[0], back[1], back[2], back[3]};
        }
        if (p.w_ref) {
            exchange(raw[r][0], raw[r][1], odd);
            uint16_t* dst = p.w_ref + (size_t)(16 * kb + k_off(i, r)) * p.n + p.n4 + col_block * 64 + 8 * jl;
            *reinterpret_cast<uint4*>(dst) = raw[r][0];
            *reinterpret_cast<uint4*>(dst + 32) = raw[r][1];
        }
    }
    uint32_t o[8];
    const size_t granule = ((size_t)kb * (p.qc / 64) + col_block) * 32 + i;      // of owner t = i; owner 4 l + i: 4 l further
    transpose_nibbles(lo, o);
#pragma unroll
    for (int m = 0; m < 8; m++) p.plane4[(granule + 4 * column_of(m)) * 4 + j] = o[m];
    transpose_nibbles(hi, o);
    // Tiles 2a and 2a + 1 share a word; they are two lanes apart (block_of).
    const bool upper = j & 1;
#pragma unroll
    for (int m = 0; m < 8; m++) {
        uint32_t v = ((o[m] >> 2) & 0x0c0c0c0cu) | (o[m] & 0x03030303u);         // each byte: [e_x, e_{x+4}] in its low four bits
        v <<= upper ? 0 : 4;
        o[m] = v | (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, true);     // quad_perm [2, 3, 0, 1]
    }
#pragma unroll
    for (int m = 0; m < 4; m++)                                          // (one lane stores columns 0, 2, 4, 6, the other the odd ones)
        p.plane2[(granule + 4 * (2 * m + (upper ? 1 : 0))) * 2 + (j >> 1)] = upper ? o[m + 4] : o[m];
}

// One launch packs both regions, the FP6 region's few workgroups first so that they run beside the others.
// 4096 x 22016, group-128 scales, 256 FP6 columns, with the check weight: scales 47 us, INT4 words 77, FP6 maxima 9, planes
// 20 as launches of one after the other; now maxima and scales 4 + 2 us, this kernel 80 (5.1 TB/s of the 0.41 GB in and
// out; a plain copy on the same box reaches 5.3).  512 threads: with one k-block per wave the weights of a
// thread are 32 registers, and four waves fit a SIMD (two k-blocks per wave spilled at four, and took 105 us at three).
template <bool GROUP128>
__global__ __launch_bounds__(512, 4) void pack_kernel(const PackArgs p)
{
    __shared__ __attribute__((aligned(16))) union {
        Int4Smem<GROUP128> int4;
        Fp6Smem fp6;
    } sm;
    const int b = blockIdx.x;
    if (b == 0 && threadIdx.x == 0 && p.verdict) {
        // One word says both that the range is known and what it is: the host relies on no order between this store and the
        // earlier kernel's store to `bad`, which has arrived when the load has returned its value.
        const int bad = __hip_atomic_load(p.bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(p.verdict, bad ? kOutOfRange : kInRange, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (b < p.wgs6) {
        const int across = p.qc / 64;
        fp6_pack(p, b % across, b / across, sm.fp6);
    } else {
        int4_pack<GROUP128>(p, (b - p.wgs6) % p.blocks4, (b - p.wgs6) / p.blocks4, sm.int4);
    }
}

// The reference harness's own layout (test.py:13-58): one thread per fragment owner of the FP6 planes.  `row` (0..qc) and
// `col` (0..k) index the [qc, k] matrix the reference's prepacker works on; that matrix is the flat [k, qc] buffer re-read
// with row length k (weight_quant pybind.cpp:52-57 does not transpose): element (row, col) is flat element row*k + col,
// normalised by the scale of *its* column in the [k, qc] view, while the check weight multiplies by the scale of `row`
// (test.py:37-38).
__global__ void fp6_pack_harness_kernel(const uint16_t* w, int k, int n, int n4, int qc, const uint16_t* s6, uint32_t* plane2,
                                        uint32_t* plane4, uint16_t* w_ref, int* bad)
{
    const size_t owner = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t groups = qc / 64, owners = (size_t)(k / 16) * groups * 32;
    if (owner >= owners) return;
    const int t = (int)(owner & 31), l = t >> 2, i = t & 3;
    const size_t g64 = (owner >> 5) % groups, kb = (owner >> 5) / groups;
    uint32_t w2[2] = {0, 0}, w4[4];
    bool any_bad = false;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        uint32_t word = 0;
#pragma unroll
        for (int x = 0; x < 8; x++) {
            const size_t row = 64 * g64 + 16 * j + l + 8 * (x >> 2);
            const size_t col = 16 * kb + k_off(i, x & 3);
            const size_t flat = row * (size_t)k + col, src_k = flat / qc, src_n = flat % qc;
            const uint32_t c = fp6_code(fp6_clamp(f2h(h2f(w[src_k * n + n4 + src_n]) / h2f(s6[scale_pos(src_n)]))));
            any_bad |= c == 0xff;
            if (w_ref) w_ref[col * n + n4 + row] = f2h(h2f(fp6_value(c)) * h2f(s6[scale_pos(row)]));
            const int b = fp6_byte_of(x), hi = x >> 2;
            word |= (c & 15u) << (28 - 4 * (2 * b + hi));
            w2[j >> 1] |= ((c >> 4) & 3u) << (30 - 2 * (4 * b + 2 * (j & 1) + hi));
        }
        w4[j] = word;
    }
    uint4 v4 = {w4[0], w4[1], w4[2], w4[3]};
    reinterpret_cast<uint4*>(plane4)[owner] = v4;
    uint2 v2 = {w2[0], w2[1]};
    reinterpret_cast<uint2*>(plane2)[owner] = v2;
    if (any_bad) *bad = 1;
}

// The FP6 range flag of a call: a line of pinned host memory that the kernels write (`bad` only when something is out of
// range) and the call reads after its wait, so that no copy back is enqueued.  kFlags lines, allocated once and kept; a
// call holds one of them, so calls on several threads and streams do not meet.  A line goes back only after a wait that
// succeeded: until then kernels of this call may still write it, and the next call's check would see that.
constexpr int kFlags = 64;
struct alignas(64) FlagLine {
    int bad, verdict;
};
std::mutex g_flag_mutex;
FlagLine* g_flags = nullptr;
unsigned long long g_flags_taken = 0, g_flags_lost = 0;                  // (lost: taken for good)
struct RangeFlag {
    int index = -1;
    bool idle = true;                                                    // nothing enqueued may still write the line
    hipError_t err = hipSuccess;
    explicit RangeFlag(bool wanted)
    {
        while (wanted) {
            {
                std::lock_guard<std::mutex> lock(g_flag_mutex);
                if (!g_flags && (err = hipHostMalloc(reinterpret_cast<void**>(&g_flags), kFlags * sizeof(FlagLine), hipHostMallocPortable | hipHostMallocMapped)) != hipSuccess)
                    return;
                if (~g_flags_taken) {
                    index = __builtin_ctzll(~g_flags_taken);
                    g_flags_taken |= 1ull << index;
                    g_flags[index] = FlagLine{0, 0};
                    return;
                }
                if (!~g_flags_lost) {                                    // (64 calls whose wait failed)
                    err = hipErrorOutOfMemory;
                    return;
                }
            }
            std::this_thread::yield();                                   // (64 other threads are inside a pack call)
        }
    }
    ~RangeFlag()
    {
        if (index < 0) return;
        std::lock_guard<std::mutex> lock(g_flag_mutex);
        if (idle)
            g_flags_taken &= ~(1ull << index);
        else
            g_flags_lost |= 1ull << index;
    }
    // All of the call's kernels.
    hipError_t wait(hipStream_t st)
    {
        const hipError_t e = hipStreamSynchronize(st);
        idle = e == hipSuccess;
        return e;
    }
    // Those that decide about the range: true once pack_kernel, which writes nothing here after that, has said that nothing is
    // out of it.  Not for long (the stream may have other work in front): false leaves it to wait().
    bool in_range_soon() const
    {
        for (int i = 0; i < 20000; i++) {
            if (const int v = __atomic_load_n(&g_flags[index].verdict, __ATOMIC_ACQUIRE)) return v == kInRange;
            __builtin_ia32_pause();
        }
        return false;
    }
    int* bad() const { return index < 0 ? nullptr : &g_flags[index].bad; }
    int* verdict() const { return index < 0 ? nullptr : &g_flags[index].verdict; }
    bool out_of_range() const { return index >= 0 && __atomic_load_n(&g_flags[index].bad, __ATOMIC_RELAXED) != 0; }
};

}  // namespace
}  // namespace fp6m

namespace fp6m {
namespace {

// whole: do not return before the call's kernels are done (where the range of the FP6 cast is checked at all).
int pack_mixed(const void* w, int k, int n, int quant_cols, int group_size, int harness_layout, void* B, void* s, void* w_ref, int dev,
               void* stream, bool whole)
{
    if (!w || !B || !s) return FP6M_ERR_ARG;
    const int qc = quant_cols == -1 ? 0 : quant_cols;
    if (k <= 0 || n <= 0 || qc < 0 || qc > n || qc % 64 || (n - qc) % 64 || k % 64 || n % 8) return FP6M_ERR_SHAPE;
    if (group_size != -1 && (group_size <= 0 || k % group_size || group_size % 16)) return FP6M_ERR_SHAPE;
    const int n4 = n - qc, g = group_size == -1 ? k : group_size;
    const bool per_column = group_size == -1;
    DeviceGuard guard(dev);                                              // the caller's current device is restored on return
    hipError_t e = guard.err;
    if (e != hipSuccess) return hip_fail(e);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint16_t* wp = static_cast<const uint16_t*>(w);
    uint16_t* sp = static_cast<uint16_t*>(s);
    uint16_t* rp = static_cast<uint16_t*>(w_ref);
    uint32_t* bp = static_cast<uint32_t*>(B);
    uint16_t* s6 = sp + (per_column ? (size_t)n4 : (size_t)(k / g) * n4);
    uint32_t* plane2 = bp + (size_t)k * n4 / 8;
    uint32_t* plane4 = plane2 + (size_t)k * qc / 16;
    PackArgs a = {wp, k, n, n4, qc, g, (int)per_column, sp, s6, bp, plane2, plane4, rp, nullptr, nullptr, 0, n4 ? (n4 + 255) / 256 : 1};
    if (qc > 0 && capturing(st)) return hip_fail(hipErrorStreamCaptureUnsupported);   // (the wait below: refused before anything is recorded)
    RangeFlag flag(qc > 0);
    if (flag.err != hipSuccess) return hip_fail(flag.err);
    if (!whole && !harness_layout) {
        a.bad = flag.bad();
        a.verdict = flag.verdict();
    }
    // Scales that span all of k (all columns with per-column scales, else the FP6 region): maxima of at most kMaxChunks row
    // ranges first.  They wait, two bytes each, in B, which is packed afterwards and larger (at least k / 2 bytes a column).
    const int first = per_column ? 0 : n4, cols = n - first;
    if (cols) {
        const int rows = ((k + kMaxChunks - 1) / kMaxChunks + 63) / 64 * 64, chunks = (k + rows - 1) / rows;
        uint16_t* part = reinterpret_cast<uint16_t*>(B);
        hipLaunchKernelGGL(column_maxima_kernel, dim3((cols + 255) / 256, chunks), dim3(256), 0, st, wp + first, k, n, cols, rows, part);
        hipLaunchKernelGGL(column_scales_kernel, dim3(cols / 64), dim3(512), 0, st, part, chunks, first, cols, n4, harness_layout, sp, s6,
                           harness_layout ? nullptr : flag.bad());
    }
    if (n4 && !per_column && g != 128)
        hipLaunchKernelGGL(int4_scales_kernel, dim3((n4 / 8 + 255) / 256, k / g), dim3(256), 0, st, wp, k, n, n4, g, sp);
    if (qc && harness_layout) {
        const size_t owners = (size_t)(k / 16) * (qc / 64) * 32;
        hipLaunchKernelGGL(fp6_pack_harness_kernel, dim3((unsigned)((owners + 255) / 256)), dim3(256), 0, st, wp, k, n, n4, qc, s6, plane2,
                           plane4, rp, flag.bad());
    } else if (qc) {
        a.wgs6 = qc / 64 * ((k + 511) / 512);
    }
    const int wgs4 = n4 ? a.blocks4 * ((k + 127) / 128) : 0;
    if (a.wgs6 + wgs4) {
        if (g == 128 && !per_column)
            hipLaunchKernelGGL(pack_kernel<true>, dim3(a.wgs6 + wgs4), dim3(512), 0, st, a);
        else
            hipLaunchKernelGGL(pack_kernel<false>, dim3(a.wgs6 + wgs4), dim3(512), 0, st, a);
    }
    e = hipGetLastError();
    if (qc) {
        // The range check of the FP6 cast is reported by value, so this call waits: for the kernels in front of pack_kernel,
        // which find the maxima, or, where the harness layout's kernel checks cast by cast, where something is out of range
        // or failed to launch (the flag's line is another call's next), and from the entry that waits, for all of them.  With
        // every call waiting for all of them the GPU is idle between one call's last kernel and the next one's first:
        // 4096 x 22016, group-128 scales, 256 FP6 columns, calls in a row 106.6 us each, 85.2 from the other entry (a call
        // that is waited for takes as long from either).
        if (e == hipSuccess && a.verdict && flag.in_range_soon()) return FP6M_OK;
        const hipError_t waited = flag.wait(st);
        if (e == hipSuccess) e = waited;
    }
    if (e != hipSuccess) return hip_fail(e);
    return flag.out_of_range() ? FP6M_ERR_RANGE : FP6M_OK;
}

}  // namespace
}  // namespace fp6m

extern "C" int fp6m_pack_mixed_device(const void* w, int k, int n, int quant_cols, int group_size, int harness_layout,
                                      void* B, void* s, void* w_ref, int dev, void* stream)
{
    return fp6m::pack_mixed(w, k, n, quant_cols, group_size, harness_layout, B, s, w_ref, dev, stream, true);
}

extern "C" int fp6m_pack_mixed_device_async(const void* w, int k, int n, int quant_cols, int group_size, int harness_layout,
                                            void* B, void* s, void* w_ref, int dev, void* stream)
{
    return fp6m::pack_mixed(w, k, n, quant_cols, group_size, harness_layout, B, s, w_ref, dev, stream, false);
}
