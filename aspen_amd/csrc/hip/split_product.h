// Single-precision products on the bfloat16 matrix cores.
//
// A float has 24 significant bits, a bfloat16 eight: x = h + m + l with h = bf16 (x), m = bf16 (x - h), l = x - h - m, and
// all three terms are exact (each rounding to nearest takes eight bits and a sign off the rest; the rest of the second
// fits a bfloat16 whole).  A product of two floats is then nine products of bfloat16 terms, each of them exact in the
// matrix core's single-precision sum.  Six are computed:
//     a b = ah bh  +  (ah bm + am bh)  +  (ah bl + al bh + am bm)      left out: am bl + al bm + al bl < 2^-24 |a b|
// (|m| <= 2^-8 |x|, |l| <= 2^-17 |x|), i.e. at worst what rounding ONE float product to a float may cost, 0.09 of that in the root mean
// square over mantissas.  The leading products are summed in one
// accumulator and the five small ones in another, added at the end: the large sum is then rounded once per 32 K positions,
// one v_mfma_f32_16x16x32_bf16 (32 addends that make 0.75 units in the last place raise the sum; each half, 0.375, would not), instead of
// once per two (v_mfma_f32_32x32x2_f32), the small sum's roundings do not count at its size, and the result is closer to the
// exact one than the single-precision matrix instruction's (relative to a 64-bit sum, 2-norm over 128 x 128 results, inputs
// normal / rectified normal: K = 64 4.8e-8 / 4.2e-8 against 1.4e-7 / 1.0e-7; K = 1024 1.8e-7 / 1.5e-7 against 5.7e-7 / 4.2e-7;
// K = 4096 4.0e-7 / 3.2e-7 against 1.1e-6 / 8.1e-7; with one accumulator for all six products 1.0e-6 / 9.5e-7).
// Speed: bfloat16 matrix instructions do sixteen times the single-precision one's work per cycle, so six products take 3 / 8 of its
// time.  In practice both are limited by power, and a product's time is its energy.  Registers alone, every compute
// unit, products in TFLOP/s of the floats' work (417 nominal): v_mfma_f32_32x32x16_bf16 300, v_mfma_f32_16x16x32_bf16 355 (half the
// accumulator traffic per product); a loop that also splits, stages and fetches what a 128 x 64 tile does, 188 and 229 (a 64 x 64
// tile's 184; whole products of 128 x 64 tiles reach 214 to 230, see PRODUCT_BAND).  So the smaller block it is.  The sums come out the same: over 1000 x 3137 and 2048 x 2048 results, K = 32 ... 4096, both
// instructions' errors against 64-bit sums agree to three digits.
// The range is float's own (bfloat16 has the same exponent) with two edges.  Terms below bfloat16's smallest number, 2^-133, do not
// exist: an input below 2^-110 enters with an absolute error of up to 2^-134.  And infinities, NaNs and floats within 0.2 % of the
// largest one, whose h rounds to infinity, leave no finite sum (inf - inf in m, inf times a zero term): the tiles look
// for sums that are not finite and compute those again from the floats themselves (single_precision_block in tile_kernels.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef float floatx16 __attribute__ ((ext_vector_type (16)));
typedef float floatx8 __attribute__ ((ext_vector_type (8)));
typedef float floatx4 __attribute__ ((ext_vector_type (4)));
typedef uint32_t u32x4 __attribute__ ((ext_vector_type (4)));
typedef __bf16 bf16x2 __attribute__ ((ext_vector_type (2)));
typedef __bf16 bf16x8 __attribute__ ((ext_vector_type (8)));
typedef float floatx2 __attribute__ ((ext_vector_type (2)));

// two floats rounded to bfloat16, the first in the low half (one v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t bf16_pair (float a, float b)
{
    return __builtin_bit_cast (uint32_t, __builtin_convertvector ((floatx2){a, b}, bf16x2));
}
__device__ __forceinline__ float bf16_low (uint32_t p) { return __builtin_bit_cast (float, p << 16); }
__device__ __forceinline__ float bf16_high (uint32_t p) { return __builtin_bit_cast (float, p & 0xffff0000u); }

// the next term of eight floats; they keep what it leaves
__device__ __forceinline__ u32x4 take_term (float4 &a, float4 &b)
{
    const u32x4 t = {bf16_pair (a.x, a.y), bf16_pair (a.z, a.w), bf16_pair (b.x, b.y), bf16_pair (b.z, b.w)};
    a.x -= bf16_low (t[0]); a.y -= bf16_high (t[0]); a.z -= bf16_low (t[1]); a.w -= bf16_high (t[1]);
    b.x -= bf16_low (t[2]); b.y -= bf16_high (t[2]); b.z -= bf16_low (t[3]); b.w -= bf16_high (t[3]);
    return t;
}

// the three terms of eight floats, as matrix-core operands (K positions 0 .. 7 of a lane)
struct split8_t { u32x4 h, m, l; };
__device__ __forceinline__ split8_t split8 (float4 a, float4 b)
{
    split8_t s;
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    #pragma unroll
    for (int q = 0; q < 4; q++)
    {
        float u = x[2 * q], v = x[2 * q + 1];
        const uint32_t h = bf16_pair (u, v);
        u -= bf16_low (h); v -= bf16_high (h);
        const uint32_t m = bf16_pair (u, v);
        u -= bf16_low (m); v -= bf16_high (m);
        s.h[q] = h; s.m[q] = m; s.l[q] = bf16_pair (u, v);
    }
    return s;
}

// The terms of weights, which the kernels have nothing else of: join2 gets every float back that is not below 2^-110.  An infinity or a
// NaN is its own h with m = l = 0, a finite float never rounds up to infinity (the largest bfloat16 and the rest instead).
__device__ __forceinline__ split8_t split8_weights (float4 a, float4 b)
{
    split8_t s = split8 (a, b);
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    #pragma unroll
    for (int q = 0; q < 4; q++)
    {
        uint32_t h = s.h[q], drop = 0;
        #pragma unroll
        for (int e = 0; e < 2; e++)
        {
            const uint32_t half = e ? 0xffff0000u : 0xffffu;
            if ((h & 0x7f807f80u & half) != (0x7f807f80u & half)) continue;
            if (fabsf (x[2 * q + e]) < INFINITY) h = (h & ~half) | (((h & 0x80008000u) | 0x7f7f7f7fu) & half);
            else drop |= half;
        }
        if (h == s.h[q] && drop == 0) continue;
        float u = x[2 * q] - bf16_low (h), v = x[2 * q + 1] - bf16_high (h);
        const uint32_t m = bf16_pair (u, v);
        u -= bf16_low (m); v -= bf16_high (m);
        s.h[q] = h; s.m[q] = m & ~drop; s.l[q] = bf16_pair (u, v) & ~drop;
    }
    return s;
}
// the two floats of one register of each term (m + l is the rest of the float behind h, exact; so is the sum of all)
__device__ __forceinline__ floatx2 join2 (uint32_t h, uint32_t m, uint32_t l)
{
    return (floatx2){bf16_low (h) + (bf16_low (m) + bf16_low (l)), bf16_high (h) + (bf16_high (m) + bf16_high (l))};
}

__device__ __forceinline__ floatx4 mfma_bf16 (const u32x4 &a, const u32x4 &b, const floatx4 &c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16 (__builtin_bit_cast (bf16x8, a), __builtin_bit_cast (bf16x8, b), c, 0, 0, 0);
}
// hi += leading products, lo += the five small ones, of COUNT neighbouring blocks of 16 x 16 x 32: rows of the result = rows of
// `a`, columns = rows of `b[j]`.  Neighbouring instructions share the operand of `a` and add to different sums.
template <int COUNT>
__device__ __forceinline__ void split_mfma (const split8_t &a, const split8_t (&b)[COUNT], floatx4 (&hi)[COUNT], floatx4 (&lo)[COUNT])
{
    #pragma unroll
    for (int j = 0; j < COUNT; j++) lo[j] = mfma_bf16 (a.h, b[j].l, lo[j]);
    #pragma unroll
    for (int j = 0; j < COUNT; j++) hi[j] = mfma_bf16 (a.h, b[j].h, hi[j]);
    #pragma unroll
    for (int j = 0; j < COUNT; j++) lo[j] = mfma_bf16 (a.h, b[j].m, lo[j]);
    #pragma unroll
    for (int j = 0; j < COUNT; j++) lo[j] = mfma_bf16 (a.m, b[j].m, lo[j]);
    #pragma unroll
    for (int j = 0; j < COUNT; j++) lo[j] = mfma_bf16 (a.m, b[j].h, lo[j]);
    #pragma unroll
    for (int j = 0; j < COUNT; j++) lo[j] = mfma_bf16 (a.l, b[j].h, lo[j]);
}
// Order of the K axis inside a slice of 32 (both operands have to agree, the sum does not care): a lane of a matrix
// instruction holds eight K positions of row lane % 16, "unit" u = lane / 16, and unit u stands for the slice's floats
// 4u .. 4u+3 and 16+4u .. 16+4u+3.  Four neighbouring threads that fetch the four units of a row then read 64 contiguous bytes
// with each of their two 16-byte requests.
#define SLICE_K 32

// Weights on the device.  SPLIT: per block of 32 rows and slice, per half of 16 rows, the terms h, m, l, each as the 64 lanes' 16 bytes in a
// row (lane l: row l % 16, unit l / 16): 6144 bytes that a wavefront fetches with contiguous 1 KB requests straight into
// the registers the matrix instructions read.  RAW: the same with the floats themselves, per half two rows of 64 x 16
// bytes (floats 4u .. and 16+4u ..): 4096 bytes per block and slice, split in registers.  A weight belongs to one
// wavefront of a tile, so nothing is staged through LDS.
// RAW is for layers that are bound by the weights' trip from memory.
#define WEIGHT_BLOCK_ROWS 32
#define SPLIT_SLICE_BYTES 6144u
#define RAW_SLICE_BYTES 4096u

// HALVES: neighbouring groups of 16 rows (2: a whole block); SETS: register sets, i.e. slices of weights in flight.
template <bool RAW, int HALVES, int SETS = 1> struct WeightFragments
{
    static constexpr uint32_t SLICE = RAW ? RAW_SLICE_BYTES : SPLIT_SLICE_BYTES, PARTS = RAW ? 2 : 3;
    typedef const char __attribute__ ((address_space (1))) *bytes_t;
    bytes_t base;               // of the wavefront's first group of 16 rows (uniform)
    uint32_t lane16;
    u32x4 f[SETS][HALVES][PARTS];
    // group: the first group of 16 rows, even where HALVES is 2
    __device__ __forceinline__ void init (const void *w, uint32_t group, uint32_t slices, uint32_t lane)
    {
        base = (bytes_t)w + ((uint64_t)(group >> 1) * ((uint64_t)slices * SLICE) + (group & 1u) * (SLICE / 2));
        lane16 = lane * 16u;
    }
    __device__ __forceinline__ void load (int it, int set = 0)
    {
        const bytes_t p = base + (uint32_t)it * SLICE;
        #pragma unroll
        for (uint32_t j = 0; j < HALVES; j++)
            #pragma unroll
            for (uint32_t q = 0; q < PARTS; q++) f[set][j][q] = *(const u32x4 __attribute__ ((address_space (1))) *)(p + (lane16 + j * (SLICE / 2) + q * 1024u));
    }
    __device__ __forceinline__ void take_second_set ()
    {
        #pragma unroll
        for (uint32_t j = 0; j < HALVES; j++)
            #pragma unroll
            for (uint32_t q = 0; q < PARTS; q++) f[0][j][q] = f[1][j][q];
    }
    __device__ __forceinline__ split8_t operand (int half, int set = 0) const
    {
        if constexpr (RAW) return split8 (__builtin_bit_cast (float4, f[set][half][0]), __builtin_bit_cast (float4, f[set][half][1]));
        else return {f[set][half][0], f[set][half][1], f[set][half][2]};
    }
};

// LDS stage of the other operand, one slice of ROWS rows: three planes (h, m, l) of ROWS x 64 bytes, the four 16-byte units
// of a row in the order unit ^ (-(row / 4) % 4).  A 16-byte access serves lanes 0-3, 12-15, 20-23 and 24-27 together (then 4-11, 16-19
// and 28-31, and the upper half alike): of a fragment read (16 rows a unit) rows 0-3 and 12-15 of one unit with rows 4-11 of the
// next, of a write (a row in four lanes) four whole rows; both touch every bank once, as sixteen lanes in a row would.  With
// unit ^ (row / 4 % 4) every read took twice the cycles (conflicts in 37 % of the cycles the LDS was busy with ResNet-50 batch 32):
// VGG-16 batch 32 5244 -> 5185 us, YOLO-v3 batch 8 3915 -> 3812, GPT-2 4 x 512 2738 -> 2689.
template <int ROWS> struct SplitStage
{
    static constexpr uint32_t PLANE = ROWS * 64u, BYTES = 3u * PLANE;
    static __device__ __forceinline__ uint32_t offset (uint32_t row, uint32_t unit) { return row * 64u + ((unit ^ ((0u - (row >> 2)) & 3u)) * 16u); }
    static __device__ __forceinline__ split8_t read (const char *stage, uint32_t off)
    {
        return {*reinterpret_cast<const u32x4 *> (stage + off), *reinterpret_cast<const u32x4 *> (stage + off + PLANE), *reinterpret_cast<const u32x4 *> (stage + off + 2 * PLANE)};
    }
};
