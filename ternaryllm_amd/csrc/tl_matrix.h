// What the matrix-core kernels share: two-bit weight codes turned into matrix operands, the matrix instruction, the
// exact walk of the index stream, and the last steps of an output.
//
// The codes (include/ternary_spmm.h) are arranged so that an operand costs two vector instructions per two weights: a
// code's sign and non-zero bits, shifted to the top of a half dword, ARE the sixteen-bit floating-point number +-2.0 or
// +-0.0, in fp16 and in bf16 alike (0x4000 is 2.0 in both).  Products with +-2.0 are exact and the factor 2 is taken
// out of the fp32 sums at the end, exactly.  The contraction is dense: a zero weight is multiplied too.  Activations
// that are not finite would spoil other columns that way (0 * inf), so every sum that comes out not finite is worked
// out again from the index stream, which names only the non-zero weights.
#pragma once
#include "tl_device.h"

namespace tl {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Weights of matrix step S (32 rows of K) of a unit, for this lane's column: eight values.
template <int S>
__device__ __forceinline__ u32x4 weight_operand(u32x4 codes)
{
    const uint32_t c = codes[S >> 1];
    constexpr int first = (S & 1) * 8;
    return u32x4{(c << first) & 0xC000C000u, (c << (first + 2)) & 0xC000C000u, (c << (first + 4)) & 0xC000C000u, (c << (first + 6)) & 0xC000C000u};
}

// acc[i] += sum over k of w[row 4 * (lane / 16) + i][k] * x[column lane % 16][k], 32 values of k, eight to a lane:
// the rows are 16 columns of the weight, the columns 16 activation rows.
template <bool BF16>
__device__ __forceinline__ f32x4 matrix_step(u32x4 w, u32x4 x, f32x4 acc)
{
    if constexpr (BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), acc, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, w), __builtin_bit_cast(half8, x), acc, 0, 0, 0);
}

// 16 bytes per lane from `base` + offset into LDS at `lds` + 16 * lane.  (As assembly, because the compiler would wait for
// all such loads before any read of LDS; here they are counted by hand.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // (m0 is a register that the compiler reserves; named all the same, as this writes it)
__device__ __forceinline__ void load_to_lds(uint32_t lds, const void* base, uint32_t offset)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(offset), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop

// An fp32 value in three bf16 parts: v = a + (b + c) / kLowScale, each part the next 8 of v's 24 significant bits, by
// truncation.  The two low parts are scaled so that they stay in bf16's range (down to 2^-133, which the matrix
// instruction keeps) for every v down to fp32's smallest, 2^-149: without that a v below 2^-110 lost bits (against fp64 4.4e-6
// at 2^-116, 1.1e-3 at 2^-124; now as exact as at any magnitude).  Their products are summed apart from the leading
// ones', which helps ordinary values too: the leading sums hardly round, and the low sums' roundings weigh 2^-8.
// Above 2^119 the low parts overflow and make the sum infinite, and the output is worked out again.
constexpr float kLowScale = 65536.0f;

// acc + low / kLowScale, in place
__device__ __forceinline__ void add_low(f32x4& acc, const f32x4& low)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = fmaf(low[i], 1.0f / kLowScale, acc[i]);
}

// The bit patterns of the parts, in the upper halves; a v that is not finite goes into the first alone.
__device__ __forceinline__ void split3(float v, uint32_t* a, uint32_t* b, uint32_t* c)
{
    const uint32_t va = __float_as_uint(v) & 0xffff0000u;
    const float r1 = (v - __uint_as_float(va)) * kLowScale;
    const bool fine = fabsf(v) < __builtin_huge_valf();
    const uint32_t vb = __float_as_uint(r1) & 0xffff0000u;
    const float r2 = r1 - __uint_as_float(vb);
    *a = va;
    *b = fine ? vb : 0u;
    *c = fine ? __float_as_uint(r2) & 0xffff0000u : 0u;
}

// One output of the product from the index stream alone: x(k) of the rows that column n names, added and subtracted.
template <typename X>
__device__ __forceinline__ float walk_column(const WeightPtrs& w, int T, int tile_rows, int n, X x)
{
    float sum = 0.f;
    for (int t = 0; t < T; ++t) {
        const uint32_t* chunk = w.stream + w.chunkstart[(size_t)(n / TL_BLOCK_COLUMNS) * T + t];
        const uint32_t d = chunk[n % TL_BLOCK_COLUMNS];
        const unsigned char* run = reinterpret_cast<const unsigned char*>(chunk + (d >> 16));
        const int n_pos = (int)(d & 0xffu), n_neg = (int)((d >> 8) & 0xffu);
        for (int i = 0; i < n_pos; ++i) sum += x(t * tile_rows + run[i]);
        run += 4 * run_pos_dwords(d);
        for (int i = 0; i < n_neg; ++i) sum -= x(t * tile_rows + run[i]);
    }
    return sum;
}

// Activation (m, k) as the caller passed it.
struct CallersX {
    const void* X;
    long long sm, sk;
    int f16, m;
    __device__ __forceinline__ float operator()(int k) const
    {
        const long long i = m * sm + k * sk;
        return f16 ? __half2float(static_cast<const __half*>(X)[i]) : static_cast<const float*>(X)[i];
    }
};

__device__ __forceinline__ CallersX callers_x(const KernelArgs& a, int m)
{
    return CallersX{a.X, a.x_kmajor ? 1 : a.ldx, a.x_kmajor ? a.ldx : 1, a.x_f16, m};
}

}  // namespace tl
