// A few activation rows (up to 48): the ternary product on the matrix cores straight from memory.
//
// Bound by latency and by the bytes of the codes: a workgroup owns one or two blocks of 16 columns over all of K, its
// waves share K out among them and meet once, in LDS, at the very end.  Nothing is staged: a lane's 16 bytes of
// activations are the matrix operand as they lie in a row, and every load of a turn (256 rows of K) is in flight before the
// first product.  fp32 rows become three bf16 parts in registers; with 48 of them that is what takes the time.
// us at 4096 -> 11008, 66 % zeros, walking the index stream / here: fp16 2 rows 16.6 / 6.1, 8 rows 20.8 / 7.9 (11.3 MB of
// codes: 1.4 TB/s), 48 rows 70 / 26 (at this width the rule in tl_kernels.hip leaves 9 to 48 fp16 rows to the walk); fp32 8
// rows 25.6 / 13.0, 48 rows 103 / 47.
#include "tl_matrix.h"

using namespace tl;

namespace {

constexpr int kSliceRows = 64;        // rows of K that one dword of a lane's codes names
constexpr int kPartFloats = 320;      // LDS floats of 16 x 16 partial sums: lane l's four at 4 * l + 16 * (l / 16), so that the
                                      // four quarters, whose columns one row's outputs take together, lie on different banks
constexpr int kMaxWaves = 16;

// How rows are read: aligned 16-byte pieces (K a multiple of 8); 16 bytes at a time from any element on, but for the turn in
// which a row ends; element by element (K-major).
enum { kRowPieces = 0, kRows = 1, kElements = 2 };

// Eight activations of a row from k on.  Past K: zeros (element by element) or the row's last whole piece again (such rows
// of K meet zero codes).  kRows: the caller has seen that k + 8 <= K.
template <typename XT, int IN>
__device__ __forceinline__ void load8(const KernelArgs& a, const XT* row, int k, XT* v)
{
    if constexpr (IN == kRowPieces) {
        const u32x4* p = reinterpret_cast<const u32x4*>(row + min(k, a.K - 8));
#pragma unroll
        for (int i = 0; i < (int)sizeof(XT) / 2; ++i) reinterpret_cast<u32x4*>(v)[i] = p[i];
    } else if constexpr (IN == kRows) {
        __builtin_memcpy(v, row + k, 8 * sizeof(XT));
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = k + i < a.K ? row[(k + i) * a.x_sk] : XT(0.f);
    }
}

// Eight fp32 values in three bf16 parts (tl_matrix.h).  What is not finite need not survive: any part that is not finite
// makes the sum so, and that output is worked out again.  (So it is above 2^112, where a scaled value overflows here.)  A
// part is taken off with a dot product of bf16 pairs -- one factor the part's, one zero; exact, as what is left is an
// fp32 number, denormals included -- in the place of a mask and a subtraction, and of the scaling for the first.  us with
// masks / so, 48 rows: 4096 -> 11008 53.2 / 46.5, 2048 -> 5504 17.0 / 15.2 (45.8 and 14.3 without the scaling); 8 rows
// 4096 -> 11008 13.2 / 13.5 (12.0).
__device__ __forceinline__ void split8(const float* v, u32x4* part)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    auto pair = [](uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); };   // the upper halves
    // value - factor * (the lower or upper number of a pair)
    auto less = [](float value, uint32_t two, uint32_t factors) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, two), __builtin_bit_cast(bf16x2, factors), value, false);
    };
    uint32_t s_lo = 0xC780u, s_hi = 0xC7800000u, o_lo = 0xBF80u, o_hi = 0xBF800000u;   // -2^16, -1 in bf16
    // in registers: folded into the instruction, -1 in the upper half becomes an inline constant, which a pair reads otherwise
    asm("" : "+v"(s_lo), "+v"(s_hi), "+v"(o_lo), "+v"(o_hi));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float lo = v[2 * i], hi = v[2 * i + 1];
        const uint32_t a = pair(__float_as_uint(lo), __float_as_uint(hi));
        const float lo1 = less(lo * kLowScale, a, s_lo), hi1 = less(hi * kLowScale, a, s_hi);
        const uint32_t b = pair(__float_as_uint(lo1), __float_as_uint(hi1));
        const float lo2 = less(lo1, b, o_lo), hi2 = less(hi1, b, o_hi);
        part[0][i] = a;
        part[1][i] = b;
        part[2][i] = pair(__float_as_uint(lo2), __float_as_uint(hi2));
    }
}

// XT: activation type.  IN: how they are read.  FM: fragments of 16 rows.  C: column blocks of a workgroup, or, TWO, one
// block of each of two weights (silu(gate) * up).  Q: slices of a wave's turn.
template <typename XT, int IN, int FM, int C, int Q, bool TWO>
__global__ __launch_bounds__(kMaxWaves * 64) void tl_matrix_few(KernelArgs a)
{
    constexpr bool F32 = sizeof(XT) == 4;
    constexpr int kTurnsOfUnit = TL_CODE_UNIT_ROWS / (kSliceRows * Q);
    extern __shared__ __align__(16) float sums[];  // [wave][C][FM][kPartFloats]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = (int)blockDim.x >> 6;
    const int g = lane >> 4, r16 = lane & 15;
    const int nb0 = (int)blockIdx.x * (TWO ? 1 : C);
    const unsigned char* codes[C];
    int units[C];                                                  // that the block's weight has
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const Codes& weight = TWO && c == 1 ? a.c1 : a.c0;
        units[c] = weight.planes * a.units;
        codes[c] = weight.base + min(TWO ? nb0 : nb0 + c, a.NB - 1) * ((long long)units[c] * TL_CODE_UNIT_BYTES) + lane * 16;
    }
    const XT* rows[FM];
#pragma unroll
    for (int f = 0; f < FM; ++f) rows[f] = static_cast<const XT*>(a.X) + min(f * 16 + r16, a.M - 1) * a.x_sm;
    // fp32: the leading parts are summed apart from the two that follow them (against fp64, 3.6e-8 where one sum of all
    // three parts had 1.1e-7 to 2.2e-7 and the walk of the index stream 0.8e-7 to 4e-7)
    f32x4 acc[C][FM], low[F32 ? C : 1][F32 ? FM : 1];
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int f = 0; f < FM; ++f) acc[c][f] = low[F32 ? c : 0][F32 ? f : 0] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int turns = a.planes == 1 ? (a.K + kSliceRows * Q - 1) / (kSliceRows * Q) : a.planes * a.units * kTurnsOfUnit;
    for (int t = wave; t < turns; t += waves) {
        const int unit = t / kTurnsOfUnit, part = t % kTurnsOfUnit;
        uint32_t w[C][4];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            if (TWO && unit >= units[c]) {                         // (the other weight has more planes)
#pragma unroll
                for (int i = 0; i < Q; ++i) w[c][i] = 0u;
                continue;
            }
            const unsigned char* src = codes[c] + (long long)unit * TL_CODE_UNIT_BYTES + part * Q * 4;
            if constexpr (Q == 4) *reinterpret_cast<u32x4*>(w[c]) = *reinterpret_cast<const u32x4*>(src);
            else if constexpr (Q == 2) *reinterpret_cast<uint2*>(w[c]) = *reinterpret_cast<const uint2*>(src);
            else w[c][0] = *reinterpret_cast<const uint32_t*>(src);
        }
        const int k0 = (unit % a.units) * TL_CODE_UNIT_ROWS + part * Q * kSliceRows + g * 8;
        XT x[Q * 2][FM][8] __attribute__((aligned(16)));
        auto load_turn = [&](auto in) {
#pragma unroll
            for (int s = 0; s < Q * 2; ++s)
#pragma unroll
                for (int f = 0; f < FM; ++f) load8<XT, decltype(in)::value>(a, rows[f], k0 + s * 32, x[s][f]);
        };
        if (IN == kRows && (unit % a.units) * TL_CODE_UNIT_ROWS + (part + 1) * Q * kSliceRows > a.K) load_turn(std::integral_constant<int, kElements>{});
        else load_turn(std::integral_constant<int, IN>{});
#pragma unroll
        for (int s = 0; s < Q * 2; ++s) {
            u32x4 op[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const u32x4 one{w[c][s >> 1], 0u, 0u, 0u};
                op[c] = (s & 1) ? weight_operand<1>(one) : weight_operand<0>(one);
            }
#pragma unroll
            for (int f = 0; f < FM; ++f) {
                if constexpr (F32) {
                    u32x4 p[3];
                    split8(x[s][f], p);
#pragma unroll
                    for (int i = 0; i < 3; ++i)
#pragma unroll
                        for (int c = 0; c < C; ++c) {
                            f32x4& sum = i == 0 ? acc[c][f] : low[c][f];
                            sum = matrix_step<true>(op[c], p[i], sum);
                        }
                } else {
#pragma unroll
                    for (int c = 0; c < C; ++c) acc[c][f] = matrix_step<false>(op[c], *reinterpret_cast<const u32x4*>(x[s][f]), acc[c][f]);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int f = 0; f < FM; ++f) {
            if constexpr (F32) add_low(acc[c][f], low[c][f]);
            *reinterpret_cast<f32x4*>(sums + ((wave * C + c) * FM + f) * kPartFloats + lane * 4 + g * 16) = acc[c][f];
        }
    __syncthreads();

    // one output after the other, 16 neighbouring columns of a row to 16 neighbouring threads
    auto total = [&](int c, int m, int col) {
        const float* s = sums + (c * FM + (m >> 4)) * kPartFloats + (col >> 2) * 80 + (m & 15) * 4 + (col & 3);
        std::conditional_t<F32, double, float> v = 0;  // (fp32: sixteen more roundings would be the largest part of the error)
        for (int i = 0; i < waves; ++i) v += s[i * C * FM * kPartFloats];
        return (float)v;
    };
    auto output = [&](const WeightPtrs& w, int c, int m, int n) {
        float v = 0.5f * total(c, m, n & 15);
        if (!(fabsf(v) < __builtin_huge_valf())) v = walk_column(w, a.T, a.tile_rows, n, callers_x(a, m));
        return v * load_scale(w.scale, a.scale_f16, n);
    };
    constexpr int COLS = TWO ? 16 : C * 16;
    for (int e = threadIdx.x; e < a.M * COLS; e += (int)blockDim.x) {
        const int m = e / COLS, col = e % COLS, n = nb0 * 16 + col;
        if (n >= a.N) continue;
        float v = output(a.w0, col >> 4, m, n);
        if constexpr (TWO) v = silu(v) * output(a.w1, 1, m, n);
        store_out(a.Y, a.y_f16, m * a.ldy + n, v);
    }
}

template <typename XT, int IN, int FM, int C, bool TWO>
int launch_few(const KernelArgs& a, hipStream_t st)
{
    const int64_t slices = a.planes == 1 ? ceil_div(a.K, kSliceRows) : (int64_t)a.planes * a.units * (TL_CODE_UNIT_ROWS / kSliceRows);
    const int most = C * FM <= 3 ? kMaxWaves : kMaxWaves / 2;   // (64 KB of sums)
    // a turn of four slices is one 16-byte load of codes; fewer where that would leave waves without a turn, and where the
    // turn's activations, loaded one by one, would not fit the registers
    constexpr int kMostSlices = IN == kRowPieces || FM == 1 ? 4 : FM == 2 ? 2 : 1;
    const int q = std::min<int>(kMostSlices, slices >= 4 * most ? 4 : slices >= 2 * most ? 2 : 1);
    const int waves = (int)std::min<int64_t>(most, ceil_div(slices, q));
    const size_t lds = (size_t)waves * C * FM * kPartFloats * sizeof(float);
    const dim3 grid((unsigned)(TWO ? a.NB : ceil_div(a.NB, C))), block((unsigned)waves * 64);
    if (q == 4) hipLaunchKernelGGL((tl_matrix_few<XT, IN, FM, C, kMostSlices, TWO>), grid, block, lds, st, a);
    else if (q == 2) hipLaunchKernelGGL((tl_matrix_few<XT, IN, FM, C, std::min(2, kMostSlices), TWO>), grid, block, lds, st, a);
    else hipLaunchKernelGGL((tl_matrix_few<XT, IN, FM, C, 1, TWO>), grid, block, lds, st, a);
    return TL_OK;
}

template <typename XT, int IN, int FM>
int launch_few_columns(const KernelArgs& a, bool two_weights, hipStream_t st)
{
    if (two_weights) return launch_few<XT, IN, FM, 2, true>(a, st);
    // Two blocks to a workgroup halve what the workgroups read of the activations, and pay once the blocks are more than the
    // compute units (fp16, us with one / two: 8 rows 4096 -> 4096 at 95 % zeros 5.2 / 5.4, 2048 -> 5504 5.2 / 4.3,
    // 4096 -> 11008 9.7 / 8.0; 48 rows 13.7 / 14.5, 13.8 / 9.2, 36 / 26).
    if (a.NB > compute_units()) return launch_few<XT, IN, FM, 2, false>(a, st);
    return launch_few<XT, IN, FM, 1, false>(a, st);
}

template <typename XT, int IN>
int launch_few_in(const KernelArgs& a, bool two_weights, hipStream_t st)
{
    if (a.M <= 16) return launch_few_columns<XT, IN, 1>(a, two_weights, st);
    if (a.M <= 32) return launch_few_columns<XT, IN, 2>(a, two_weights, st);
    return launch_few_columns<XT, IN, 3>(a, two_weights, st);
}

template <typename XT>
int launch_few_type(const KernelArgs& a, bool pieces, bool two_weights, hipStream_t st)
{
    if (a.x_kmajor) return launch_few_in<XT, kElements>(a, two_weights, st);
    return pieces ? launch_few_in<XT, kRowPieces>(a, two_weights, st) : launch_few_in<XT, kRows>(a, two_weights, st);
}

}  // namespace

int tl::launch_matrix_few(KernelArgs a, int x_dtype, bool two_weights, hipStream_t st)
{
    const int es = x_dtype == TL_F16 ? 2 : 4;
    a.x_sm = a.x_kmajor ? 1 : a.ldx;
    a.x_sk = a.x_kmajor ? a.ldx : 1;
    const bool pieces = a.K % 8 == 0 && (a.M == 1 || (a.ldx * es) % 16 == 0) && reinterpret_cast<uintptr_t>(a.X) % 16 == 0;
    return x_dtype == TL_F16 ? launch_few_type<_Float16>(a, pieces, two_weights, st) : launch_few_type<float>(a, pieces, two_weights, st);
}
