// A few activation rows (up to 48): the ternary product on the matrix cores straight from memory.
//
// Bound by latency, by the bytes of the codes and by what the workgroups read of the activations: a workgroup owns one or two
// blocks of 16 columns over all of K, its waves share K out among them and meet once, in LDS, at the very end.  Every load of a
// turn (up to 256 rows of K) is in flight before the first product.  A lane's operand is 16 bytes of a row, and such a load
// touches 16 rows, four clocks each; so the rows go through LDS, whole slices of 8 rows a load, into a part that is the wave's
// own: no barrier.  fp32 rows become three bf16 parts in registers.
// us at 4096 -> 11008, 66 % zeros, walking the index stream / operands straight from memory / through LDS: fp16 8 rows 20.1 / 8.1 / 6.7
// (11.3 MB of codes: 1.7 TB/s), 16 rows 25.7 / 10.8 / 7.1, 48 rows 68.9 / 26 / 15.5; fp32 16 rows 24.7 / 18.3 / 13.7, 48 rows
// 100 / 48 / 41.
#include "tl_matrix.h"

using namespace tl;

namespace {

constexpr int kSliceRows = 64;        // rows of K that one dword of a lane's codes names
constexpr int kPartFloats = 320;      // LDS floats of 16 x 16 partial sums: lane l's four at 4 * l + 16 * (l / 16), so that the
                                      // four quarters, whose columns one row's outputs take together, lie on different banks
constexpr int kMaxWaves = 16;
// Waves of a workgroup: 16 for one column block; 8 for two, whose workgroups share compute units (us with 16 / 8, 16 fp16 rows with
// all steps: 2048 -> 11008 11.0 / 9.3, 4096 -> 11008 14.6 / 12.9, 2048 -> 6144 6.7 / 6.6), and as 64 KB of sums hold no more.
constexpr __host__ __device__ int most_waves(int C, int stage_bytes) { return C == 1 && stage_bytes <= 8192 ? kMaxWaves : kMaxWaves / 2; }


// How rows are read: aligned 16-byte pieces (K a multiple of 8), as operands; through registers and LDS, 16 bytes at a time
// from any element on; element by element (K-major); aligned pieces straight to LDS; as operands from any element on, but for the
// turn in which a row ends.
enum { kRowPieces = 0, kRows = 1, kElements = 2, kStaged = 3, kOperands = 4 };

// Eight activations of a row from k on.  Past K: zeros (element by element) or the row's last whole piece again (such rows
// of K meet zero codes).  kOperands: the caller has seen that k + 8 <= K.
template <typename XT, int IN>
__device__ __forceinline__ void load8(const KernelArgs& a, const XT* row, int k, XT* v)
{
    if constexpr (IN == kRowPieces) {
        const u32x4* p = reinterpret_cast<const u32x4*>(row + min(k, a.K - 8));
#pragma unroll
        for (int i = 0; i < (int)sizeof(XT) / 2; ++i) reinterpret_cast<u32x4*>(v)[i] = p[i];
    } else if constexpr (IN == kOperands) {
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

// What a call does besides the product: nothing; one block of each of two weights, silu(gate) * up; what a decoder layer does
// around a product (tl_spmm_chain_rows, tl_spmm_gated), by the argument block: the rows' normalisation factors, the gate of column
// pairs, the residual rows, the next norm's image and sums of squares; and the norm of the rows on their way in
// (tl_spmm_normed_rows), with the gate by the argument block.
enum { kPlain = 0, kTwo = 1, kSteps = 2, kNormed = 3 };

// Eight activations times their row's factor times the norm's weights, in fp32, then rounded to fp16: five instructions for two
// (v_fma_mix_f32 takes fp16 factors as they are).
__device__ __forceinline__ u32x4 normed8(u32x4 x, float factor, u32x4 w)
{
    const half8 xs = __builtin_bit_cast(half8, x), ws = __builtin_bit_cast(half8, w);
    half8 out;
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = (_Float16)__builtin_fmaf(__builtin_fmaf((float)xs[i], factor, 0.f), (float)ws[i], 0.f);
    return __builtin_bit_cast(u32x4, out);
}

// Rows that the sums of squares of M rows have room for: a lane's four are the same in every block it reads.
constexpr __host__ __device__ int squares_rows(int M) { return M <= 16 ? 16 : M <= 32 ? 32 : 64; }

// One value as it lies in memory, for loads that nothing waits for until the very end, and what it is.
__device__ __forceinline__ uint32_t raw_value(const void* p, int f16, long long i) { return f16 ? static_cast<const unsigned short*>(p)[i] : static_cast<const uint32_t*>(p)[i]; }
__device__ __forceinline__ float value_of(uint32_t raw, int f16) { return f16 ? __half2float(__ushort_as_half((unsigned short)raw)) : __uint_as_float(raw); }

// The sum over the lanes whose number differs in the bits from FROM to below TO only (powers of two), on the vector unit.
template <int FROM, int TO>
__device__ __forceinline__ float sum_over_lanes(float v)
{
    auto turned = [](float x, auto by) {   // from `by` lanes further on among 16, around
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + decltype(by)::value, 0xf, 0xf, true));
    };
    auto both = [](auto pair) { return __uint_as_float(pair[0]) + __uint_as_float(pair[1]); };
    if constexpr (FROM <= 8 && TO > 8) v += turned(v, std::integral_constant<int, 8>{});
    if constexpr (FROM <= 4 && TO > 4) v += turned(v, std::integral_constant<int, 4>{});
    if constexpr (FROM <= 2 && TO > 2) v += turned(v, std::integral_constant<int, 2>{});
    if constexpr (FROM <= 1 && TO > 1) v += turned(v, std::integral_constant<int, 1>{});
    if constexpr (TO > 16) v = both(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false));
    if constexpr (TO > 32) v = both(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false));
    return v;
}

// LDS of a wave: its activations of a turn (kStaged, kRows), then its sums.
template <typename XT, int IN, int FM>
constexpr __host__ __device__ int stage_bytes(int Q) { return IN == kStaged || IN == kRows ? Q * FM * 16 * kSliceRows * (int)sizeof(XT) : 0; }
template <typename XT, int IN, int FM, int C, int Q>
constexpr __host__ __device__ int wave_floats() { return std::max(C * FM * kPartFloats, stage_bytes<XT, IN, FM>(Q) / 4); }

// XT: activation type.  IN: how they are read.  FM: fragments of 16 rows.  C: column blocks of a workgroup (kTwo: one of each
// weight).  Q: slices of a wave's turn.
// (33 to 48 staged fp32 rows run with eight waves and may take the registers of sixteen.)
template <typename XT, int IN, int FM, int C, int Q, int STEPS>
__global__ __launch_bounds__(64 * (stage_bytes<XT, IN, FM>(1) > 8192 ? most_waves(C, stage_bytes<XT, IN, FM>(1)) : kMaxWaves)) void tl_matrix_few(KernelArgs a)
{
    constexpr bool F32 = sizeof(XT) == 4, TWO = STEPS == kTwo, NORMED = STEPS == kNormed;
    constexpr int kTurnsOfUnit = TL_CODE_UNIT_ROWS / (kSliceRows * Q);
    // [wave] its stage of activations (kStaged, kRows), where its sums [C][FM][kPartFloats] lie afterwards; and, kSteps and kNormed, [wave][SR] sums of squares
    extern __shared__ __align__(16) float sums[];
    constexpr int OWN = wave_floats<XT, IN, FM, C, Q>();
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

    // What the last steps need is asked for now, for a thread's first output (its only one, mostly).  Squares lie as [block of
    // 16][SR rows], pieces of four rows.
    constexpr int SR = squares_rows(FM * 16), U = FM == 3 ? 4 : 2, COLS = TWO ? 16 : C * 16;
    const bool pairs = STEPS >= kSteps && a.gated;
    const int first_m = (int)threadIdx.x / (pairs ? COLS / 2 : COLS), first_col = pairs ? (int)threadIdx.x % (COLS / 2) * 2 : (int)threadIdx.x % COLS;
    const int first_n = nb0 * 16 + first_col;
    uint32_t early_scale[2] = {0u, 0u};
    if (a.w0.scale && first_m < a.M && first_n < a.N) {
        early_scale[0] = raw_value(a.w0.scale, a.scale_f16, first_n);
        if (pairs) early_scale[1] = raw_value(a.w0.scale, a.scale_f16, first_n + 1);
        if (TWO) early_scale[1] = raw_value(a.w1.scale, a.scale_f16, first_n);
    }
    [[maybe_unused]] float4 squares[U];
    const int square_pieces = STEPS >= kSteps && a.chain_sq_in ? a.chain_sq_blocks * (SR / 4) : 0;
    [[maybe_unused]] uint32_t early_residual = 0, early_weight = 0;
    if constexpr (STEPS >= kSteps) {
        const float4* pieces = reinterpret_cast<const float4*>(a.chain_sq_in);
        if (NORMED || square_pieces)
#pragma unroll
            for (int u = 0; u < U; ++u) squares[u] = pieces[min((int)threadIdx.x + u * (int)blockDim.x, square_pieces - 1)];
        if (!pairs && first_m < a.M && first_n < a.N) {
            if (a.chain_res) early_residual = raw_value(a.chain_res, 1, first_m * a.chain_ldres + first_n);
            if (a.chain_image) early_weight = raw_value(a.chain_w, 1, first_n);
        }
    }

    const int turns = a.planes == 1 ? (a.K + kSliceRows * Q - 1) / (kSliceRows * Q) : a.planes * a.units * kTurnsOfUnit;
    constexpr bool STAGED = IN == kStaged || IN == kRows;
    struct Turn {
        uint32_t w[C][4];
        XT x[STAGED ? 1 : Q * 2][FM][8] __attribute__((aligned(16)));
        u32x4 norm[NORMED ? Q * 2 : 1];   // the norm's weights
    };
    // kStaged: a load takes whole slices (128 or 256 bytes) of 8 or 4 rows.  A row's pieces lie rotated so that 16 lanes that
    // read one piece of 16 rows find them on different banks.
    constexpr int PIECES = kSliceRows * (int)sizeof(XT) / 16, BLOCK = 16 * kSliceRows * (int)sizeof(XT);   // bytes of 16 rows of a slice
    auto turned = [](int r) { return F32 ? r & 15 : (r >> 1) & 7; };
    [[maybe_unused]] const uint32_t own = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)(sums + wave * OWN);
    [[maybe_unused]] auto stage = [&](int t) {
        const int k0 = t / kTurnsOfUnit % a.units * TL_CODE_UNIT_ROWS + t % kTurnsOfUnit * Q * kSliceRows;
        const uint32_t last = (uint32_t)a.K * (uint32_t)sizeof(XT) - 16;
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");       // (what was read of the turn before has been read)
#pragma unroll
        for (int i = 0; i < FM * BLOCK / 1024; ++i) {
            const int r = (i * 64 + lane) / PIECES;
            const uint32_t row = (uint32_t)min(r, a.M - 1) * (uint32_t)(a.x_sm * (int)sizeof(XT)), piece = (uint32_t)(lane % PIECES ^ turned(r)) * 16;
#pragma unroll
            for (int q = 0; q < Q; ++q)
                load_to_lds(own + q * FM * BLOCK + i * 1024, a.X, row + min((uint32_t)((k0 + q * kSliceRows) * (int)sizeof(XT)) + piece, last));
        }
    };
    // One lane writes what others of its wave read: a wave's LDS instructions run in order, and nothing may move across here.
    [[maybe_unused]] auto lanes_meet = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    // kRows: the same through registers, 16 bytes from any element on, and element by element where a row ends.  us as operands
    // straight from memory / so: fp16 16 rows 4095 -> 11008 26.5 / 9.3, 48 rows 67.6 / 23.0, 37 rows 1003 -> 777 8.0 / 6.2; fp32 16 rows
    // 24.7 / 14.7, 48 rows 54.6 / 42.8, but 37 rows 1003 -> 777 7.7 / 8.8 (eight waves, whose 12 KB fill the LDS, in the place of 16).
    [[maybe_unused]] auto stage_any = [&](int t) {
        constexpr int E = 16 / (int)sizeof(XT), LOADS = FM * BLOCK / 1024;
        const int k0 = t / kTurnsOfUnit % a.units * TL_CODE_UNIT_ROWS + t % kTurnsOfUnit * Q * kSliceRows;
        const XT* x = static_cast<const XT*>(a.X);
        u32x4 v[LOADS][Q];
        auto read = [&](auto whole) {
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                const int r = (i * 64 + lane) / PIECES;
                const XT* row = x + min(r, a.M - 1) * a.x_sm;
                const int piece = (lane % PIECES ^ turned(r)) * E;
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const int k = k0 + q * kSliceRows + piece;
                    XT e[E] __attribute__((aligned(16)));
                    if (decltype(whole)::value || k + E <= a.K) __builtin_memcpy(e, row + k, 16);
                    else {
#pragma unroll
                        for (int j = 0; j < E; ++j) e[j] = k + j < a.K ? row[k + j] : XT(0.f);
                    }
                    v[i][q] = *reinterpret_cast<const u32x4*>(e);
                }
            }
        };
        if (k0 + Q * kSliceRows <= a.K) read(std::true_type{});
        else read(std::false_type{});
        lanes_meet();                                              // (what was read of the turn before has been read)
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
#pragma unroll
            for (int q = 0; q < Q; ++q)
                *reinterpret_cast<u32x4*>(reinterpret_cast<unsigned char*>(sums + wave * OWN) + q * FM * BLOCK + i * 1024 + lane * 16) = v[i][q];
    };
    [[maybe_unused]] auto staged = [&](int s, int f, XT* v) {      // the eight activations of step s that are this lane's
        const unsigned char* row = reinterpret_cast<const unsigned char*>(sums + wave * OWN) + ((s >> 1) * FM + f) * BLOCK + r16 * (PIECES * 16);
#pragma unroll
        for (int i = 0; i < (int)sizeof(XT) / 2; ++i)
            reinterpret_cast<u32x4*>(v)[i] = *reinterpret_cast<const u32x4*>(row + ((((s & 1) * 4 + g) * ((int)sizeof(XT) / 2) + i) ^ turned(r16)) * 16);
    };
    auto load = [&](int t, Turn& to) {
        const int unit = t / kTurnsOfUnit, part = t % kTurnsOfUnit;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            if (TWO && unit >= units[c]) {                         // (the other weight has more planes)
#pragma unroll
                for (int i = 0; i < Q; ++i) to.w[c][i] = 0u;
                continue;
            }
            const unsigned char* src = codes[c] + (long long)unit * TL_CODE_UNIT_BYTES + part * Q * 4;
            if constexpr (Q == 4) *reinterpret_cast<u32x4*>(to.w[c]) = *reinterpret_cast<const u32x4*>(src);
            else if constexpr (Q == 2) *reinterpret_cast<uint2*>(to.w[c]) = *reinterpret_cast<const uint2*>(src);
            else to.w[c][0] = *reinterpret_cast<const uint32_t*>(src);
        }
        const int k0 = (unit % a.units) * TL_CODE_UNIT_ROWS + part * Q * kSliceRows + g * 8;
        if constexpr (NORMED) {
#pragma unroll
            for (int s = 0; s < Q * 2; ++s) to.norm[s] = *reinterpret_cast<const u32x4*>(static_cast<const _Float16*>(a.norm_w) + min(k0 + s * 32, a.K - 8));
        }
        if constexpr (IN == kStaged) stage(t);
        else if constexpr (IN == kRows) stage_any(t);
        else {
            auto load_turn = [&](auto in) {
#pragma unroll
                for (int s = 0; s < Q * 2; ++s)
#pragma unroll
                    for (int f = 0; f < FM; ++f) load8<XT, decltype(in)::value>(a, rows[f], k0 + s * 32, to.x[s][f]);
            };
            if (IN == kOperands && (unit % a.units) * TL_CODE_UNIT_ROWS + (part + 1) * Q * kSliceRows > a.K) load_turn(std::integral_constant<int, kElements>{});
            else load_turn(std::integral_constant<int, IN>{});
        }
    };
    auto arrived = [&] {
        if constexpr (IN == kStaged) asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        if constexpr (IN == kRows) lanes_meet();
    };
    [[maybe_unused]] float* wave_squares = sums + waves * OWN;
    auto add_squares = [&] {                                       // into wave_squares
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
        auto add = [&](const float4& v, bool there) {
            sum.x += there ? v.x : 0.f; sum.y += there ? v.y : 0.f; sum.z += there ? v.z : 0.f; sum.w += there ? v.w : 0.f;
        };
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // (without this the first is added to zero, and waited for, where it is asked for: before the first turn's loads)
            asm volatile("" : "+v"(squares[u].x), "+v"(squares[u].y), "+v"(squares[u].z), "+v"(squares[u].w));
            add(squares[u], (int)threadIdx.x + u * (int)blockDim.x < square_pieces);
        }
        for (int i = (int)threadIdx.x + U * (int)blockDim.x; i < square_pieces; i += (int)blockDim.x) add(reinterpret_cast<const float4*>(a.chain_sq_in)[i], true);
        for (float* v : {&sum.x, &sum.y, &sum.z, &sum.w}) *v = sum_over_lanes<SR / 4, 64>(*v);   // the lanes with the same rows
        if (lane < SR / 4) reinterpret_cast<float4*>(wave_squares + wave * SR)[lane] = sum;
    };
    // (The waves' sums are read at once: one after the other each is a trip to LDS; and no more than there are: 37 fp32 rows of 301 ->
    // 1024, five waves, 6.5 us with sixteen reads always, 6.1.)
    auto over_waves = [&](const float* s, int stride) {
        auto read = [&](auto most) {
            constexpr int MOST = decltype(most)::value;
            float part[MOST];
#pragma unroll
            for (int i = 0; i < MOST; ++i) part[i] = s[min(i, waves - 1) * stride];
            std::conditional_t<F32, double, float> v = 0;  // (fp32: sixteen more roundings would be the largest part of the error)
#pragma unroll
            for (int i = 0; i < MOST; ++i) v += i < waves ? part[i] : 0.f;
            return (float)v;
        };
        constexpr int MOST = most_waves(C, stage_bytes<XT, IN, FM>(Q));
        if (waves <= 4) return read(std::integral_constant<int, 4>{});
        if (MOST > 8 && waves <= 8) return read(std::integral_constant<int, 8>{});
        return read(std::integral_constant<int, MOST>{});
    };
    auto row_factor = [&](int m) { return rsqrtf(over_waves(wave_squares + m, SR) * (1.0f / (float)a.K) + a.eps); };
    [[maybe_unused]] float factors[FM];                            // (kNormed: of the rows of this lane's operands)
    auto multiply = [&](const Turn& turn) {
#pragma unroll
        for (int s = 0; s < Q * 2; ++s) {
            u32x4 op[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const u32x4 one{turn.w[c][s >> 1], 0u, 0u, 0u};
                op[c] = (s & 1) ? weight_operand<1>(one) : weight_operand<0>(one);
            }
#pragma unroll
            for (int f = 0; f < FM; ++f) {
                XT x[8] __attribute__((aligned(16)));
                if constexpr (STAGED) staged(s, f, x);
                else __builtin_memcpy(x, turn.x[s][f], sizeof(x));
                if constexpr (NORMED) *reinterpret_cast<u32x4*>(x) = normed8(*reinterpret_cast<const u32x4*>(x), factors[f], turn.norm[s]);
                if constexpr (F32) {
                    u32x4 p[3];
                    split8(x, p);
#pragma unroll
                    for (int i = 0; i < 3; ++i)
#pragma unroll
                        for (int c = 0; c < C; ++c) {
                            f32x4& sum = i == 0 ? acc[c][f] : low[c][f];
                            sum = matrix_step<true>(op[c], p[i], sum);
                        }
                } else {
#pragma unroll
                    for (int c = 0; c < C; ++c) acc[c][f] = matrix_step<false>(op[c], *reinterpret_cast<const u32x4*>(x), acc[c][f]);
                }
            }
        }
    };
    if constexpr (NORMED) {
        // the factors are needed before the first product: what the first turn reads is on its way while they meet.  (There are
        // no more waves than turns.)
        Turn turn;
        load(wave, turn);
        add_squares();
        __syncthreads();
#pragma unroll
        for (int f = 0; f < FM; ++f) factors[f] = row_factor(f * 16 + r16);
        arrived();
        multiply(turn);
        for (int t = wave + waves; t < turns; t += waves) {
            load(t, turn);
            arrived();
            multiply(turn);
        }
    } else {
        for (int t = wave; t < turns; t += waves) {
            Turn turn;
            load(t, turn);
            arrived();
            multiply(turn);
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int f = 0; f < FM; ++f) {
            if constexpr (F32) add_low(acc[c][f], low[c][f]);
            *reinterpret_cast<f32x4*>(sums + wave * OWN + (c * FM + f) * kPartFloats + lane * 4 + g * 16) = acc[c][f];
        }
    if (STEPS == kSteps && square_pieces) add_squares();
    __syncthreads();

    // one output after the other, 16 neighbouring columns of a row to 16 neighbouring threads
    auto output = [&](const WeightPtrs& w, int c, int m, int n, uint32_t early, bool first) {
        const int col = n & 15;
        float v = 0.5f * over_waves(sums + (c * FM + (m >> 4)) * kPartFloats + (col >> 2) * 80 + (m & 15) * 4 + (col & 3), OWN);
        if (!(fabsf(v) < __builtin_huge_valf())) {
            const CallersX x = callers_x(a, m);
            if constexpr (NORMED) {
                const float factor = row_factor(m);
                v = walk_column(w, a.T, a.tile_rows, n, [&](int k) { return as_output(x(k) * factor * value_of(raw_value(a.norm_w, 1, k), 1), 1); });
            } else {
                v = walk_column(w, a.T, a.tile_rows, n, x);
            }
        }
        return w.scale ? v * value_of(first ? early : raw_value(w.scale, a.scale_f16, n), a.scale_f16) : v;
    };
    if constexpr (STEPS >= kSteps) {
        auto factor = [&](int m) { return NORMED || !square_pieces ? 1.0f : row_factor(m); };
        if (a.gated) {
            // column pairs; a K-major image's rows past M are zeroed
            const int rows = a.y_kld ? (int)a.y_kld : a.M;
            for (int e = threadIdx.x; e < rows * (COLS / 2); e += (int)blockDim.x) {
                const int m = e / (COLS / 2), col = e % (COLS / 2) * 2, n = nb0 * 16 + col;
                if (n >= a.N) continue;
                float v = 0.f;
                if (m < a.M) {
                    const float f = factor(m);
                    const bool first = e == (int)threadIdx.x;
                    const float gate = output(a.w0, col >> 4, m, n, early_scale[0], first) * f, up = output(a.w0, col >> 4, m, n + 1, early_scale[1], first) * f;
                    v = gate_pair(as_output(gate, a.y_f16), as_output(up, a.y_f16), a.y_f16);
                }
                store_out(a.Y, a.y_f16, a.y_kld ? n / 2 * a.y_kld + m : m * a.ldy + n / 2, v);
            }
            return;
        }
        for (int e = threadIdx.x; e < a.M * COLS; e += (int)blockDim.x) {   // (a row's 16 columns of a block: 16 lanes of one wave)
            const int m = e / COLS, col = e % COLS, n = nb0 * 16 + col;
            const bool first = e == (int)threadIdx.x;
            float v = 0.f;
            if (n < a.N) {
                v = output(a.w0, col >> 4, m, n, early_scale[0], first) * factor(m);
                if (a.chain_res) v = as_output(v, 1) + value_of(first ? early_residual : raw_value(a.chain_res, 1, m * a.chain_ldres + n), 1);
                v = as_output(v, 1);
                store_out(a.Y, 1, m * a.ldy + n, v);
                if (a.chain_image) store_out(a.chain_image, 1, m * a.chain_ild + n, v * value_of(first ? early_weight : raw_value(a.chain_w, 1, n), 1));
            }
            if (a.chain_sq_out) {
                const float square = sum_over_lanes<1, 16>(v * v);
                if (col % 16 == 0 && n < a.N) a.chain_sq_out[(nb0 + (col >> 4)) * SR + m] = square;
            }
        }
        return;
    }
    for (int e = threadIdx.x; e < a.M * COLS; e += (int)blockDim.x) {
        const int m = e / COLS, col = e % COLS, n = nb0 * 16 + col;
        if (n >= a.N) continue;
        const bool first = e == (int)threadIdx.x;
        float v = output(a.w0, col >> 4, m, n, early_scale[0], first);
        if constexpr (TWO) v = silu(v) * output(a.w1, 1, m, n, early_scale[1], first);
        store_out(a.Y, a.y_f16, m * a.ldy + n, v);
    }
}

template <typename XT, int IN, int FM, int C, int STEPS>
int launch_few(const KernelArgs& a, hipStream_t st)
{
    const int64_t slices = a.planes == 1 ? ceil_div(a.K, kSliceRows) : (int64_t)a.planes * a.units * (TL_CODE_UNIT_ROWS / kSliceRows);
    const int most = most_waves(C, stage_bytes<XT, IN, FM>(1));
    // a turn of four slices is one 16-byte load of codes; fewer where that would leave waves without a turn, and where the
    // turn's activations, loaded one by one, would not fit the registers
    constexpr int kMostSlices = stage_bytes<XT, IN, FM>(1) ? std::max(1, 8192 / stage_bytes<XT, IN, FM>(1)) : IN == kOperands ? (FM == 3 ? 1 : 2) : IN == kRowPieces || FM == 1 ? 4 : FM == 2 ? 2 : 1;
    const int q = std::min<int>(kMostSlices, slices >= 4 * most ? 4 : slices >= 2 * most ? 2 : 1);
    const int waves = (int)std::min<int64_t>(most, ceil_div(slices, q));
    const dim3 grid((unsigned)(STEPS == kTwo ? a.NB : ceil_div(a.NB, C))), block((unsigned)waves * 64);
    auto launch = [&](auto q_tag) {
        constexpr int Q = decltype(q_tag)::value;
        const size_t lds = (size_t)waves * (wave_floats<XT, IN, FM, C, Q>() + (STEPS >= kSteps ? squares_rows(FM * 16) : 0)) * sizeof(float);
        auto kernel = tl_matrix_few<XT, IN, FM, C, Q, STEPS>;
        if (IN == kStaged || IN == kRows) {
            static LdsLimit raised;
            if (int rc = raised.raise(kernel, 160 * 1024)) return rc;
        }
        hipLaunchKernelGGL(kernel, grid, block, lds, st, a);
        return (int)TL_OK;
    };
    if (q == 4) return launch(std::integral_constant<int, kMostSlices>{});
    if (q == 2) return launch(std::integral_constant<int, std::min(2, kMostSlices)>{});
    return launch(std::integral_constant<int, 1>{});
}

template <typename XT, int IN, int FM>
int launch_few_columns(const KernelArgs& a, bool two_weights, hipStream_t st)
{
    if (two_weights) return launch_few<XT, IN, FM, 2, kTwo>(a, st);
    // Two blocks to a workgroup halve what the workgroups read of the activations, and pay once the blocks are more than the
    // compute units (fp16, us with one / two: 8 rows 4096 -> 4096 at 95 % zeros 5.2 / 5.4, 2048 -> 5504 5.2 / 4.3,
    // 4096 -> 11008 9.7 / 8.0; 48 rows 13.7 / 14.5, 13.8 / 9.2, 36 / 26).
    const bool pairs = a.NB > compute_units();
    if constexpr (sizeof(XT) == 2 && (IN == kStaged || (IN == kRowPieces && FM == 1))) {
        if (a.norm_w) return pairs ? launch_few<XT, IN, FM, 2, kNormed>(a, st) : launch_few<XT, IN, FM, 1, kNormed>(a, st);
    }
    if constexpr (sizeof(XT) == 2) {
        if (a.gated || a.chain_res || a.chain_sq_out || a.chain_sq_in) return pairs ? launch_few<XT, IN, FM, 2, kSteps>(a, st) : launch_few<XT, IN, FM, 1, kSteps>(a, st);
    }
    return pairs ? launch_few<XT, IN, FM, 2, kPlain>(a, st) : launch_few<XT, IN, FM, 1, kPlain>(a, st);
}

template <typename XT, int IN>
int launch_few_in(const KernelArgs& a, bool two_weights, hipStream_t st)
{
    if (a.M <= 16) return launch_few_columns<XT, IN, 1>(a, two_weights, st);
    if (a.M <= 32) return launch_few_columns<XT, IN, 2>(a, two_weights, st);
    return launch_few_columns<XT, IN, 3>(a, two_weights, st);
}

constexpr int64_t kMostStagedLd = 1 << 24;   // (a lane's byte offset inside 48 rows has 32 bits)

template <typename XT>
int launch_few_type(const KernelArgs& a, bool pieces, bool two_weights, hipStream_t st)
{
    if (a.x_kmajor) return launch_few_in<XT, kElements>(a, two_weights, st);
    // Through LDS once the rows are many enough, over a K that is long enough, that reading them as operands costs more.  us, as operands /
    // through LDS.  Aligned, fp16: K = 1000 -> 4096 8 rows 3.11 / 3.15, 16 rows 3.35 / 3.26; 2048 -> 2048 3 rows 3.26 / 3.18, 8 rows 3.72 / 3.23;
    // 11008 -> 4096 2 rows 6.4 / 6.4, 16 rows 12.5 / 6.8.  fp32: 8 rows 1000 -> 4096 3.78 / 3.76, 2048 -> 2048 5.03 / 4.83, 4096 -> 4096 7.4 / 6.7,
    // 4096 -> 11008 12.5 / 12.5, but 2048 -> 6144, whose workgroups of two blocks have eight waves, 5.17 / 5.53 (12 rows 5.87 / 5.66); 6 rows
    // 4096 -> 4096 6.7 / 6.7, 2048 -> 6144 4.9 / 5.4.
    // On no boundary, fp16: 2 rows 1003 -> 4096 4.4 / 4.3, 16 rows 5.5 / 4.1: always LDS.  fp32: 1003 -> 4096 2 rows 4.35 / 4.45, 8 rows 4.58 / 4.51,
    // 16 rows 5.1 / 4.7, 37 rows, whose stages fill the LDS with eight waves, 8.1 / 9.2; 2047 -> 2048 2 rows 5.6 / 5.3, 37 rows 13.3 / 13.0.
    const int64_t depth = (int64_t)a.planes * a.K;
    const bool wide = a.NB > compute_units();
    if (pieces) {
        const int enough = sizeof(XT) == 2 ? (depth > 1024 ? 4 : 9) : wide && depth < 4096 ? 12 : 8;
        if (a.M >= enough && a.ldx <= kMostStagedLd) return launch_few_in<XT, kStaged>(a, two_weights, st);   // (a lane's offset has 32 bits)
        return launch_few_in<XT, kRowPieces>(a, two_weights, st);
    }
    if constexpr (sizeof(XT) == 4) {
        if (depth <= 1024 && (a.M < 8 || a.M > 16)) return launch_few_in<XT, kOperands>(a, two_weights, st);
    }
    return launch_few_in<XT, kRows>(a, two_weights, st);
}

}  // namespace

int tl::launch_matrix_few(KernelArgs a, int x_dtype, bool two_weights, hipStream_t st)
{
    const int es = x_dtype == TL_F16 ? 2 : 4;
    const bool steps = a.gated || a.chain_res || a.chain_sq_out || a.chain_sq_in;
    if (steps && x_dtype != TL_F16) return fail(TL_ERR_UNSUPPORTED, "the gated and chained steps of few rows are for fp16 activations");
    a.x_sm = a.x_kmajor ? 1 : a.ldx;
    a.x_sk = a.x_kmajor ? a.ldx : 1;
    const bool pieces = a.K % 8 == 0 && (a.M == 1 || (a.ldx * es) % 16 == 0) && reinterpret_cast<uintptr_t>(a.X) % 16 == 0;
    if (a.norm_w && (!pieces || a.ldx > kMostStagedLd || reinterpret_cast<uintptr_t>(a.norm_w) % 16))
        return fail(TL_ERR_UNSUPPORTED, "rows that are normalised on their way in, and the norm's weight, are read in aligned pieces of 16 bytes");
    return x_dtype == TL_F16 ? launch_few_type<_Float16>(a, pieces, two_weights, st) : launch_few_type<float>(a, pieces, two_weights, st);
}
