// Many activation rows: the ternary product as a dense contraction on the matrix cores.
//
// tl_matrix_rows computes whole output tiles.  The activations of a tile and of a stage of 64 rows of K are copied into LDS
// by direct loads (`global_load_lds_dwordx4`: no register holds them on the way), a few stages ahead; the weights' two-bit
// codes arrive the same way, a unit of 256 rows of K ahead.  A wave turns the codes of its columns into operands in
// registers, where they serve all of its activation rows.  tl_x_image makes the row-major, padded copy of activations that
// come in another layout, and the three bf16 parts of fp32 ones.  tl_walk_rows multiplies from the index stream, for blobs
// without codes and K-major rows without a workspace.
#include "tl_matrix.h"

using namespace tl;

namespace {

typedef u32x4 u32x4_out __attribute__((aligned(8)));
typedef f32x4 f32x4_out __attribute__((aligned(8)));

constexpr int kStageRows = 64;                       // rows of K of a stage
constexpr int kStageRowBytes = kStageRows * 2;       // bytes of one activation row in a stage
// Row tiles whose column tiles a part of the chip works through together.  An activation tile is eight times the bytes of
// a code tile along the same K (24 times for fp32 in three parts), so few row tiles against many column tiles is least traffic: 8192 x 2048 -> 11008 took 456 us
// with all 64 row tiles in one group (every column tile streamed all activations through an L2), 300 / 300 / 310 with 2 / 4 / 8 (gated, as
// it is now, 248 / 247 / 248 and 254 with 16).
constexpr int kRowGroup = 4;
constexpr int kUnitStages = TL_CODE_UNIT_ROWS / kStageRows;
__device__ __align__(16) const unsigned char kNoCodes[TL_CODE_UNIT_BYTES] = {};   // a unit of zero weights

template <int N, typename F, int... I>
__device__ __forceinline__ void static_for(F f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void static_for(F f) { static_for<N>(f, std::make_integer_sequence<int, N>{}); }

// All but this wave's last N loads have come, and, where waves share what they copy, every other wave's.
template <bool SHARED, int N>
__device__ __forceinline__ void loads_here()
{
    if constexpr (SHARED) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(N) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// Where an activation row's 16-byte piece p of a stage lies among the row's eight: rotated by the row so that the 16 lanes
// the LDS serves together (rows r and r + 1 share 256 bytes, all 64 banks) find their pieces on different banks.
__device__ __forceinline__ int piece_place(int row, int p) { return p ^ ((row >> 1) & 7); }

// Where column c of the 16 of a wave's column block b lies in a quarter of the block's codes: four columns to 64 bytes, turned by
// the block, as the 16 lanes that the LDS serves together read four columns of each of four blocks, or eight of each of two.
__device__ __forceinline__ int code_place(int c, int b) { return c ^ ((b & 3) * 4); }

// COUNT neighbouring outputs of row m from column n on, of N: 16 bytes at a time where they lie so (vector_out), else one by one.
template <int COUNT>
__device__ __forceinline__ void store_piece(const KernelArgs& a, int m, int n, int N, const float* v)
{
    const long long at = (long long)m * a.ldy + n;
    if (a.vector_out && n + COUNT <= N) {
        if (a.y_f16) {
            static_assert(COUNT == 4 || COUNT % 8 == 0);
            __align__(16) __half o[COUNT];
#pragma unroll
            for (int i = 0; i < COUNT; ++i) o[i] = __float2half(settled(v[i]));
#pragma unroll
            for (int i = 0; i < COUNT / 8; ++i) reinterpret_cast<u32x4_out*>(static_cast<__half*>(a.Y) + at)[i] = reinterpret_cast<const u32x4*>(o)[i];
            if constexpr (COUNT == 4) *reinterpret_cast<uint2*>(static_cast<__half*>(a.Y) + at) = *reinterpret_cast<const uint2*>(o);
        } else {
#pragma unroll
            for (int i = 0; i < COUNT / 4; ++i) reinterpret_cast<f32x4_out*>(static_cast<float*>(a.Y) + at)[i] = f32x4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < COUNT; ++i)
        if (n + i < N) store_out(a.Y, a.y_f16, at + i, v[i]);
}

// `factor` times the scales of COUNT columns from n on, of N (past N: of the last column again; nothing of such columns is stored).
// Read at once: a load for each column under its own condition, and a wait for each, took 2 us of a launch.
template <int COUNT>
__device__ __forceinline__ void read_scales(const void* scale, int is_f16, int n, int N, float factor, float (&s)[COUNT])
{
    auto read = [&](auto type) {
        using T = decltype(type);
        const T* p = static_cast<const T*>(scale);
        T raw[COUNT];
        if (n + COUNT <= N) __builtin_memcpy(raw, p + n, sizeof(raw));
        else {
#pragma unroll
            for (int i = 0; i < COUNT; ++i) raw[i] = p[min(n + i, N - 1)];
        }
#pragma unroll
        for (int i = 0; i < COUNT; ++i) s[i] = factor * (float)raw[i];
    };
    if (!scale) {
#pragma unroll
        for (int i = 0; i < COUNT; ++i) s[i] = factor;
    } else if (is_f16) read(_Float16{});
    else read(float{});
}

enum { kPlain = 0, kPairs = 1, kTwoWeights = 2, kSteps = 3 };   // (kSteps: with what a decoder layer does around a product)

// The product of one output: from the index stream where the matrix cores' sum is not finite.
__device__ __forceinline__ float exact_output(const KernelArgs& a, const WeightPtrs& w, int m, int n) { return walk_column(w, a.T, a.tile_rows, n, callers_x(a, m)); }

// The last steps of COUNT neighbouring outputs of a row (kSteps): residual row, output, the next norm's image; returns the sum of
// the outputs' squares.  Rounded as separate operators would round.
template <int COUNT>
__device__ __forceinline__ float put_steps(const KernelArgs& a, int row, int n, float (&v)[COUNT])
{
    const bool whole = a.vector_out && n + COUNT <= a.N;             // (16-byte pieces of every array: the launcher has looked)
    auto read = [&](const void* p, long long at, float (&to)[COUNT]) {
        const __half* h = static_cast<const __half*>(p) + at;
        __align__(16) __half raw[COUNT];
        if (whole) {
#pragma unroll
            for (int i = 0; i < COUNT / 8; ++i) reinterpret_cast<u32x4*>(raw)[i] = reinterpret_cast<const u32x4_out*>(h)[i];
        } else {
#pragma unroll
            for (int i = 0; i < COUNT; ++i) raw[i] = n + i < a.N ? h[i] : __half(0.f);
        }
#pragma unroll
        for (int i = 0; i < COUNT; ++i) to[i] = __half2float(raw[i]);
    };
    float other[COUNT], sum = 0.f;
    if (a.chain_res) {
        read(a.chain_res, (long long)row * a.chain_ldres + n, other);
#pragma unroll
        for (int i = 0; i < COUNT; ++i) v[i] = as_output(v[i], 1) + other[i];
    }
#pragma unroll
    for (int i = 0; i < COUNT; ++i) v[i] = n + i < a.N ? as_output(v[i], 1) : 0.f;
    store_piece<COUNT>(a, row, n, a.N, v);
    if (a.chain_image) {
        read(a.chain_w, n, other);
#pragma unroll
        for (int i = 0; i < COUNT; ++i) {
            sum = fmaf(v[i], v[i], sum);
            v[i] *= other[i];
        }
        KernelArgs image = a;
        image.Y = a.chain_image;
        image.ldy = a.chain_ild;
        store_piece<COUNT>(image, row, n, a.N, v);
    }
    return sum;
}

// A lane's sums of G rows on their way out: C = 4 * CF neighbouring columns of each row from each CF fragments, of one weight or of
// two (fragments FW and on).  lane_m0 and lane_n0: its first row, of rows 16 apart, and its first column, of groups 4 * C apart.
// A sum that is not finite is worked out again by the lane that holds it, before anything is stored: the outputs of
// finite rows keep their bits whatever another row of the tile holds.  (The sums that need it go into a mask that a
// loop takes bit by bit, so that the walk stands here once and the sums stay in registers.)
template <int CF, int FW, int F, int G, int MODE>
__device__ __forceinline__ void put_out(const KernelArgs& a, f32x4 (&acc)[F][G], int lane_m0, int lane_n0)
{
    constexpr int C = 4 * CF, GROUPS = FW / CF, ALL = F / CF * G;
    static_assert(F == (MODE == kTwoWeights ? 2 : 1) * FW && FW % CF == 0);
    bool fine = true;
    float half = 0.5f;                                            // (the products are with +-2)
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
        for (int m = 0; m < G; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) fine = fine && fabsf(acc[f][m][e]) < __builtin_huge_valf();
    if (!fine) {
        half = 1.0f;
#pragma unroll 1
        for (int i = 0; i < ALL; ++i) {
            const int group = i / G, m = i % G, n = lane_n0 + group % GROUPS * 4 * C;
            float v[C];
            uint32_t redo = 0;
#pragma unroll
            for (int e = 0; e < C; ++e) {
                v[e] = acc[e / 4][0][e % 4];
#pragma unroll
                for (int o = 1; o < ALL; ++o) v[e] = o == i ? acc[o / G * CF + e / 4][o % G][e % 4] : v[e];
                const bool mine = lane_m0 + m * 16 < a.M && n + e < a.N;
                redo |= mine && !(fabsf(v[e]) < __builtin_huge_valf()) ? 1u << e : 0u;
                v[e] *= 0.5f;                                     // (twice what is worked out again might overflow)
            }
            while (redo != 0) {
                const int at = __builtin_ctz(redo);
                redo &= redo - 1;
                const float y = exact_output(a, group >= GROUPS ? a.w1 : a.w0, lane_m0 + m * 16, n + at);
#pragma unroll
                for (int e = 0; e < C; ++e) v[e] = e == at ? y : v[e];
            }
#pragma unroll
            for (int e = 0; e < C; ++e)
#pragma unroll
                for (int o = 0; o < ALL; ++o) acc[o / G * CF + e / 4][o % G][e % 4] = o == i ? v[e] : acc[o / G * CF + e / 4][o % G][e % 4];
        }
    }
    float s0[GROUPS][C], s1[MODE == kTwoWeights ? GROUPS : 1][C];
#pragma unroll
    for (int group = 0; group < GROUPS; ++group) {
        read_scales(a.w0.scale, a.scale_f16, lane_n0 + group * 4 * C, a.N, half, s0[group]);
        if constexpr (MODE == kTwoWeights) read_scales(a.w1.scale, a.scale_f16, lane_n0 + group * 4 * C, a.N, half, s1[group]);
    }
#pragma unroll
    for (int m = 0; m < G; ++m) {
        const int row = lane_m0 + m * 16;
#pragma unroll
        for (int group = 0; group < GROUPS; ++group) {
            const int n = lane_n0 + group * 4 * C;
            float v[C];
            if constexpr (MODE == kSteps) {
                static_assert(C == 8, "four lanes hold 32 columns of a row");
                float sum = 0.f;
                const float factor = a.chain_factors && row < a.M ? a.chain_factors[row] : 1.0f;
#pragma unroll
                for (int i = 0; i < C; ++i) v[i] = acc[group * CF + i / 4][m][i % 4] * s0[group][i] * factor;
                if (row < a.M && n < a.N) sum = put_steps(a, row, n, v);
                if (a.chain_image) {
                    auto pair = __builtin_amdgcn_permlane16_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
                    sum = __uint_as_float(pair[0]) + __uint_as_float(pair[1]);
                    pair = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
                    sum = __uint_as_float(pair[0]) + __uint_as_float(pair[1]);
                    if (n % 32 == 0 && row < a.M && n < a.N) a.chain_sq_out[(long long)row * ((a.N + 31) / 32) + n / 32] = sum;
                }
                continue;
            }
            if (row >= a.M || n >= a.N) continue;
#pragma unroll
            for (int i = 0; i < C; ++i) {
                v[i] = acc[group * CF + i / 4][m][i % 4] * s0[group][i];
                if constexpr (MODE == kTwoWeights) v[i] = silu(v[i]) * (acc[FW + group * CF + i / 4][m][i % 4] * s1[group][i]);
            }
            if constexpr (MODE == kPairs) {
                if (a.chain_factors) {
#pragma unroll
                    for (int i = 0; i < C; ++i) v[i] *= a.chain_factors[row];
                }
#pragma unroll
                for (int i = 0; i < C / 2; ++i) v[i] = gate_pair(as_output(v[2 * i], a.y_f16), as_output(v[2 * i + 1], a.y_f16), a.y_f16);
                store_piece<C / 2>(a, row, n / 2, a.N / 2, v);
            } else {
                store_piece<C>(a, row, n, a.N, v);
            }
        }
    }
}

// Bound by the matrix cores and, at the large sizes, by the power that they draw, so by the instruction: on such operands alone, and no
// memory, 16 x 16 x 32 products run at 2200 TFLOP/s in fp16 and 2230 in bf16, 32 x 32 x 16 ones at 1750 and 1880 (with the weights as
// the second operand 1970; at 66 % zeros).  With all that stands around them 8192 x 5504 -> 2048 runs at 1600, or 1760 without what a
// launch costs; without making operands and reading LDS it would take 8 % less.  A wave owns 64 columns: each fragment of
// activations that it reads from LDS serves four products.  us with 32 x 32 x 16 / now: 8192 x 2048 -> 11008 gated 280 / 247, 8192 x 2048 -> 6144
// 152 / 136, 8192 x 5504 -> 2048 133 / 115, 1024 x 4096 -> 11008 76 / 69; fp32 4096 x 4096 -> 4096 301 / 257, 1024 x 4096 -> 4096 88 / 74 (one run; by a tenth
// more or less on other cards).
// A lone wave on its SIMD is bound by what it issues, of which twice as many products are more: the load side's addresses
// are scalar and follow from the turn (fp32 1024 x 4096 -> 4096 82 us while they were worked out for every load).
//
// Output tiles of (WM * FM * 32) activation rows x (WN * FN * 32) columns, one per workgroup; a wave owns FM * 32 rows x
// FN * 32 columns.  WK = 1: WM x WN waves over all of K that share what they copy.  WK > 1: one tile of a wave, whose WK waves
// share K out by units, copy for themselves, wait for nobody and add up at the end; or, WN > 1, two groups of waves that share K out
// and whose waves share what they copy.  PARTS: 1 for fp16 activations, 3 for fp32
// ones in bf16 parts (a stage's three parts one after the other, with the same codes).
template <int PARTS, int WM, int WN, int WK, int FM, int FN, int MODE>
__global__ __launch_bounds__(WM * WN * WK * 64, 2) void tl_matrix_rows(KernelArgs a)
{
    constexpr int W = WM * WN;                                    // waves that work on the same rows of K, and share what is copied
    constexpr bool SHARED = W > 1;
    constexpr int TM = WM * FM * 32, TN = WN * FN * 32;
    static_assert(WK == 1 || (W == 1 && 2 * FM <= WK) || (WM == 1 && WK == 2), "how the sums of waves that share out K meet");
    constexpr int STAGES = kUnitStages;                           // buffers of activations: a stage's place in its unit names its buffer
    constexpr int XB = TM * kStageRowBytes;                       // bytes of a stage of activations
    constexpr int XL = TM / 8 / W;                                // activation loads of a wave per stage (8 rows each)
    constexpr int CL = (TN / 16 + W - 1) / W;                     // code loads of a wave per unit
    static_assert(TM % (8 * W) == 0, "every wave loads the same number of row groups");
    extern __shared__ __align__(16) unsigned char all_lds[];
    const int lane = threadIdx.x & 63;
    const int wg_wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave = wg_wave % W, wk = wg_wave / W;
    const int wm = wave / WN, wn = wave % WN;
    constexpr int OWN = STAGES * XB + (TN / 16) * TL_CODE_UNIT_BYTES;   // LDS of the waves that share
    unsigned char* lds = all_lds + wk * OWN;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;

    // Each part of the chip (ids equal modulo 8), which has an L2 of its own, owns a contiguous run of the list of tiles; the
    // list goes through all column tiles for a few row tiles at a time.
    constexpr int OUT_TN = MODE == kTwoWeights ? TN / 2 : TN;     // output columns of a tile
    const int row_tiles = (a.M + TM - 1) / TM;
    const int total_tiles = (int)gridDim.x;
    const int part = (int)blockIdx.x & 7, in_part = (int)blockIdx.x >> 3;
    const int base = total_tiles >> 3, extra = total_tiles & 7;
    const int tile = part * base + min(part, extra) + in_part;
    const int col_tiles = total_tiles / row_tiles;
    const int group = tile / (kRowGroup * col_tiles), in_group = tile - group * kRowGroup * col_tiles;
    const int group_rows = min(kRowGroup, row_tiles - group * kRowGroup);
    const int m0 = (group * kRowGroup + in_group % group_rows) * TM;
    const int nb0 = (in_group / group_rows) * (OUT_TN / 16);      // first column block

    // ---- what this wave copies ----
    // activations: its load i covers rows (i * W + wave) * 8 .. + 7 of the tile; lane -> row lane / 8, place lane % 8
    uint32_t xrow[XL];                                            // byte offset of this lane's row from the tile's base
    const uint32_t limit = (uint32_t)((a.K + 7) / 8 * 16 - 16);          // last whole piece of a row: pieces past it meet zero weights
    const int lane_row = lane >> 3;

    const uint32_t piece = (uint32_t)piece_place(wave * 8 + lane_row, lane & 7) * 16;
    static_assert(W % 2 == 0 || W == 1, "a lane's pieces lie at one place, or at two in turn");
#pragma unroll
    for (int i = 0; i < XL; ++i) xrow[i] = (uint32_t)(min(m0 + (i * W + wave) * 8 + lane_row, a.M - 1) - m0) * (uint32_t)(a.image_ld * 2);
    const unsigned char* image = static_cast<const unsigned char*>(a.image) + (long long)m0 * a.image_ld * 2;
    const long long unit_stride = TL_CODE_UNIT_BYTES;

    const int stages_k = (a.K + kStageRows - 1) / kStageRows;     // stages of K that hold anything
    const int all_units = a.planes * a.units;
    // this wave's units, and its turns: the last stage of the only plane may end a unit early
    const int unit0 = all_units * wk / WK, units = all_units * (wk + 1) / WK - unit0;
    const int all_stages = a.planes == 1 ? stages_k : all_units * kUnitStages;
    auto turns_of = [&](int first, int count) { return PARTS * (min((first + count) * kUnitStages, all_stages) - first * kUnitStages); };
    const int total = turns_of(unit0, units);

    // load side: the unit, within its plane, of the next activations to ask for; their stage and part follow from the turn
    int lk = unit0 % a.units, issued = 0;
    // (rows of a lane's loads differ by 8 * W: by a multiple of 16, or, W = 1, by 8, which turns the place by half)
    const unsigned char* part_image[PARTS];
#pragma unroll
    for (int p = 0; p < PARTS; ++p) part_image[p] = image + (PARTS > 1 ? (long long)p * a.image_plane * 2 : 0ll);
    // Turn TURN of a unit's activations.  WHOLE: all of the stage's pieces lie within K; else those past it are its last (and meet zero weights).
    auto issue_x = [&](auto turn_tag, auto whole_tag) {
        constexpr int TURN = decltype(turn_tag)::value, STAGE = TURN / PARTS;
        constexpr bool WHOLE = decltype(whole_tag)::value;
        const uint32_t k_bytes = (uint32_t)(lk * TL_CODE_UNIT_ROWS + STAGE * kStageRows) * 2;
        const unsigned char* src = part_image[TURN % PARTS] + (WHOLE ? k_bytes : 0);
#pragma unroll
        for (int i = 0; i < XL; ++i) {
            const uint32_t mine = W == 1 && i % 2 ? piece ^ 64u : piece;
            load_to_lds(lds0 + TURN % STAGES * XB + (i * W + wave) * 1024, src, xrow[i] + (WHOLE ? mine : min(k_bytes + mine, limit)));
        }
        ++issued;
        if (TURN == kUnitStages * PARTS - 1 && ++lk == a.units) lk = 0;   // (the last unit may be shorter: nothing is asked for after it)
    };
    const unsigned char* code_src[CL];                            // (wave-uniform)
    uint32_t code_to[CL];
    int code_units[CL];                                           // units that the block's weight has
#pragma unroll
    for (int i = 0; i < CL; ++i) {
        const int c = min(i * W + wave, TN / 16 - 1);             // column block of the tile
        const int owner = c / (2 * FN), f = c % (2 * FN);         // its wave column and place there
        const Codes& w = (MODE == kTwoWeights && f >= FN) ? a.c1 : a.c0;
        const int nb = MODE == kTwoWeights ? nb0 + owner * FN + f % FN : nb0 + c;
        code_units[i] = w.planes * a.units;
        code_src[i] = w.base + min(nb, a.NB - 1) * (code_units[i] * unit_stride);
        code_to[i] = lds0 + STAGES * XB + c * TL_CODE_UNIT_BYTES;
    }
    auto issue_codes = [&](int u) {
#pragma unroll
        for (int i = 0; i < CL; ++i) {
            const unsigned char* src = code_src[i] + (unit0 + u) * unit_stride;
            if (MODE == kTwoWeights && unit0 + u >= code_units[i]) src = kNoCodes;   // (the other weight has more planes)
            load_to_lds(code_to[i], src, (uint32_t)((lane & 48) + code_place(lane & 15, min(i * W + wave, TN / 16 - 1) % (MODE == kTwoWeights ? FN : 2 * FN))) * 16);
        }
    };

    // ---- what it reads ----
    constexpr int F = 2 * FN, G = 2 * FM;                         // fragments of 16 columns, of 16 rows
    constexpr int FW = MODE == kTwoWeights ? FN : F;              // fragments of columns of one weight
    const int q = lane >> 4, r16 = lane & 15;
    const uint32_t x_read = (uint32_t)((wm * FM * 32 + r16) * kStageRowBytes);
    const uint32_t swz = (uint32_t)(piece_place(r16, q) * 16);    // rows of a wave's fragments differ by multiples of 16: same place
    // Fragments whose columns a lane holds side by side, so that its sums of a row are 16 bytes of output (of fp16 ones for fp16
    // activations), and four lanes' 64.  (Where each lane held 16 columns, fp32 took 4 % longer: 4096 x 4096 -> 4096 274 us / 263.)
    constexpr int CF = (PARTS > 1 ? 1 : 2) * (MODE == kPairs ? 2 : 1) > FW ? FW : (PARTS > 1 ? 1 : 2) * (MODE == kPairs ? 2 : 1);
    // where the codes of this lane's row of fragment f's operand lie: column 16 * CF * (f / CF) + 4 * CF * (r16 / 4) + 4 * (f % CF) + r16 % 4
    const int col = 4 * CF * (r16 >> 2) + (r16 & 3);
    const uint32_t c_read = (uint32_t)(STAGES * XB + (wn * F + (col >> 4)) * TL_CODE_UNIT_BYTES + (q * 16 + code_place(col & 15, col >> 4)) * 16);
    constexpr bool F32 = PARTS > 1;
    f32x4 acc[F][G], low[F32 ? F : 1][F32 ? G : 1];               // low: the sums of the parts after the first
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
        for (int m = 0; m < G; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[f][m][e] = low[F32 ? f : 0][F32 ? m : 0][e] = 0.f;

    constexpr int R = 4, AHEAD = R - 1;                           // fragments of activations in registers; read ahead
    constexpr int STEPS = 2 * G;                                  // of a stage: a fragment of 16 rows x 32 rows of K each
    u32x4 x[R], codes[F], w[2][F];
    uint32_t last[F];                                             // the unit's last 64 rows of K, while the next unit's codes come
    auto read_x = [&](int buffer, int step) {                     // (constants)
        x[step % R] = *reinterpret_cast<const u32x4*>(lds + x_read + (swz ^ (uint32_t)(step / G * 64)) + buffer * XB + step % G * 16 * kStageRowBytes);
    };
    auto read_codes = [&]() {
#pragma unroll
        for (int f = 0; f < F; ++f) {
            const int first = f % FW / CF * CF;                   // column block of the weight's fragments that stand beside f
            codes[f] = *reinterpret_cast<const u32x4*>(lds + (c_read ^ (uint32_t)(code_place(4 * (f % CF), first) * 16)) + (first + f / FW * FN) * TL_CODE_UNIT_BYTES);
        }
    };
    // dword d % 4 of fragment d / 4's operand of the 32 rows of K number j of a unit (constants)
    auto operand_dword = [&](int j, int d, u32x4* to) {
        to[d / 4][d % 4] = ((j >= 6 ? last[d / 4] : codes[d / 4][j >> 1]) << ((j & 1) * 8 + 2 * (d % 4))) & 0xC000C000u;
    };
    if (units > 0) issue_codes(0);
    static_for<STAGES - 1>([&](auto s) {
        if (issued < total) issue_x(s, std::false_type{});
    });
    if (total >= STAGES - 1) loads_here<SHARED, (STAGES - 2) * XL>();
    else loads_here<SHARED, 0>();
    read_codes();
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) read_x(0, s);
#pragma unroll
    for (int d = 0; d < 4 * F; ++d) operand_dword(0, d, w[0]);
    int t = 0;
    // Turn Q of unit u: part Q % PARTS of its stage Q / PARTS.  STEADY: turns up to t + STAGES - 1 exist, and those asked for are whole.
    constexpr int TURNS = kUnitStages * PARTS;
    auto turn = [&](auto q_tag, auto steady_tag, int u) {
        constexpr int Q = decltype(q_tag)::value, J = Q / PARTS, P = Q % PARTS;
        constexpr bool STEADY = decltype(steady_tag)::value, FIRST = P == 0;
        constexpr int PER = 4 * F / G;                            // operand dwords made in a step
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int m = s % G, k = s / G;                       // k: 32 rows of K of the stage
            if (s == STEPS - AHEAD) {
                // turn t + 1's activations have come; every wave is done with turn t - 1, whose buffer takes turn t + STAGES - 1
                if (STEADY) loads_here<SHARED, (STAGES - 3) * XL>();
                else if (t + 1 < total) loads_here<SHARED, 0>();
                if (Q == 0 && (STEADY || u + 1 < units)) issue_codes(u + 1);
                if (STEADY || issued < total) issue_x(std::integral_constant<int, (Q + STAGES - 1) % TURNS>{}, steady_tag);
            }
            if (s + AHEAD < STEPS) read_x(Q % STAGES, s + AHEAD);
            else read_x((Q + 1) % STAGES, s + AHEAD - STEPS);
            if (Q == TURNS - PARTS - 1 && s == STEPS / 2) {       // (what the unit's last 64 rows of K are made from)
#pragma unroll
                for (int f = 0; f < F; ++f) last[f] = codes[f][3];
            }
            if (Q == TURNS - 1 && s == 0) read_codes();
#pragma unroll
            for (int f = 0; f < F; ++f) {
                f32x4& sum = FIRST ? acc[f][m] : low[F32 ? f : 0][F32 ? m : 0];
                sum = matrix_step<F32>(w[k & 1][f], x[s % R], sum);
            }
            if (k < 1 ? P == 0 : P == PARTS - 1) {                // (a stage's parts meet the same weights)
#pragma unroll
                for (int i = 0; i < PER; ++i) operand_dword((k < 1 ? 2 * J + 1 : 2 * J + 2) % 8, m * PER + i, w[(k + 1) & 1]);
            }
#pragma unroll
            for (int f = 0; f < F; ++f) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);               // a product,
                __builtin_amdgcn_sched_group_barrier(0x2, (2 * PER + F - 1) / F, 0);  // then vector instructions
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        ++t;
    };
    auto turns = [&](auto steady_tag, int u, int count) {
        static_for<TURNS>([&](auto q) {
            if (decltype(steady_tag)::value || decltype(q)::value < count) turn(q, steady_tag, u);
        });
    };
    int u = 0;
    // turns before one that might reach past K: the last stage, or, of several planes, those that fill up every plane's last unit
    const int whole = a.planes == 1 ? total - (a.K % kStageRows ? PARTS : 0) : a.K % TL_CODE_UNIT_ROWS == 0 ? total : 0;
    for (; (u + 1) * TURNS + STAGES - 1 <= whole; ++u) turns(std::true_type{}, u, TURNS);
    for (; u < units; ++u) turns(std::false_type{}, u, min(total - u * TURNS, TURNS));

    // (waves that meet at barriers take as many of them: a group whose share of K is shorter waits for the longest)
    if constexpr (SHARED && WK > 1) {
        int most = 0;
#pragma unroll
        for (int o = 0; o < WK; ++o) most = max(most, turns_of(all_units * o / WK, all_units * (o + 1) / WK - all_units * o / WK));
        for (int i = max(total, 1); i < most; ++i) __builtin_amdgcn_s_barrier();
    }

    // ---- out ----
    constexpr int WAVE_N = MODE == kTwoWeights ? FN * 16 : FN * 32;   // output columns of a wave
    if constexpr (SHARED && WK > 1) {
        // A wave and the other group's wave of the same outputs give each other half of their sums, by rows, through LDS (all of the
        // workgroup's, which every wave is done with); fp32 activations' are added up in 64 bits.
        constexpr int FRAGMENT = 64 * 4 * 4, HALF = G / 2, GIVEN = (F32 ? 2 : 1) * F * HALF * FRAGMENT;
        f32x4 v[F][HALF], v_low[F32 ? F : 1][F32 ? HALF : 1];
        unsigned char* mine = all_lds + wg_wave * GIVEN + lane * 16;
        const unsigned char* other = all_lds + ((1 - wk) * W + wave) * GIVEN + lane * 16;
        __syncthreads();
#pragma unroll
        for (int f = 0; f < F; ++f)
#pragma unroll
            for (int g = 0; g < HALF; ++g) {
                v[f][g] = wk ? acc[f][HALF + g] : acc[f][g];
                *reinterpret_cast<f32x4*>(mine + (f * HALF + g) * FRAGMENT) = wk ? acc[f][g] : acc[f][HALF + g];
                if constexpr (F32) {
                    v_low[f][g] = wk ? low[f][HALF + g] : low[f][g];
                    *reinterpret_cast<f32x4*>(mine + (F * HALF + f * HALF + g) * FRAGMENT) = wk ? low[f][g] : low[f][HALF + g];
                }
            }
        __syncthreads();
#pragma unroll
        for (int f = 0; f < F; ++f)
#pragma unroll
            for (int g = 0; g < HALF; ++g) {
                const f32x4 high = *reinterpret_cast<const f32x4*>(other + (f * HALF + g) * FRAGMENT);
                if constexpr (F32) {
                    const f32x4 rest = *reinterpret_cast<const f32x4*>(other + (F * HALF + f * HALF + g) * FRAGMENT);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        v[f][g][e] = (float)(((double)v_low[f][g][e] + rest[e]) * (1.0 / kLowScale) + ((double)v[f][g][e] + high[e]));
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[f][g][e] += high[e];
                }
            }
        put_out<CF, FW, F, HALF, MODE>(a, v, m0 + wk * HALF * 16 + r16, nb0 * 16 + wn * WAVE_N + q * 4 * CF);
    } else if constexpr (WK > 1) {
        // every wave has sums of the whole tile, of its own rows of K: they meet in LDS (a wave's in its own part, which it is
        // done with), and each goes on with 16 rows, or, where those are fewer than waves, with a group of their columns.  fp32
        // activations' are added up in 64 bits: roundings in 32 would weigh.
        constexpr int FRAGMENT = 64 * 4 * 4, PIECES = F32 ? 2 : 1;
        static_assert(PIECES * F * G * FRAGMENT <= OWN, "a wave's sums fit its part of LDS");
#pragma unroll
        for (int f = 0; f < F; ++f)
#pragma unroll
            for (int g = 0; g < G; ++g) {
                *reinterpret_cast<f32x4*>(lds + (f * G + g) * FRAGMENT + lane * 16) = acc[f][g];
                if constexpr (F32) *reinterpret_cast<f32x4*>(lds + (F * G + f * G + g) * FRAGMENT + lane * 16) = low[f][g];
            }
        __syncthreads();
        constexpr int MINE = CF > FW * G / WK ? CF : FW * G / WK; // fragments of a weight that a wave goes on with
        static_assert(FW % MINE == 0 && FW / MINE * G <= WK, "the waves take all of the tile");
        const int rows = wk % G, group = wk / G;
        if (group >= FW / MINE) return;
        f32x4 v[F / FW * MINE][1];
#pragma unroll
        for (int f = 0; f < F / FW * MINE; ++f) {
            const int from = (f / MINE * FW + group * MINE + f % MINE) * G + rows;
            std::conditional_t<F32, double, float> sum[4] = {};
#pragma unroll
            for (int piece = PIECES - 1; piece >= 0; --piece) {
#pragma unroll
                for (int o = 0; o < WK; ++o) {
                    const f32x4 part = *reinterpret_cast<const f32x4*>(all_lds + o * OWN + (piece * F * G + from) * FRAGMENT + lane * 16);
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[e] += part[e];
                }
                if (piece == 1)
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[e] *= 1.0f / kLowScale;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[f][0][e] = (float)sum[e];
        }
        put_out<CF, MINE, F / FW * MINE, 1, MODE>(a, v, m0 + rows * 16 + r16, nb0 * 16 + group * 16 * MINE + q * 4 * CF);
    } else {
        if constexpr (F32) {
#pragma unroll
            for (int f = 0; f < F; ++f)
#pragma unroll
                for (int m = 0; m < G; ++m) add_low(acc[f][m], low[f][m]);
        }
        put_out<CF, FW, F, G, MODE>(a, acc, m0 + wm * FM * 32 + r16, nb0 * 16 + wn * WAVE_N + q * 4 * CF);
    }
}

// Eight neighbouring activations of a row into the image: fp16 as they are, fp32 in three bf16 parts.
template <typename XT>
__device__ __forceinline__ void put8(const KernelArgs& a, unsigned short* image, int m, int k, const XT* v)
{
    if constexpr (sizeof(XT) == 2) {
        *reinterpret_cast<u32x4*>(image + m * a.image_ld + k) = *reinterpret_cast<const u32x4*>(v);
    } else {
        u32x4 part[3];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t lo[3], hi[3];
            split3(v[2 * i], &lo[0], &lo[1], &lo[2]);
            split3(v[2 * i + 1], &hi[0], &hi[1], &hi[2]);
#pragma unroll
            for (int p = 0; p < 3; ++p) part[p][i] = (lo[p] >> 16) | hi[p];
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4*>(image + p * a.image_plane + m * a.image_ld + k) = part[p];
    }
}

// The activations as a row-major image of rows of whole 16-byte pieces, zeros past K.  Bound by memory: each value read
// once and written once (three times two bytes of four for fp32).  Row-major: a thread takes eight values of a row.
template <typename XT>
__global__ __launch_bounds__(256) void tl_x_image(KernelArgs a, unsigned short* image)
{
    const unsigned pieces = (unsigned)(a.K + 7) / 8;
    const unsigned e = blockIdx.x * 256 + threadIdx.x;
    if (e >= pieces * (unsigned)a.M) return;
    const int m = (int)(e / pieces), k = (int)(e % pieces) * 8;
    const XT* row = static_cast<const XT*>(a.X) + m * a.ldx;
    __align__(16) XT v[8];
    if (k + 8 <= a.K && ((uintptr_t)(row + k) & 15) == 0) {
#pragma unroll
        for (int i = 0; i < (int)sizeof(XT) / 2; ++i) reinterpret_cast<u32x4*>(v)[i] = reinterpret_cast<const u32x4*>(row + k)[i];
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = k + i < a.K ? row[k + i] : XT(0.f);
    }
    put8<XT>(a, image, m, k, v);
}

// The same from K-major activations: 64 x 64 tiles turned in LDS.
template <typename XT>
__global__ __launch_bounds__(256) void tl_x_image_k(KernelArgs a, unsigned short* image)
{
    __shared__ XT tile[64][65];  // [row][k]
    const int k0 = (int)blockIdx.x * 64, m0 = (int)blockIdx.y * 64;
    const int c = threadIdx.x & 63, q = threadIdx.x >> 6;
    const XT* X = static_cast<const XT*>(a.X);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int k = k0 + q * 16 + i, m = m0 + c;
        tile[c][q * 16 + i] = k < a.K && m < a.M ? X[k * a.ldx + m] : XT(0.f);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int item = i * 256 + (int)threadIdx.x, r = item >> 3, p = (item & 7) * 8;
        if (m0 + r >= a.M || k0 + p >= (a.K + 7) / 8 * 8) continue;
        __align__(16) XT v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = tile[r][p + e];
        put8<XT>(a, image, m0 + r, k0 + p, v);
    }
}

// The product from the index stream alone, for blobs without codes and for K-major rows without a workspace.  A wave owns
// 64 * R rows and four columns, so indices are wave-uniform (scalar loads); R neighbouring rows of a lane are one 8-byte
// piece.  Bound by those loads: 16 waves, 64 columns, share the pieces of a tile of K-major activations in LDS (us, 80 %
// zeros, fp16 / fp32: 1024 x 4096 -> 11008 967 / 1259, 200 x 2048 -> 2048 143 / 87; one thread per output took 46038 / 46556
// and 625 / 699, four waves that read the pieces from the caches 1115 / 2066 and 114 / 99).
// R = 1 reads single elements of any layout: the last resort, without a workspace for row-major ones.
template <typename XT, int R, int MODE>
__global__ __launch_bounds__(R > 1 ? 1024 : 256) void tl_walk_rows(KernelArgs a)
{
    constexpr bool STAGED = R > 1;
    extern __shared__ __align__(16) unsigned char lds[];  // STAGED: [row of K][lane], 8 bytes each
    uint2* staged = reinterpret_cast<uint2*>(lds);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    constexpr int COLS = TL_BLOCK_COLUMNS / 4, BLOCKS = STAGED ? 4 : 1;   // columns of a wave, blocks of a workgroup
    const int groups = (a.NB + BLOCKS - 1) / BLOCKS;
    const int nb = (int)blockIdx.x % groups * BLOCKS + wave / 4, c0 = wave % 4 * COLS;
    const int m0 = ((int)blockIdx.x / groups * 64 + lane) * R;
    const XT* x = static_cast<const XT*>(a.X) + (R > 1 ? m0 : min(m0, a.M - 1) * a.x_sm);   // (wide rows are padded to whole waves)
    float acc[MODE == kTwoWeights ? 2 : 1][COLS][R] = {};
    auto walk = [&](const WeightPtrs& w, int t, float (&sum)[COLS][R]) {
        const_u32_ptr chunk = as_const(w.stream) + as_const(w.chunkstart)[(size_t)nb * a.T + t];
        const XT* tile = x + (long long)t * a.tile_rows * a.x_sk;
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
            const uint32_t d = chunk[c0 + c];
            auto run = [&](const_u32_ptr p, int n, float sign) {
                auto value = [&](uint32_t k, XT* v) {
                    if constexpr (STAGED) *reinterpret_cast<uint2*>(v) = staged[k * 64 + lane];
                    else v[0] = tile[k * a.x_sk];
                };
                auto add = [&](const XT* v) {
#pragma unroll
                    for (int j = 0; j < R; ++j) sum[c][j] = fmaf((float)v[j], sign, sum[c][j]);
                };
                // (four dwords of the stream are always there: the blob has spare bytes behind it)
                for (; n >= 16; n -= 16, p += 4) {
                    __align__(8) XT v[16][R];
#pragma unroll
                    for (int i = 0; i < 16; ++i) value(p[i >> 2] >> (8 * (i & 3)) & 0xffu, v[i]);
#pragma unroll
                    for (int i = 0; i < 16; ++i) add(v[i]);
                }
                const uint32_t rest[4] = {p[0], p[1], p[2], p[3]};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (4 * q >= n) break;
                    __align__(8) XT v[4][R];
#pragma unroll
                    for (int i = 0; i < 4; ++i) value(4 * q + i < n ? rest[q] >> (8 * i) & 0xffu : rest[q] & 0xffu, v[i]);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (4 * q + i < n) add(v[i]);
                }
            };
            run(chunk + (d >> 16), (int)(d & 0xffu), 1.0f);
            run(chunk + (d >> 16) + run_pos_dwords(d), (int)((d >> 8) & 0xffu), -1.0f);
        }
    };
    for (int t = 0; t < a.T; ++t) {
        if constexpr (STAGED) {
            const XT* tile = x + (long long)t * a.tile_rows * a.x_sk;
            const int rows = min(a.tile_rows, a.K - t * a.tile_rows);
            __syncthreads();                                      // (every wave is done with the tile before)
            for (int k = wave; k < rows; k += 16) staged[k * 64 + lane] = *reinterpret_cast<const uint2*>(tile + k * a.x_sk);
            __syncthreads();
        }
        if (STAGED && nb >= a.NB) continue;
        walk(a.w0, t, acc[0]);
        if constexpr (MODE == kTwoWeights) walk(a.w1, t, acc[1]);
    }
#pragma unroll
    for (int c = 0; c < COLS; c += MODE == kPairs ? 2 : 1) {
        const int n = nb * TL_BLOCK_COLUMNS + c0 + c;
        if (n >= a.N) break;
        const float s0 = load_scale(a.w0.scale, a.scale_f16, n);
        const float s1 = MODE == kTwoWeights ? load_scale(a.w1.scale, a.scale_f16, n) : MODE == kPairs ? load_scale(a.w0.scale, a.scale_f16, n + 1) : 0.f;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            if (m0 + j >= a.M) break;
            float v = acc[0][c][j] * s0;
            if constexpr (MODE == kTwoWeights) v = silu(v) * (acc[1][c][j] * s1);
            if constexpr (MODE == kPairs) v = gate_pair(as_output(v, a.y_f16), as_output(acc[0][c + 1][j] * s1, a.y_f16), a.y_f16);
            store_out(a.Y, a.y_f16, (long long)(m0 + j) * a.ldy + (MODE == kPairs ? n / 2 : n), v);
        }
    }
}

// Activations of any layout as the K-major image [K][ld] that tl_walk_rows reads, zeros from row M to ld: 64 x 64 tiles,
// row-major ones turned in LDS.
template <typename XT>
__global__ __launch_bounds__(256) void tl_k_image(KernelArgs a, XT* image, int ld)
{
    __shared__ XT tile[64][65];  // [k][row]
    const int k_tiles = (a.K + 63) / 64;
    const int k0 = (int)(blockIdx.x % k_tiles) * 64, m0 = (int)(blockIdx.x / k_tiles) * 64;
    const int c = threadIdx.x & 63, q = threadIdx.x >> 6;
    const XT* X = static_cast<const XT*>(a.X);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int k = k0 + (a.x_kmajor ? q * 16 + i : c), m = m0 + (a.x_kmajor ? c : q * 16 + i);
        const XT v = k < a.K && m < a.M ? X[k * a.x_sk + m * a.x_sm] : XT(0.f);
        if (a.x_kmajor) tile[q * 16 + i][c] = v;
        else tile[c][q * 16 + i] = v;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int k = k0 + q * 16 + i;
        if (k < a.K) image[(long long)k * ld + m0 + c] = tile[q * 16 + i][c];
    }
}

// Whether tl_walk_rows can read 8 bytes of a row of K at a time, up to a whole wave's rows.
bool walk_reads_directly(const KernelArgs& a)
{
    const int64_t rows = a.x_f16 ? 256 : 128;
    return a.x_kmajor && a.ldx % rows == 0 && a.ldx >= round_up(a.M, rows) && reinterpret_cast<uintptr_t>(a.X) % 16 == 0;
}

template <typename XT, int R, int MODE>
int launch_walk_mode(const KernelArgs& a, hipStream_t st)
{
    const int64_t groups = ceil_div(a.NB, R > 1 ? 4 : 1) * ceil_div(a.M, 64 * R);
    if (groups > INT32_MAX) return fail(TL_ERR_SHAPE, "%d rows are more than one launch takes", a.M);
    const size_t lds = R > 1 ? (size_t)kMaxTileRows * 512 : 0;
    auto kernel = tl_walk_rows<XT, R, MODE>;
    static LdsLimit raised;
    if (lds)
        if (int rc = raised.raise(kernel, lds)) return rc;
    hipLaunchKernelGGL(kernel, dim3((unsigned)groups), dim3(R > 1 ? 1024 : 256), lds, st, a);
    return TL_OK;
}

template <typename XT, int R>
int launch_walk(const KernelArgs& a, bool two_weights, hipStream_t st)
{
    if (two_weights) return launch_walk_mode<XT, R, kTwoWeights>(a, st);
    return a.gated ? launch_walk_mode<XT, R, kPairs>(a, st) : launch_walk_mode<XT, R, kPlain>(a, st);
}

// Rows that lie K-major, aligned and padded to whole waves are read where they are; others through an image, where the
// workspace holds it.
template <typename XT>
int walk_rows(KernelArgs a, void* workspace, int64_t workspace_bytes, bool two_weights, hipStream_t st)
{
    constexpr int R = 8 / (int)sizeof(XT);
    const int64_t ld = round_up(a.M, 64 * R);
    if (walk_reads_directly(a)) return launch_walk<XT, R>(a, two_weights, st);
    const int64_t tiles = ceil_div(a.K, 64) * (ld / 64);
    if (!workspace || workspace_bytes < a.K * ld * (int64_t)sizeof(XT) || reinterpret_cast<uintptr_t>(workspace) % 16 || tiles > INT32_MAX)
        return launch_walk<XT, 1>(a, two_weights, st);
    hipLaunchKernelGGL(tl_k_image<XT>, dim3((unsigned)tiles), dim3(256), 0, st, a, static_cast<XT*>(workspace), (int)ld);
    a.X = workspace;
    a.x_sm = 1;
    a.x_sk = ld;
    return launch_walk<XT, R>(a, two_weights, st);
}

template <int PARTS, int WM, int WN, int WK, int FM, int FN, int MODE>
int launch_tile(const KernelArgs& a, hipStream_t st)
{
    constexpr int TM = WM * FM * 32, TN = WN * FN * 32, OUT_TN = MODE == kTwoWeights ? TN / 2 : TN;
    constexpr size_t copied = WK * ((size_t)kUnitStages * TM * kStageRowBytes + (TN / 16) * TL_CODE_UNIT_BYTES);
    constexpr size_t given = WK > 1 && WN > 1 ? (size_t)TM * TN * sizeof(float) * (PARTS > 1 ? 2 : 1) : 0;   // half of each group's sums
    constexpr size_t lds = copied > given ? copied : given;
    static_assert(lds <= 160 * 1024, "the stages fit a compute unit's LDS");
    auto kernel = tl_matrix_rows<PARTS, WM, WN, WK, FM, FN, MODE>;
    static LdsLimit raised;
    if (int rc = raised.raise(kernel, lds)) return rc;
    const int64_t tiles = ceil_div(a.M, TM) * ceil_div(a.N, OUT_TN);
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(WM * WN * WK * 64), lds, st, a);
    return TL_OK;
}

}  // namespace

// Which tile, by how many there are and by the units of 256 rows of K (a multiple of the units is shared out evenly).  us, fp16, graphs of
// a call (`tl_spmm`, `tl_mlp_gate_up`), both sides of a line in turn:
//   "shared", K shared out among four waves, up to one 64 x 64 tile a compute unit.  Bound by what a compute unit copies (some 40 bytes a clock, of
//     which each wave's activations are most), so the smallest tile of which each compute unit has at most one, and 32 x 64 two to a unit for fp32.
//     32 x 32 / 32 x 64 / 64 x 64, 64 rows -> 4096: K = 512 4.1 / 4.6 / 5.8, 4096 6.6 / 8.1 / 10.6; fp32 512 9.4 / 10.3 / 12.0, 4096 17.7 / 19.0 / 24.6.  Two
//     32 x 64 tiles a unit / one 64 x 64, 256 rows -> 4096: 1024 6.3 / 6.4, 1536 7.4 / 8.0, 2048 8.1 / 8.2, 4096 11.5 / 11.2; fp32 1024 13.7 / 14.5, 2048
//     19.1 / 20.9; two weights, 128 rows -> 4096: 512 5.6 / 6.0, 768 6.3 / 6.2, 1536 7.8 / 7.8, 2048 8.4 / 8.1, 4096 11.7 / 10.9.
//   "small", 64 x 64, a wave 32 x 32, where K is one unit, of which three waves that share it have none, and for fp16 up to three where shared ones are two
//     to a unit.  32 x 64 / small, 128 rows -> 4096: K = 64 3.9 / 3.6, 256 4.7 / 4.2, but 512 4.7 / 4.8; 256 rows 256 5.3 / 4.3, 768 6.1 / 5.8, 1024 6.3 / 6.5; fp32,
//     128 rows 64 7.0 / 6.4, 256 10.0 / 9.6, 512 10.6 / 12.2; 256 rows 64 7.8 / 6.8, 256 10.8 / 10.2, 512 11.6 / 13.0.  (32 x 32, one to a unit, are as fast:
//     64 rows 64 3.6 / 3.5, 256 4.0 / 4.1.)  Two weights, 128 rows -> 4096, 32 x 64 / wide: 256 5.5 / 5.3, 512 5.6 / 6.4, 768 6.3 / 7.4.
//   "wide", 64 x 128, a wave 64 x 32 (two weights: 32 x 64), up to three a unit; two weights of fp16 rows up to eight units of K only; one weight
//     of fp16 rows up to three units of K as many as fit the units at once, four each.  Shared (which fits a unit once) / wide / flat, 512 rows -> 4096: K = 256 10.0 / 5.4 / 6.7, 1024
//     11.2 / 8.3 / 11.0, 4096 23.0 / 22.0 / 27.3; fp32 21.6 / 13.1 / 14.8, 25.8 / 23.1 / 28.1, 61.5 / 58.0 / 75.5.  Wide / flat, two or three a unit: 1024 rows -> 5504 256
//     8.0 / 9.1, 1024 13.3 / 15.7, 5504 49.1 / 55.6; two weights, 768 rows -> 4096 256 8.5 / 8.9, 1536 20.0 / 20.3, 2048 25.0 / 25.1, 5504 59.4 / 57.2.  Four, 2048 rows -> 4096:
//     256 9.6 / 9.8, 512 11.7 / 12.2, 768 13.8 / 14.3, 1024 16.5 / 16.6; more, 1024 rows of 256 -> 11008 12.1 / 11.8.
//   "halves", 64 x 128 for four waves, two for each 64 columns, which share K out, in the place of wide ones that are one a unit, for two weights from four
//     units of K on: a wave's 64 columns meet each fragment of activations four times, as it makes half the operands a product, and twice as much is
//     asked for ahead.  Wide / halves, 512 rows -> 2048: 768 7.7 / 8.3, 1024 8.8 / 8.2, 2048 13.1 / 11.3, 5504 29.5 / 23.1; fp32 768 17.7 / 19.8, 1024 20.7 / 19.8, 5504 68.2 / 58.0.
//     One weight, fp16 rows, from eight units on where the groups' shares are alike, and past twelve at all: wide ones had become up to 6 % slower with products
//     of 16 x 16 x 32 (with those before / wide / halves, 640 rows -> 2048: 1536 9.1 / 9.5 / 9.5, 2048 11.3 / 11.7 / 11.4, 2304 12.2 / 12.6 / 13.1, 2560 13.1 / 13.5 / 13.0, 2816
//     14.1 / 14.5 / 14.7, 3328 16.3 / 17.3 / 16.7, 4096 20.3 / 20.9 / 18.1, 8192 36.8 / 36.0 / 29.4; 512 rows -> 4096: 1536 9.9 / 9.8 / 9.8, 2048 12.2 / 11.9 / 11.7, 5504 26.5 / 26.3 / 23.0).
//   "groups", 64 x 256 for eight waves, two for each 64 columns, which share K out, while such tiles are one a unit and K is long: with flat ones a unit has
//     four waves, one on each SIMD.  Wide / groups, 1024 rows -> 4096: 1024 10.3 / 11.2, 2816 20.6 / 20.5, 4096 28.1 / 26.8, 5504 37.0 / 34.7; 768 rows 2816 19.0 / 19.7, 4096
//     25.5 / 25.1; fp32, 1024 rows 1536 38.0 / 38.7, 2048 46.2 / 46.6, 4096 79.1 / 73.0; 768 rows 1536 36.1 / 36.4, 2048 43.9 / 43.3.  Two weights, wide / flat / groups, 512 rows -> 4096: 256
//     6.9 / 7.2 / 7.8, 768 10.2 / 10.2 / 10.2, 1024 11.8 / 11.7 / 11.1, 2048 18.4 / 17.4 / 15.9.
//   "tall", 128 x 256, a wave 128 rows x 64, where there are two of them a unit, so that one multiplies while the other waits or stores, and where flat ones
//     (64 x 256) would not spread the rows better.  Tall / flat: 2048 x 4096 -> 11008 122 / 128, 8192 x 2048 -> 11008 gated 244 / 253, 8192 x 5504 -> 2048 114 / 120,
//     but 1024 x 4096 -> 11008 80 / 68 (344 tall tiles are two for some units, 688 flat ones five halves).  Not for fp32, whose second
//     set of sums does not fit.
MatrixTile tl::matrix_tile(int64_t rows, int64_t columns, int64_t depth, bool f32, bool two, int64_t units)
{
    auto tiles = [&](int height, int width) { return ceil_div(rows, height) * ceil_div(columns * (two ? 2 : 1), width); };
    if (tiles(64, 64) <= units) {
        const bool one_each = tiles(32, 64) <= units;
        if (tiles(32, 32) <= units) return kShared32x32;
        if (!two && depth <= (f32 || one_each ? 1 : 3)) return kSmall;
        if (f32 || one_each || (depth > 1 && depth <= (two ? 6 : 8))) return kShared32x64;
        if (depth > 1) return kShared64x64;
    }
    const int64_t wide = tiles(64, 128);
    if (wide <= units) return (two ? depth > 3 : !f32 && (depth > 12 || (depth >= 8 && depth % 2 == 0))) ? kHalves : kWide;
    if (tiles(64, 256) <= units && depth > (f32 ? two ? 4 : 6 : two ? 3 : 12)) return kGroups;
    if (wide <= 3 * units && (f32 || !two || depth <= 8)) return kWide;
    if (wide <= 4 * units && !f32 && !two && depth <= 3) return kWide;
    if (!f32 && tiles(128, 256) >= 2 * units && ceil_div(tiles(64, 256), units) >= 2 * ceil_div(tiles(128, 256), units)) return kTall;
    return kFlat;
}

namespace {

// The rows are the whole call's: a row's result does not depend on how many rows at a time a workspace holds.
template <int PARTS, int MODE>
int launch_mode(const KernelArgs& a, hipStream_t st)
{
    constexpr bool TWO = MODE == kTwoWeights, F32 = PARTS > 1;
    switch (matrix_tile(a.call_rows, a.N, (int64_t)a.planes * a.units, F32, TWO, compute_units())) {
    case kShared32x32: return launch_tile<PARTS, 1, 1, 4, 1, 1, MODE>(a, st);
    case kShared32x64: return launch_tile<PARTS, 1, 1, 4, 1, 2, MODE>(a, st);
    case kShared64x64:
        if constexpr (!F32) return launch_tile<PARTS, 1, 1, 4, 2, 2, MODE>(a, st);
        break;
    case kSmall:
        if constexpr (!TWO) return launch_tile<PARTS, 2, 2, 1, 1, 1, MODE>(a, st);
        break;
    case kWide:
        if constexpr (TWO) return launch_tile<PARTS, 2, 2, 1, 1, 2, MODE>(a, st);
        else return launch_tile<PARTS, 1, 4, 1, 2, 1, MODE>(a, st);
    case kHalves:
        if constexpr (TWO || !F32) return launch_tile<PARTS, 1, 2, 2, 2, 2, MODE>(a, st);
        break;
    case kGroups: return launch_tile<PARTS, 1, 4, 2, 2, 2, MODE>(a, st);
    case kFlat: return launch_tile<PARTS, 1, 4, 1, 2, 2, MODE>(a, st);
    case kTall:
        if constexpr (!F32) return launch_tile<PARTS, 1, 4, 1, 4, 2, MODE>(a, st);
        break;
    }
    return fail(TL_ERR_UNSUPPORTED, "no such tile");
}

template <int PARTS>
int launch_parts(const KernelArgs& a, bool two_weights, hipStream_t st)
{
    if (two_weights) return launch_mode<PARTS, kTwoWeights>(a, st);
    if constexpr (PARTS == 1) {
        if (!a.gated && (a.chain_res || a.chain_image || a.chain_factors)) return launch_mode<PARTS, kSteps>(a, st);
    }
    return a.gated ? launch_mode<PARTS, kPairs>(a, st) : launch_mode<PARTS, kPlain>(a, st);
}

// The image of a call's activations (a.image_ld and a.image_plane say how it lies).
void make_image(const KernelArgs& a, int x_dtype, unsigned short* image, hipStream_t st)
{
    if (a.x_kmajor) {
        const dim3 grid((unsigned)ceil_div(a.K, 64), (unsigned)ceil_div(a.M, 64));
        if (x_dtype == TL_F16) hipLaunchKernelGGL(tl_x_image_k<__half>, grid, dim3(256), 0, st, a, image);
        else hipLaunchKernelGGL(tl_x_image_k<float>, grid, dim3(256), 0, st, a, image);
        return;
    }
    const int64_t pieces = ceil_div(a.K, 8);
    const int64_t rows = std::max<int64_t>(1, ((int64_t)1 << 30) / pieces);  // of a launch, which counts its pieces in 32 bits
    for (int64_t m = 0; m < a.M; m += rows) {
        KernelArgs some = a;
        some.X = static_cast<const unsigned char*>(a.X) + m * a.ldx * (x_dtype == TL_F16 ? 2 : 4);
        some.M = (int)std::min<int64_t>(a.M - m, rows);
        const dim3 grid((unsigned)ceil_div(pieces * some.M, 256));
        if (x_dtype == TL_F16) hipLaunchKernelGGL(tl_x_image<__half>, grid, dim3(256), 0, st, some, image + m * a.image_ld);
        else hipLaunchKernelGGL(tl_x_image<float>, grid, dim3(256), 0, st, some, image + m * a.image_ld);
    }
}

}  // namespace

constexpr int64_t kMostLd = 1 << 24;  // (a lane's byte offset inside the 128 rows of a tile has 32 bits)

bool tl::matrix_reads_rows(const KernelArgs& a, int x_dtype)
{
    return x_dtype == TL_F16 && !a.x_kmajor && a.K % 8 == 0 && a.ldx % 8 == 0 && a.ldx <= kMostLd && reinterpret_cast<uintptr_t>(a.X) % 16 == 0;
}

int tl::launch_matrix_rows(KernelArgs a, int x_dtype, void* workspace, int64_t workspace_bytes, bool two_weights, hipStream_t st)
{
    a.call_rows = a.M;
    a.x_sm = a.x_kmajor ? 1 : a.ldx;
    a.x_sk = a.x_kmajor ? a.ldx : 1;
    const int64_t need = least_image_bytes(a.K, a.M, x_dtype);
    // Without codes, and for K-major rows that need no workspace, the index stream is walked.
    if (!a.c0.base || (two_weights && !a.c1.base) || ((!workspace || workspace_bytes < need) && walk_reads_directly(a)))
        return x_dtype == TL_F16 ? walk_rows<__half>(a, workspace, workspace_bytes, two_weights, st)
                                 : walk_rows<float>(a, workspace, workspace_bytes, two_weights, st);
    a.vector_out = a.ldy % (a.y_f16 ? 4 : 2) == 0 && reinterpret_cast<uintptr_t>(a.Y) % 8 == 0;
    if (a.chain_image)                                            // (the image is stored, and the residual rows read, in the same pieces)
        a.vector_out = a.vector_out && a.chain_ild % 4 == 0 && reinterpret_cast<uintptr_t>(a.chain_image) % 8 == 0 && reinterpret_cast<uintptr_t>(a.chain_w) % 8 == 0;
    if (a.chain_res) a.vector_out = a.vector_out && a.chain_ldres % 4 == 0 && reinterpret_cast<uintptr_t>(a.chain_res) % 8 == 0;
    // rows that lie as the kernel reads them are read where they are; any other layout, and fp32, goes through the image
    const bool direct = matrix_reads_rows(a, x_dtype);
    a.image_ld = direct ? a.ldx : round_up(a.K, 8);
    if (a.image_ld > kMostLd)
        return fail(TL_ERR_ARG, "rows of %lld activations are too long for one call", (long long)a.image_ld);
    if (direct) {
        a.image = a.X;
        return launch_parts<1>(a, two_weights, st);
    }
    if (!workspace || workspace_bytes < need)
        return fail(TL_ERR_SIZE, "workspace has %lld bytes, %lld needed", (long long)workspace_bytes, (long long)need);
    if (reinterpret_cast<uintptr_t>(workspace) % 16) return fail(TL_ERR_ALIGN, "workspace must be 16-byte aligned");
    // all rows at once where their image fits (and its launch's second dimension holds them), else as many whole row tiles as do
    int64_t rows = std::min<int64_t>(a.M, workspace_bytes / image_row_bytes(a.K, x_dtype));
    if (a.x_kmajor) rows = std::min<int64_t>(rows, 65535 * 64);
    if (rows < a.M && rows > 128) rows = rows / 128 * 128;
    a.image = workspace;
    for (int64_t m = 0; m < a.M; m += rows) {
        KernelArgs some = a;
        some.M = (int)std::min<int64_t>(a.M - m, rows);
        some.X = static_cast<const unsigned char*>(a.X) + m * (a.x_kmajor ? 1 : a.ldx) * (x_dtype == TL_F16 ? 2 : 4);
        some.Y = static_cast<unsigned char*>(a.Y) + m * a.ldy * (a.y_f16 ? 2 : 4);
        some.image_plane = a.image_ld * some.M;
        make_image(some, x_dtype, static_cast<unsigned short*>(workspace), st);
        if (int rc = x_dtype == TL_F16 ? launch_parts<1>(some, two_weights, st) : launch_parts<3>(some, two_weights, st)) return rc;
    }
    return TL_OK;
}
