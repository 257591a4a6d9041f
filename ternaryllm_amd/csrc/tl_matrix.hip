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

constexpr int kStageRows = 64;                       // rows of K of a stage
constexpr int kStageRowBytes = kStageRows * 2;       // bytes of one activation row in a stage
// Row tiles whose column tiles a part of the chip works through together.  An activation tile is eight times the bytes of
// a code tile along the same K (24 times for fp32 in three parts), so few row tiles against many column tiles is least traffic: 8192 x 2048 -> 11008 took 456 us
// with all 64 row tiles in one group (every column tile streamed all activations through an L2), 300 / 300 / 310 with 2 / 4 / 8.
constexpr int kRowGroup = 4;
constexpr int kUnitStages = TL_CODE_UNIT_ROWS / kStageRows;
__device__ __align__(16) const unsigned char kNoCodes[TL_CODE_UNIT_BYTES] = {};   // a unit of zero weights

// 16 bytes per lane from `base` + offset into LDS at `lds` + 16 * lane.  (As assembly, because the compiler would wait for
// all such loads before any read of LDS; here they are counted by hand.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // (m0 is a register that the compiler reserves; named all the same, as this writes it)
__device__ __forceinline__ void load_to_lds(uint32_t lds, const void* base, uint32_t offset)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(offset), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop

template <int N>
__device__ __forceinline__ void wait_loads_and_barrier()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

// Where an activation row's 16-byte piece p of a stage lies among the row's eight: rotated by the row so that the 16 lanes
// the LDS serves together (rows r and r + 1 share 256 bytes, all 64 banks) find their pieces on different banks.
__device__ __forceinline__ int piece_place(int row, int p) { return p ^ ((row >> 1) & 7); }

// Four neighbouring outputs of one row, v[i] in column n + i: scale, SiLU gate of column pairs, store.
template <bool PAIRS>
__device__ __forceinline__ void store4(const KernelArgs& a, int m, int n, f32x4 v, const float* scale4)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= scale4[i];
    if constexpr (PAIRS) {
        float o[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) o[i] = gate_pair(as_output(v[2 * i], a.y_f16), as_output(v[2 * i + 1], a.y_f16), a.y_f16);
        const long long at = (long long)m * a.ldy + n / 2;
        if (n < a.N) store_out(a.Y, a.y_f16, at, o[0]);
        if (n + 2 < a.N) store_out(a.Y, a.y_f16, at + 1, o[1]);
        return;
    }
    const long long at = (long long)m * a.ldy + n;
    if (n + 3 < a.N && (a.vector_out)) {
        if (a.y_f16) {
            __half h[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = __float2half(settled(v[i]));
            *reinterpret_cast<uint2*>(static_cast<__half*>(a.Y) + at) = *reinterpret_cast<const uint2*>(h);
        } else {
            *reinterpret_cast<f32x4*>(static_cast<float*>(a.Y) + at) = v;
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (n + i < a.N) store_out(a.Y, a.y_f16, at + i, v[i]);
}

enum { kPlain = 0, kPairs = 1, kTwoWeights = 2 };

// The product of one output: from the index stream where the matrix cores' sum is not finite.
__device__ __forceinline__ float exact_output(const KernelArgs& a, const WeightPtrs& w, int m, int n) { return walk_column(w, a.T, a.tile_rows, n, callers_x(a, m)); }

// Bound by the matrix cores: 1024 x 4096 -> 11008 in fp16 is 92 GFLOP dense, 80 us = 1155 TFLOP/s (8192 x 2048 -> 11008:
// 1230; a library fp16 product of that size 1090, the matrix instruction alone on trivial operands 2000).  What it took, at
// 1024 x 12288 -> 8192: sums kept in their registers (fences around the barrier) 190 -> 161 us; operands made between the
// products instead of in front of them 161 -> 152.  The same product by adding activation rows up, one vector lane per row
// and non-zero, took 457 us at 80 % zeros (1024 x 4096 -> 11008), 133 at 99 %; this one takes 80 at any.
//
// Output tiles of (WM * FM * 16) activation rows x (WN * FN * 16) columns, one per workgroup of WM x WN waves; a wave owns
// FM * 16 rows x FN * 16 columns.  PARTS: 1 for fp16 activations, 3 for fp32 ones in bf16 parts (all three are multiplied by
// the same operands while a unit's codes are at hand).  STAGES of activations in LDS.
template <int PARTS, int WM, int WN, int FM, int FN, int STAGES, int MODE>
__global__ __launch_bounds__(WM * WN * 64) void tl_matrix_rows(KernelArgs a)
{
    constexpr int W = WM * WN, TM = WM * FM * 16, TN = WN * FN * 16;
    constexpr int XB = TM * kStageRowBytes;                       // bytes of a stage of activations
    constexpr int CB = (TN / 16) * TL_CODE_UNIT_BYTES;            // bytes of a unit of codes
    constexpr int XL = TM / 8 / W;                                // activation loads of a wave per stage (8 rows each)
    constexpr int CL = (TN / 16 + W - 1) / W;                     // code loads of a wave per unit
    static_assert(TM % (8 * W) == 0, "every wave loads the same number of row groups");
    extern __shared__ __align__(16) unsigned char lds[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN;

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
    uint32_t piece[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int r = (i * W + wave) * 8 + lane_row;
        xrow[i] = (uint32_t)(min(m0 + r, a.M - 1) - m0) * (uint32_t)(a.image_ld * 2);
        piece[i] = (uint32_t)piece_place(r, lane & 7) * 16;
    }
    const unsigned char* image = static_cast<const unsigned char*>(a.image) + (long long)m0 * a.image_ld * 2;
    const long long unit_stride = TL_CODE_UNIT_BYTES;

    const int stages_k = (a.K + kStageRows - 1) / kStageRows;     // stages of K that hold anything
    const int all_units = a.planes * a.units;
    // stages of unit u: the last one of the only plane may be shorter
    const int last_stages = a.planes == 1 ? stages_k - (a.units - 1) * kUnitStages : kUnitStages;
    const int total = PARTS * ((all_units - 1) * kUnitStages + last_stages);

    // load side: where the next activations to ask for lie, and the buffer they go to
    int lu = 0, lk = 0, lp = 0, lj = 0, issued = 0;               // unit, unit within its plane, part, stage
    uint32_t lbuf = lds0 + (uint32_t)wave * 1024;
    auto issue_x = [&]() {
        const uint32_t k_bytes = (uint32_t)(lk * TL_CODE_UNIT_ROWS + lj * kStageRows) * 2;
        const unsigned char* src = image + (PARTS > 1 ? (long long)lp * a.image_plane * 2 : 0ll);
#pragma unroll
        for (int i = 0; i < XL; ++i) load_to_lds(lbuf + i * W * 1024, src, xrow[i] + min(k_bytes + piece[i], limit));
        ++issued;
        lbuf = lbuf + XB >= lds0 + STAGES * XB ? lbuf - (STAGES - 1) * XB : lbuf + XB;
        if (++lj == (lu == all_units - 1 ? last_stages : kUnitStages)) {
            lj = 0;
            if (++lp == PARTS) {
                lp = 0;
                ++lu;
                if (++lk == a.units) lk = 0;
            }
        }
    };
    const unsigned char* code_src[CL];                            // (wave-uniform)
    uint32_t code_to[CL];
    int code_units[CL];                                           // units that the block's weight has
#pragma unroll
    for (int i = 0; i < CL; ++i) {
        const int c = min(i * W + wave, TN / 16 - 1);             // column block of the tile
        const int owner = c / FN, f = c % FN;                     // its wave column and fragment
        const Codes& w = (MODE == kTwoWeights && f >= FN / 2) ? a.c1 : a.c0;
        const int nb = MODE == kTwoWeights ? nb0 + owner * (FN / 2) + f % (FN / 2) : nb0 + c;
        code_units[i] = w.planes * a.units;
        code_src[i] = w.base + min(nb, a.NB - 1) * (code_units[i] * unit_stride);
        code_to[i] = lds0 + STAGES * XB + c * TL_CODE_UNIT_BYTES;
    }
    auto issue_codes = [&](int u) {
#pragma unroll
        for (int i = 0; i < CL; ++i) {
            const unsigned char* src = code_src[i] + u * unit_stride;
            if (MODE == kTwoWeights && u >= code_units[i]) src = kNoCodes;   // (the other weight has more planes)
            load_to_lds(code_to[i] + (u & 1) * CB, src, (uint32_t)lane * 16);
        }
    };

    // ---- what it reads ----
    const int g = lane >> 4, r16 = lane & 15;
    const uint32_t x_read = (uint32_t)((wm * FM * 16 + r16) * kStageRowBytes);
    const uint32_t swz = (uint32_t)(piece_place(r16, g) * 16);    // rows of a wave's fragments differ by multiples of 16: same place
    constexpr bool F32 = PARTS > 1;
    f32x4 acc[FN][FM], low[F32 ? FN : 1][F32 ? FM : 1];           // low: the sums of the parts after the first
#pragma unroll
    for (int f = 0; f < FN; ++f)
#pragma unroll
        for (int m = 0; m < FM; ++m) acc[f][m] = low[F32 ? f : 0][F32 ? m : 0] = f32x4{0.f, 0.f, 0.f, 0.f};

    // A stage is worked on in two halves of 32 rows of K, each half's activations read from LDS while the other half is
    // multiplied, across stages too: the barrier that says that the next stage has come stands between the halves.
    issue_codes(0);
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
        if (issued < total) issue_x();
    u32x4 codes[FN], x0[FM], x1[FM];
    uint32_t xbuf = x_read;                                       // this stage's activations
    auto read_half = [&](u32x4* x, uint32_t half) {
#pragma unroll
        for (int m = 0; m < FM; ++m) x[m] = *reinterpret_cast<const u32x4*>(lds + xbuf + (swz ^ half) + m * 16 * kStageRowBytes);
    };
    auto read_codes = [&](u32x4* c, int u) {
        const unsigned char* cs = lds + STAGES * XB + (u & 1) * CB + (wn * FN) * TL_CODE_UNIT_BYTES + lane * 16;
#pragma unroll
        for (int f = 0; f < FN; ++f) c[f] = *reinterpret_cast<const u32x4*>(cs + f * TL_CODE_UNIT_BYTES);
    };
    if (total >= STAGES) wait_loads_and_barrier<(STAGES - 1) * XL>();
    else wait_loads_and_barrier<0>();
    read_codes(codes, 0);
    read_half(x0, 0);
    int t = 0;
    u32x4 w = weight_operand<0>(codes[0]);                        // operand of the next products
    // The products of one half with the operands of all FN column fragments.  The operand of the next fragment -- at the
    // end, of the next half's first -- is made between a fragment's products: a product keeps the matrix core busy for 16
    // clocks, and the wave can issue three vector instructions meanwhile.
    auto products = [&](auto step_tag, auto first_tag, const u32x4* x, auto next) {
        constexpr int S = decltype(step_tag)::value;
#pragma unroll
        for (int f = 0; f < FN; ++f) {
            const u32x4 now = w;
#pragma unroll
            for (int m = 0; m < FM; ++m) {
                f32x4& sum = decltype(first_tag)::value ? acc[f][m] : low[F32 ? f : 0][F32 ? m : 0];
                sum = matrix_step<F32>(now, x[m], sum);
            }
            if (f + 1 < FN) w = weight_operand<S>(codes[f + 1 < FN ? f + 1 : 0]);
            else w = next();
#pragma unroll
            for (int m = 0; m < FM; ++m) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);               // a product,
                __builtin_amdgcn_sched_group_barrier(0x2, FM >= 8 ? 1 : 2, 0);  // then vector instructions
            }
        }
    };
    // Stage J of part p of unit u (first: whether p is the leading part).  STEADY: stages t + 1 .. t + STAGES exist, so
    // nothing needs to be asked.
    auto turn = [&](auto j_tag, auto steady_tag, auto first_tag, int u, int p, bool part_ends) {
        const bool unit_ends = part_ends && p == PARTS - 1;
        constexpr int J = decltype(j_tag)::value;
        constexpr bool STEADY = decltype(steady_tag)::value;
        read_half(x1, 64);
        if (J == 0 && decltype(first_tag)::value && u + 1 < all_units) issue_codes(u + 1);
        __builtin_amdgcn_sched_barrier(0);
        products(std::integral_constant<int, 2 * J>{}, first_tag, x0, [&]() { return weight_operand<2 * J + 1>(codes[0]); });
        // (without the fences the scheduler moves these products behind the barrier and pays for it with copies of the sums)
        __builtin_amdgcn_sched_barrier(0);
        u32x4 fresh[FN];
        if (STEADY || t + 1 < total) {
            // after this barrier every wave has read all of stage t: its buffer takes the stage STAGES further on
            if (STEADY || total - t >= STAGES) wait_loads_and_barrier<(STAGES - 2) * XL>();
            else wait_loads_and_barrier<0>();
            if (STEADY || issued < total) issue_x();
            xbuf = xbuf + XB >= STAGES * XB ? xbuf - (STAGES - 1) * XB : xbuf + XB;
            read_half(x0, 0);
            if (unit_ends) read_codes(fresh, u + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        constexpr int AFTER = J == kUnitStages - 1 ? 0 : 2 * J + 2;   // (of the unit's next stage; a part that ends starts it again)
        products(std::integral_constant<int, 2 * J + 1>{}, first_tag, x1, [&]() {
            if (unit_ends) {
#pragma unroll
                for (int f = 0; f < FN; ++f) codes[f] = fresh[f];
                return weight_operand<0>(codes[0]);
            }
            return AFTER != 0 && part_ends ? weight_operand<0>(codes[0]) : weight_operand<AFTER>(codes[0]);
        });
        __builtin_amdgcn_sched_barrier(0);
        ++t;
    };
    constexpr std::integral_constant<int, 0> s0t; constexpr std::integral_constant<int, 1> s1t;
    constexpr std::integral_constant<int, 2> s2t; constexpr std::integral_constant<int, 3> s3t;
    auto one_part = [&](auto steady_tag, auto first_tag, int u, int p, int stages) {
        turn(s0t, steady_tag, first_tag, u, p, stages == 1);
        if (stages > 1) turn(s1t, steady_tag, first_tag, u, p, stages == 2);
        if (stages > 2) turn(s2t, steady_tag, first_tag, u, p, stages == 3);
        if (stages > 3) turn(s3t, steady_tag, first_tag, u, p, true);
    };
    auto one_unit = [&](auto steady_tag, int u, int stages) {
        one_part(steady_tag, std::true_type{}, u, 0, stages);
        if constexpr (F32)
            for (int p = 1; p < PARTS; ++p) one_part(steady_tag, std::false_type{}, u, p, stages);
    };
    int u = 0;
    for (; (u + 1) * PARTS * kUnitStages + STAGES <= total; ++u) one_unit(std::true_type{}, u, kUnitStages);
    for (; u < all_units; ++u) one_unit(std::false_type{}, u, u == all_units - 1 ? last_stages : kUnitStages);

    // ---- out ----
    // A sum that is not finite is worked out again by the lane that holds it, before anything is stored: the outputs of
    // finite rows keep their bits whatever another row of the tile holds.  (The sums that need it go into a mask that a
    // loop takes bit by bit, so that the walk stands here once and the sums stay in registers.)
    constexpr int OUT_FN = MODE == kTwoWeights ? FN / 2 : FN;
    const int wave_n0 = (nb0 + wn * OUT_FN) * 16, wave_m0 = m0 + wm * FM * 16;
    static_assert(FN * FM * 4 <= 32, "a bit for each of a lane's sums");
    bool fine = true;
    float half = 0.5f;                                            // (the products are with +-2)
#pragma unroll
    for (int f = 0; f < FN; ++f)
#pragma unroll
        for (int m = 0; m < FM; ++m) {
            if constexpr (F32) add_low(acc[f][m], low[f][m]);
            fine = fine && finite4(acc[f][m]);
        }
    if (!fine) {
        uint32_t redo = 0;
#pragma unroll
        for (int e = 0; e < FN * FM * 4; ++e) {
            const int f = e / (FM * 4), m = e / 4 % FM, i = e % 4;
            const bool mine = wave_m0 + m * 16 + r16 < a.M && wave_n0 + f % OUT_FN * 16 + g * 4 + i < a.N;
            redo |= mine && !(fabsf(acc[f][m][i]) < __builtin_huge_valf()) ? 1u << e : 0u;
            acc[f][m][i] *= half;                                 // (twice what is worked out again might overflow)
        }
        half = 1.0f;
        while (redo != 0) {
            const int at = __builtin_ctz(redo), f = at / (FM * 4), m = at / 4 % FM;
            redo &= redo - 1;
            const float v = exact_output(a, f >= OUT_FN ? a.w1 : a.w0, wave_m0 + m * 16 + r16, wave_n0 + f % OUT_FN * 16 + g * 4 + at % 4);
#pragma unroll
            for (int e = 0; e < FN * FM * 4; ++e) acc[e / (FM * 4)][e / 4 % FM][e % 4] = e == at ? v : acc[e / (FM * 4)][e / 4 % FM][e % 4];
        }
    }
#pragma unroll
    for (int f = 0; f < OUT_FN; ++f) {
        const int n = wave_n0 + f * 16 + g * 4;
        float s0[4], s1[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s0[i] = half * (n + i < a.N ? load_scale(a.w0.scale, a.scale_f16, n + i) : 0.f);
            if constexpr (MODE == kTwoWeights) s1[i] = half * (n + i < a.N ? load_scale(a.w1.scale, a.scale_f16, n + i) : 0.f);
        }
#pragma unroll
        for (int m = 0; m < FM; ++m) {
            const int row = wave_m0 + m * 16 + r16;
            f32x4 v = acc[f][m];
            if constexpr (MODE == kTwoWeights) {
                const f32x4 u = acc[f + FN / 2][m];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = silu(v[i] * s0[i]) * (u[i] * s1[i]);
                const float one[4] = {1.f, 1.f, 1.f, 1.f};
                if (row < a.M && n < a.N) store4<false>(a, row, n, v, one);
            } else {
                if (row < a.M && n < a.N) store4<MODE == kPairs>(a, row, n, v, s0);
            }
        }
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
    static std::atomic<bool> raised{false};  // per instantiation; a repeated call is harmless
    if (lds && !raised.load(std::memory_order_relaxed)) {
        if (int rc = raise_lds_limit(kernel, lds)) return rc;
        raised.store(true, std::memory_order_relaxed);
    }
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

template <int PARTS, int WM, int WN, int FM, int FN, int STAGES, int MODE>
int launch_tile(const KernelArgs& a, hipStream_t st)
{
    constexpr int TM = WM * FM * 16, TN = WN * FN * 16, OUT_TN = MODE == kTwoWeights ? TN / 2 : TN;
    constexpr size_t lds = (size_t)STAGES * TM * kStageRowBytes + 2 * (TN / 16) * TL_CODE_UNIT_BYTES;
    static_assert(lds <= 160 * 1024, "the stages fit a compute unit's LDS");
    auto kernel = tl_matrix_rows<PARTS, WM, WN, FM, FN, STAGES, MODE>;
    static std::atomic<bool> raised{false};  // per instantiation; a repeated call is harmless
    if (!raised.load(std::memory_order_relaxed)) {
        if (int rc = raise_lds_limit(kernel, lds)) return rc;
        raised.store(true, std::memory_order_relaxed);
    }
    const int64_t tiles = ceil_div(a.M, TM) * ceil_div(a.N, OUT_TN);
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(WM * WN * 64), lds, st, a);
    return TL_OK;
}

template <int PARTS>
int launch_parts(const KernelArgs& a, bool two_weights, hipStream_t st)
{
    // 128 x 128 tiles, eight waves of 64 x 32: two workgroups share a compute unit in fp16 (114 registers, 80 KB of LDS each), one of
    // which multiplies while the other waits at a barrier or stores (fp32, with its second set of sums, takes 188 registers:
    // one workgroup a unit).  Best of the shapes tried at every size (fp16, us at
    // 1024 x 4096 -> 11008 / 1024 x 4096 -> 4096 / 8192 x 2048 -> 11008): 80 / 34 / 300; four waves of 64 x 64 86 / 40 / 306 or
    // 128 x 32 86 / 40 / 301; 128 x 256 tiles, eight waves of 64 x 64, one workgroup a unit 105 / 52 / 310; 256 x 192, eight of
    // 128 x 48, 84 / 72 / 370.
    if (two_weights) return launch_tile<PARTS, 2, 4, 4, 2, 4, kTwoWeights>(a, st);
    return a.gated ? launch_tile<PARTS, 2, 4, 4, 2, 4, kPairs>(a, st) : launch_tile<PARTS, 2, 4, 4, 2, 4, kPlain>(a, st);
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

int tl::launch_matrix_rows(KernelArgs a, int x_dtype, void* workspace, int64_t workspace_bytes, bool two_weights, hipStream_t st)
{
    a.x_sm = a.x_kmajor ? 1 : a.ldx;
    a.x_sk = a.x_kmajor ? a.ldx : 1;
    const int64_t need = least_image_bytes(a.K, a.M, x_dtype);
    // Without codes, and for K-major rows that need no workspace, the index stream is walked.
    if (!a.c0.base || (two_weights && !a.c1.base) || ((!workspace || workspace_bytes < need) && walk_reads_directly(a)))
        return x_dtype == TL_F16 ? walk_rows<__half>(a, workspace, workspace_bytes, two_weights, st)
                                 : walk_rows<float>(a, workspace, workspace_bytes, two_weights, st);
    const uintptr_t y_align = a.y_f16 ? 8 : 16;
    a.vector_out = a.ldy % 4 == 0 && reinterpret_cast<uintptr_t>(a.Y) % y_align == 0;
    // rows that lie as the kernel reads them are read where they are; any other layout, and fp32, goes through the image
    constexpr int64_t kMostLd = 1 << 24;  // (a lane's byte offset inside the 128 rows of a tile has 32 bits)
    const bool direct = x_dtype == TL_F16 && !a.x_kmajor && a.K % 8 == 0 && a.ldx % 8 == 0 && a.ldx <= kMostLd && reinterpret_cast<uintptr_t>(a.X) % 16 == 0;
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
