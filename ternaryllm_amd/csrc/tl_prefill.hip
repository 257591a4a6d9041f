// What stands around the products of a pass over whole prompts: rotary tables, the rotation of a prompt's keys on their
// way into a cache, and causal softmax attention of many queries on the matrix cores (the reference's
// apply_rotary_pos_emb, Cache.update and eager matmul / softmax / matmul, ternaryLLM_GPU/TernaryLLM/TernaryAttn.py:93-113).
#include <climits>

#include "tl_common.h"
#include "tl_matrix.h"
#include "tl_rope.h"

using namespace tl;

namespace {

// cos and sin of position * theta^(-2i / head_dim), i = d modulo head_dim / 2, one thread per position and i.
template <typename T>
__global__ __launch_bounds__(256) void tl_rope_table_k(const long long* __restrict__ positions, long long first, long long count, int half,
                                                       float theta, T* __restrict__ cos_t, T* __restrict__ sin_t)
{
    const long long e = blockIdx.x * 256ll + threadIdx.x;
    if (e >= count * half) return;
    const long long r = e / half;
    const int i = (int)(e - r * half);
    const float pos = (float)(positions ? positions[r] : first + r);
    const float angle = pos * (1.0f / powf(theta, (float)(2 * i) / (float)(2 * half)));
    float s, c;
    sincosf(angle, &s, &c);
    const long long at = r * 2 * half + i;
    cos_t[at] = cos_t[at + half] = from_f<T>(c);
    sin_t[at] = sin_t[at + half] = from_f<T>(s);
}

template <typename T>
struct __align__(16) Eight {
    T v[8];
};

struct RopeRows {
    const void *k, *v, *cos_t, *sin_t;
    void *k_out, *v_out;                      // v_out null: only the keys
    long long in_b, in_s, table_b;            // elements between batch rows and tokens (heads lie side by side), and tables
    long long out_b, out_s, out_h;
    unsigned seq, heads, eighths, total;      // eighths: groups of eight values in half a head
};

// Keys rotated, values copied, to wherever they are kept.  A thread takes eight values of the lower half of a head and
// their partners: whole 16-byte pieces (two for fp32) in and out.  Bound by memory: each value is read and written once.
template <typename T>
__global__ __launch_bounds__(256) void tl_rope_rows_k(RopeRows a)
{
    const unsigned e = blockIdx.x * 256u + threadIdx.x;
    if (e >= a.total) return;
    const unsigned p = e % a.eighths, t = e / a.eighths, h = t % a.heads, row = t / a.heads, s = row % a.seq, b = row / a.seq;
    const int half = (int)a.eighths * 8, d = (int)p * 8;
    const long long in = b * a.in_b + s * a.in_s + (long long)h * 2 * half + d;
    const long long out = b * a.out_b + s * a.out_s + h * a.out_h + d;
    const long long tab = b * a.table_b + (long long)s * 2 * half + d;
    auto load = [](const void* base, long long at) { return *reinterpret_cast<const Eight<T>*>(static_cast<const T*>(base) + at); };
    auto store = [](void* base, long long at, const Eight<T>& x) { *reinterpret_cast<Eight<T>*>(static_cast<T*>(base) + at) = x; };
    const Eight<T> lo = load(a.k, in), hi = load(a.k, in + half);
    const Eight<T> c0 = load(a.cos_t, tab), c1 = load(a.cos_t, tab + half), s0 = load(a.sin_t, tab), s1 = load(a.sin_t, tab + half);
    Eight<T> v0, v1;
    if (a.v_out) v0 = load(a.v, in), v1 = load(a.v, in + half);
    Eight<T> r0, r1;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        r0.v[i] = from_f<T>(rope_value(to_f(lo.v[i]), to_f(hi.v[i]), to_f(c0.v[i]), to_f(s0.v[i]), -1.0f));
        r1.v[i] = from_f<T>(rope_value(to_f(hi.v[i]), to_f(lo.v[i]), to_f(c1.v[i]), to_f(s1.v[i]), 1.0f));
    }
    store(a.k_out, out, r0);
    store(a.k_out, out + half, r1);
    if (a.v_out) store(a.v_out, out, v0), store(a.v_out, out + half, v1);
}

struct PrefillAttn {
    const __half *q, *k, *v, *cos_t, *sin_t;  // tables null: q is rotated already
    __half* out;
    tl_attention_strides s;
    int heads, group, bh, q_len, kv_len, q_tiles;
    float scale_log2;                          // 1 / sqrt(head_dim) * log2(e)
};

// f over the four lanes with the same number modulo 16, on the vector unit (16 x 512 of 16 heads took 48.4 us with shuffles, 47.6).
template <typename F>
__device__ __forceinline__ float with_other_rows(float v, F f)
{
    const auto near = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = f(__uint_as_float(near[0]), __uint_as_float(near[1]));
    const auto far = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return f(__uint_as_float(far[0]), __uint_as_float(far[1]));
}

// Causal attention: query i of a batch row sees keys 0 .. i + (kv_len - q_len).  A workgroup of four waves owns 64 * QF
// queries of one head, a wave QF fragments of 16; it walks the keys that its queries see in tiles of 64, one pass, with a
// running maximum, sum and weighted sum in fp32 (rescaled when the maximum moves).
// The scores are computed transposed, keys x queries: a lane then holds, for ONE query (lane % 16), four neighbouring keys
// of every fragment -- the maximum and sum take two cross-lane steps a tile, and what it holds is already its operand of
// the second product (values^T x probabilities): the order of the keys within a product step is free, so the values are
// laid out to match (keys 4g .. 4g + 3 of two fragments in one 16-byte piece) and the probabilities cross no lanes.
// LDS: two buffers of a tile of keys (rows, pieces of 16 bytes swizzled so that the 16 lanes of a read hit all banks) and
// of values (turned while they are written, pieces swizzled by d so that both the writes and the reads spread over the
// banks).  The next tile is on its way into registers while this one is worked on; one barrier a tile.
// Workgroup ids go through the (batch row, head) pairs first: those of one head are equal modulo 8 where the pairs divide
// by it, so they share an L2; later query tiles, which see the most keys, come first.
template <int HD, int QF>
__global__ __launch_bounds__(256, 2) void tl_prefill_attn(PrefillAttn a)
{
    constexpr int KT = 64, PIECES = HD / 8, KS = HD / 32, DF = HD / 16, TQ = 64 * QF;
    constexpr int KB = KT * HD * 2, BUF = 2 * KB;                 // bytes of a tile of keys, and of keys + values
    constexpr int KL = KT * PIECES / 256;                         // key pieces of a thread
    constexpr bool kAllTurn = 16 * PIECES == 256;                 // every thread turns one piece of four keys' values
    __shared__ __align__(16) unsigned char lds[2 * BUF];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, r16 = lane & 15;
    const int bh = (int)blockIdx.x % a.bh, qt = a.q_tiles - 1 - (int)blockIdx.x / a.bh;
    const int b = bh / a.heads, h = bh % a.heads;
    const int q0 = qt * TQ, offset = a.kv_len - a.q_len;
    const int wq0 = q0 + wave * 16 * QF;                          // the wave's first query
    const __half* kp = a.k + b * a.s.k_batch + (h / a.group) * a.s.k_head;
    const __half* vp = a.v + b * a.s.v_batch + (h / a.group) * a.s.v_head;
    const int tiles = (min(q0 + TQ, a.q_len) + offset + KT - 1) / KT;

    // ---- tiles on their way ----
    auto key_place = [](int key, int p) { return HD == 128 ? p ^ (key & 15) : p ^ ((key >> 1) & 7); };
    const int vc = tid % PIECES, vg = tid / PIECES;               // this thread's piece of d and its four keys, 4 * vg ...
    u32x4 kreg[KL], vreg[4];
    auto fetch = [&](int t) {
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            const int id = i * 256 + tid, key = min(t * KT + id / PIECES, a.kv_len - 1);
            kreg[i] = *reinterpret_cast<const u32x4*>(kp + key * a.s.k_seq + id % PIECES * 8);
        }
        if (kAllTurn || tid < 16 * PIECES) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int key = t * KT + vg * 4 + j;
                // (a key past the end weighs 0, which would make NaN of a value that is not finite)
                vreg[j] = key < a.kv_len ? *reinterpret_cast<const u32x4*>(vp + key * a.s.v_seq + vc * 8) : u32x4{0u, 0u, 0u, 0u};
            }
        }
    };
    auto value_place = [](int d, int piece) { return d * KT * 2 + ((piece ^ (d >> 3) ^ d) & 7) * 16; };
    auto put = [&](int buf) {
        unsigned char* kd = lds + buf * BUF;
        unsigned char* vd = kd + KB;
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            const int id = i * 256 + tid, key = id / PIECES;
            *reinterpret_cast<u32x4*>(kd + key * HD * 2 + key_place(key, id % PIECES) * 16) = kreg[i];
        }
        if (kAllTurn || tid < 16 * PIECES) {
            // four-key group vg = 8 * step + 4 * half + g: piece (step, g), its lower or upper 8 bytes
            const int piece = (vg >> 3) * 4 + (vg & 3), at = ((vg >> 2) & 1) * 8;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t sel = i & 1 ? 0x07060302u : 0x05040100u;
                uint2 four;
                four.x = __builtin_amdgcn_perm(vreg[1][i >> 1], vreg[0][i >> 1], sel);
                four.y = __builtin_amdgcn_perm(vreg[3][i >> 1], vreg[2][i >> 1], sel);
                *reinterpret_cast<uint2*>(vd + value_place(vc * 8 + i, piece) + at) = four;
            }
        }
    };
    fetch(0);

    // ---- the wave's queries ----
    u32x4 qx[QF][KS];
#pragma unroll
    for (int f = 0; f < QF; ++f) {
        const int qi = min(wq0 + f * 16 + r16, a.q_len - 1);
        const __half* row = a.q + b * a.s.q_batch + qi * a.s.q_seq + h * a.s.q_head + g * 8;
#pragma unroll
        for (int s = 0; s < KS; ++s) qx[f][s] = *reinterpret_cast<const u32x4*>(row + s * 32);
        if (a.cos_t) {
            const long long tab = b * a.s.table_batch + (long long)qi * HD + g * 8;
#pragma unroll
            for (int s = 0; s < KS / 2; ++s) {                    // d and its partner half a head away are in one lane
                auto eight = [&](const __half* t, int at) { return *reinterpret_cast<const Eight<__half>*>(t + tab + at * 32); };
                const Eight<__half> c0 = eight(a.cos_t, s), c1 = eight(a.cos_t, s + KS / 2), s0 = eight(a.sin_t, s), s1 = eight(a.sin_t, s + KS / 2);
                Eight<__half> lo = __builtin_bit_cast(Eight<__half>, qx[f][s]), hi = __builtin_bit_cast(Eight<__half>, qx[f][s + KS / 2]);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float x = to_f(lo.v[i]), y = to_f(hi.v[i]);
                    lo.v[i] = from_f<__half>(rope_value(x, y, to_f(c0.v[i]), to_f(s0.v[i]), -1.0f));
                    hi.v[i] = from_f<__half>(rope_value(y, x, to_f(c1.v[i]), to_f(s1.v[i]), 1.0f));
                }
                qx[f][s] = __builtin_bit_cast(u32x4, lo);
                qx[f][s + KS / 2] = __builtin_bit_cast(u32x4, hi);
            }
        }
    }
    f32x4 o[DF][QF];
    float top[QF], sum[QF];
#pragma unroll
    for (int f = 0; f < QF; ++f) {
        top[f] = -__builtin_huge_valf();
        sum[f] = 0.f;
#pragma unroll
        for (int d = 0; d < DF; ++d) o[d][f] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    put(0);
    __syncthreads();
    // The queries are here before the loop: waited for inside it, at the first products of every turn, the next tile's loads are too (16 x 512 tokens,
    // 16 heads of 128: 44.6 us, 42.5 so).
#pragma unroll
    for (int f = 0; f < QF; ++f)
#pragma unroll
        for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qx[f][s]));

    for (int t = 0; t < tiles; ++t) {
        if (t + 1 < tiles) fetch(t + 1);
        const unsigned char* ks = lds + (t & 1) * BUF;
        const unsigned char* vs = ks + KB;
        if (t * KT <= wq0 + 16 * QF - 1 + offset) {               // (a tile of which the wave's queries see nothing is skipped)
            f32x4 sc[4][QF];
#pragma unroll
            for (int i = 0; i < 4 * KS; ++i) {
                // heads of 128: the four steps of keys in turn, so that a product waits for its sum's last one three products before; of 64, whose
                // sums have two, one step after the other (2 x 4096 tokens, 16 heads: 123.7 us in turn, 108.3 so; of 128 183.5 / 184.7)
                const int s = HD == 128 ? i / 4 : i % KS, n = HD == 128 ? i % 4 : i / KS, key = n * 16 + r16;
                const u32x4 kx = *reinterpret_cast<const u32x4*>(ks + key * HD * 2 + key_place(key, s * 4 + g) * 16);
#pragma unroll
                for (int f = 0; f < QF; ++f) sc[n][f] = matrix_step<false>(kx, qx[f][s], s == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sc[n][f]);
            }
            if (t * KT + KT - 1 > wq0 + offset) {                 // some query of the wave does not see all of the tile
#pragma unroll
                for (int f = 0; f < QF; ++f) {
                    const int last = wq0 + f * 16 + r16 + offset - t * KT - g * 4;   // last key seen, from this lane's first
#pragma unroll
                    for (int n = 0; n < 4; ++n)
#pragma unroll
                        for (int i = 0; i < 4; ++i) sc[n][f][i] = n * 16 + i <= last ? sc[n][f][i] : -__builtin_huge_valf();
                }
            }
            u32x4 px[QF][2];
#pragma unroll
            for (int f = 0; f < QF; ++f) {
                float most = sc[0][f][0];
#pragma unroll
                for (int n = 0; n < 4; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i) most = fmaxf(most, sc[n][f][i]);
                most = with_other_rows(most, [](float x, float y) { return fmaxf(x, y); });
                const float now = fmaxf(top[f], most);
                const float base = now == -__builtin_huge_valf() ? 0.f : now * a.scale_log2;   // (nothing but -inf so far)
                const float shrink = __builtin_amdgcn_exp2f(fmaf(top[f], a.scale_log2, -base));
                top[f] = now;
                float part = 0.f;
#pragma unroll
                for (int n = 0; n < 4; ++n) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        typedef float float2v __attribute__((ext_vector_type(2)));
                        typedef _Float16 half2v __attribute__((ext_vector_type(2)));
                        float2v e;
#pragma unroll
                        for (int j = 0; j < 2; ++j) e[j] = __builtin_amdgcn_exp2f(fmaf(sc[n][f][2 * i + j], a.scale_log2, -base));
                        part += e[0];
                        part += e[1];
                        px[f][n >> 1][(n & 1) * 2 + i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(e, half2v));
                    }
                }
                sum[f] = fmaf(sum[f], shrink, part);
                if (__builtin_amdgcn_ballot_w64(shrink != 1.0f) != 0) {
#pragma unroll
                    for (int d = 0; d < DF; ++d)
#pragma unroll
                        for (int i = 0; i < 4; ++i) o[d][f][i] *= shrink;
                }
            }
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int d = 0; d < DF; ++d) {
                    const u32x4 vx = *reinterpret_cast<const u32x4*>(vs + value_place(d * 16 + r16, s * 4 + g));
#pragma unroll
                    for (int f = 0; f < QF; ++f) o[d][f] = matrix_step<false>(vx, px[f][s], o[d][f]);
                }
        }
        if (t + 1 < tiles) {
            put((t + 1) & 1);                                     // (read last before the barrier of the turn before)
            __syncthreads();
        }
    }
#pragma unroll
    for (int f = 0; f < QF; ++f) {
        const int qi = wq0 + f * 16 + r16;
        const float all = with_other_rows(sum[f], [](float x, float y) { return x + y; });
        if (qi >= a.q_len) continue;
        const float inv = 1.0f / all;
        __half* row = a.out + ((long long)b * a.q_len + qi) * a.heads * HD + h * HD + g * 4;
#pragma unroll
        for (int d = 0; d < DF; ++d) {
            __half r[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) r[i] = __float2half(o[d][f][i] * inv);
            *reinterpret_cast<uint2*>(row + d * 16) = *reinterpret_cast<const uint2*>(r);
        }
    }
}

bool pieces(const void* p, std::initializer_list<int64_t> strides, int dtype)
{
    const int64_t es = dtype == TL_F16 ? 2 : 4;
    if (reinterpret_cast<uintptr_t>(p) % 16) return false;
    for (int64_t s : strides)
        if (s * es % 16) return false;
    return true;
}

}  // namespace

extern "C" int tl_rope_table(const int64_t* positions, int64_t first, int64_t count, int head_dim, float theta, int dtype, void* cos_table,
                             void* sin_table, void* stream)
{
    if (int rc = check_dtype(dtype, "table")) return rc;
    if (!cos_table || !sin_table) return fail(TL_ERR_ARG, "device pointer is null");
    if (head_dim <= 0 || head_dim % 2 || count <= 0 || count > (1ll << 30)) return fail(TL_ERR_SHAPE, "count must be positive, head_dim=%d positive and even", head_dim);
    const int64_t groups = ceil_div(count * (head_dim / 2), 256);
    if (groups > INT32_MAX) return fail(TL_ERR_SHAPE, "%lld positions are more than one launch takes", (long long)count);
    const long long* pos = reinterpret_cast<const long long*>(positions);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (dtype == TL_F16)
        hipLaunchKernelGGL(tl_rope_table_k<__half>, dim3((unsigned)groups), dim3(256), 0, st, pos, (long long)first, (long long)count, head_dim / 2, theta,
                           static_cast<__half*>(cos_table), static_cast<__half*>(sin_table));
    else
        hipLaunchKernelGGL(tl_rope_table_k<float>, dim3((unsigned)groups), dim3(256), 0, st, pos, (long long)first, (long long)count, head_dim / 2, theta,
                           static_cast<float*>(cos_table), static_cast<float*>(sin_table));
    return finish_launch();
}

extern "C" int tl_rope_rows(const void* k, const void* v, int dtype, int64_t batch, int64_t seq, int heads, int head_dim, int64_t in_batch,
                            int64_t in_seq, const void* cos_table, const void* sin_table, int64_t table_batch, void* k_out, void* v_out,
                            int64_t out_batch, int64_t out_seq, int64_t out_head, void* stream)
{
    if (int rc = check_dtype(dtype, "k")) return rc;
    if (!k || !cos_table || !sin_table || !k_out || (v_out && !v)) return fail(TL_ERR_ARG, "device pointer is null");
    if (batch <= 0 || seq <= 0 || heads <= 0 || head_dim <= 0 || batch > (1 << 24) || seq > (1 << 24)) return fail(TL_ERR_SHAPE, "batch, seq, heads and head_dim must be positive");
    if (head_dim % 16) return fail(TL_ERR_UNSUPPORTED, "head_dim=%d (multiples of 16 supported)", head_dim);
    if (!pieces(k, {in_batch, in_seq}, dtype) || !pieces(v, {}, dtype) || !pieces(k_out, {out_batch, out_seq, out_head}, dtype) || !pieces(v_out, {}, dtype) ||
        !pieces(cos_table, {table_batch}, dtype) || !pieces(sin_table, {}, dtype))
        return fail(TL_ERR_ALIGN, "addresses and strides must be whole 16-byte pieces");
    const int64_t total = batch * seq * heads * (head_dim / 16);
    if (total > INT32_MAX) return fail(TL_ERR_SHAPE, "%lld tokens are more than one launch takes", (long long)(batch * seq));
    RopeRows a{k, v, cos_table, sin_table, k_out, v_out, in_batch, in_seq, table_batch, out_batch, out_seq, out_head,
               (unsigned)seq, (unsigned)heads, (unsigned)head_dim / 16, (unsigned)total};
    const dim3 grid((unsigned)ceil_div(total, 256));
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (dtype == TL_F16) hipLaunchKernelGGL(tl_rope_rows_k<__half>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(tl_rope_rows_k<float>, grid, dim3(256), 0, st, a);
    return finish_launch();
}

extern "C" int tl_prefill_attention(const void* q, const void* k, const void* v, const void* cos_table, const void* sin_table, int dtype,
                                    int64_t batch, int heads, int kv_heads, int head_dim, int64_t q_len, int64_t kv_len,
                                    const tl_attention_strides* strides, void* out, void* stream)
{
    if (int rc = check_dtype(dtype, "q")) return rc;
    if (!q || !k || !v || !strides || !out || !cos_table != !sin_table) return fail(TL_ERR_ARG, "null pointer");
    if (dtype != TL_F16 || (head_dim != 64 && head_dim != 128)) return fail(TL_ERR_UNSUPPORTED, "fp16 heads of 64 or 128 values only");
    if (batch <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads) return fail(TL_ERR_SHAPE, "batch and heads must be positive, kv_heads a divisor of heads");
    if (q_len <= 0 || kv_len < q_len || kv_len > (1 << 30)) return fail(TL_ERR_SHAPE, "q_len=%lld, kv_len=%lld: every query needs a key", (long long)q_len, (long long)kv_len);
    const tl_attention_strides& s = *strides;
    if (!pieces(q, {s.q_batch, s.q_seq, s.q_head}, dtype) || !pieces(k, {s.k_batch, s.k_seq, s.k_head}, dtype) || !pieces(v, {s.v_batch, s.v_seq, s.v_head}, dtype) ||
        !pieces(cos_table, {s.table_batch}, dtype) || !pieces(sin_table, {}, dtype) || !pieces(out, {}, dtype))
        return fail(TL_ERR_ALIGN, "addresses and strides must be whole 16-byte pieces");
    PrefillAttn a{static_cast<const __half*>(q), static_cast<const __half*>(k), static_cast<const __half*>(v), static_cast<const __half*>(cos_table),
                  static_cast<const __half*>(sin_table), static_cast<__half*>(out), s, heads, heads / kv_heads, 0, (int)q_len, (int)kv_len, 0,
                  1.4426950408889634f / sqrtf((float)head_dim)};
    const int64_t pairs = batch * heads;
    // 128 queries to a workgroup halve what is read from LDS per product, and pay once there are enough of them for every compute
    // unit to have two at a time until the end (us with 128 / 64, workgroups of 128: 16 x 512 of 16 heads, 1024: 47.6 / 59.7;
    // 1 x 2048 of 32, 512: 81.7 / 78.9; 8 x 128 of 32, 256: 10.0 / 8.9; 4 x 1000 of 8, 256: 40.5 / 30.5).
    // (A few queries over a long past leave most of a workgroup idle and a head's keys in series; the attention block of 32 heads,
    // one query, past of 2048 / 8192 keys: 125 / 334 us, with the torch operator in its place 220 / 483.)
    const bool tall = pairs * ceil_div(q_len, 128) >= 3 * compute_units();
    const int64_t q_tiles = ceil_div(q_len, tall ? 128 : 64);
    if (pairs * q_tiles > INT32_MAX) return fail(TL_ERR_SHAPE, "%lld queries are more than one launch takes", (long long)(batch * q_len));
    a.bh = (int)pairs;
    a.q_tiles = (int)q_tiles;
    auto kernel = head_dim == 128 ? (tall ? tl_prefill_attn<128, 2> : tl_prefill_attn<128, 1>) : (tall ? tl_prefill_attn<64, 2> : tl_prefill_attn<64, 1>);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(pairs * q_tiles)), dim3(256), 0, static_cast<hipStream_t>(stream), a);
    return finish_launch();
}
