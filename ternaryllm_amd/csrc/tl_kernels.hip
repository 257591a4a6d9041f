// Entry points of libternary_spmm's device code (include/ternary_spmm.h): the checks in front of every launch, the
// choice between the kernels for few rows (tl_small_m.hip) and the matrix-core kernel (tl_matrix.hip), the tuning
// knobs, the scratch of the entry point that allocates nothing, and the measurement helpers.
#include "tl_device.h"

using namespace tl;

namespace tl {
// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
int check_header(const tl_layout_header* h)
{
    if (!h) return fail(TL_ERR_ARG, "layout header is null");
    if (h->magic != TL_LAYOUT_MAGIC || (h->version != TL_LAYOUT_VERSION && h->version != TL_LAYOUT_VERSION_NO_CODES)) return fail(TL_ERR_FORMAT, "bad layout magic/version");
    if (h->tile_rows == 0 || h->tile_rows > (uint32_t)kMaxTileRows || h->n_tiles != (uint32_t)ceil_div(h->inners, h->tile_rows) ||
        h->n_blocks != (uint32_t)ceil_div(h->columns, TL_BLOCK_COLUMNS) || h->max_chunk_dwords < TL_BLOCK_COLUMNS ||
        (int64_t)h->max_chunk_dwords * 4 > kMaxChunkBytes + 16)
        return fail(TL_ERR_FORMAT, "layout header geometry is inconsistent");
    const uint64_t code_bytes = (uint64_t)h->n_blocks * h->code_planes * h->code_units * TL_CODE_UNIT_BYTES;
    const bool codes = h->version == TL_LAYOUT_VERSION;
    if (codes ? h->code_planes == 0 || h->code_planes > 255 || h->code_units != (uint32_t)ceil_div(h->inners, TL_CODE_UNIT_ROWS) || h->off_codes < 256 ||
                    h->off_codes % 16 || h->off_codes > h->total_bytes || h->total_bytes - h->off_codes < code_bytes
              : h->code_planes != 0 || h->code_units != 0 || h->off_codes != 0)
        return fail(TL_ERR_FORMAT, "layout header: the code section is inconsistent");
    return TL_OK;
}

int check_dtype(int d, const char* what)
{
    if (d != TL_F32 && d != TL_F16) return fail(TL_ERR_DTYPE, "%s dtype code %d unknown", what, d);
    return TL_OK;
}

const char* const kKnobNames[kKnobCount] = {"TL_SMALL_LDS", "TL_TILE_GROUP", "TL_QUAD_SHARE", "TL_LW", "TL_SPMV_SHARE", "TL_SPMV_WIDE",
                                            "TL_SMALL_MT", "TL_SPMV_DIRECT", "TL_BLOCK_SET", "TL_OCTET", "TL_QUAD_WIDE", "TL_SPMV_TILES", "TL_RES16",
                                            "TL_FEW"};
struct Knobs {
    bool set[kKnobCount];
    int value[kKnobCount];
};
std::atomic<const Knobs*> g_knobs{nullptr};

const Knobs* read_knobs()
{
    Knobs* k = new Knobs;
    for (int i = 0; i < kKnobCount; ++i) {
        const char* v = std::getenv(kKnobNames[i]);
        k->set[i] = v && *v;
        k->value[i] = k->set[i] ? std::atoi(v) : 0;
    }
    return k;
}

int knob(Knob which, int fallback)
{
    const Knobs* k = g_knobs.load(std::memory_order_acquire);
    if (!k) {
        const Knobs* fresh = read_knobs();
        if (g_knobs.compare_exchange_strong(k, fresh, std::memory_order_acq_rel)) k = fresh;
        else delete fresh;  // another thread was first; k now holds its table
    }
    return k->set[which] ? k->value[which] : fallback;
}

// Compute units of the current device, asked once per device.  Launch shapes are sized by it.
int compute_units()
{
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return kMaxComputeUnits;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = kMaxComputeUnits;
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

WeightPtrs weight_ptrs(const tl_layout_header* h, const void* blob_dev, const void* scale)
{
    const unsigned char* b = static_cast<const unsigned char*>(blob_dev);
    WeightPtrs w;
    w.chunkstart = reinterpret_cast<const uint32_t*>(b + h->off_chunkstart);
    w.stream = reinterpret_cast<const uint32_t*>(b + h->off_stream);
    w.scale = scale;
    return w;
}


int finish_launch()
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(TL_ERR_LAUNCH, "kernel launch failed: %s", hipGetErrorString(e));
    return TL_OK;
}

int check_io(const void* blob_dev, const void* X, void* Y, int x_dtype, int x_layout, int64_t ldx, int64_t M, int y_dtype,
             int64_t ldy, const void* scale, int scale_dtype, const tl_layout_header* h)
{
    if (!blob_dev || !X || !Y) return fail(TL_ERR_ARG, "device pointer is null");
    if (reinterpret_cast<uintptr_t>(blob_dev) % 256) return fail(TL_ERR_ALIGN, "weight blob must be 256-byte aligned");
    if (int rc = check_dtype(x_dtype, "x")) return rc;
    if (int rc = check_dtype(y_dtype, "y")) return rc;
    if (scale)
        if (int rc = check_dtype(scale_dtype, "scale")) return rc;
    if (x_layout != TL_X_ROW_MAJOR && x_layout != TL_X_K_MAJOR) return fail(TL_ERR_ARG, "x_layout=%d unknown", x_layout);
    if (M <= 0 || M > (1 << 30)) return fail(TL_ERR_SHAPE, "M=%lld out of range", (long long)M);
    const int64_t min_ldx = x_layout == TL_X_ROW_MAJOR ? h->inners : M;
    if (ldx < min_ldx) return fail(TL_ERR_SHAPE, "ldx=%lld smaller than the %lld elements of a row", (long long)ldx, (long long)min_ldx);
    if (ldy < (int64_t)h->columns) return fail(TL_ERR_SHAPE, "ldy=%lld smaller than N=%u", (long long)ldy, h->columns);
    return TL_OK;
}

}  // namespace tl

extern "C" int tl_reload_options(void)
{
    const Knobs* old = g_knobs.exchange(read_knobs(), std::memory_order_acq_rel);
    (void)old;  // a launch on another thread may still be reading it: the few bytes are left alone
    return TL_OK;
}

extern "C" int tl_spmm_workspace(const tl_layout_header* header, int64_t M, int x_dtype, int x_layout, int64_t* workspace_bytes)
{
    if (int rc = check_header(header)) return rc;
    if (int rc = check_dtype(x_dtype, "x")) return rc;
    if (!workspace_bytes) return fail(TL_ERR_ARG, "workspace_bytes is null");
    if (M <= 0) return fail(TL_ERR_SHAPE, "M=%lld must be positive", (long long)M);
    if (M <= kSmallMaxM) {  // room for the aligned K-major image of the activations (more than 4 rows)
        (void)x_layout;  // K-major activations need it too when they are not aligned vectors
        *workspace_bytes = small_kmajor_bytes(header, M, x_dtype);
        return TL_OK;
    }
    // the image of all rows, in whole 256 of them, so that a caller's buffer serves nearby row counts too, and the bytes
    // by which a buffer of any alignment may have to be moved
    *workspace_bytes = round_up(M, 256) * image_row_bytes(header->inners, x_dtype) + 256;
    return TL_OK;
}

namespace {
// Whether a product is tl_few.hip's.  It costs the bytes of the codes (two bits an entry) whatever the weight; the kernels
// that walk the index stream cost its bytes, and some of them start from a K-major image that a K-major caller has at hand.
// us, walk / codes, 4096 -> 11008 at 66 % and at 95 % zeros:
//   one row         fp16 8.0 / 5.9, 5.4 / 6.1;  fp32 8.2 / 11.0, 5.4 / 11.1: never.  One row's gated and fused products are the
//                   walk's and equal the plain one bit for bit; that costs the fp16 rows of dense weights.
//   8 rows          fp16 20.1 / 6.7, 14.3 / 6.7;  fp32 24.3 / 13.5, 17.2 / 13.5: always
//   16 rows         fp16 25.7 / 7.1, 14.8 / 7.1: always;  fp32 24.7 / 13.7, 13.1 / 13.7 (2048 -> 2048 at 95 % 9.8 / 5.0): by bytes
//                   at such widths
//   48 rows         fp16 68.9 / 15.5, 42.4 / 15.5;  fp32 100 / 41, 75 / 41: always
//   K-major         3 and 4 rows, which the walk does not take from an image, fp16 38 / 15, 31 / 15: always;  8 rows fp16 16.9 / 15.0,
//                   11.5 / 15.2, fp32 21.3 / 19.0, 14.6 / 19.1: by bytes;  16 fp16 rows 23.1 / 15.6, 11.9 / 15.6: where the walk would do
//                   the gate too, from half the bytes on;  32 rows fp16 42 / 22, 23.1 / 21.8, fp32 66 / 35, 49 / 34: always at such
//                   widths (2048 -> 2048 at 95 %: fp16 5.2 / 6.9, by bytes)
// The gated product goes where the plain one goes, so that they are equal bit for bit.
// A knob that names another kernel for few rows keeps the call with it.
bool few_on_matrix_cores(const KernelArgs& a, const tl_layout_header* h, int64_t M, bool chained)
{
    if (M > kSmallMaxM || chained || !a.c0.base || (M == 1 && (a.gated || knob(TL_FEW, 0) == 0))) return false;
    for (Knob other : {TL_SMALL_MT, TL_OCTET, TL_QUAD_WIDE, TL_RES16, TL_SPMV_DIRECT, TL_SPMV_TILES})
        if (knob(other, -1) >= 0) return false;
    if (a.gated && !walk_has_gated(a, h)) return false;   // (refused there, as it is not the walk's)
    bool use = M > 1;
    const uint64_t code_bytes = (uint64_t)a.NB * a.units * a.planes * TL_CODE_UNIT_BYTES;
    const bool wide = a.NB > 2 * compute_units();
    if (use && (a.x_kmajor ? (M < 3 || M > 4) && !(wide && M > 16) : M > 8 && M <= 16 && !a.x_f16 && wide))
        use = code_bytes < h->stream_bytes * (a.x_kmajor && walk_has_gated(a, h) ? 2 : 1);
    return knob(TL_FEW, use ? 1 : 0) != 0;
}

// tl_spmm, or (y_layout >= 0) tl_spmm_gated with that output layout
int spmm_call(const tl_layout_header* header, const void* blob_dev, const void* X, int x_dtype, int x_layout, int64_t ldx, int64_t M,
              void* Y, int y_dtype, int64_t ldy, int y_layout, const void* scale, int scale_dtype, void* workspace, int64_t workspace_bytes,
              void* stream, const tl_chain* chain = nullptr)
{
    if (int rc = check_header(header)) return rc;
    const bool gated = y_layout >= 0;
    // the checks of tl_spmm, with the width of the gated output where ldy is compared
    if (int rc = check_io(blob_dev, X, Y, x_dtype, x_layout, ldx, M, y_dtype, gated ? (int64_t)header->columns : ldy, scale, scale_dtype, header)) return rc;
    if (gated) {
        if (y_layout != TL_X_ROW_MAJOR && y_layout != TL_X_K_MAJOR) return fail(TL_ERR_ARG, "y_layout=%d unknown", y_layout);
        if (header->columns % 2) return fail(TL_ERR_SHAPE, "N=%u: gate and up columns come in pairs", header->columns);
        const int64_t min_ldy = y_layout == TL_X_K_MAJOR ? M : (int64_t)header->columns / 2;
        if (ldy < min_ldy) return fail(TL_ERR_SHAPE, "ldy=%lld smaller than %lld", (long long)ldy, (long long)min_ldy);
        if (y_layout == TL_X_K_MAJOR && (M <= 8 || M > 16)) return fail(TL_ERR_UNSUPPORTED, "a K-major gated output is written for 9 to 16 rows");
    }
    KernelArgs a;
    std::memset(&a, 0, sizeof(a));
    a.gated = gated;
    if (gated && y_layout == TL_X_K_MAJOR) a.y_kld = ldy;
    if (chain) {
        const bool out = chain->next_norm_weight || chain->image_out || chain->squares_out;
        if (out && !(chain->next_norm_weight && chain->image_out && chain->squares_out))
            return fail(TL_ERR_ARG, "next_norm_weight, image_out and squares_out come together");
        if ((out || chain->residual) && gated) return fail(TL_ERR_ARG, "a gated product has no residual or image epilogue");
        if (M < 9 || M > 16) return fail(TL_ERR_UNSUPPORTED, "chained products are for 9 to 16 fp16 rows");
        if (chain->residual && chain->residual_ld < (int64_t)header->columns) return fail(TL_ERR_SHAPE, "residual_ld=%lld smaller than N", (long long)chain->residual_ld);
        if (out && (chain->image_ld < M || chain->image_ld > 16))  // the epilogue writes (and zeroes) 16 rows of the image at most
            return fail(TL_ERR_SHAPE, "image_ld=%lld outside M=%lld .. 16", (long long)chain->image_ld, (long long)M);
        if (chain->squares_in && chain->squares_blocks <= 0) return fail(TL_ERR_ARG, "squares_blocks must be positive");
        const uintptr_t es = y_dtype == TL_F16 ? 2 : 4;
        for (const void* p : {chain->residual, chain->next_norm_weight, static_cast<const void*>(chain->image_out)})
            if (reinterpret_cast<uintptr_t>(p) % es) return fail(TL_ERR_ALIGN, "residual, next_norm_weight and image_out must be aligned to y_dtype");
        for (const void* p : {static_cast<const void*>(chain->squares_out), static_cast<const void*>(chain->squares_in)})
            if (reinterpret_cast<uintptr_t>(p) % 16) return fail(TL_ERR_ALIGN, "squares_out and squares_in must be 16-byte aligned");
        a.chain_res = chain->residual; a.chain_ldres = chain->residual_ld;
        a.chain_w = chain->next_norm_weight; a.chain_image = chain->image_out; a.chain_ild = chain->image_ld; a.chain_sq_out = chain->squares_out;
        a.chain_sq_in = chain->squares_in; a.chain_sq_blocks = chain->squares_blocks; a.eps = chain->eps;
    }
    a.w0 = weight_ptrs(header, blob_dev, scale);
    a.X = X; a.Y = Y;
    a.ldx = ldx; a.ldy = ldy;
    a.M = (int)M; a.N = (int)header->columns; a.K = (int)header->inners; a.T = (int)header->n_tiles; a.tile_rows = (int)header->tile_rows;
    a.NB = (int)header->n_blocks; a.c0 = weight_codes(header, blob_dev); a.units = (int)header->code_units; a.planes = a.c0.planes;
    a.x_f16 = x_dtype == TL_F16; a.x_kmajor = x_layout == TL_X_K_MAJOR; a.y_f16 = y_dtype == TL_F16; a.scale_f16 = scale_dtype == TL_F16;
    a.one = 1.0f;
    hipStream_t st = static_cast<hipStream_t>(stream);
    int rc = few_on_matrix_cores(a, header, M, chain != nullptr) ? launch_matrix_few(a, x_dtype, false, st)
             : (M <= kSmallMaxM) ? launch_small(a, header, x_dtype, workspace, workspace_bytes, st)
                               : launch_matrix_rows(a, x_dtype, workspace, workspace_bytes, false, st);
    if (rc) return rc;
    return finish_launch();
}
}  // namespace

extern "C" int tl_spmm(const tl_layout_header* header, const void* blob_dev,
                       const void* X, int x_dtype, int x_layout, int64_t ldx, int64_t M,
                       void* Y, int y_dtype, int64_t ldy,
                       const void* scale, int scale_dtype,
                       void* workspace, int64_t workspace_bytes, void* stream)
{
    return spmm_call(header, blob_dev, X, x_dtype, x_layout, ldx, M, Y, y_dtype, ldy, -1, scale, scale_dtype, workspace, workspace_bytes, stream);
}

extern "C" int tl_spmm_chain(const tl_layout_header* header, const void* blob_dev,
                             const void* X, int x_dtype, int x_layout, int64_t ldx, int64_t M,
                             void* Y, int y_dtype, int64_t ldy, int y_layout,
                             const void* scale, int scale_dtype, const tl_chain* chain,
                             void* workspace, int64_t workspace_bytes, void* stream)
{
    if (!chain) return fail(TL_ERR_ARG, "chain is null");
    return spmm_call(header, blob_dev, X, x_dtype, x_layout, ldx, M, Y, y_dtype, ldy, y_layout, scale, scale_dtype, workspace, workspace_bytes, stream, chain);
}

namespace {
// The argument block of a row-major product without a workspace, of checked arguments.
KernelArgs rows_call(const tl_layout_header* h, const void* blob_dev, const void* X, int x_dtype, int64_t ldx, int64_t M, void* Y, int y_dtype, int64_t ldy,
                     int gated, const void* scale, int scale_dtype)
{
    KernelArgs a;
    std::memset(&a, 0, sizeof(a));
    a.w0 = weight_ptrs(h, blob_dev, scale);
    a.X = X; a.Y = Y;
    a.ldx = ldx; a.ldy = ldy;
    a.M = (int)M; a.N = (int)h->columns; a.K = (int)h->inners; a.T = (int)h->n_tiles; a.tile_rows = (int)h->tile_rows;
    a.NB = (int)h->n_blocks; a.c0 = weight_codes(h, blob_dev); a.units = (int)h->code_units; a.planes = a.c0.planes;
    a.x_f16 = x_dtype == TL_F16; a.y_f16 = y_dtype == TL_F16; a.scale_f16 = scale_dtype == TL_F16;
    a.one = 1.0f;
    a.gated = gated != 0;
    return a;
}

int check_gated_rows(const tl_layout_header* h, int gated, int64_t ldy)
{
    const int64_t N = h->columns;
    if (gated && N % 2) return fail(TL_ERR_SHAPE, "N=%lld: gate and up columns come in pairs", (long long)N);
    if (gated && ldy < N / 2) return fail(TL_ERR_SHAPE, "ldy=%lld smaller than %lld", (long long)ldy, (long long)(N / 2));
    return TL_OK;
}
}  // namespace

extern "C" int tl_spmm_chain_rows(const tl_layout_header* header, const void* blob_dev,
                                  const void* X, int x_dtype, int64_t ldx, int64_t M, void* Y, int y_dtype, int64_t ldy, int gated,
                                  const void* scale, int scale_dtype, const tl_chain* chain, void* stream)
{
    if (int rc = check_header(header)) return rc;
    if (!chain) return fail(TL_ERR_ARG, "chain is null");
    const int64_t N = header->columns;
    if (int rc = check_io(blob_dev, X, Y, x_dtype, TL_X_ROW_MAJOR, ldx, M, y_dtype, gated ? N : ldy, scale, scale_dtype, header)) return rc;
    if (int rc = check_gated_rows(header, gated, ldy)) return rc;
    const bool few = M <= kSmallMaxM;
    if (M < 2 || x_dtype != TL_F16 || y_dtype != TL_F16 || !header->off_codes)
        return fail(TL_ERR_UNSUPPORTED, "products chained row by row are for 2 and more fp16 rows and blobs with codes");
    const bool image = chain->next_norm_weight || chain->image_out, out = image || chain->squares_out;
    if (out && !(chain->squares_out && (!image || (chain->next_norm_weight && chain->image_out)) && (few || image)))
        return fail(TL_ERR_ARG, "next_norm_weight, image_out and squares_out come together, or squares_out alone for up to %d rows", kSmallMaxM);
    if ((out || chain->residual) && gated) return fail(TL_ERR_ARG, "a gated product has no residual or image epilogue");
    if (chain->residual && chain->residual_ld < N) return fail(TL_ERR_SHAPE, "residual_ld=%lld smaller than N", (long long)chain->residual_ld);
    if (image && chain->image_ld < N) return fail(TL_ERR_SHAPE, "image_ld=%lld smaller than N", (long long)chain->image_ld);
    if (few && chain->squares_in && chain->squares_blocks <= 0) return fail(TL_ERR_ARG, "squares_blocks must be positive");
    for (const void* p : {chain->residual, chain->next_norm_weight, static_cast<const void*>(chain->image_out)})
        if (reinterpret_cast<uintptr_t>(p) % 2) return fail(TL_ERR_ALIGN, "residual, next_norm_weight and image_out must be aligned to y_dtype");
    for (const void* p : {static_cast<const void*>(chain->squares_out), static_cast<const void*>(chain->squares_in)})
        if (reinterpret_cast<uintptr_t>(p) % 16) return fail(TL_ERR_ALIGN, "squares_out and squares_in must be 16-byte aligned");
    KernelArgs a = rows_call(header, blob_dev, X, x_dtype, ldx, M, Y, y_dtype, ldy, gated, scale, scale_dtype);
    a.chain_res = chain->residual; a.chain_ldres = chain->residual_ld;
    a.chain_w = chain->next_norm_weight; a.chain_image = chain->image_out; a.chain_ild = chain->image_ld; a.chain_sq_out = chain->squares_out;
    a.chain_sq_in = chain->squares_in; a.chain_sq_blocks = chain->squares_blocks; a.eps = chain->eps;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (!few) {
        if (!matrix_reads_rows(a, x_dtype)) return fail(TL_ERR_UNSUPPORTED, "more than %d chained rows are read where they lie: aligned, K and ldx multiples of 8", kSmallMaxM);
        a.chain_factors = chain->squares_in;
        a.chain_sq_in = nullptr;
    }
    if (int rc = few ? launch_matrix_few(a, x_dtype, false, st) : launch_matrix_rows(a, x_dtype, nullptr, 0, false, st)) return rc;
    return finish_launch();
}

extern "C" int tl_spmm_normed_rows(const tl_layout_header* header, const void* blob_dev,
                                   const void* X, int x_dtype, int64_t ldx, int64_t M, void* Y, int y_dtype, int64_t ldy, int gated,
                                   const void* scale, int scale_dtype, const void* norm_weight, const float* squares, int squares_blocks, float eps,
                                   void* stream)
{
    if (int rc = check_header(header)) return rc;
    if (int rc = check_io(blob_dev, X, Y, x_dtype, TL_X_ROW_MAJOR, ldx, M, y_dtype, gated ? (int64_t)header->columns : ldy, scale, scale_dtype, header)) return rc;
    if (int rc = check_gated_rows(header, gated, ldy)) return rc;
    if (!norm_weight || !squares) return fail(TL_ERR_ARG, "norm_weight or squares is null");
    if (squares_blocks <= 0) return fail(TL_ERR_ARG, "squares_blocks must be positive");
    if (reinterpret_cast<uintptr_t>(squares) % 16) return fail(TL_ERR_ALIGN, "squares must be 16-byte aligned");
    if (M < 2 || M > kSmallMaxM || x_dtype != TL_F16 || y_dtype != TL_F16 || !header->off_codes)
        return fail(TL_ERR_UNSUPPORTED, "rows are normalised on their way in for 2 to %d fp16 rows and blobs with codes", kSmallMaxM);
    KernelArgs a = rows_call(header, blob_dev, X, x_dtype, ldx, M, Y, y_dtype, ldy, gated, scale, scale_dtype);
    a.norm_w = norm_weight; a.chain_sq_in = squares; a.chain_sq_blocks = squares_blocks; a.eps = eps;
    if (int rc = launch_matrix_few(a, x_dtype, false, static_cast<hipStream_t>(stream))) return rc;
    return finish_launch();
}

extern "C" int tl_spmm_gated(const tl_layout_header* header, const void* blob_dev,
                             const void* X, int x_dtype, int x_layout, int64_t ldx, int64_t M,
                             void* Y, int y_dtype, int64_t ldy, int y_layout,
                             const void* scale, int scale_dtype,
                             void* workspace, int64_t workspace_bytes, void* stream)
{
    return spmm_call(header, blob_dev, X, x_dtype, x_layout, ldx, M, Y, y_dtype, ldy, y_layout, scale, scale_dtype, workspace, workspace_bytes, stream);
}

namespace {
// tl_mlp_gate_up, or (few) tl_mlp_gate_up_few
int gate_up_call(bool few, const tl_layout_header* gate_header, const void* gate_blob_dev,
                 const tl_layout_header* up_header, const void* up_blob_dev,
                 const void* X, int x_dtype, int x_layout, int64_t ldx, int64_t M,
                 void* H, int h_dtype, int64_t ldh,
                 const void* gate_scale, const void* up_scale, int scale_dtype,
                 int activation,
                 void* workspace, int64_t workspace_bytes, void* stream)
{
    if (int rc = check_header(gate_header)) return rc;
    if (int rc = check_header(up_header)) return rc;
    if (gate_header->inners != up_header->inners || gate_header->columns != up_header->columns ||
        gate_header->tile_rows != up_header->tile_rows)
        return fail(TL_ERR_SHAPE, "gate and up weights must share K, N and tile height");
    if (activation != TL_ACT_SILU_GATE) return fail(TL_ERR_UNSUPPORTED, "activation code %d (only TL_ACT_SILU_GATE)", activation);
    if (!up_blob_dev || reinterpret_cast<uintptr_t>(up_blob_dev) % 256) return fail(TL_ERR_ALIGN, "up blob null or not 256-byte aligned");
    if (int rc = check_io(gate_blob_dev, X, H, x_dtype, x_layout, ldx, M, h_dtype, ldh, gate_scale, scale_dtype, gate_header)) return rc;
    if ((gate_scale == nullptr) != (up_scale == nullptr)) return fail(TL_ERR_ARG, "pass both scales or neither");
    if (!few && M <= kSmallMaxM) return fail(TL_ERR_UNSUPPORTED, "fused gate/up needs M > %d; use two tl_spmm calls below that", kSmallMaxM);
    if (few && (M > kSmallMaxM || !gate_header->off_codes || !up_header->off_codes))
        return fail(TL_ERR_UNSUPPORTED, "fused gate/up of few rows is for M <= %d and blobs with codes", kSmallMaxM);
    KernelArgs a;
    std::memset(&a, 0, sizeof(a));
    a.w0 = weight_ptrs(gate_header, gate_blob_dev, gate_scale);
    a.w1 = weight_ptrs(up_header, up_blob_dev, up_scale);
    a.X = X; a.Y = H;
    a.ldx = ldx; a.ldy = ldh;
    a.NB = (int)gate_header->n_blocks; a.units = (int)gate_header->code_units;
    a.c0 = weight_codes(gate_header, gate_blob_dev);
    a.c1 = weight_codes(up_header, up_blob_dev);
    a.planes = std::max(a.c0.planes, a.c1.planes);
    a.M = (int)M; a.N = (int)gate_header->columns; a.K = (int)gate_header->inners; a.T = (int)gate_header->n_tiles;
    a.tile_rows = (int)gate_header->tile_rows;
    a.x_f16 = x_dtype == TL_F16; a.x_kmajor = x_layout == TL_X_K_MAJOR; a.y_f16 = h_dtype == TL_F16; a.scale_f16 = scale_dtype == TL_F16;
    a.one = 1.0f;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (int rc = few ? launch_matrix_few(a, x_dtype, true, st) : launch_matrix_rows(a, x_dtype, workspace, workspace_bytes, true, st)) return rc;
    return finish_launch();
}
}  // namespace

extern "C" int tl_mlp_gate_up(const tl_layout_header* gate_header, const void* gate_blob_dev,
                              const tl_layout_header* up_header, const void* up_blob_dev,
                              const void* X, int x_dtype, int x_layout, int64_t ldx, int64_t M,
                              void* H, int h_dtype, int64_t ldh,
                              const void* gate_scale, const void* up_scale, int scale_dtype,
                              int activation,
                              void* workspace, int64_t workspace_bytes, void* stream)
{
    return gate_up_call(false, gate_header, gate_blob_dev, up_header, up_blob_dev, X, x_dtype, x_layout, ldx, M, H, h_dtype, ldh, gate_scale,
                        up_scale, scale_dtype, activation, workspace, workspace_bytes, stream);
}

extern "C" int tl_mlp_gate_up_few(const tl_layout_header* gate_header, const void* gate_blob_dev,
                                  const tl_layout_header* up_header, const void* up_blob_dev,
                                  const void* X, int x_dtype, int x_layout, int64_t ldx, int64_t M,
                                  void* H, int h_dtype, int64_t ldh,
                                  const void* gate_scale, const void* up_scale, int scale_dtype,
                                  int activation, void* stream)
{
    return gate_up_call(true, gate_header, gate_blob_dev, up_header, up_blob_dev, X, x_dtype, x_layout, ldx, M, H, h_dtype, ldh, gate_scale,
                        up_scale, scale_dtype, activation, nullptr, 0, stream);
}



// Scratch of tl_spmm_noalloc: device memory that belongs to the library's code object, one copy per GPU,
// there from the moment the library is loaded on a device until the process ends.
constexpr int64_t kActivationBytes = 32ll << 20;
constexpr int64_t kStaticScratchBytes = kActivationBytes / 2 * 3;  // fp32 rows in three bf16 parts
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
// Device address of `scratch` on the current device.  In host code the array's name is only a handle
// for the runtime; the address comes from hipGetSymbolAddress, asked once per device with that device
// current, and differs from GPU to GPU.
int static_scratch(void** out)
{
    static std::atomic<void*> address[64];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(TL_ERR_LAUNCH, "hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= 64) return fail(TL_ERR_UNSUPPORTED, "device ordinal %d: the static scratch serves ordinals 0 to 63", dev);
    void* p = address[dev].load(std::memory_order_acquire);
    if (!p) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return fail(TL_ERR_LAUNCH, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        address[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return TL_OK;
}
}  // namespace

extern "C" int tl_spmm_noalloc(const tl_layout_header* header, const void* blob_dev,
                               const void* X, int x_dtype, int x_layout, int64_t ldx, int64_t M,
                               void* Y, int y_dtype, int64_t ldy,
                               const void* scale, int scale_dtype, void* stream)
{
    if (int rc = check_header(header)) return rc;
    if (int rc = check_dtype(x_dtype, "x")) return rc;
    if (M <= 0) return fail(TL_ERR_SHAPE, "M=%lld must be positive", (long long)M);
    // what the kernels stage in the scratch: the image of the activations (none for 4 rows and fewer).  32 MiB of
    // activations are always taken, as an image that does not fit is made some rows at a time.
    const int64_t image = M * image_row_bytes(header->inners, x_dtype);
    int64_t need = M <= kSmallMaxM ? small_kmajor_bytes(header, M, x_dtype) : image;
    if (M > kSmallMaxM && image > kStaticScratchBytes && least_image_bytes(header->inners, M, x_dtype) <= kActivationBytes) need = kStaticScratchBytes;
    if (need > kStaticScratchBytes)
        return fail(TL_ERR_SIZE, "M=%lld rows of K=%u need %lld bytes of scratch; tl_spmm_noalloc has %lld (use tl_spmm with a workspace)",
                    (long long)M, header->inners, (long long)need, (long long)kStaticScratchBytes);
    void* ws = nullptr;
    if (int rc = static_scratch(&ws)) return rc;
    return tl_spmm(header, blob_dev, X, x_dtype, x_layout, ldx, M, Y, y_dtype, ldy, scale, scale_dtype, ws, kStaticScratchBytes, stream);
}

// Reads `pieces` 16-byte pieces and folds them: what streaming that much memory costs a launch that writes next to
// nothing.  256 threads a workgroup, eight pieces of a thread in flight per turn.
__global__ __launch_bounds__(256) void tl_read_probe(const u32x4* __restrict__ src, long long pieces, uint32_t* __restrict__ out)
{
    constexpr int U = 8;
    const long long stride = (long long)gridDim.x * 256;
    uint32_t fold = 0;
    for (long long first = (long long)blockIdx.x * 256 + threadIdx.x; first < pieces; first += stride * U) {
        u32x4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = first + u * stride < pieces ? src[first + u * stride] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int u = 0; u < U; ++u) fold ^= v[u][0] ^ v[u][1] ^ v[u][2] ^ v[u][3];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) fold ^= __shfl_xor(fold, off, 64);
    __shared__ uint32_t part[4];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = fold;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = part[0] ^ part[1] ^ part[2] ^ part[3];
}

extern "C" int tl_matrix_tile(int64_t M, int columns, int inners, int planes, int x_dtype, int two_weights, int units)
{
    if (int rc = check_dtype(x_dtype, "x_dtype")) return rc;
    if (M < 1 || columns < 1 || inners < 1 || planes < 1 || units < 1) return fail(TL_ERR_SHAPE, "sizes must be positive");
    return matrix_tile(M, columns, (int64_t)planes * ceil_div(inners, TL_CODE_UNIT_ROWS), x_dtype == TL_F32, two_weights != 0, units);
}

extern "C" int tl_read_probe_workgroups(void) { return 8 * compute_units(); }

extern "C" int tl_stream_read_probe(const void* src, int64_t bytes, void* out, void* stream)
{
    if (!src || !out) return fail(TL_ERR_ARG, "device pointer is null");
    if (bytes <= 0 || bytes % 16) return fail(TL_ERR_SIZE, "bytes=%lld must be a positive multiple of 16", (long long)bytes);
    if (reinterpret_cast<uintptr_t>(src) % 16 || reinterpret_cast<uintptr_t>(out) % 4) return fail(TL_ERR_ALIGN, "src must be 16-byte, out 4-byte aligned");
    const long long pieces = bytes / 16;
    const int groups = (int)std::min<long long>(tl_read_probe_workgroups(), ceil_div(pieces, 256));
    hipLaunchKernelGGL(tl_read_probe, dim3((unsigned)groups), dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<const u32x4*>(src), pieces,
                       static_cast<uint32_t*>(out));
    return finish_launch();
}

extern "C" int tl_spmm_time(const tl_layout_header* header, const void* blob_dev,
                            const void* X, int x_dtype, int x_layout, int64_t ldx, int64_t M,
                            void* Y, int y_dtype, int64_t ldy,
                            const void* scale, int scale_dtype,
                            void* workspace, int64_t workspace_bytes, void* stream,
                            int iters, float* mean_ms)
{
    if (iters <= 0 || !mean_ms) return fail(TL_ERR_ARG, "iters must be positive and mean_ms non-null");
    hipStream_t st = static_cast<hipStream_t>(stream);
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) return fail(TL_ERR_LAUNCH, "hipEventCreate failed");
    int rc = TL_OK;
    (void)hipEventRecord(e0, st);
    for (int i = 0; i < iters && rc == TL_OK; ++i)
        rc = tl_spmm(header, blob_dev, X, x_dtype, x_layout, ldx, M, Y, y_dtype, ldy, scale, scale_dtype, workspace, workspace_bytes, stream);
    (void)hipEventRecord(e1, st);
    if (rc == TL_OK) {
        hipError_t e = hipEventSynchronize(e1);
        float ms = 0.f;
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
        if (e != hipSuccess) rc = fail(TL_ERR_LAUNCH, "event timing failed: %s", hipGetErrorString(e));
        *mean_ms = ms / iters;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return rc;
}

