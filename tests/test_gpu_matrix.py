"""The matrix-core kernels at the sizes where they can go wrong: edges of their tiles, stages and code units, weights
whose entries are not ternary, activations that are not finite, blobs without codes."""
import numpy as np
import pytest
import torch

from tests.test_matrix_tiles_cpu import SIZES
from tests.util import activations, ternary_weight

pytestmark = pytest.mark.gpu


def _device(w, cuda):
    from ternaryllm_amd import ops
    from ternaryllm_amd.packing import PackedWeight
    return ops.DeviceWeight(PackedWeight.from_dense(w), cuda)


# rows: the 64-row tile and the 32-row fragment; K: the 64-row stage, the stages asked for ahead, the 256-row unit,
# rows that are not whole 16-byte pieces; N: the 16-column block, a wave's 64 columns
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(49, 1, 1), (49, 8, 16), (127, 64, 31), (128, 72, 128), (129, 192, 129), (145, 256, 113), (64, 264, 144),
                                   (300, 320, 257), (640, 520, 300), (257, 1100, 1000), (129, 1280, 700)])
def test_many_rows_at_the_edges(cuda, oracle, M, K, N, dtype):
    """Integer activations: every sum is exact, whatever its order."""
    from ternaryllm_amd import ops
    w = ternary_weight(K, N, 0.6, M + K + N)
    dw = _device(w, cuda)
    x = activations(M, K, M, dtype, integer=True)
    ref = oracle.fast_product(x.double().numpy(), w)
    for name, xin, layout in (("rows", x.to(cuda), 0), ("k-major", x.t().contiguous().to(cuda), 1)):
        print(f"case M={M} K={K} N={N} {dtype} {name}", flush=True)
        y = ops.spmm(dw, xin, out_dtype=torch.float32, x_layout=layout)
        assert np.array_equal(y.cpu().numpy().astype(np.float64), ref), name
    if dtype == torch.float32:  # all 24 bits of an fp32 value (its three bf16 parts) pass through a column with one entry
        rng = np.random.default_rng(M)
        rows, one = rng.integers(0, K, N), np.zeros((K, N), np.int32)
        one[rows, np.arange(N)] = rng.choice([-1, 1], N)
        x = activations(M, K, M + 1, dtype)
        y = ops.spmm(_device(one, cuda), x.to(cuda)).cpu().numpy()
        assert np.array_equal(y, x.numpy()[:, rows] * one[rows, np.arange(N)].astype(np.float32))


# tiles of 32 x 32 with five units and a stage shared out over four waves; tiles of 128 x 256 and of 64 x 256 with rows, columns
# and stages left over (4093 x 4090 is 512 of the tall ones, as many as two for each compute unit)
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(65, 1344, 66), (200, 2048, 1032), (1030, 330, 2100), (4093, 200, 4090)])
def test_tiles_of_every_shape(cuda, M, K, N, dtype):
    from ternaryllm_amd import ops
    w, w2 = ternary_weight(K, N, 0.6, M), ternary_weight(K, N, 0.7, N)
    dw, dw2 = _device(w, cuda), _device(w2, cuda)
    x = activations(M, K, M, dtype, integer=True).to(cuda)
    wd, wd2 = torch.from_numpy(w).double().to(cuda), torch.from_numpy(w2).double().to(cuda)
    scale = torch.rand(N, device=cuda).to(dtype)
    print(f"case M={M} K={K} N={N} {dtype}", flush=True)
    want = x.double() @ wd
    assert torch.equal(ops.spmm(dw, x, out_dtype=torch.float32).double(), want)           # whole numbers
    ragged = torch.full((M, N + 3), 7.0, dtype=torch.float32, device=cuda)
    ops.spmm(dw, x, out=ragged[:, 1:N + 1], out_dtype=torch.float32)                      # rows that lie on no boundary
    assert torch.equal(ragged[:, 1:N + 1].double(), want) and bool((ragged[:, 0] == 7).all()) and bool((ragged[:, N + 1:] == 7).all())
    x = x / 16
    assert torch.equal(ops.spmm_gated(dw, x, scale), ops.silu_mul(ops.spmm(dw, x, scale), pairs=True))
    got = ops.mlp_gate_up(dw, dw2, x, scale, scale, out_dtype=torch.float32).double()
    sd = scale.double()
    want = torch.nn.functional.silu((x.double() @ wd) * sd) * ((x.double() @ wd2) * sd)
    assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())              # exact sums; __expf and the division


# few units of K, of which four waves' 32 x 32 tiles leave some without a share (one, two, three and, beside it, four); one and two 64 x 128
# tiles a unit (two weights: 32 x 64 a wave); 64 x 256 ones that are not enough for 128 x 256
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(65, 250, 66), (63, 264, 34), (150, 768, 98), (150, 776, 98), (520, 250, 2058), (520, 1100, 2058), (769, 330, 4090), (2110, 264, 4090)])
def test_tiles_of_few_units(cuda, M, K, N, dtype):
    test_tiles_of_every_shape(cuda, M, K, N, dtype)


@pytest.mark.parametrize("M,K,N,N2", [(49, 8, 1, 34), (65, 1344, 66, 40), (200, 2048, 1032, 130), (1030, 336, 2100, 66), (4096, 200, 4096, 2048)])
def test_chained_rows(cuda, M, K, N, N2):
    """More than 48 rows: a product that adds residual rows and leaves the next norm's image and sums of squares, bit for bit as
    separate operators do, and products that multiply by the rows' factors, plain and gated."""
    from ternaryllm_amd import ops
    K2 = N - N % 8
    w1, w2 = ternary_weight(K, N, 0.7, 1), ternary_weight(max(K2, 8), N2, 0.7, 2)
    d1, d2 = _device(w1, cuda), _device(w2, cuda)
    g = torch.Generator(device=cuda).manual_seed(M)
    x, res = torch.randn((M, K), generator=g, device=cuda).half(), torch.randn((M, N), generator=g, device=cuda).half()
    nw, sc1 = (1 + 0.1 * torch.randn(N, generator=g, device=cuda)).half(), (0.05 + 0.01 * torch.rand(N, generator=g, device=cuda)).half()
    sc2 = (0.05 + 0.01 * torch.rand(N2, generator=g, device=cuda)).half()
    print(f"case M={M} K={K} N={N} N2={N2}", flush=True)
    y, image, squares = ops.spmm_chain_rows(d1, x, sc1, residual=res, next_norm_weight=nw)
    assert torch.equal(y, ops.spmm(d1, x, sc1) + res)
    assert torch.equal(image, (y.float() * nw.float()).half())
    blocks = -(-N // 32)
    padded = torch.zeros((M, blocks * 32), dtype=torch.float64, device=cuda)
    padded[:, :N] = y.double().pow(2)
    # (32 squares and 31 additions, each rounded to 2^-24)
    assert torch.allclose(squares.double(), padded.view(M, blocks, 32).sum(-1), rtol=63 * 2.0 ** -24, atol=0)
    factors = ops.row_factors(squares, N, 1e-5)
    # (the sums' roundings halved by the root, and rsqrt's own)
    assert torch.allclose(factors.double(), torch.rsqrt(y.double().pow(2).mean(-1) + 1e-5), rtol=(64 + blocks) * 2.0 ** -24, atol=0)
    rows = image[:, :K2].contiguous() if K2 else x
    out = ops.spmm_chain_rows(d2, rows, sc2, squares_in=factors)
    want = (ops.spmm(d2, rows, sc2, out_dtype=torch.float32) * factors[:, None]).half()
    assert float((out.double() - want.double()).abs().max()) <= 2.0 ** -10 * float(want.double().abs().max())   # a unit in the last place of fp16
    gated = ops.spmm_chain_rows(d2, rows, sc2, squares_in=factors, gated=True)
    assert torch.equal(gated, ops.silu_mul(out, pairs=True))
    assert torch.equal(ops.spmm_chain_rows(d2, rows, sc2, gated=True), ops.spmm_gated(d2, rows, sc2))
    with pytest.raises(RuntimeError, match="UNSUPPORTED"):
        wide = torch.zeros((M, K + 1), dtype=torch.float16, device=cuda)[:, :K]
        ops.spmm_chain_rows(d1, wide, sc1, residual=res)               # rows that are not read where they lie


def _repeated(w):
    """The packed weight of tiled-CSC arrays that name a row |entry| times."""
    from ternaryllm_amd.packing import PackedWeight
    K, N = w.shape
    neg, pos, neg_off, pos_off = [], [], np.zeros((N, 1, 2), np.int32), np.zeros((N, 1, 2), np.int32)
    for y in range(N):
        for rows, off, sign in ((neg, neg_off, -1), (pos, pos_off, 1)):
            off[y, 0, 0] = len(rows)
            for k in range(K):
                rows += [k] * max(0, sign * int(w[k, y]))
            off[y, 0, 1] = len(rows)
    return PackedWeight.from_tiled_csc(np.array(neg, np.int32), neg_off.reshape(-1), np.array(pos, np.int32), pos_off.reshape(-1), N, K, K)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M", [2, 16, 48, 49, 130])
def test_gate_and_up_of_different_planes(cuda, M, dtype):
    """A gate that names rows three times beside an up weight that does not, and the other way round."""
    from ternaryllm_amd import ops
    K, N = 600, 72
    rng = np.random.default_rng(7)
    often, once = rng.integers(-3, 4, (K, N)) * (rng.random((K, N)) < 0.3), ternary_weight(K, N, 0.7, 8)
    pw = _repeated(often)
    assert pw.header.code_planes == 3
    d_often, d_once = ops.DeviceWeight(pw, cuda), _device(once, cuda)
    x = activations(M, K, 6, dtype, integer=True) / 16
    for (dg, wg), (du, wu) in (((d_often, often), (d_once, once)), ((d_once, once), (d_often, often))):
        print(f"case M={M} {dtype} gate planes {dg.header.code_planes}", flush=True)
        got = ops.mlp_gate_up(dg, du, x.to(cuda), out_dtype=torch.float32).double().cpu()
        want = torch.nn.functional.silu(x.double() @ torch.from_numpy(wg).double()) * (x.double() @ torch.from_numpy(wu).double())
        # exact sums; a few units in the last place of __expf and of the division
        assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())


@pytest.mark.parametrize("M", [1, 5, 16, 40, 64, 200])
def test_entries_beyond_one(cuda, M):
    """Arrays that name a row several times make entries up to 3: the codes hold a plane for each mention."""
    from ternaryllm_amd import ops
    rng = np.random.default_rng(5)
    for K, N in ((100, 20), (600, 40)):
        w = rng.integers(-3, 4, (K, N)) * (rng.random((K, N)) < 0.3)
        pw = _repeated(w)
        pw.validate()
        assert pw.header.code_planes == 3 and np.array_equal(pw.to_dense(), w)
        x = activations(M, K, 6, torch.float32, integer=True)
        print(f"case M={M} K={K}", flush=True)
        y = ops.spmm(ops.DeviceWeight(pw, cuda), x.to(cuda))
        assert np.array_equal(y.cpu().numpy().astype(np.float64), x.double().numpy() @ w)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M", [1, 3, 16, 33, 130])
def test_activations_that_are_not_finite(cuda, M, dtype):
    """A column that does not name a row is not touched by what that row holds, infinities and NaN included."""
    from ternaryllm_amd import ops
    K, N = 300, 50
    w = ternary_weight(K, N, 0.9, 8)
    x = activations(M, K, 9, dtype, integer=True)
    x[0, 7], x[M // 2, 100], x[M - 1, 299] = float("inf"), float("-inf"), float("nan")
    want = np.zeros((M, N))
    xn = x.double().numpy()
    for n in range(N):
        rows = np.nonzero(w[:, n])[0]
        want[:, n] = (xn[:, rows] * w[rows, n]).sum(1)
    print(f"case M={M} {dtype}", flush=True)
    dw = _device(w, cuda)
    got = ops.spmm(dw, x.to(cuda), out_dtype=torch.float32).double().cpu().numpy()
    assert np.array_equal(got, want, equal_nan=True)
    if M > 48:
        pairs = ops.spmm_gated(dw, x.to(cuda)).float()
        assert torch.equal(torch.nan_to_num(pairs), torch.nan_to_num(ops.silu_mul(ops.spmm(dw, x.to(cuda)), pairs=True).float()))
        both = ops.mlp_gate_up(dw, dw, x.to(cuda), out_dtype=torch.float32).double().cpu()
        g = torch.from_numpy(want)
        assert torch.allclose(both, torch.nn.functional.silu(g) * g, rtol=1e-4, atol=1e-4, equal_nan=True)


@pytest.mark.parametrize("M", [1, 4, 16, 48, 200])
def test_activations_of_every_magnitude(cuda, M):
    """Denormal and very large activations keep all their bits: exactly where a column has one entry, and in sums to what
    their roundings give (2^-24 of the sum of magnitudes, once for each of the column's entries)."""
    from ternaryllm_amd import ops
    K, N = 520, 70
    rng = np.random.default_rng(M)
    rows, one = rng.integers(0, K, N), np.zeros((K, N), np.int32)
    one[rows, np.arange(N)] = rng.choice([-1, 1], N)
    w = ternary_weight(K, N, 0.6, 21)
    d_one, dw = _device(one, cuda), _device(w, cuda)
    for dtype, exponents in ((torch.float32, (-149, -140, -130, -126, -118, -110, -60, 60, 100, 115)), (torch.float16, (-24, -20, -14, 10))):
        for e in exponents:
            x = (activations(M, K, 22, torch.float64) * 2.0 ** e).to(dtype)
            print(f"case M={M} {dtype} 2^{e}", flush=True)
            y = ops.spmm(d_one, x.to(cuda)).cpu().numpy()
            assert np.array_equal(y, x.numpy()[:, rows] * one[rows, np.arange(N)].astype(x.numpy().dtype)), e
            xd, wd = x.double(), torch.from_numpy(w).double()
            y = ops.spmm(dw, x.to(cuda), out_dtype=torch.float32).cpu().double()
            bound = 2.0 ** -24 * (wd != 0).sum(0) * (xd.abs() @ wd.abs())
            assert bool(((y - xd @ wd).abs() <= bound).all()), e


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_finite_rows_keep_their_bits_beside_rows_that_are_not(cuda, dtype):
    """What a row holds does not show in the bits of another row's outputs."""
    from ternaryllm_amd import ops
    M, K, N = 150, 700, 90
    dg, du = _device(ternary_weight(K, N, 0.5, 11), cuda), _device(ternary_weight(K, N, 0.5, 12), cuda)
    x = activations(M, K, 13, dtype).to(cuda)
    spoilt = x.clone()
    spoilt[3, 5], spoilt[70, 600], spoilt[149, 0] = float("inf"), float("nan"), float("-inf")
    keep = [m for m in range(M) if m not in (3, 70, 149)]
    for name, call in (("plain", lambda t: ops.spmm(dg, t)), ("pairs", lambda t: ops.spmm_gated(dg, t)), ("two weights", lambda t: ops.mlp_gate_up(dg, du, t))):
        print(f"case {name} {dtype}", flush=True)
        assert torch.equal(call(x)[keep], call(spoilt)[keep]), name


def _without_codes(new, cuda):
    """The device weight of the blob that the version before the codes would have made."""
    from ternaryllm_amd import _lib, ops
    old = new.blob[:new.header.off_codes].copy()
    h = _lib.LayoutHeader.from_buffer_copy(old[:256].tobytes())
    h.version, h.off_codes, h.code_units, h.code_planes, h.total_bytes = 5, 0, 0, 0, old.size
    old[:256] = np.frombuffer(bytes(h), np.uint8)
    dev = ops.DeviceWeight.__new__(ops.DeviceWeight)
    dev.header, dev.blob = h, torch.from_numpy(old).to(cuda)
    return dev


def _product(dw, x, layout, M, ldx, ws):
    """tl_spmm with just this workspace."""
    import ctypes
    from ternaryllm_amd import _lib
    y = torch.full((M, dw.columns), 7.0, dtype=torch.float32, device=x.device)
    rc = _lib.lib().tl_spmm(ctypes.byref(dw.header), dw.blob.data_ptr(), x.data_ptr(), _lib.TL_F16 if x.dtype == torch.float16 else _lib.TL_F32,
                            layout, ldx, M, y.data_ptr(), _lib.TL_F32, dw.columns, None, _lib.TL_F32, ws.data_ptr() if ws is not None else None,
                            ws.numel() if ws is not None else 0, ctypes.c_void_p(torch.cuda.current_stream(x.device).cuda_stream))
    return rc, y


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(49, 3, 5), (128, 250, 16), (129, 248, 66), (257, 600, 131), (300, 1003, 64)])
def test_the_index_stream_alone(cuda, oracle, M, K, N, dtype):
    """More than 48 rows of a weight without codes, and K-major rows without a workspace: padded to whole waves they need
    none, as other layouts do where there are codes."""
    from ternaryllm_amd import _lib, ops
    from ternaryllm_amd.packing import PackedWeight
    w, w2 = ternary_weight(K, N, 0.6, M + K), ternary_weight(K, N, 0.7, M + N)
    new = PackedWeight.from_dense(w)
    dw, old, old2 = ops.DeviceWeight(new, cuda), _without_codes(new, cuda), _without_codes(PackedWeight.from_dense(w2), cuda)
    x = activations(M, K, M, dtype, integer=True)
    ref = oracle.fast_product(x.double().numpy(), w)
    ld = (M + 255) // 256 * 256
    padded = torch.full((K, ld), 9.0, dtype=dtype)
    padded[:, :M] = x.t()
    forms = {"rows": (x.to(cuda), 0, K), "k-major": (x.t().contiguous().to(cuda), 1, M), "k-major padded": (padded.to(cuda), 1, ld)}
    ws = torch.empty(K * ld * 4, dtype=torch.uint8, device=cuda)
    for name, (xd, layout, ldx) in forms.items():
        for weight, space in ((old, None), (old, ws), (dw, None)):
            print(f"case {name} {dtype} codes={weight is dw} workspace={space is not None}", flush=True)
            rc, y = _product(weight, xd, layout, M, ldx, space)
            if weight is dw and (name == "k-major" and ldx % (256 if dtype == torch.float16 else 128) or name == "rows" and not (dtype == torch.float16 and K % 8 == 0)):
                assert _lib.ERROR_NAMES[rc] == "TL_ERR_SIZE"
            else:
                assert rc == 0 and np.array_equal(y.cpu().numpy().astype(np.float64), ref)
    xd = x.to(cuda) / 16
    if N % 2 == 0:
        assert torch.equal(ops.spmm_gated(old, xd), ops.silu_mul(ops.spmm(old, xd), pairs=True))
    for g, u in ((old, old2), (dw, old2), (old, dw)):
        got = ops.mlp_gate_up(g, u, xd, out_dtype=torch.float32).double().cpu()
        want = torch.nn.functional.silu(xd.double().cpu() @ torch.from_numpy(w).double()) * (xd.double().cpu() @ torch.from_numpy(w2 if u is old2 else w).double())
        assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())   # exact sums; __expf and the division


@pytest.mark.parametrize("M,K,N", [(2048, 4096, 2048), (1100, 1100, 2100)])
def test_a_row_s_bits_do_not_depend_on_the_workspace(cuda, M, K, N):
    """An image of fp32 rows that does not fit is made and multiplied some rows at a time, the last time with few (768 of 2048,
    460 of 1100): with the tile of the whole call, whose sums are taken in one order."""
    dw = _device(ternary_weight(K, N, 0.7, 5), cuda)
    x = activations(M, K, 6, torch.float32).to(cuda)
    print(f"case M={M} K={K} N={N}", flush=True)
    rc, some = _product(dw, x, 0, M, K, torch.empty(M * K * 4, dtype=torch.uint8, device=cuda))
    rc2, whole = _product(dw, x, 0, M, K, torch.empty(M * (K + 8) * 6, dtype=torch.uint8, device=cuda))
    assert rc == rc2 == 0 and torch.equal(some, whole)


def test_loading_a_blob_without_codes_from_the_device(cuda):
    """load_state_dict(assign=True) keeps the device of what it is given, also where the blob is brought up to date."""
    from ternaryllm_amd import TernaryLinear
    from ternaryllm_amd.packing import PackedWeight
    K, N = 264, 40
    new = PackedWeight.from_dense(ternary_weight(K, N, 0.6, 41))
    module = TernaryLinear(K, N, sparsity=0.9, bias=False, reference_buffers=False).to(cuda)
    module.load_state_dict({"w_packed": _without_codes(new, cuda).blob}, assign=True)
    assert module.w_packed.device == cuda and np.array_equal(module.w_packed.cpu().numpy(), new.blob)
    x = activations(60, K, 1, torch.float32, integer=True).to(cuda)
    assert torch.equal(module(x), x @ torch.from_numpy(new.to_dense()).float().to(cuda))   # exact: whole numbers


@pytest.mark.parametrize("M,K,ld", [(60, 64, 1 << 23), (60, 64, (1 << 24) + 8), (4300000, 16, 0)])
def test_rows_far_apart_and_very_many_of_them(cuda, M, K, ld):
    """Row-major rows whose distance the kernel cannot address go through the image; K-major ones in several passes where one
    launch's image cannot hold them (ld = 0)."""
    from ternaryllm_amd import ops
    N = 24
    w = ternary_weight(K, N, 0.5, 31)
    x = torch.randint(-8, 9, (K, M) if ld == 0 else (M, K), generator=torch.Generator(device=cuda).manual_seed(1), device=cuda).half()
    want = (x.t() if ld == 0 else x).float() @ torch.from_numpy(w).float().to(cuda)   # exact: whole numbers
    if ld:
        far = torch.empty((M - 1) * ld + K, dtype=torch.float16, device=cuda).as_strided((M, K), (ld, 1))
        far.copy_(x)
        x = far
    print(f"case M={M} ld={ld}", flush=True)
    assert torch.equal(ops.spmm(_device(w, cuda), x, out_dtype=torch.float32, x_layout=1 if ld == 0 else 0), want)


def test_a_blob_without_codes(cuda, oracle):
    """What an older version packed: the packed-weight object brings it up to date, and a device blob that was not is
    multiplied by the general kernel."""
    import ctypes
    from ternaryllm_amd import _lib, ops
    from ternaryllm_amd.packing import PackedWeight
    K, N = 520, 96
    w = ternary_weight(K, N, 0.7, 3)
    new = PackedWeight.from_dense(w)
    old = new.blob[:new.header.off_codes].copy()
    h = _lib.LayoutHeader.from_buffer_copy(old[:256].tobytes())
    h.version, h.off_codes, h.code_units, h.code_planes, h.total_bytes = 5, 0, 0, 0, old.size
    old[:256] = np.frombuffer(bytes(h), np.uint8)
    _lib.check(_lib.lib().tl_layout_validate(old.ctypes.data, old.size))
    assert np.array_equal(PackedWeight(old).blob, new.blob)
    dev = ops.DeviceWeight.__new__(ops.DeviceWeight)
    dev.header, dev.blob = h, torch.from_numpy(old).to(cuda)
    for M in (1, 6, 60):
        x = activations(M, K, M, torch.float16, integer=True)
        print(f"case M={M}", flush=True)
        y = ops.spmm(dev, x.to(cuda), out_dtype=torch.float32)
        assert np.array_equal(y.cpu().numpy().astype(np.float64), oracle.fast_product(x.double().numpy(), w))


# few tiles (one of 64 x 64 a compute unit at most), whose waves share K: 64 x 64 of nine units, and of three, which they own parts of;
# 32 x 64 two to a compute unit; 32 x 32 with rows, columns and a stage left over, and of one unit, which leaves waves without a share; of one unit,
# 64 x 64 that share nothing; two weights of three units, 32 x 64
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(250, 2304, 4000), (250, 520, 4000), (253, 1100, 3970), (97, 1412, 1001), (49, 130, 33), (130, 250, 4000), (130, 600, 2000)])
def test_tiles_whose_waves_share_k(cuda, M, K, N, dtype):
    """Integer activations: every sum is exact, whatever its order; two weights and pairs against the gate of the products."""
    from ternaryllm_amd import ops
    N2 = N // 2 * 2
    w, w2 = ternary_weight(K, N, 0.6, M), ternary_weight(K, N, 0.7, N)
    dw, dw2 = _device(w, cuda), _device(w2, cuda)
    x = activations(M, K, K, dtype, integer=True).to(cuda)
    print(f"case M={M} K={K} N={N} {dtype}", flush=True)
    one, two = x.double() @ torch.from_numpy(w).double().to(cuda), x.double() @ torch.from_numpy(w2).double().to(cuda)
    assert torch.equal(ops.spmm(dw, x, out_dtype=torch.float32).double(), one)
    x, one, two = x / 16, one / 16, two / 16
    got, want = ops.mlp_gate_up(dw, dw2, x, out_dtype=torch.float32).double(), torch.nn.functional.silu(one) * two
    assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())              # exact sums; __expf and the division
    even = _device(w[:, :N2].copy(), cuda)
    assert torch.equal(ops.spmm_gated(even, x), ops.silu_mul(ops.spmm(even, x), pairs=True))


# two groups of four waves that share K: eleven units (five and six), fp16 fourteen, and a last one of one stage or of eight rows, for one weight
# and, at half the rows, for two; two groups of two waves, for two weights: the same and five units
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(900, 2568, 4090), (500, 2616, 4090), (1000, 2816, 3850), (900, 3336, 4090), (500, 2616, 2040), (450, 1032, 2000)])
def test_groups_of_waves_that_share_k(cuda, M, K, N, dtype):
    test_tiles_whose_waves_share_k(cuda, M, K, N, dtype)


# planes of rows that are named again, where K is whole stages of 64 rows but not whole units of 256 (the stages that fill up a plane's last
# unit lie past K), and where it is both
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K", [(60, 192), (130, 1088), (130, 1024)])
def test_entries_beyond_one_of_whole_stages(cuda, M, K, dtype):
    from ternaryllm_amd import ops
    rng = np.random.default_rng(K)
    w = rng.integers(-3, 4, (K, 40)) * (rng.random((K, 40)) < 0.3)
    x = activations(M, K, 6, dtype, integer=True)
    y = ops.spmm(ops.DeviceWeight(_repeated(w), cuda), x.to(cuda), out_dtype=torch.float32)
    assert np.array_equal(y.cpu().numpy().astype(np.float64), x.double().numpy() @ w)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_nothing_past_k_is_read_for_entries_beyond_one(cuda, dtype):
    """What lies behind a row's K values -- for fp16 rows read where they are the gap to the next row, in the fp32 rows' image the next row's
    head -- shows in no bit: NaN there would meet zero weights, and the sum be worked out again in another order."""
    from ternaryllm_amd import ops
    M, K, ld, N = 130, 1088, 1344, 40
    rng = np.random.default_rng(K)
    w = rng.integers(-3, 4, (K, N)) * (rng.random((K, N)) < 0.3)
    dw = ops.DeviceWeight(_repeated(w), cuda)
    values = activations(M, K, 6, dtype).to(cuda)
    rows = torch.zeros((M + 1, ld), dtype=dtype, device=cuda)
    rows[:M, :K] = values
    print(f"case {dtype}", flush=True)
    want = ops.spmm(dw, rows[:M, :K], out_dtype=torch.float32)
    assert bool(want.isfinite().all())
    rows[:, K:] = float("nan")
    assert torch.equal(ops.spmm(dw, rows[:M, :K], out_dtype=torch.float32), want)
    spoilt = values.clone()
    spoilt[1::2, :192] = float("nan")
    assert torch.equal(ops.spmm(dw, spoilt, out_dtype=torch.float32)[0::2], want[0::2])


def _of_every_tile(two):
    return [pytest.param(dtype, tile, *size, id=f"{kind}-{tile}") for kind, dtype in (("fp16", torch.float16), ("fp32", torch.float32)) for tile, size in SIZES[kind, two].items()]


def _spoilt_rows(M):
    """Rows in each fragment of 16 of a tile's first 128, at its edges and between (groups of waves exchange half of a tile's fragments), and the last."""
    return [m for m in (0, 15, 21, 40, 63, 70, 90, 101, 127) if m < M - 1] + [M - 1]


@pytest.mark.parametrize("dtype,tile,M,K,N", _of_every_tile(False))
def test_sums_that_are_not_finite_on_every_tile(cuda, dtype, tile, M, K, N):
    """One infinity or NaN a row, at rows of K of every stage's parts: outputs that name it have it, all others are exact (whole numbers); gated
    outputs are the gate of those; and with other activations, rows without one keep their bits."""
    from ternaryllm_amd import ops
    w = ternary_weight(K, N, 0.6, M)
    dw, wd = _device(w, cuda), torch.from_numpy(w).double().to(cuda)
    x = activations(M, K, K, dtype, integer=True).to(cuda)
    want = x.double() @ wd
    spoilt, rows = x.clone(), _spoilt_rows(M)
    for i, m in enumerate(rows):
        k, v = (i * 37 + i * K // len(rows)) % K, (float("inf"), float("nan"), float("-inf"))[i % 3]
        want[m] += torch.where(wd[k] != 0, v * wd[k], 0.0) - x[m, k].double() * wd[k]
        spoilt[m, k] = v
    print(f"case {tile} M={M} K={K} N={N} {dtype}", flush=True)
    got = ops.spmm(dw, spoilt, out_dtype=torch.float32).double()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0, 1e30, -1e30), want.nan_to_num(7.0, 1e30, -1e30))
    pairs, both = ops.spmm_gated(dw, spoilt), ops.silu_mul(ops.spmm(dw, spoilt), pairs=True)
    assert torch.equal(pairs.isnan(), both.isnan()) and torch.equal(pairs.nan_to_num(7.0), both.nan_to_num(7.0))
    keep = torch.ones(M, dtype=torch.bool, device=cuda)
    keep[rows] = False
    x = activations(M, K, 13, dtype).to(cuda)
    beside = torch.where(spoilt.isfinite(), x, spoilt)
    assert torch.equal(ops.spmm(dw, x)[keep], ops.spmm(dw, beside)[keep])
    assert torch.equal(ops.spmm_gated(dw, x)[keep], ops.spmm_gated(dw, beside)[keep])


@pytest.mark.parametrize("dtype,tile,M,K,N", _of_every_tile(True))
def test_two_weights_sums_that_are_not_finite_on_every_tile(cuda, dtype, tile, M, K, N):
    from ternaryllm_amd import ops
    wg, wu = ternary_weight(K, N, 0.6, M), ternary_weight(K, N, 0.7, N)
    dg, du = _device(wg, cuda), _device(wu, cuda)
    x = (activations(M, K, K, dtype, integer=True) / 16).to(cuda)
    spoilt, rows, products = x.clone(), _spoilt_rows(M), []
    for i, m in enumerate(rows):
        spoilt[m, (i * 37 + i * K // len(rows)) % K] = (float("inf"), float("nan"), float("-inf"))[i % 3]
    for w in (wg, wu):
        wd = torch.from_numpy(w).double().to(cuda)
        y = torch.where(spoilt.isfinite(), x, 0).double() @ wd
        for i, m in enumerate(rows):
            k = (i * 37 + i * K // len(rows)) % K
            y[m] += torch.where(wd[k] != 0, spoilt[m, k].double() * wd[k], 0.0)
        products.append(y)
    print(f"case {tile} M={M} K={K} N={N} {dtype}", flush=True)
    want = products[0] / (1 + torch.exp(-products[0])) * products[1]
    got = ops.mlp_gate_up(dg, du, spoilt, out_dtype=torch.float32).double()
    assert torch.equal(got.isnan(), want.isnan())
    got, want = got.nan_to_num(0.0, 1e30, -1e30), want.nan_to_num(0.0, 1e30, -1e30)
    largest = float(want[want.abs() < 1e29].abs().max())
    assert float((got - want).abs().max()) <= 1e-5 * largest                  # exact sums; __expf and the division (infinities are equal)
    keep = torch.ones(M, dtype=torch.bool, device=cuda)
    keep[rows] = False
    x = activations(M, K, 13, dtype).to(cuda)
    beside = torch.where(spoilt.isfinite(), x, spoilt)
    assert torch.equal(ops.mlp_gate_up(dg, du, x)[keep], ops.mlp_gate_up(dg, du, beside)[keep])


@pytest.mark.parametrize("tile", list(SIZES["fp16", False]))
def test_chained_rows_on_every_tile(cuda, tile):
    test_chained_rows(cuda, *SIZES["fp16", False][tile], 66)


# few rows and many
@pytest.mark.parametrize("M,N", [(32, 11008), (1024, 4096)])
def test_a_gate_rounded_to_fp16_is_the_fp32_gate_rounded(cuda, M, N):
    """The SiLU in front of an fp16 result is the fp32 one, a division's quotient: an approximate one shows where the product with the up
    column is near a tie (a unit of fp32 moves one in some 10^4 results by one of fp16)."""
    from ternaryllm_amd import ops
    K = 64
    g = torch.Generator(device=cuda).manual_seed(M)
    dg, du = _device(ternary_weight(K, N, 0.5, 51), cuda), _device(ternary_weight(K, N, 0.5, 52), cuda)
    x = torch.randn((M, K), generator=g, device=cuda).half()
    scale = 0.1 + 0.3 * torch.rand(N, generator=g, device=cuda)
    print(f"case M={M}", flush=True)
    full = ops.mlp_gate_up(dg, du, x, scale, scale, out_dtype=torch.float32)
    assert torch.equal(ops.mlp_gate_up(dg, du, x, scale, scale, out_dtype=torch.float16), full.half())
