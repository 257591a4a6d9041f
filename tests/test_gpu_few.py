"""The matrix-core kernel for a few rows at the sizes where it can go wrong: its 16-row fragments, turns of one, two and
four slices of 64 rows of K, more turns than waves, one and two column blocks to a workgroup, every way of reading rows."""
import numpy as np
import pytest
import torch

from tests.util import activations, ternary_weight

pytestmark = pytest.mark.gpu


# K: below one 16-byte piece, whole and ragged slices, 32 and 64 slices, more than 16 units; N: the 16-column block, and
# 8200 columns are more blocks than twice the compute units
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(2, 1, 1), (16, 8, 16), (3, 72, 31), (5, 1003, 77), (17, 1024, 33), (32, 2048, 16), (48, 2056, 40), (33, 4100, 50),
                                   (9, 4352, 24), (48, 11008, 17), (16, 520, 8200), (34, 300, 8195)])
def test_few_rows_at_the_edges(cuda, oracle, M, K, N, dtype):
    """Integer activations: every sum is exact, whatever its order.  fp32 ones use all 24 bits where a column has one entry."""
    from ternaryllm_amd import ops
    from ternaryllm_amd.packing import PackedWeight
    w = ternary_weight(K, N, 0.6, M + K + N)
    dw = ops.DeviceWeight(PackedWeight.from_dense(w), cuda)
    x = activations(M, K, M, dtype, integer=True)
    ref = oracle.fast_product(x.double().numpy(), w)
    wide = torch.zeros((M, K + 3), dtype=dtype)
    wide[:, :K] = x
    for name, xin, layout in (("rows", x.to(cuda), 0), ("strided rows", wide.to(cuda)[:, :K], 0), ("k-major", x.t().contiguous().to(cuda), 1)):
        print(f"case M={M} K={K} N={N} {dtype} {name}", flush=True)
        out = torch.full((M, N + 5), 7.0, dtype=torch.float32, device=cuda)
        ops.spmm(dw, xin, out_dtype=torch.float32, x_layout=layout, out=out[:, :N])
        assert np.array_equal(out[:, :N].cpu().numpy().astype(np.float64), ref), name
        assert bool((out[:, N:] == 7.0).all()), name
    one = np.zeros((K, N), np.int32)
    rng = np.random.default_rng(M)
    rows = rng.integers(0, K, N)
    one[rows, np.arange(N)] = rng.choice([-1, 1], N)
    x = activations(M, K, M + 1, dtype)
    y = ops.spmm(ops.DeviceWeight(PackedWeight.from_dense(one), cuda), x.to(cuda)).cpu().numpy()
    assert np.array_equal(y, x.numpy()[:, rows] * one[rows, np.arange(N)].astype(x.numpy().dtype))


# where rows go through LDS and where they are read as operands: fp16 from 4 or, up to 1024 of K, 9 rows on; fp32 from 8 or 12; on no
# boundary fp32 rows up to 1024 of K but for 8 to 16
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(2, 520, 8200), (4, 1024, 40), (7, 1032, 40), (9, 1024, 40), (11, 2048, 6150), (12, 2048, 6150), (8, 4096, 6150), (24, 1003, 8200), (37, 65, 40), (40, 1003, 4200), (7, 1025, 17)])
def test_few_rows_of_every_path(cuda, oracle, M, K, N, dtype):
    test_few_rows_at_the_edges(cuda, oracle, M, K, N, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K", [(3, 1003), (20, 301), (37, 1000), (44, 1001)])
def test_gate_and_up_of_short_rows(cuda, M, K, dtype):
    """silu(gate) * up of two weights over up to 1024 of K, whole numbers / 16: exact sums, then __expf and a division."""
    from ternaryllm_amd import ops
    from ternaryllm_amd.packing import PackedWeight
    wg, wu = ternary_weight(K, 83, 0.8, 3), ternary_weight(K, 83, 0.8, 4)
    dg, du = (ops.DeviceWeight(PackedWeight.from_dense(w), cuda) for w in (wg, wu))
    x = activations(M, K, 5, dtype, integer=True).to(cuda) / 16
    print(f"case M={M} K={K} {dtype}", flush=True)
    got = ops.mlp_gate_up(dg, du, x, out_dtype=torch.float32).double()
    g, u = (x.double() @ torch.from_numpy(w).double().to(cuda) for w in (wg, wu))
    want = torch.nn.functional.silu(g) * u
    assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M", [2, 16, 31, 48])
def test_gate_and_up_of_few_rows(cuda, M, dtype):
    """silu(gate) * up of two weights in one launch, infinities included: a column sees only the rows that it names."""
    from ternaryllm_amd import ops
    from ternaryllm_amd.packing import PackedWeight
    K, N = 1100, 83
    wg, wu = ternary_weight(K, N, 0.8, 3), ternary_weight(K, N, 0.8, 4)
    dg, du = (ops.DeviceWeight(PackedWeight.from_dense(w), cuda) for w in (wg, wu))
    x = activations(M, K, 5, dtype)
    x[M - 1, 9] = float("inf")
    sg = (0.5 + torch.rand(N, generator=torch.Generator().manual_seed(6))).to(dtype)
    g, u = (torch.zeros(M, N, dtype=torch.float64) for _ in range(2))
    for n in range(N):
        for w, out in ((wg, g), (wu, u)):
            rows = np.nonzero(w[:, n])[0]
            out[:, n] = (x[:, rows].double() * torch.from_numpy(w[rows, n]).double()).sum(1)
    g, u = g * sg.double(), u * sg.double()
    want = torch.nn.functional.silu(g) * u
    print(f"case M={M} {dtype}", flush=True)
    got = ops.mlp_gate_up(dg, du, x.to(cuda), sg.to(cuda), sg.to(cuda), out_dtype=torch.float32).double().cpu()
    # K fp32 roundings of sums of magnitude sqrt(K) at most, and __expf's few units: far below 1e-4 of the result's size
    fine = torch.isfinite(want)
    assert torch.equal(fine, torch.isfinite(got))
    assert float((got[fine] - want[fine]).abs().max()) <= 1e-4 * float(want[fine].abs().max())


@pytest.mark.parametrize("M,K,N,N2", [(2, 8, 16, 2), (13, 1000, 272, 96), (16, 520, 270, 8200), (17, 2048, 43, 34), (31, 72, 4128, 40), (48, 1100, 78, 4200), (33, 5504, 2048, 64)])
def test_chained_rows(cuda, M, K, N, N2):
    """A product that ends a block (residual rows, the next norm's image and sums of squares) and the products behind the norm,
    plain and gated: each step bit for bit what the separate operators give, the norm against float64."""
    from tests.util import max_rel_err
    from ternaryllm_amd import ops
    from ternaryllm_amd.packing import PackedWeight
    w1, w2 = ternary_weight(K, N, 0.7, 1), ternary_weight(N, N2, 0.7, 2)
    d1, d2 = (ops.DeviceWeight(PackedWeight.from_dense(w), cuda) for w in (w1, w2))
    g = torch.Generator().manual_seed(M)
    x, res = torch.randn((M, K), generator=g).half().to(cuda), torch.randn((M, N), generator=g).half().to(cuda)
    nw = (1 + 0.1 * torch.randn(N, generator=g)).half().to(cuda)
    sc1, sc2 = (0.05 + 0.01 * torch.rand(N, generator=g)).half().to(cuda), (0.5 + torch.rand(N2, generator=g)).half().to(cuda)
    print(f"case M={M} K={K} N={N} N2={N2}", flush=True)
    y, image, squares = ops.spmm_chain_rows(d1, x, sc1, residual=res, next_norm_weight=nw)
    assert torch.equal(y, ops.spmm(d1, x, sc1) + res)
    assert torch.equal(image, (y.float() * nw.float()).half())
    blocks = -(-N // 16)
    padded = torch.zeros((M, blocks * 16), dtype=torch.float64, device=cuda)
    padded[:, :N] = y.double().pow(2)
    # (16 squares and 15 additions, each rounded to 2^-24)
    assert torch.allclose(squares[:, :M].double(), padded.reshape(M, blocks, 16).sum(-1).t(), rtol=31 * 2.0 ** -24, atol=0)
    out = ops.spmm_chain_rows(d2, image, sc2, squares_in=squares, eps=1e-5)
    h64 = y.double() * torch.rsqrt(y.double().pow(2).mean(-1, keepdim=True) + 1e-5) * nw.double()
    ref = (h64.cpu().numpy() @ w2.astype("float64")) * sc2.double().cpu().numpy()[None, :]
    assert max_rel_err(out.double().cpu().numpy(), ref, h64.cpu().numpy(), w2) <= 4e-3
    assert torch.equal(ops.spmm_chain_rows(d2, image, sc2, squares_in=squares, eps=1e-5, gated=True), ops.silu_mul(out, pairs=True))
    assert torch.equal(ops.spmm_chain_rows(d2, image, sc2), ops.spmm(d2, image, sc2))
    # the gated product is the plain one and the gate, rows and a K-major result with its padding rows
    plain = ops.silu_mul(ops.spmm(d2, image, sc2), pairs=True)
    assert torch.equal(ops.spmm_gated(d2, image, sc2), plain)
    if 9 <= M <= 16:
        turned = ops.spmm_gated(d2, image, sc2, kmajor=True)
        assert torch.equal(turned.t(), plain) and not turned.as_strided((N2 // 2, 16), (16, 1))[:, M:].any()
    x[M - 1, 7] = float("inf")          # a column that does not name the row is not touched
    assert torch.equal(ops.spmm_chain_rows(d1, x, sc1, residual=res).isfinite(), (ops.spmm(d1, x, sc1) + res).isfinite())
    with pytest.raises(RuntimeError, match="UNSUPPORTED"):
        ops.spmm_chain_rows(d1, x[:1], sc1, residual=res[:1])


@pytest.mark.parametrize("M,K,N", [(2, 16, 34), (3, 1104, 4200), (4, 72, 16), (13, 2048, 272), (16, 520, 8200), (17, 2064, 66), (31, 72, 4128), (33, 264, 40), (48, 5504, 2048)])
def test_rows_normalised_on_their_way_in(cuda, M, K, N):
    """RMSNorm and product in one against the two kernels, over magnitudes that leave fp16's middle, with a row that is not
    finite, plain and gated; and the sums of squares without an image."""
    from ternaryllm_amd import ops
    from ternaryllm_amd.packing import PackedWeight
    dw = ops.DeviceWeight(PackedWeight.from_dense(ternary_weight(K, N, 0.7, M)), cuda)
    up = ops.DeviceWeight(PackedWeight.from_dense(ternary_weight(40, K, 0.7, 1)), cuda)
    g = torch.Generator().manual_seed(M)
    sc, res = (0.5 + torch.rand(N, generator=g)).half().to(cuda), torch.randn((M, K), generator=g).half().to(cuda)
    nw = (1 + 0.1 * torch.randn(K, generator=g)).half().to(cuda)
    few = torch.randn((M, 40), generator=g).half().to(cuda)
    print(f"case M={M} K={K} N={N}", flush=True)
    for rows, weights in ((1.0, 1.0), (2e-3, 0.02), (1e-5, 1.0), (1500.0, 40.0)):   # (1500: up to five times 5400, and times 40 beyond fp16)
        r = res * rows
        x, squares = ops.spmm_chain_rows(up, few * rows, residual=r, squares_out=True)
        assert torch.equal(x, ops.spmm(up, few * rows) + r)
        norm = nw * weights
        h = ops.add_rmsnorm(x, None, norm, 1e-5)[1]
        got, want = ops.spmm_normed_rows(dw, x, norm, squares, 1e-5, sc), ops.spmm(dw, h, sc)
        # the squares' sum in another order moves a row by 2^-22 and few of its values across a rounding: by 2^-10 of them
        assert float((got.double() - want.double()).norm()) <= 2.0 ** -11 * float(want.double().norm())
        assert torch.equal(ops.spmm_normed_rows(dw, x, norm, squares, 1e-5, sc, gated=True), ops.silu_mul(got, pairs=True))
    x[M - 1, 7] = float("inf")                  # (squares as they were: the value, not its row, is infinite)
    got = ops.spmm_normed_rows(dw, x, norm, squares, 1e-5, sc)
    assert torch.equal(got.isfinite(), ops.spmm(dw, x, sc * 1e-5).isfinite())
    with pytest.raises(RuntimeError, match="UNSUPPORTED"):
        ops.spmm_normed_rows(dw, torch.zeros((M, K + 1), dtype=torch.float16, device=cuda)[:, :K], norm, squares, 1e-5, sc)
    if M > 8:
        with pytest.raises(ValueError):
            ops.spmm_normed_rows(dw, x, norm, torch.zeros((K // 16, 8), device=cuda), 1e-5, sc)


@pytest.mark.parametrize("B,width", [(1, 16), (1, 2048), (5, 2064), (16, 4096), (17, 48), (48, 2048), (49, 48), (300, 2064)])
def test_embedding_rows(cuda, B, width):
    """A token's row, its image for the product behind the first norm and its sums of squares; tokens counted from the end, and
    tokens that the table does not have."""
    from ternaryllm_amd import ops
    g = torch.Generator().manual_seed(B)
    table, nw = torch.randn((37, width), generator=g).half().to(cuda), torch.rand(width, generator=g).half().to(cuda)
    token = torch.randint(-37, 37, (B,), generator=g).to(cuda)
    print(f"case B={B} width={width}", flush=True)
    x, image, squares = ops.embed_rows(table, token, nw)
    want = table[token]
    assert torch.equal(x, want) and torch.equal(image, (want.float() * nw.float()).half())
    run = 16 if B <= 48 else 32
    padded = torch.zeros((B, -(-width // run) * run), dtype=torch.float64, device=cuda)
    padded[:, :width] = want.double().pow(2)
    got = squares.view(1, -1) if B == 1 else squares[:, :B].t() if B <= 48 else squares
    assert torch.allclose(got.double(), padded.view(B, -1, run).sum(-1), rtol=run * 2.0 ** -24, atol=0)   # a rounding for each value
    token[B - 1] = 37
    x, image, squares = ops.embed_rows(table, token, nw)
    assert bool(x[B - 1].isnan().all()) and torch.equal(x[:B - 1], want[:B - 1])
