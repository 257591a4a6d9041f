"""The short way from torch calls to a product (csrc/tl_torch.cpp) against the general one, over the forms of activations that it
takes and those that it leaves."""
import pytest
import torch

from tests.util import ternary_weight

pytestmark = pytest.mark.gpu


def _forms(K, M, dtype, cuda, g):
    x = torch.randn((M, K), generator=g).to(dtype).to(cuda)
    wide = torch.randn((M + 1, K + 24), generator=g).to(dtype).to(cuda)
    yield "rows", x, 0
    yield "strided rows", wide[:M, :K], 0
    yield "rows from an odd element", wide[:M, 3:K + 3], 0
    yield "every other column", torch.randn((M, 2 * K), generator=g).to(dtype).to(cuda)[:, ::2], 0
    yield "k-major", x.t().contiguous(), 1
    yield "strided k-major", torch.randn((K, M + 5), generator=g).to(dtype).to(cuda)[:, :M], 1
    if M > 1:
        yield "columns of rows", x.t().contiguous().t(), 0
        yield "one row for all", x[:1].expand(M, K), 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(1, 72, 40), (3, 1003, 77), (16, 64, 5000), (48, 264, 33), (49, 264, 48), (200, 1000, 130)])
def test_products(cuda, M, K, N, dtype):
    from ternaryllm_amd import TernaryLinear, ops
    g = torch.Generator().manual_seed(M)
    w = torch.from_numpy(ternary_weight(K, N, 0.6, M))
    for scale in (None, torch.rand(N, generator=g).half(), torch.rand(N, generator=g)):
        module = TernaryLinear(K, N, weight=w, scale=scale, bias=False, reference_buffers=False).to(cuda)
        dw, sc = module.device_weight(), module.w_scale
        for name, x, layout in _forms(K, M, dtype, cuda, g):
            print(f"case {name} M={M} K={K} N={N} {dtype} scale {None if scale is None else scale.dtype}", flush=True)
            if name == "one row for all":
                with pytest.raises(ValueError):
                    ops.spmm(dw, x, sc, out_dtype=dtype)                      # (rows of no distance are refused either way)
                with pytest.raises(ValueError):
                    ops.spmm(dw, x, sc)
                continue
            want = ops.spmm(dw, x, sc, out_dtype=dtype, x_layout=layout)      # the general way, which leaves the scratch behind
            short = ops.product(dw, x, sc, layout == 1)
            assert (short is not None) == (x.stride(-1) == 1), name
            assert short is None or torch.equal(short, want), name
            assert torch.equal(ops.spmm(dw, x, sc, x_layout=layout), want), name
            if K != M:
                assert torch.equal(module(x), want) and torch.equal(module(x[None]), want[None]), name
            if layout == 0:
                assert torch.equal(module(x[0]), ops.spmm(dw, x[:1].contiguous(), sc, out_dtype=dtype)[0]), name


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M", [1, 2, 48, 49, 130])
def test_gate_and_up(cuda, M, dtype):
    from ternaryllm_amd import LlamaTernaryMLP, TernaryConfig, ops
    g = torch.Generator().manual_seed(M)
    block = LlamaTernaryMLP(TernaryConfig(hidden_size=264, intermediate_size=136, num_attention_heads=4, num_key_value_heads=4, sparsity=0.7), generator=g, reference_buffers=False).to(cuda)
    gate, up = block.gate_proj.device_weight(), block.up_proj.device_weight()
    sg, su = torch.rand(136, generator=g).to(dtype).to(cuda), torch.rand(136, generator=g).to(dtype).to(cuda)
    x = torch.randn((1, M, 264), generator=g).to(dtype).to(cuda)
    for a, b in ((None, None), (sg, su)):
        print(f"case M={M} {dtype} scaled {a is not None}", flush=True)
        want = ops.mlp_gate_up(gate, up, x[0], a, b, out_dtype=dtype)
        short = ops.gate_up(gate, up, x, a, b)
        assert (short is None) == (M == 1) and (short is None or torch.equal(short[0], want))
    want = block.down_proj(ops.mlp_gate_up(gate, up, x[0], out_dtype=dtype))
    assert torch.equal(block(x)[0], want) and torch.equal(block(x[0]), want)


def test_what_is_not_plain(cuda):
    """Types, devices and wrappers that the short way leaves to the general one, whose errors and results stay; other streams and
    threads, each with scratch of its own."""
    import threading
    from ternaryllm_amd import TernaryLinear, ops
    g = torch.Generator().manual_seed(1)
    w = torch.from_numpy(ternary_weight(264, 40, 0.6, 1))
    module = TernaryLinear(264, 40, weight=w, bias=False, reference_buffers=False).to(cuda)
    dw = module.device_weight()
    x = torch.randn((60, 264), generator=g).to(cuda)
    for bad, error in ((x.double(), ValueError), (x.cpu(), RuntimeError), (x[:, :200], ValueError)):
        with pytest.raises(error):
            ops.spmm(dw, bad)
    with pytest.raises(ValueError):
        ops.spmm(dw, x, torch.rand(39, device=cuda))
    assert ops.spmm(dw, x[:0]).shape == (0, 40) and module(x.view(1, 60, 264)[:, :0]).shape == (1, 0, 40)
    with pytest.raises(AssertionError):
        module(x.view(1, 1, 60, 264))

    class Own(torch.Tensor):
        pass

    want = ops.spmm(dw, x, out_dtype=torch.float32)
    assert ops.product(dw, x.as_subclass(Own)) is None and torch.equal(ops.spmm(dw, x.as_subclass(Own)).as_subclass(torch.Tensor), want)
    x.requires_grad_()
    assert torch.equal(module(x), want) and not module(x).requires_grad
    x = x.detach()
    results, streams = {}, [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()

    def work(i):
        with torch.cuda.stream(streams[i]):
            results[i] = [module(x) for _ in range(20)]
            streams[i].synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(torch.equal(y, want) for ys in results.values() for y in ys) and len(results) == 3
    ops.release_workspaces()
    assert torch.equal(module(x), want)
