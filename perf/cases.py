"""What a user of this framework has it do, as a list of cases that can be timed and compared.

Four kinds of work, all through the public entry points:
  linear     one ternary product: `TernaryLinear` (the module) or `ter_spmm.ter_spmm` on merged tiled-CSC arrays (the drop-in)
  mlp        the SiLU-gated block of three ternary products, `LlamaTernaryMLP`
  attention  the attention block with ternary projections, `LlamaTernaryAttention`
  prefill / decode  a decoder whose linear layers are all ternary, `TernaryLlamaDecoder`: a prompt, or one step of a
             serving loop that samples on its own and hands the next token over (the step replayed from its HIP graph)

The path has inference only: prefill (many rows) and decode (few rows) are its two directions.  A case is a dict of
plain values; `draw` makes more of the same ranges.
"""
import math

import torch

import ter_spmm
from ternaryllm_amd import LlamaTernaryAttention, LlamaTernaryMLP, TernaryConfig, TernaryLinear, TernaryLlamaDecoder, convert_ternary_weights

DTYPES = {"float16": torch.float16, "float32": torch.float32}
MAX_WEIGHTS = 46_000_000     # ternary weights of a drawn product: the largest single weight that is listed
CACHE_ROWS = 640             # 512 prompt tokens and 128 new ones


def _linear(name, rows, K, N, sparsity, dtype="float16", entry="module", layout="rows", scaled=True):
    case = {"kind": "linear", "rows": rows, "K": K, "N": N, "sparsity": sparsity, "dtype": dtype, "entry": entry, "layout": layout, "scaled": scaled}
    return dict(case, name=name) if name else case


def _mlp(name, rows, hidden, inner, sparsity, dtype="float16"):
    case = {"kind": "mlp", "rows": rows, "hidden": hidden, "inner": inner, "sparsity": sparsity, "dtype": dtype}
    return dict(case, name=name) if name else case


def _attention(name, batch, seq, heads, sparsity, dtype="float16"):
    case = {"kind": "attention", "batch": batch, "seq": seq, "heads": heads, "sparsity": sparsity, "dtype": dtype}
    return dict(case, name=name) if name else case


def _decoder(name, kind, batch, prompt, heads, inner, layers, vocab, sparsity=0.66):
    case = {"kind": kind, "batch": batch, "prompt": prompt, "heads": heads, "inner": inner, "layers": layers, "vocab": vocab, "sparsity": sparsity}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one token through a square projection: the smallest call a decode loop makes, where launch and latency count
        _linear("row_4096x4096", 1, 4096, 4096, 0.66),
        # one token through a wide-K projection of a very sparse weight
        _linear("row_11008x4096_sparse", 1, 11008, 4096, 0.95),
        # the drop-in extension call on a small fp32 batch
        _linear("dropin_16rows_fp32", 16, 4096, 4096, 0.5, "float32", "dropin", scaled=False),
        # odd sizes everywhere: 37 rows, K and N that divide by nothing
        _linear("ragged_37x1003x777", 37, 1003, 777, 0.7),
        # the layout the reference kernel itself reads, [batch, K, rows], fp32, a few hundred rows
        _linear("kmajor_200rows_fp32", 200, 2048, 2048, 0.8, "float32", "dropin", "kmajor", scaled=False),
        # a prompt's worth of fp32 rows, the reference's own activation type
        _linear("rows1024_fp32", 1024, 4096, 4096, 0.9, "float32"),
        # the MLP block on 8 x 128 tokens at the reference's benchmark width
        _mlp("mlp_1024", 1024, 4096, 11008, 0.8),
        # the MLP block on a handful of tokens (speculative tokens, a small batch)
        _mlp("mlp_8", 8, 2048, 5504, 0.8),
        # the attention block on 8 x 128 tokens
        _attention("attention_8x128", 8, 128, 32, 0.9),
        # one decode step, a single sequence and a batch of 16
        _decoder("decode_1", "decode", 1, 512, 16, 5504, 2, 8000),
        _decoder("decode_16", "decode", 16, 512, 16, 5504, 2, 8000),
        # a batch of 16 prompts of 512 tokens: the largest pass
        _decoder("prefill_16x512", "prefill", 16, 512, 16, 5504, 2, 8000),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _size(rng, low, high):
    """A width: mostly whole multiples of 64, one in four odd."""
    n = _log_int(rng, low, high)
    return n if rng.random() < 0.25 else max(64, n // 64 * 64)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "mlp", "mlp", "attention", "decode", "decode", "prefill"])
    sparsity = round(rng.uniform(0.5, 0.97), 3)
    dtype = rng.choice(["float16", "float16", "float16", "float32"])
    if kind == "linear":
        K, N = _size(rng, 256, 11008), _size(rng, 128, 11008)
        while K * N > MAX_WEIGHTS:
            K, N = _size(rng, 256, 11008), _size(rng, 128, 11008)
        rows = rng.choice([1, _log_int(rng, 2, 48), _log_int(rng, 2, 48), _log_int(rng, 49, 4096)])
        entry = rng.choice(["module", "module", "dropin"])
        layout = "kmajor" if rows > 1 and rows != K and rng.random() < 0.2 else "rows"
        if rows == K:
            rows += 1
        return _linear(None, rows, K, N, sparsity, dtype, entry, layout, entry == "module" and rng.random() < 0.7)
    if kind == "mlp":
        return _mlp(None, rng.choice([_log_int(rng, 1, 48), _log_int(rng, 49, 2048)]), _size(rng, 512, 4096), _size(rng, 1024, 5504), sparsity, dtype)
    if kind == "attention":
        return _attention(None, _log_int(rng, 1, 8), _log_int(rng, 1, 256), rng.randint(4, 32), sparsity, dtype)
    heads = rng.randint(4, 16)
    inner = max(512, _log_int(rng, 1024, 5504) // 8 * 8)
    if kind == "decode":
        return _decoder(None, kind, _log_int(rng, 1, 32), _log_int(rng, 16, 600), heads, inner, rng.randint(1, 2), rng.randint(500, 8000), sparsity)
    batch = _log_int(rng, 1, 16)
    return _decoder(None, kind, batch, _log_int(rng, 16, 8192 // max(16, batch)), heads, inner, rng.randint(1, 2), rng.randint(500, 8000), sparsity)


def _weight(K, N, sparsity, gen):
    """Ternary [K, N] drawn on the GPU by the reference's rule: sparsity zeros, the rest half +1 and half -1, i.i.d."""
    r = torch.rand((K, N), generator=gen, device="cuda")
    return ((r >= (sparsity + 1) / 2).to(torch.int32) - ((r >= sparsity) & (r < (sparsity + 1) / 2)).to(torch.int32)).cpu()


def _scale(K, N, sparsity, gen, dtype):
    """Per-output-channel factors U(0.5, 1.5) / sqrt(non-zeros of a column): outputs keep the magnitude of the inputs."""
    return ((0.5 + torch.rand(N, generator=gen, device="cuda")) / math.sqrt(max(1.0, K * (1 - sparsity)))).to(dtype).cpu()


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    cpu_gen = torch.Generator().manual_seed(seed)
    kind = case["kind"]

    def normal(*shape, dtype):
        return torch.randn(shape, generator=gen, device="cuda").to(dtype)

    if kind == "linear":
        K, N, rows, dtype = case["K"], case["N"], case["rows"], DTYPES[case["dtype"]]
        w = _weight(K, N, case["sparsity"], gen)
        x = normal(1, K, rows, dtype=dtype) if case["layout"] == "kmajor" else normal(1, rows, K, dtype=dtype)
        if case["entry"] == "module":
            scale = _scale(K, N, case["sparsity"], gen, dtype) if case["scaled"] else None
            return {"case": case, "x": x, "module": TernaryLinear(K, N, weight=w, scale=scale, bias=False, reference_buffers=False).to("cuda")}
        rows_idx, offsets, tiles = convert_ternary_weights(w, dtype=torch.int16, device="cuda")
        ter_spmm.prepare(rows_idx, offsets, N, K)
        return {"case": case, "x": x, "arrays": (rows_idx, offsets, tiles)}
    if kind == "mlp":
        H, inner, dtype = case["hidden"], case["inner"], DTYPES[case["dtype"]]
        cfg = TernaryConfig(hidden_size=H, intermediate_size=inner, sparsity=case["sparsity"])
        scales = {"gate": _scale(H, inner, case["sparsity"], gen, dtype), "up": _scale(H, inner, case["sparsity"], gen, dtype),
                  "down": _scale(inner, H, case["sparsity"], gen, dtype)}
        block = LlamaTernaryMLP(cfg, generator=cpu_gen, scales=scales, reference_buffers=False).to("cuda")
        return {"case": case, "x": normal(1, case["rows"], H, dtype=dtype), "module": block}
    if kind == "attention":
        H, dtype = case["heads"] * 128, DTYPES[case["dtype"]]
        cfg = TernaryConfig(hidden_size=H, num_attention_heads=case["heads"], num_key_value_heads=case["heads"], sparsity=case["sparsity"])
        block = LlamaTernaryAttention(cfg, generator=cpu_gen, reference_buffers=False).to("cuda")
        for p in (block.q_proj, block.k_proj, block.v_proj, block.o_proj):
            p.w_scale = _scale(H, H, case["sparsity"], gen, dtype).to("cuda")
        with torch.no_grad():
            block(normal(1, 2, H, dtype=dtype))  # the block lays its q | k | v weight side by side at its first call
        return {"case": case, "x": normal(case["batch"], case["seq"], H, dtype=dtype), "module": block}
    H = case["heads"] * 128
    cache_rows = CACHE_ROWS if kind == "decode" else case["prompt"]
    cfg = TernaryConfig(hidden_size=H, intermediate_size=case["inner"], num_hidden_layers=case["layers"], num_attention_heads=case["heads"],
                        num_key_value_heads=case["heads"], vocab_size=case["vocab"], max_position_embeddings=cache_rows, sparsity=case["sparsity"])
    model = TernaryLlamaDecoder(cfg, seed=seed, device="cuda", pack_threads=8)
    B = case["batch"]
    tokens = torch.randint(0, case["vocab"], (B, case["prompt"]), generator=gen, device="cuda")
    state = {"case": case, "module": model, "tokens": tokens, "cache": model.allocate_cache(B)}
    if kind == "decode":
        model.prefill(tokens)
        steps = {"token": torch.zeros(B, dtype=torch.long, device="cuda"), "pos": torch.zeros(1, dtype=torch.long, device="cuda"),
                 "mask": torch.zeros((1, 1, 1, cache_rows), dtype=torch.bool, device="cuda")}

        def at_the_end_of_the_prompt():
            steps["token"].copy_(tokens[:, -1])
            steps["pos"].fill_(case["prompt"])
            steps["mask"].copy_((torch.arange(cache_rows, device="cuda") <= case["prompt"])[None, None, None])

        at_the_end_of_the_prompt()
        model.decode_once(steps)  # captures the step's graph, which a program keeps for all its steps
        at_the_end_of_the_prompt()
        state["steps"] = steps
        state["sampled"] = torch.randint(0, case["vocab"], (B,), generator=gen, device="cuda")
    return state


@torch.no_grad()
def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "linear":
        if "module" in state:
            return state["module"](state["x"])
        rows_idx, offsets, tiles = state["arrays"]
        return ter_spmm.ter_spmm(state["x"], rows_idx, offsets, tiles, 1, case["rows"], case["N"], case["K"], False, False,
                                 x_layout="k_major" if case["layout"] == "kmajor" else None)
    if kind == "mlp":
        return state["module"](state["x"])
    if kind == "attention":
        out, _, (k, v) = state["module"](state["x"], use_cache=True)
        return out, k, v
    model = state["module"]
    if kind == "prefill":
        return model.prefill(state["tokens"]), state["cache"]
    # the caller's own sampler chose the token; the step itself moves the position on (and stays at the cache's last row)
    state["steps"]["token"].copy_(state["sampled"])
    model.decode_once(state["steps"])
    return model.last_logits, state["cache"]


def _weight_bytes(K, N, sparsity):
    """What a random ternary matrix of this sparsity cannot be told in less than: its entropy."""
    s = sparsity
    bits = -s * math.log2(s) - (1 - s) * math.log2((1 - s) / 2)
    return K * N * bits / 8


def work(case):
    """Bytes: every weight at its entropy, every activation, scale and cache row once.  Operations: one addition per row
    and non-zero weight, and two per multiply-add of the attention."""
    kind, s = case["kind"], case["sparsity"]
    if kind == "linear":
        K, N, M = case["K"], case["N"], case["rows"]
        es = 2 if case["dtype"] == "float16" else 4
        return {"bytes": _weight_bytes(K, N, s) + (M * K + M * N + (N if case["scaled"] else 0)) * es, "flops": M * K * N * (1 - s)}
    if kind == "mlp":
        H, inner, M = case["hidden"], case["inner"], case["rows"]
        es = 2 if case["dtype"] == "float16" else 4
        return {"bytes": 3 * _weight_bytes(H, inner, s) + (2 * M * H + 2 * inner + H) * es, "flops": 3 * M * H * inner * (1 - s)}
    if kind == "attention":
        H, B, S = case["heads"] * 128, case["batch"], case["seq"]
        es = 2 if case["dtype"] == "float16" else 4
        return {"bytes": 4 * _weight_bytes(H, H, s) + (4 * B * S * H + 4 * H) * es, "flops": 4 * B * S * H * H * (1 - s) + 2 * B * S * (S + 1) * H}
    H, inner, L, V, B = case["heads"] * 128, case["inner"], case["layers"], case["vocab"], case["batch"]
    per_layer = 4 * H * H + 3 * H * inner
    weights = L * (4 * _weight_bytes(H, H, s) + 3 * _weight_bytes(H, inner, s)) + _weight_bytes(H, V, s)
    small = (L * (9 * H + 3 * inner) + H + V) * 2 + B * (H + V) * 2
    if kind == "decode":
        rows = case["prompt"] + 1
        return {"bytes": weights + small + L * 2 * B * rows * H * 2,
                "flops": B * (L * per_layer + H * V) * (1 - s) + L * B * 4 * rows * H}
    S = case["prompt"]
    return {"bytes": weights + small + B * S * (H + L * 2 * H) * 2,
            "flops": B * (S * L * per_layer + H * V) * (1 - s) + L * B * 2 * S * (S + 1) * H}


def tolerance(case):
    """Four times the largest error against float64 that was measured over the listed cases and fourteen drawn ones
    (rel: fp32 3.7e-7 and, with the attention in between, 5.4e-7; fp16 2.1e-4 for a product, whose result is rounded
    once, 3.0e-4 for the MLP block, 5.9e-4 for the attention block, 1.5e-3 for the logits of a decoder)."""
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return {"rel": 6e-3}
    if case["dtype"] == "float32":
        return {"rel": 2e-6}
    return {"rel": {"linear": 8e-4, "mlp": 1.2e-3, "attention": 2.4e-3}[kind]}
