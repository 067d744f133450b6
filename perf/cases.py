"""What the framework is measured on: generation with quantized decoder graphs -- prompt prefill, greedy decode and
batch decode through GoldenModel -- and the two device entry points its producers and tests call directly, the INT8
GEMM (llhip_linear) and the per-channel weight quantizer (llhip_quant_rows_i8).

The models are the seeded synthetic graphs of llaccel_amd.synth at the repository's own shapes, written once to
$LLACCEL_BENCH_DIR (default: the temporary folder) and loaded from there; a graph's weights are a program's fixed
data, the prompts, tokens and KV-cache contents come from the seed.  "qwen3" runs 8 of its 28 layers, which keeps
loading quick; every layer is alike.  All outputs are integers of an exactly specified datapath (or, for the
quantizer's scales, one double division), so every case is compared exactly."""
from __future__ import annotations

import ctypes
import dataclasses
import functools
import os
import shutil
import tempfile
from pathlib import Path

import numpy as np
import torch

from llaccel_amd import _lib, golden, synth

# graph name -> (configuration, layers or None for all, fused epilogues).  "smol_v1" is the same shape written for
# the accelerator's first target: add, silu and mul as ops of their own.
GRAPHS = {"tiny": ("tiny", None, True), "smol": ("smol", None, True), "smol_v1": ("smol", None, False),
          "qwen25": ("qwen25", None, True), "qwen3": ("qwen3", 8, True)}
# (K, N) of the linear layers of the "qwen25" shape and of odd widths beside them
GEMM_SHAPES = ((896, 151936), (896, 4864), (4864, 896), (896, 896), (576, 1536), (1536, 576), (1000, 777))


def config(graph):
    name, layers, _ = GRAPHS[graph]
    cfg = synth.CONFIGS[name]
    return cfg if layers is None else dataclasses.replace(cfg, n_layers=layers)


def graph_dir(graph):
    """The graph's folder, written by the first process that needs it."""
    root = Path(os.environ.get("LLACCEL_BENCH_DIR", Path(tempfile.gettempdir()) / "llaccel_bench"))
    _, layers, fusion = GRAPHS[graph]
    final = root / f"case_{graph}_l{layers or 'all'}_s0"
    if not (final / "qgraph.json").exists():
        root.mkdir(parents=True, exist_ok=True)
        part = Path(tempfile.mkdtemp(prefix=final.name, dir=root))
        synth.build_qgraph(part, config(graph), seed=0, fusion=fusion)
        try:
            os.rename(part, final)
        except OSError:  # another process was first
            shutil.rmtree(part, ignore_errors=True)
    return final


def listed():
    return [
        # the whole call a small program makes, record and all: launches and host work, no bandwidth
        {"name": "generate_tiny", "do": "generate", "graph": "tiny", "prompt": 8, "steps": 16},
        # one user, a short chat turn on the small model
        {"name": "decode_smol", "do": "decode", "graph": "smol", "pos": 40, "steps": 16},
        # one user after a 512-token prompt: the benchmark's headline workload
        {"name": "decode_qwen25", "do": "decode", "graph": "qwen25", "pos": 760, "steps": 8},
        # one user at the end of a long context, with Q/K norm and head_dim 128
        {"name": "decode_qwen3_long", "do": "decode", "graph": "qwen3", "pos": 4077, "steps": 8},
        # a few users of an unfused graph, at unequal positions
        {"name": "decode_batch3_smol_v1", "do": "batch", "graph": "smol_v1", "batch": 3, "pos": 61, "spread": 7,
         "steps": 8},
        # a full decode batch, at unequal positions
        {"name": "decode_batch16_qwen25", "do": "batch", "graph": "qwen25", "batch": 16, "pos": 512, "spread": 13,
         "steps": 8},
        # a short prompt of odd length
        {"name": "prefill_smol_53", "do": "prefill", "graph": "smol", "prompt": 53},
        # the benchmark's prompt
        {"name": "prefill_qwen25_512", "do": "prefill", "graph": "qwen25", "prompt": 512},
        # a long prompt of odd length, Q/K norm and head_dim 128
        {"name": "prefill_qwen3_1531", "do": "prefill", "graph": "qwen3", "prompt": 1531},
        # sixteen prompts at once
        {"name": "prefill_batch16_qwen25", "do": "prefill_batch", "graph": "qwen25", "batch": 16, "prompt": 512},
        # one large linear layer by itself: the output head over a long prompt
        {"name": "linear_2048x896x151936", "do": "linear", "rows": 2048, "k": 896, "n": 151936, "out": "i8", "aux": False},
        # the quantizer on the output head's weights
        {"name": "quantize_151936x896", "do": "quantize", "n": 151936, "k": 896},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    do = rng.choice(("generate", "decode", "decode", "batch", "batch", "prefill", "prefill", "prefill_batch", "linear",
                     "linear", "quantize"))
    if do == "generate":
        prompt = _log_int(rng, 1, 40)
        return {"do": do, "graph": "tiny", "prompt": prompt, "steps": _log_int(rng, 1, 63 - prompt)}
    if do == "decode":
        graph = rng.choice(("tiny", "smol", "smol_v1", "qwen25", "qwen3"))
        steps = rng.randint(4, 8)
        return {"do": do, "graph": graph, "pos": _log_int(rng, 1, config(graph).max_seq - steps), "steps": steps}
    if do == "batch":
        graph = rng.choice(("smol", "smol_v1", "qwen25"))
        batch, spread, steps = _log_int(rng, 2, 16), rng.randint(0, 13), rng.randint(4, 8)
        top = min(512, config(graph).max_seq - steps - spread * 15)
        return {"do": do, "graph": graph, "batch": batch, "pos": _log_int(rng, 1, top), "spread": spread, "steps": steps}
    if do == "prefill":
        graph = rng.choice(("smol", "smol_v1", "qwen25", "qwen3"))
        return {"do": do, "graph": graph, "prompt": _log_int(rng, 3, min(config(graph).max_seq, 1600))}
    if do == "prefill_batch":
        graph = rng.choice(("smol", "qwen25"))
        return {"do": do, "graph": graph, "batch": rng.randint(2, 16),
                "prompt": _log_int(rng, 17, min(512, config(graph).max_seq))}
    if do == "linear":
        k, n = rng.choice(GEMM_SHAPES)
        out = rng.choice(("i8", "i16"))
        return {"do": do, "rows": _log_int(rng, 1, 2048), "k": k, "n": n, "out": out,
                "aux": out == "i16" and rng.random() < 0.5}
    return {"do": do, "n": _log_int(rng, 64, 151936), "k": rng.choice((576, 777, 896, 1024, 3072, 4864 // 4))}


# --------------------------------------------------------------------------------------
# prepare
# --------------------------------------------------------------------------------------
def _tokens(cfg, rng, n):
    return [int(t) for t in rng.integers(0, cfg.vocab, n)]


def _linear_inputs(case, seed):
    """A [rows][k] and W [n][k] int8, per-column requantization that spreads the outputs over their type, and the
    residual rows of the resadd epilogue."""
    M, K, N = case["rows"], case["k"], case["n"]
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 11)
    r8 = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device="cuda", generator=g)  # noqa: E731
    a, w = r8(M, K), r8(N, K)
    mult = torch.randint(1 << 30, (1 << 31) - 1, (N,), dtype=torch.int64, device="cuda", generator=g)
    # accumulators have a spread of about 73 * 73 * sqrt(K); M * 2^-S takes that to a third of the output's range
    shift = 30 + round(np.log2(73 * 73 * K ** 0.5 * 1.5 / (42 if case["out"] == "i8" else 10900)))
    rq = torch.stack([mult.to(torch.int32), torch.full((N,), shift, dtype=torch.int32, device="cuda")], 1).contiguous()
    aux = torch.randint(-9000, 9001, (M, N), dtype=torch.int16, device="cuda", generator=g) if case["aux"] else None
    return a, w, rq, aux


def _quantize_input(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 17)
    w = torch.randn((case["n"], case["k"]), dtype=torch.float32, device="cuda", generator=g) * 0.02
    w[seed % case["n"]] = 0.0  # a dead output channel
    return w


def prepare(case, seed):
    do = case["do"]
    if do == "linear":
        a, w, rq, aux = _linear_inputs(case, seed)
        out = torch.empty((case["rows"], case["n"]), dtype=torch.int8 if case["out"] == "i8" else torch.int16, device="cuda")
        ws = torch.zeros(int(_lib.lib().llhip_workspace_bytes()), dtype=torch.uint8, device="cuda")
        return {"case": case, "a": a, "w": w, "rq": rq, "aux": aux, "out": out, "ws": ws}
    if do == "quantize":
        n, k = case["n"], case["k"]
        return {"case": case, "w": _quantize_input(case, seed), "q": torch.empty((n, k), dtype=torch.int8, device="cuda"),
                "scales": torch.empty(n, dtype=torch.float64, device="cuda"),
                "status": torch.zeros(1, dtype=torch.int32, device="cuda")}
    cfg = config(case["graph"])
    rng = np.random.default_rng(seed)
    g = golden.GoldenModel(graph_dir(case["graph"]))
    state = {"case": case, "model": g}
    if do in ("generate", "prefill"):
        state["prompt"] = _tokens(cfg, rng, case["prompt"])
    elif do == "prefill_batch":
        state["prompts"] = [_tokens(cfg, rng, case["prompt"]) for _ in range(case["batch"])]
    elif do == "decode":
        # a context in the cache, as an earlier prefill leaves it; what lies past it is stale
        shape = (cfg.n_kv_heads, cfg.max_seq, cfg.head_dim)
        for layer in range(cfg.n_layers):
            g.set_kv(layer, rng.integers(-100, 101, shape, dtype=np.int8), rng.integers(-100, 101, shape, dtype=np.int8))
        state["token"] = _tokens(cfg, rng, 1)[0]
    else:  # batch: the prompts are prefilled, the decode starts where each ends
        state["positions"] = [case["pos"] + case["spread"] * (b * 7 % case["batch"]) for b in range(case["batch"])]
        g.prefill_batch([_tokens(cfg, rng, p) for p in state["positions"]])
        state["tokens"] = _tokens(cfg, rng, case["batch"])
    return state


# --------------------------------------------------------------------------------------
# run
# --------------------------------------------------------------------------------------
def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _cache(g):
    """The K/V caches of all layers and slots: the one device allocation that they are views of."""
    return next(iter(g._kv.values()))[0]._base


def run(state):
    case = state["case"]
    do = case["do"]
    if do == "linear":
        M, K, N = case["rows"], case["k"], case["n"]
        _lib.call("llhip_linear", _p(state["a"]), M, K, K, _p(state["w"]), N, _p(state["rq"]), None, int(case["aux"]),
                  _p(state["aux"]), N, 0, 0, 0, 0, int(case["out"] == "i8"), _p(state["out"]), N, _p(state["ws"]), _stream())
        return state["out"]
    if do == "quantize":
        n, k = case["n"], case["k"]
        _lib.call("llhip_quant_rows_i8", _p(state["w"]), n, k, k, _p(state["q"]), k, _p(state["scales"]),
                  _p(state["status"]), _stream())
        return [state["q"], state["scales"], state["status"]]
    g = state["model"]
    if do == "generate":
        rec = g.generate(state["prompt"], case["steps"])
        return {"argmax": np.array(rec["argmax_per_step"]), "logits": np.array(rec["logits_last_rows"]), "kv": _cache(g)}
    if do == "decode":
        g.decode_loop(state["token"], case["pos"], case["steps"], sync=False)
        return [*g.decode_ring(case["steps"]), _cache(g)]
    if do == "batch":  # the device record that decode_batch_loop downloads when it is asked to wait
        n = case["steps"]
        g.decode_batch_loop(state["tokens"], state["positions"], n, sync=False)
        return [g._b_ring_tok[:n], g._b_ring_rows[:n], _cache(g)]
    if do == "prefill":
        rows = g.prefill(state["prompt"])
        return [rows._rows if isinstance(rows, golden.DeviceRows) else np.stack(rows), _cache(g)]
    rows = g.prefill_batch(state["prompts"])
    return [r._rows if isinstance(r, golden.DeviceRows) else np.stack(r) for r in rows] + [_cache(g)]


# --------------------------------------------------------------------------------------
# work, tolerance, exact
# --------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _sizes(graph):
    c = config(graph)
    layer = c.dim * (c.n_heads + 2 * c.n_kv_heads) * c.head_dim + c.n_heads * c.head_dim * c.dim + 3 * c.dim * c.ffn
    columns = (c.n_heads + 2 * c.n_kv_heads) * c.head_dim + 2 * c.ffn + 2 * c.dim
    weights = c.n_layers * layer + c.vocab * c.dim  # int8: bytes and values alike
    tables = 8 * (c.n_layers * columns + c.vocab)  # requantization pairs
    kv = 2 * c.n_layers * c.n_kv_heads * c.head_dim  # cache bytes of one position
    pair = 4 * c.n_layers * c.n_heads * c.head_dim  # operations of one (query, key) pair, all heads and layers
    return c, weights, tables, kv, pair


def _launch(graph, contexts):
    """One launch of a row per context length in `contexts` (each row its own sequence)."""
    c, weights, tables, kv, pair = _sizes(graph)
    rows, keys = len(contexts), sum(contexts)
    return np.array([weights + tables + kv * (keys + rows) + rows * 2 * (c.dim + c.vocab),
                     2 * rows * weights + pair * keys], dtype=np.float64)


def _prompts(graph, batch, length):
    c, weights, tables, kv, pair = _sizes(graph)
    rows = batch * length
    return np.array([weights + tables + 2 * kv * rows + rows * 2 * (c.dim + c.vocab),
                     2 * rows * weights + pair * batch * length * (length + 1) / 2], dtype=np.float64)


def work(case):
    do = case["do"]
    if do == "linear":
        M, K, N = case["rows"], case["k"], case["n"]
        out = 1 if case["out"] == "i8" else 2
        return {"bytes": M * K + N * K + 8 * N + M * N * (out + (2 if case["aux"] else 0)), "flops": 2 * M * N * K}
    if do == "quantize":
        return {"bytes": case["n"] * (5 * case["k"] + 8), "flops": 3 * case["n"] * case["k"]}
    graph = case["graph"]
    if do == "generate":
        w = _prompts(graph, 1, case["prompt"]) + sum(_launch(graph, [case["prompt"] + i + 1]) for i in range(case["steps"]))
    elif do == "decode":
        w = sum(_launch(graph, [case["pos"] + i + 1]) for i in range(case["steps"]))
    elif do == "batch":
        at = [case["pos"] + case["spread"] * (b * 7 % case["batch"]) for b in range(case["batch"])]
        w = sum(_launch(graph, [p + i + 1 for p in at]) for i in range(case["steps"]))
    else:
        w = _prompts(graph, case.get("batch", 1), case["prompt"])
    return {"bytes": float(w[0]), "flops": float(w[1])}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The two single operations in 64 bits.  The model calls compute integers that have one right value; restating
    the whole datapath over a model takes longer than a case may."""
    if case["do"] == "linear":
        a, w, rq, aux = _linear_inputs(case, seed)
        lo, hi = (-128, 127) if case["out"] == "i8" else (-32768, 32767)
        wt = w.double().t().contiguous()
        parts = []
        for i in range(0, case["rows"], 128):
            acc = (a[i:i + 128].double() @ wt).to(torch.int64)  # below 2^53: exact
            y = (acc * rq[:, 0].to(torch.int64) + (1 << (int(rq[0, 1]) - 1))) >> int(rq[0, 1])
            y = y.clamp(lo, hi)
            if aux is not None:
                y = (y + aux[i:i + 128]).clamp(lo, hi)
            parts.append(y.to(torch.int16))
        return torch.cat(parts)
    if case["do"] == "quantize":
        w = _quantize_input(case, seed).double()
        top = w.abs().amax(1)
        scales = torch.where(top > 0, top / torch.full_like(top, 127.0), torch.ones_like(top))
        v = (w / scales[:, None]).clamp(-128, 127)
        q = torch.where(v < 0, torch.ceil(v - 0.5), torch.floor(v + 0.5))
        return [q.to(torch.int8), scales, torch.zeros(1, dtype=torch.int32)]
    return None
