"""Fused decoder-block launches (llaccel_amd.fusion -> llhip_attn_in / llhip_mlp_in /
llhip_norm_linear) against the per-op path and the CPU oracle, bit-exact, on every
configuration shape: tiny Llama (fused and unfused graphs), SmolLM2-135M, Qwen2.5-0.5B
(QKV bias) and Qwen3-0.6B (head_dim 128, Q/K RMSNorm)."""
from __future__ import annotations

import numpy as np
import pytest

from llaccel_amd import golden as G
from llaccel_amd import synth
from oracle import golden_np as O

pytestmark = pytest.mark.gpu

_CACHE = {}


def _qgraph(tmp_path_factory, cfg, fusion=True, seed=1):
    key = (cfg, fusion, seed)
    if key not in _CACHE:
        d = tmp_path_factory.mktemp(f"{cfg}_{int(fusion)}")
        _CACHE[key] = synth.build_qgraph(d, cfg, seed=seed, fusion=fusion)
    return _CACHE[key]


def _kinds(g):
    return [getattr(s, "kind", "?") for s in g._plan]


@pytest.mark.parametrize("name", ["ref_tiny_v2", "ref_tiny_v1"])
def test_tiny_plan_is_fused_and_exact(golden_dir, name):
    qdir = golden_dir / name / "qgraph"
    g = G.GoldenModel(qdir)
    k = _kinds(g)
    assert k.count("attn_in") == 2 and k.count("mlp_in") == 2 and k.count("norm_linear") == 1
    u = G.GoldenModel(qdir, fuse=False)
    prompt = list(range(3, 23))
    a1, a2 = [], []
    assert g.generate(prompt, 6, a1) == u.generate(prompt, 6, a2)
    for s1, s2 in zip(a1, a2):
        assert set(s1["acts"]) == set(s2["acts"])
        for n in s1["acts"]:
            assert np.array_equal(s1["acts"][n], s2["acts"][n]), (s1["kind"], s1["pos"], n)


@pytest.mark.parametrize("cfg,fusion", [("smol", True), ("smol", False), ("qwen25", True), ("qwen3", True)])
def test_model_shapes_fused_vs_oracle(tmp_path_factory, cfg, fusion):
    qdir = _qgraph(tmp_path_factory, cfg, fusion)
    g = G.GoldenModel(qdir)
    k = _kinds(g)
    L = g.n_layers
    assert k.count("attn_in") == L and k.count("mlp_in") == L and k.count("norm_linear") == 1, k[:20]
    o = O.OracleModel(qdir, backend="c")
    prompt = synth.seeded_prompt(cfg, 19, 5)
    acts_g, acts_o = [], []
    rg = g.generate(prompt, 3, acts_g)      # eager launches (activations collected)
    ro = o.generate(prompt, 3, acts_o)
    assert rg == ro
    for sg, so in zip(acts_g, acts_o):
        for n in so["acts"]:
            assert np.array_equal(sg["acts"][n], so["acts"][n]), (sg["kind"], sg["pos"], n)
    for layer in (0, L - 1):
        assert np.array_equal(g.kv[layer][0], o.kv[layer][0]) and np.array_equal(g.kv[layer][1], o.kv[layer][1])
    # graph decode path (no activations requested) gives the same record
    assert g.generate(prompt, 3) == ro


def test_qwen3_preinitialised_long_context(tmp_path_factory):
    """Config 5: KV of every layer filled with seeded int8 at positions 0..4094, one decode
    launch at position 4095 (T = 4096 = 16 tiles of 256 keys)."""
    qdir = _qgraph(tmp_path_factory, "qwen3", True)
    g = G.GoldenModel(qdir)
    o = O.OracleModel(qdir, backend="c")
    rng = np.random.default_rng(4095)
    for layer in g.kv:
        shape = o.kv[layer][0].shape
        k = np.zeros(shape, np.int8)
        v = np.zeros(shape, np.int8)
        k[:, :4095] = rng.integers(-128, 128, (shape[0], 4095, shape[2]))
        v[:, :4095] = rng.integers(-128, 128, (shape[0], 4095, shape[2]))
        g.set_kv(layer, k, v)
        o.kv[layer][0][...] = k
        o.kv[layer][1][...] = v
    tok = 12345
    want = o.decode(tok, 4095)
    assert np.array_equal(g.decode(tok, 4095), want)
    kv = g.kv  # every layer's K and V region after the launch (one host snapshot)
    assert sorted(kv) == sorted(o.kv) and len(kv) == 28
    for layer in kv:
        assert np.array_equal(kv[layer][0], o.kv[layer][0]), f"K cache, layer {layer}"
        assert np.array_equal(kv[layer][1], o.kv[layer][1]), f"V cache, layer {layer}"
    # the graph decode launch at the same position rewrites the same KV row and gives the same logits
    toks, rows = g.decode_loop(tok, 4095, 1)
    assert np.array_equal(rows[0], want[:g.vocab]) and toks[0] == int(np.argmax(want[:g.vocab]))


@pytest.mark.parametrize("cfg", ["smol", "qwen25", "qwen3"])
def test_whole_prompt_prefill_large_models(tmp_path_factory, cfg):
    """Config 3-5 shapes: one M = 64 prefill launch (tiled MFMA GEMM, M-row attention; at head_dim 64
    the q/k/v GEMM with the rope/quant/kv_write epilogue) == the chunked M = 16 launches (fused
    kernels), logits and KV."""
    qdir = _qgraph(tmp_path_factory, cfg, True)
    prompt = synth.seeded_prompt(cfg, 61, 3)
    g1, g2 = G.GoldenModel(qdir), G.GoldenModel(qdir)
    g2.whole_prompt_prefill = False
    r1, r2 = g1.prefill(prompt), g2.prefill(prompt)
    assert all(np.array_equal(a, b) for a, b in zip(r1, r2))
    for layer in (0, g1.n_layers // 2, g1.n_layers - 1):
        assert np.array_equal(g1.kv[layer][0], g2.kv[layer][0]) and np.array_equal(g1.kv[layer][1], g2.kv[layer][1])
    from llaccel_amd.fusion import _GroupRopeStep

    gr = [w for st in g1._plan for w in getattr(st, "wide", None) or [] if isinstance(w, _GroupRopeStep)]
    if cfg == "qwen25":  # head_dim 64, K % 128 == 0: q, k, v with their rope, quant and kv_write in one launch
        assert gr and all(w.fused and w.launched > 0 for w in gr)
    if cfg == "smol":  # K = 576: the fused launch refuses and the two launches run
        assert gr and not any(w.fused for w in gr)


def test_prefill_graph_replays_equal_eager_launches(tmp_path_factory):
    """The second whole-prompt prefill of a shape is captured as a HIP graph and later ones replay
    it: four prefills (eager, capture + replay, replay, replay of another prompt of the same
    length), with eager decode launches between them, each equal to the eager model's logits and
    KV; a prompt of another length runs eagerly again."""
    qdir = _qgraph(tmp_path_factory, "qwen25", True)
    g, e = G.GoldenModel(qdir), G.GoldenModel(qdir)
    e.use_graph = False
    prompts = [synth.seeded_prompt("qwen25", 40, 1)] * 3 + [synth.seeded_prompt("qwen25", 40, 2),
                                                           synth.seeded_prompt("qwen25", 37, 3)]
    for i, p in enumerate(prompts):
        g.reset()
        e.reset()
        r1, r2 = g.prefill(p), e.prefill(p)
        assert all(np.array_equal(a, b) for a, b in zip(r1, r2)), i
        for layer in (0, g.n_layers - 1):
            assert np.array_equal(g.kv[layer][0], e.kv[layer][0]) and np.array_equal(g.kv[layer][1], e.kv[layer][1])
        assert np.array_equal(g.decode(5, len(p)), e.decode(5, len(p)))
    assert len(g._pf_graphs) == 1


def test_fused_and_unfused_graph_decode_agree(tmp_path_factory):
    qdir = _qgraph(tmp_path_factory, "smol", True)
    prompt = synth.seeded_prompt("smol", 33, 9)
    g, u = G.GoldenModel(qdir), G.GoldenModel(qdir, fuse=False)
    assert g.generate(prompt, 24) == u.generate(prompt, 24)


@pytest.mark.parametrize("cfg", ["smol", "qwen25", "qwen3"])
def test_prefill_batch_one_launch_equals_separate_prefills(tmp_path_factory, cfg):
    """prefill_batch of prompts of one length runs ONE launch of B x padded rows (sequence-major
    positions, slot per sequence); its logits rows and every slot's KV equal separate prefill()
    calls (each the whole-prompt launch into slot 0 of its own model)."""
    qdir = _qgraph(tmp_path_factory, cfg, True)
    B, L = 3, 61
    prompts = [synth.seeded_prompt(cfg, L, 10 + b) for b in range(B)]
    g = G.GoldenModel(qdir)
    calls = []
    one = g._prefill_seqs
    g._prefill_seqs = lambda *a: calls.append(1) or one(*a)
    rows = g.prefill_batch(prompts)
    assert calls == [1] and len(rows) == B
    for b, p in enumerate(prompts):
        s = G.GoldenModel(qdir)
        want = s.prefill(p)
        assert len(rows[b]) == L == len(want)
        assert np.array_equal(rows[b].numpy(), want.numpy()), b
        got_kv, want_kv = g.kv_of(b), s.kv
        for layer in want_kv:
            assert np.array_equal(got_kv[layer][0], want_kv[layer][0]), (b, layer)
            assert np.array_equal(got_kv[layer][1], want_kv[layer][1]), (b, layer)


def test_prefill_batch_other_lengths_run_separately(tmp_path_factory):
    """Prompts of different lengths (or one chunk long) take one prefill() per prompt."""
    qdir = _qgraph(tmp_path_factory, "qwen25", True)
    g = G.GoldenModel(qdir)
    calls = []
    one = g._prefill_seqs
    g._prefill_seqs = lambda *a: calls.append(1) or one(*a)
    prompts = [synth.seeded_prompt("qwen25", 40, 1), synth.seeded_prompt("qwen25", 33, 2)]
    rows = g.prefill_batch(prompts)
    assert calls == [] and [len(r) for r in rows] == [40, 33]
    s = G.GoldenModel(qdir)
    assert np.array_equal(np.asarray(rows[1][32]), np.asarray(s.prefill(prompts[1])[32]))


@pytest.mark.parametrize("K,N", [(576, 1536), (896, 4880), (1024, 48), (16, 32)])
@pytest.mark.parametrize("M", [2, 3, 4, 5, 7, 8, 9, 13, 16, 17, 33, 128])
def test_rows_normalised_in_the_prologue(M, K, N):
    """llhip_mlp_in of several rows normalising them in every workgroup (several waves to a row, one
    wave to one, two or more rows; from 8 rows on, past one workgroup per CU, a launch of its own) writes
    what llhip_rmsnorm_quant followed by the prequantised form writes."""
    import ctypes

    from llaccel_amd import _lib
    from tests.gpu_helpers import ptr, random_rq, stream, torch, up

    t = torch()
    rng = np.random.default_rng(100 * M + K)
    x, g = up(rng.integers(-32768, 32768, (M, K)), np.int16), up(rng.integers(-32768, 32768, K), np.int16)
    wg, wu = (up(rng.integers(-127, 128, (N, K)), np.int8) for _ in range(2))
    rqg, rqu = (up(random_rq(rng, N, K, False), np.int32) for _ in range(2))
    outs = []
    for pre in (0, 1):
        h, hq = t.zeros((M, K), dtype=t.int16, device="cuda"), t.zeros((M, K), dtype=t.int8, device="cuda")
        sg, f = (t.zeros((M, N), dtype=t.int16, device="cuda") for _ in range(2))
        fq = t.zeros((M, N), dtype=t.int8, device="cuda")
        d = _lib.MlpInDesc()
        n = d.pre
        n.x, n.gamma, n.h_out, n.hq_out, n.ldx, n.K = ptr(x), ptr(g), ptr(h), ptr(hq), K, K
        n.eps_t, n.C, n.sh_post, n.Mq, n.Sq, n.prequant = 999, int(2**24 * K**0.5), 24, 1234567891, 38, pre
        d.Wg, d.Wu, d.rqg, d.rqu = ptr(wg), ptr(wu), ptr(rqg), ptr(rqu)
        d.sg_out, d.f_out, d.fq_out = ptr(sg), ptr(f), ptr(fq)
        d.silu_Mi, d.silu_Si, d.silu_sh, d.mul_sh, d.fq_M, d.fq_S, d.M, d.N = 1 << 30, 30, 16, 11, 1 << 30, 37, M, N
        if pre:
            _lib.call("llhip_rmsnorm_quant", ctypes.byref(n), M, stream())
        if M <= 16 or not pre:
            _lib.call("llhip_mlp_in" if M <= 16 else "llhip_mlp_in_blocks", ctypes.byref(d), stream())
        else:
            for m in range(0, M, 16):
                n.x, n.h_out, n.hq_out, d.M = ptr(x[m:]), ptr(h[m:]), ptr(hq[m:]), min(16, M - m)
                d.sg_out, d.f_out, d.fq_out = ptr(sg[m:]), ptr(f[m:]), ptr(fq[m:])
                _lib.call("llhip_mlp_in", ctypes.byref(d), stream())
        outs.append([a.cpu().numpy() for a in (h, hq, sg, f, fq)])
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
    assert np.abs(outs[0][4]).max() > 0


@pytest.mark.parametrize("K,H,Hkv,D,norm", [(64, 4, 2, 16, 0), (576, 9, 3, 64, 0), (896, 14, 2, 64, 0), (1024, 4, 2, 128, 1),
                                            (768, 4, 2, 256, 1)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 12, 13, 16])
def test_attn_in_rows_normalised_in_the_prologue(M, K, H, Hkv, D, norm):
    """llhip_attn_in of one to 16 rows normalising them itself (one wave per workgroup up to sixteen, several waves
    to a row, one wave to one, two or more rows) writes what llhip_rmsnorm_quant followed by the prequantised
    form writes, rows at positions of their own."""
    import ctypes

    from llaccel_amd import _lib
    from tests.gpu_helpers import ptr, random_rq, stream, torch, up

    t = torch()
    rng = np.random.default_rng(100 * M + K)
    max_seq = 64
    x, g = up(rng.integers(-32768, 32768, (M, K)), np.int16), up(rng.integers(-32768, 32768, K), np.int16)
    cols = (H * D, Hkv * D, Hkv * D)
    w = [up(rng.integers(-127, 128, (n, K)), np.int8) for n in cols]
    rq = [up(random_rq(rng, n, K, i == 2), np.int32) for i, n in enumerate(cols)]
    hg = [up(rng.integers(-32768, 32768, D), np.int16) for _ in range(2)]
    tab = [up(rng.integers(-16384, 16385, (max_seq, D // 2)), np.int16) for _ in range(2)]
    pos = up(rng.permutation(max_seq)[:M], np.int32)
    outs = []
    for pre in (0, 1):
        def z(*shape, dt=t.int16):
            return t.zeros(shape, dtype=dt, device="cuda")

        h, hq = z(M, K), z(M, K, dt=t.int8)
        lin = [z(M, n, dt=t.int8 if i == 2 else t.int16) for i, n in enumerate(cols)]
        nrm, rope, quant = ([z(M, n, dt=dt) for n in cols[:2]] for dt in (t.int16, t.int16, t.int8))
        kc, vc = (z(M, Hkv, max_seq, D, dt=t.int8) for _ in range(2))
        d = _lib.AttnInDesc()
        n = d.pre
        n.x, n.gamma, n.h_out, n.hq_out, n.ldx, n.K = ptr(x), ptr(g), ptr(h), ptr(hq), K, K
        n.eps_t, n.C, n.sh_post, n.Mq, n.Sq, n.prequant = 999, int(2**24 * K**0.5), 24, 1234567891, 38, pre
        for i in range(3):
            d.W[i], d.rq[i], d.bias[i], d.lin_out[i] = ptr(w[i]), ptr(rq[i]), None, ptr(lin[i])
        for i in range(2):
            d.nrm_gamma[i], d.nrm_out[i] = ptr(hg[i]), ptr(nrm[i])
            d.nrm_eps[i], d.nrm_C[i], d.nrm_sh[i] = 99, int(2**22 * D**0.5), 22
            d.rope_out[i], d.quant_out[i], d.quant_M[i], d.quant_S[i] = ptr(rope[i]), ptr(quant[i]), 1234567891, 38
        d.cos_tab, d.sin_tab, d.row_pos, d.slot_stride = ptr(tab[0]), ptr(tab[1]), ptr(pos), Hkv * max_seq * D
        d.kc, d.vc, d.max_seq, d.M, d.H, d.Hkv, d.D, d.has_norm = ptr(kc), ptr(vc), max_seq, M, H, Hkv, D, norm
        if pre:
            _lib.call("llhip_rmsnorm_quant", ctypes.byref(n), M, stream())
        _lib.call("llhip_attn_in", ctypes.byref(d), stream())
        outs.append([a.cpu().numpy() for a in (h, hq, *lin, *nrm, *rope, *quant, kc, vc)])
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
    assert np.abs(outs[0][1]).max() > 0 and np.abs(outs[0][-1]).max() > 0


@pytest.mark.parametrize("K,N", [(64, 256), (576, 1040), (896, 65600)])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 16])
def test_norm_linear_rows_normalised_in_the_prologue(M, K, N):
    """llhip_norm_linear in its three forms of the rows (few and many tiles per workgroup): one launch writes what
    llhip_rmsnorm_quant followed by the prequantised form writes."""
    import ctypes

    from llaccel_amd import _lib
    from tests.gpu_helpers import ptr, random_rq, stream, torch, up

    t = torch()
    rng = np.random.default_rng(100 * M + K)
    x, g = up(rng.integers(-32768, 32768, (M, K)), np.int16), up(rng.integers(-32768, 32768, K), np.int16)
    w, rq = up(rng.integers(-127, 128, (N, K)), np.int8), up(random_rq(rng, N, K, False), np.int32)
    outs = []
    for pre in (0, 1):
        h, hq = t.zeros((M, K), dtype=t.int16, device="cuda"), t.zeros((M, K), dtype=t.int8, device="cuda")
        out = t.zeros((M, N), dtype=t.int16, device="cuda")
        d = _lib.NormLinearDesc()
        n = d.pre
        n.x, n.gamma, n.h_out, n.hq_out, n.ldx, n.K = ptr(x), ptr(g), ptr(h), ptr(hq), K, K
        n.eps_t, n.C, n.sh_post, n.Mq, n.Sq, n.prequant = 999, int(2**24 * K**0.5), 24, 1234567891, 38, pre
        d.W, d.rq, d.out, d.M, d.N, d.silu_Mi, d.silu_Si, d.silu_sh = ptr(w), ptr(rq), ptr(out), M, N, 1 << 30, 30, 16
        if pre:
            _lib.call("llhip_rmsnorm_quant", ctypes.byref(n), M, stream())
        _lib.call("llhip_norm_linear", ctypes.byref(d), stream())
        outs.append([a.cpu().numpy() for a in (h, hq, out)])
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
    assert np.abs(outs[0][2]).max() > 0


@pytest.mark.parametrize("K,N", [(64, 192), (128, 400), (896, 4128)])
@pytest.mark.parametrize("M", [4, 5, 7, 8, 12, 13, 16, 17, 40])
def test_waves_of_the_prologue(M, K, N):
    """Workgroups whose GEMM takes two and four waves, with more of them for the rows, and the rows in a launch of their own:
    eight rows and more with more workgroups than compute units."""
    test_rows_normalised_in_the_prologue(M, K, N)


def test_rows_normalised_without_quantised_rows_out():
    """Without hq_out the rows cannot come from a launch of their own: they are normalised in the workgroups."""
    import ctypes

    from llaccel_amd import _lib
    from tests.gpu_helpers import ptr, random_rq, stream, torch, up

    t = torch()
    rng = np.random.default_rng(5)
    M, K, N = 16, 64, 4128
    x, g = up(rng.integers(-32768, 32768, (M, K)), np.int16), up(rng.integers(-32768, 32768, K), np.int16)
    wg, wu = (up(rng.integers(-127, 128, (N, K)), np.int8) for _ in range(2))
    rqg, rqu = (up(random_rq(rng, N, K, False), np.int32) for _ in range(2))
    outs = []
    for out in (True, False):
        hq = t.zeros((M, K), dtype=t.int8, device="cuda") if out else None
        sg, f = (t.zeros((M, N), dtype=t.int16, device="cuda") for _ in range(2))
        fq = t.zeros((M, N), dtype=t.int8, device="cuda")
        d = _lib.MlpInDesc()
        n = d.pre
        n.x, n.gamma, n.h_out, n.hq_out, n.ldx, n.K = ptr(x), ptr(g), None, ptr(hq), K, K
        n.eps_t, n.C, n.sh_post, n.Mq, n.Sq, n.prequant = 999, int(2**24 * K**0.5), 24, 1234567891, 38, 0
        d.Wg, d.Wu, d.rqg, d.rqu = ptr(wg), ptr(wu), ptr(rqg), ptr(rqu)
        d.sg_out, d.f_out, d.fq_out = ptr(sg), ptr(f), ptr(fq)
        d.silu_Mi, d.silu_Si, d.silu_sh, d.mul_sh, d.fq_M, d.fq_S, d.M, d.N = 1 << 30, 30, 16, 11, 1 << 30, 37, M, N
        _lib.call("llhip_mlp_in", ctypes.byref(d), stream())
        outs.append([a.cpu().numpy() for a in (sg, f, fq)])
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
    assert np.abs(outs[0][2]).max() > 0


def test_short_prompt_with_misaligned_mlp_weights(golden_dir, tmp_path):
    """Weights at offsets that are no multiple of 16 bytes: a prompt of 17 to 128 rows is prefilled by the launches that
    take them, as a longer one is."""
    import json
    import shutil

    qdir = tmp_path / "q"
    shutil.copytree(golden_dir / "ref_tiny_v2" / "qgraph", qdir)
    prompt = list(range(2, 42))
    want = np.stack(list(G.GoldenModel(qdir).prefill(prompt)))
    q = json.loads((qdir / "qgraph.json").read_text())
    gate = next(o for o in q["ops"] if o["op"] == "linear" and o.get("epilogue") == "silu")["w"]
    blob = (qdir / q["weights_file"]).read_bytes()
    spec = q["tensors"][gate]
    data = blob[spec["offset"]:spec["offset"] + int(np.prod(spec["shape"]))]
    blob += bytes(-len(blob) % 16 + 8)
    spec["offset"] = len(blob)
    (qdir / q["weights_file"]).write_bytes(blob + data)
    (qdir / "qgraph.json").write_text(json.dumps(q))
    assert np.array_equal(np.stack(list(G.GoldenModel(qdir).prefill(prompt))), want)


@pytest.mark.parametrize("fuse", [True, False])
def test_prefill_rows_outlive_later_calls(golden_dir, fuse):
    """The rows that prefill() returns stay what they are: those of an eager, a captured and a replayed prefill of one
    length, read only after another prefill and a decode have run (with fuse=False the plan ends in a
    linear of its own, whose rows are copied)."""
    qdir = golden_dir / "ref_tiny_v2" / "qgraph"
    g, e = G.GoldenModel(qdir, fuse=fuse), G.GoldenModel(qdir, fuse=fuse)
    e.use_graph = False
    assert (g._head_step(32) is not None) == fuse
    prompts = [[(7 * i + 3 * j) % 60 for j in range(30)] for i in range(4)]
    kept = []
    for p in prompts:
        g.reset()
        kept.append(g.prefill(p))
    g.decode(5, 30)
    assert len(g._pf_graphs) == 1
    for i, (p, rows) in enumerate(zip(prompts, kept)):
        e.reset()
        assert np.array_equal(rows.numpy(), np.stack(list(e.prefill(p)))), i


def test_prefill_batch_rows_of_every_prompt(tmp_path_factory):
    """Prompts of other lengths, each prefilled by itself: every prompt's rows, not the last one's alone."""
    qdir = _qgraph(tmp_path_factory, "qwen25", True)
    prompts = [synth.seeded_prompt("qwen25", n, n) for n in (40, 33, 47)]
    rows = G.GoldenModel(qdir).prefill_batch(prompts)
    s = G.GoldenModel(qdir)
    for p, r in zip(prompts, rows):
        s.reset()
        assert np.array_equal(np.asarray(r[len(p) - 1]), np.asarray(s.prefill(p)[len(p) - 1]))
