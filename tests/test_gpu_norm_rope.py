"""llhip_norm_rope_quant2 (Q/K norm, rope, quant and the K/V cache write of a prompt chunk in one launch)
against llhip_rmsnorm over the heads followed by llhip_rope_quant2, bit-exact in every output and both
caches: every head_dim it takes, rows that fill no wave, extreme values, every form of positions, rows
past the table, and the optional outputs left out."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from llaccel_amd import _lib
from tests.gpu_helpers import down, ptr, stream, torch, up

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,M,H,HKV,mode", [(128, 1, 16, 8, "pos"), (128, 37, 16, 8, "pos"), (128, 64, 3, 1, "seq_rows"),
                                            (64, 5, 9, 3, "row_pos"), (256, 9, 4, 2, "pos_dev"), (64, 130, 14, 2, "past"),
                                            (128, 33, 16, 8, "lean")])
def test_equals_rmsnorm_then_rope_quant2(D, M, H, HKV, mode):
    t = torch()
    rng = np.random.default_rng(D + M)
    max_seq, rows_tab = 256, 256
    slots = M if mode == "row_pos" else M // 16 if mode == "seq_rows" else 1
    stride = HKV * max_seq * D if slots > 1 else 0
    lo, hi = (-32768, 32768) if M % 2 else (-900, 901)
    xs = [rng.integers(lo, hi, (M, h * D)) for h in (H, HKV)]
    xs[0][0, :D] = -32768
    xs[1][0, :D] = 0
    g = [up(rng.integers(-32768, 32768, D), np.int16) for _ in range(2)]
    tab = [up(rng.integers(-16384, 16385, (rows_tab, D // 2)), np.int16) for _ in range(2)]
    tab[1][3] = -32768
    v = up(rng.integers(-128, 128, (M, HKV * D)), np.int8)
    caches = [rng.integers(-128, 128, (slots, HKV, max_seq, D)) for _ in range(2)]
    row_pos = up(rng.integers(0, max_seq, M), np.int32)
    pos_dev = up(np.array([200 if mode == "past" else 7]), np.int32)  # 200: the last rows lie past the table
    norm = ((12345, int(2**22 * D**0.5), 22), (1, int(2**23 * D**0.5), 24))
    results = []
    for fused in (0, 1):
        x = [up(a, np.int16) for a in xs]
        nrm, y = ([t.full((M, h * D), 11, dtype=t.int16, device="cuda") for h in (H, HKV)] for _ in range(2))
        yq = [t.full((M, h * D), 11, dtype=t.int8, device="cuda") for h in (H, HKV)]
        kc, vc = (up(c, np.int8) for c in caches)
        d, n = [_lib.RopeQuantDesc() for _ in range(2)], [_lib.HeadNormDesc() for _ in range(2)]
        for i, h in enumerate((H, HKV)):
            d[i].x, d[i].M, d[i].H, d[i].D, d[i].ldx = ptr(x[i] if fused else nrm[i]), M, h, D, h * D
            d[i].cos_tab, d[i].sin_tab, d[i].table_rows, d[i].pos = ptr(tab[0]), ptr(tab[1]), rows_tab, 5
            d[i].pos_dev = ptr(pos_dev) if mode in ("pos_dev", "past") else None
            d[i].row_pos = ptr(row_pos) if mode == "row_pos" else None
            d[i].seq_rows = 16 if mode == "seq_rows" else 0
            d[i].y, d[i].yq, d[i].qM, d[i].qS = ptr(y[i]), ptr(yq[i]), 1234567891, 38
            d[i].max_seq, d[i].slot_stride = max_seq, stride
            n[i].gamma, n[i].out = ptr(g[i]), ptr(nrm[i])
            n[i].eps_t, n[i].C, n[i].sh_post = norm[i]
            if fused and mode == "lean":
                d[i].y = n[i].out = None
        d[1].kc, d[1].v, d[1].ldv, d[1].vc = ptr(kc), ptr(v), HKV * D, ptr(vc)
        if fused:
            _lib.call("llhip_norm_rope_quant2", ctypes.byref(d[0]), ctypes.byref(n[0]), ctypes.byref(d[1]),
                      ctypes.byref(n[1]), stream())
        else:
            for i, h in enumerate((H, HKV)):
                _lib.call("llhip_rmsnorm", ptr(x[i]), M * h, D, D, ptr(g[i]), *norm[i], ptr(nrm[i]), D, stream())
            _lib.call("llhip_rope_quant2", ctypes.byref(d[0]), ctypes.byref(d[1]), stream())
        keep = yq + [kc, vc] + ([] if mode == "lean" else nrm + y)
        results.append([down(a) for a in keep])
    for a, b in zip(*results):
        assert np.array_equal(a, b)
    d[0].D = 32
    with pytest.raises(ValueError):
        _lib.call("llhip_norm_rope_quant2", ctypes.byref(d[0]), ctypes.byref(n[0]), ctypes.byref(d[1]), ctypes.byref(n[1]),
                  stream())


@pytest.mark.parametrize("M,n,dim", [(1, 1, 64), (16, 5, 576), (300, 300, 896), (7, 0, 8), (5, 3, 12)])
def test_embedding_rows(M, n, dim):
    rng = np.random.default_rng(M + dim)
    table = rng.integers(-32768, 32768, (50, dim))
    tok = rng.integers(0, 50, max(n, 1))
    out = torch().full((M, dim), 7, dtype=torch().int16, device="cuda")
    td, ed = up(tok, np.int32), up(table, np.int16)
    _lib.call("llhip_embed_rows", ptr(ed), 50, dim, ptr(td), n, M, ptr(out), stream())
    want = np.zeros((M, dim), np.int64)
    want[:n] = table[tok[:n]]
    assert np.array_equal(down(out), want)
