"""Host logic of llaccel_amd.fusion, no GPU: the rule for a short prompt's MLP in blocks of rows, and the
fused q/k/v + rope step (_GroupRopeStep): when the one-launch entry refuses a call, the two-launch path
runs; the fused entry is switched off only when those two launches take the operands (a refusal that is a
property of the graph), and an error of the call itself propagates and leaves the fused entry on."""
from __future__ import annotations

import pytest

from llaccel_amd import _lib, fusion, golden


class _Rec:
    def __init__(self, log, name, fail=False):
        self.log, self.name, self.fail = log, name, fail

    def __call__(self, M, pos, pd=None):
        self.log.append(self.name)
        if self.fail:
            raise ValueError(f"{self.name}: refused")


class _Group(_Rec):
    lins = [{"in": "x", "K": 896}]
    probs = None

    def fill(self):
        pass


class _Rope(_Rec):
    desc = (object(), object())
    parts = ()

    def _fill(self, *a):
        pass


class _Model:
    _ws = None

    def _buf(self, name):
        return None

    def _stream_handle(self):
        return None


def _step(log, monkeypatch, fused_ok, fallback_fails=False):
    def call(name, *args):
        log.append(name)
        if name == "llhip_linear_group_rope" and not fused_ok:
            raise ValueError("linear_group_rope: refused")

    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(fusion, "_vp", lambda t: None)
    monkeypatch.setattr(fusion.ctypes, "byref", lambda x: x)
    return fusion._GroupRopeStep(_Model(), _Group(log, "group", fallback_fails), _Rope(log, "rope"))


def test_fused_entry_taken(monkeypatch):
    log = []
    st = _step(log, monkeypatch, fused_ok=True)
    st(512, 0)
    st(512, 0)
    assert log == ["llhip_linear_group_rope"] * 2 and st.fused and st.launched == 2


def test_refusal_of_the_graph_switches_the_fused_entry_off(monkeypatch):
    log = []
    st = _step(log, monkeypatch, fused_ok=False)
    st(512, 0)
    assert log == ["llhip_linear_group_rope", "group", "rope"] and not st.fused
    log.clear()
    st(512, 0)  # not tried again
    assert log == ["group", "rope"]


def test_error_of_the_call_propagates_and_keeps_the_fused_entry(monkeypatch):
    log = []
    st = _step(log, monkeypatch, fused_ok=False, fallback_fails=True)
    with pytest.raises(ValueError, match="group: refused"):
        st(512, 0)
    assert st.fused and log == ["llhip_linear_group_rope", "group"]


class _Tensor:
    def __init__(self, ptr):
        self.ptr = ptr

    def data_ptr(self):
        return self.ptr


def _mlp_step(K, N, gate_up=True, at=4096):
    st = object.__new__(fusion.FusedStep)
    st.kind, st.K = "mlp_in", K
    st.ops = [{"op": "rmsnorm", "gamma": "g"}, {"op": "quant"}, {"op": "linear", "w": "wg", "N": N, "K": K},
              {"op": "linear", "w": "wu", "N": N, "K": K}]
    st.model = type("M", (), {"_dt": {"g": _Tensor(4096), "wg": _Tensor(4096), "wu": _Tensor(at)}})()
    st.wide = [object.__new__(fusion._GateUpStep)] if gate_up else [object()]
    st.blocks = st._blocks_limit()
    return st


@pytest.mark.parametrize("K,N,gate_up,most", [(576, 1536, True, 64), (768, 2048, True, 32), (1024, 1024, True, 64), (896, 4864, True, 16),
                                              (128, 384, True, 16), (64, 172, True, 128), (592, 1000, True, 128),
                                              (576, 1536, False, 128), (1024, 3072, False, 64)])
def test_mlp_rows_in_blocks(K, N, gate_up, most):
    """The largest number of rows (in whole blocks) that a short prompt's MLP runs in blocks: by the workgroups and the
    K of the GEMM it replaces, by the weights read again where there is none, 128 at most, 16 for none."""
    st = _mlp_step(K, N, gate_up)
    for M in range(17, 161):
        assert st.in_blocks(M) == (M <= most), M
        assert st.takes_wide(M) == (M > most)
    assert not st.in_blocks(16) and not st.takes_wide(16)
    assert not st.in_blocks(32, golden._SeqRows(32, 0))  # sequences of rows: the wide launches


def test_mlp_rows_in_blocks_as_the_kernel_takes_them():
    """Weights at an address that is no multiple of 16 bytes, or a width that is none, are refused by the fused kernel."""
    assert _mlp_step(576, 1536).in_blocks(32)
    assert not _mlp_step(576, 1536, at=4096 + 8).in_blocks(32)
    assert not _mlp_step(584, 1536).in_blocks(32) and not _mlp_step(1040, 1536).in_blocks(32)
