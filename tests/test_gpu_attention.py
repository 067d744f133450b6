"""GPU parity of the attn engine (kv_write + causal GQA attention) against the CPU oracle,
bit-exact, including BASELINE config 5's long-context shapes (T = 4096 = 16 tiles of 256,
head_dim 128 and the head_dim-256 extra case)."""
from __future__ import annotations

import numpy as np
import pytest

from llaccel_amd import _lib
from oracle import golden_np as O
from tests.gpu_helpers import down, ptr, stream, up, workspace

pytestmark = pytest.mark.gpu


def gpu_attention(q, kc, vc, pos, H, Hkv, D, Ms, Ss, Mo, So, pb):
    t = __import__("torch")
    M = q.shape[0]
    qd, kd, vd = up(q, np.int8), up(kc, np.int8), up(vc, np.int8)
    out = t.empty((M, H * D), dtype=t.int8, device="cuda")
    _lib.call("llhip_attention", ptr(qd), M, H, Hkv, D, H * D, pos, None, None, 0, ptr(kd), ptr(vd), kc.shape[1], Ms,
              Ss, Mo, So, pb, ptr(out), H * D, ptr(workspace()), stream())
    return down(out)


CASES = [
    # M, H, Hkv, D, pos, max_seq
    (1, 4, 2, 16, 47, 64),
    (16, 4, 2, 16, 0, 64),
    (16, 9, 3, 64, 112, 256),
    (1, 14, 2, 64, 767, 1024),
    (16, 14, 2, 64, 496, 1024),
    (1, 16, 8, 128, 4095, 4096),
    (1, 8, 2, 256, 4095, 4096),
    (16, 8, 2, 256, 4080, 4096),
    (3, 2, 1, 32, 254, 260),
    # multi-row launches (the 16-row MFMA kernel): prompt-sized blocks, ragged row counts, every D
    (200, 14, 2, 64, 0, 256),
    (512, 14, 2, 64, 0, 512),
    (33, 16, 8, 128, 100, 256),
    (17, 4, 2, 32, 40, 64),
    (2, 8, 2, 256, 61, 128),
    (45, 2, 2, 16, 3, 64),
    # long contexts with few (row block, head) pairs: the key tiles split over workgroups
    (16, 16, 8, 128, 4080, 4096),
    (20, 8, 2, 64, 3000, 4096),
    (3, 4, 2, 32, 2500, 3000),
    (1, 2, 1, 16, 2047, 2048),
    # launches of more waves than fit three to a SIMD (a batched prefill's size)
    (2048, 14, 2, 64, 0, 2048),
    (1024, 8, 2, 16, 0, 1024),
    (1024, 8, 4, 32, 0, 1024),
    # four waves with more tiles than their registers hold (probabilities in LDS), and eight waves with
    # more than the LDS holds as well (recomputed in the value pass); a ragged last row block
    (800, 14, 2, 64, 0, 1024),
    (602, 16, 8, 128, 0, 640),
    (250, 16, 8, 128, 3840, 4096),
]


@pytest.mark.parametrize("M,H,Hkv,D,pos,max_seq", CASES)
def test_attention_matches_oracle(M, H, Hkv, D, pos, max_seq):
    rng = np.random.default_rng(M * 1000 + H * 10 + D + pos)
    kc = rng.integers(-128, 128, (Hkv, max_seq, D)).astype(np.int8)
    vc = rng.integers(-128, 128, (Hkv, max_seq, D)).astype(np.int8)
    q = rng.integers(-128, 128, (M, H * D))
    # score scale chosen so softmax is neither one-hot nor flat: the score spread
    # (std ~ 5372 sqrt(D) for uniform i8 operands) maps to z ~ 768, i.e. e^-3
    Ms, Ss = int(rng.integers(1 << 30, 1 << 31)), 31 + int(round(np.log2(5372 * np.sqrt(D) / 768)))
    Mo, So = int(rng.integers(1 << 30, 1 << 31)), 38
    for pb in (15, 8):
        got = gpu_attention(q, kc, vc, pos, H, Hkv, D, Ms, Ss, Mo, So, pb)
        want = O.attention_c(q, kc, vc, pos, H, Hkv, D, Ms, Ss, Mo, So, pb)
        assert np.array_equal(got, want), pb
    assert np.abs(got).max() > 0


@pytest.mark.parametrize("D,H,Hkv", [(16, 4, 2), (64, 14, 2), (128, 16, 8), (256, 8, 2)])
def test_one_row_context_edges(D, H, Hkv):
    """One row, whose threads take its values two keys at a time: contexts of one key, and on both sides of a
    whole pair, of the prefetched keys and of the loop past them; one-hot and flat probabilities."""
    rng = np.random.default_rng(D)
    max_seq = 1300
    kc, vc = (rng.integers(-128, 128, (Hkv, max_seq, D)).astype(np.int8) for _ in range(2))
    vc[:, ::3] = np.where(vc[:, ::3] < 0, -128, 127)
    q = rng.integers(-128, 128, (1, H * D))
    tg = 512 * 16 // D  # keys of one pass of the workgroup
    for T in sorted({1, 2, 3, tg - 1, tg, tg + 1, 2 * tg + 1, 8 * tg, 8 * tg + 1, 9 * tg + 5, 1299} & set(range(1, max_seq))):
        for Ss in (20, 31 + int(round(np.log2(5372 * np.sqrt(D) / 768))), 50):
            got = gpu_attention(q, kc, vc, T - 1, H, Hkv, D, (1 << 31) - 1, Ss, 1 << 30, 38, 15)
            want = O.attention_c(q, kc, vc, T - 1, H, Hkv, D, (1 << 31) - 1, Ss, 1 << 30, 38, 15)
            assert np.array_equal(got, want), (T, Ss)


def test_kv_write_and_positions():
    rng = np.random.default_rng(3)
    t = __import__("torch")
    Hkv, D, max_seq, M = 3, 64, 256, 16
    k = rng.integers(-128, 128, (M, Hkv * D))
    v = rng.integers(-128, 128, (M, Hkv * D))
    kc = t.zeros((Hkv, max_seq, D), dtype=t.int8, device="cuda")
    vc = t.zeros_like(kc)
    kd, vd = up(k, np.int8), up(v, np.int8)
    _lib.call("llhip_kv_write", ptr(kd), ptr(vd), M, Hkv, D, Hkv * D, Hkv * D, 100, None, None, 0, ptr(kc), ptr(vc),
              max_seq, stream())
    want = np.zeros((Hkv, max_seq, D), np.int64)
    want[:, 100:116] = k.reshape(M, Hkv, D).transpose(1, 0, 2)
    assert np.array_equal(down(kc), want)
    want[:, 100:116] = v.reshape(M, Hkv, D).transpose(1, 0, 2)
    assert np.array_equal(down(vc), want)
    with pytest.raises(ValueError, match="max_seq"):
        _lib.call("llhip_kv_write", ptr(kd), ptr(vd), M, Hkv, D, Hkv * D, Hkv * D, 250, None, None, 0, ptr(kc),
                  ptr(vc), max_seq, stream())


def test_device_position():
    """pos read from device memory (decode state inside a captured graph) == host pos."""
    t = __import__("torch")
    rng = np.random.default_rng(11)
    H, Hkv, D, max_seq = 14, 2, 64, 1024
    kc = rng.integers(-128, 128, (Hkv, max_seq, D))
    vc = rng.integers(-128, 128, (Hkv, max_seq, D))
    q = rng.integers(-128, 128, (1, H * D))
    qd, kd, vd = up(q, np.int8), up(kc, np.int8), up(vc, np.int8)
    posd = t.tensor([600], dtype=t.int32, device="cuda")
    out = t.empty((1, H * D), dtype=t.int8, device="cuda")
    _lib.call("llhip_attention", ptr(qd), 1, H, Hkv, D, H * D, 0, ptr(posd), None, 0, ptr(kd), ptr(vd), max_seq,
              1 << 30, 40, 1 << 30, 38, 15, ptr(out), H * D, ptr(workspace()), stream())
    assert np.array_equal(down(out), O.attention_c(q, kc.astype(np.int8), vc.astype(np.int8), 600, H, Hkv, D,
                                                   1 << 30, 40, 1 << 30, 38, 15))


@pytest.mark.parametrize("pos", [0, 5, 2100, 4095])
def test_device_position_long_context(pos):
    """Device position with a long cache (the split-context path sizes its grid for max_seq):
    splits past the position find no keys and contribute nothing."""
    t = __import__("torch")
    rng = np.random.default_rng(12 + pos)
    H, Hkv, D, max_seq = 16, 8, 128, 4096
    kc = rng.integers(-128, 128, (Hkv, max_seq, D))
    vc = rng.integers(-128, 128, (Hkv, max_seq, D))
    q = rng.integers(-128, 128, (1, H * D))
    qd, kd, vd = up(q, np.int8), up(kc, np.int8), up(vc, np.int8)
    posd = t.tensor([pos], dtype=t.int32, device="cuda")
    out = t.empty((1, H * D), dtype=t.int8, device="cuda")
    for pb in (15, 8):
        _lib.call("llhip_attention", ptr(qd), 1, H, Hkv, D, H * D, 0, ptr(posd), None, 0, ptr(kd), ptr(vd), max_seq,
                  1 << 30, 41, 1 << 30, 38, pb, ptr(out), H * D, ptr(workspace()), stream())
        want = O.attention_c(q, kc.astype(np.int8), vc.astype(np.int8), pos, H, Hkv, D, 1 << 30, 41, 1 << 30, 38, pb)
        assert np.array_equal(down(out), want), pb


@pytest.mark.parametrize("D,H,Hkv", [(64, 14, 2), (128, 16, 8), (16, 4, 2)])
def test_rows_as_sequences(D, H, Hkv):
    """Batch decode form: row m is its own sequence at position row_pos[m] with its caches in slot m.
    Each row equals a single-row launch over its own caches (oracle), and kv_write stores each row
    in its own slot at its own position."""
    t = __import__("torch")
    rng = np.random.default_rng(D + H)
    B, max_seq = 5, 300
    positions = np.array([0, 17, 299, 128, 63], np.int32)
    kc = rng.integers(-128, 128, (B, Hkv, max_seq, D))
    vc = rng.integers(-128, 128, (B, Hkv, max_seq, D))
    q = rng.integers(-128, 128, (B, H * D))
    kd, vd, qd = up(kc, np.int8), up(vc, np.int8), up(q, np.int8)
    rp = t.tensor(positions, dtype=t.int32, device="cuda")
    stride = Hkv * max_seq * D
    # the new K/V rows go to each sequence's slot at its position
    knew = rng.integers(-128, 128, (B, Hkv * D))
    vnew = rng.integers(-128, 128, (B, Hkv * D))
    knd, vnd = up(knew, np.int8), up(vnew, np.int8)  # held until the launch has run
    _lib.call("llhip_kv_write", ptr(knd), ptr(vnd), B, Hkv, D, Hkv * D, Hkv * D, 0, None, ptr(rp), stride, ptr(kd),
              ptr(vd), max_seq, stream())
    for b in range(B):
        kc[b][:, positions[b]] = knew[b].reshape(Hkv, D)
        vc[b][:, positions[b]] = vnew[b].reshape(Hkv, D)
    assert np.array_equal(down(kd), kc) and np.array_equal(down(vd), vc)
    out = t.empty((B, H * D), dtype=t.int8, device="cuda")
    _lib.call("llhip_attention", ptr(qd), B, H, Hkv, D, H * D, 0, None, ptr(rp), stride, ptr(kd), ptr(vd), max_seq,
              1 << 30, 40, 1 << 30, 38, 8, ptr(out), H * D, ptr(workspace()), stream())
    got = down(out)
    for b in range(B):
        want = O.attention_c(q[b:b + 1], kc[b].astype(np.int8), vc[b].astype(np.int8), int(positions[b]), H, Hkv, D,
                             1 << 30, 40, 1 << 30, 38, 8)
        assert np.array_equal(got[b:b + 1], want), b
    with pytest.raises(ValueError, match="slots overlap"):
        _lib.call("llhip_attention", ptr(qd), B, H, Hkv, D, H * D, 0, None, ptr(rp), stride - 1, ptr(kd), ptr(vd),
                  max_seq, 1 << 30, 40, 1 << 30, 38, 8, ptr(out), H * D, ptr(workspace()), stream())


@pytest.mark.parametrize("M,D", [(16, 64), (1, 64), (40, 128), (5, 256)])
@pytest.mark.parametrize("regime", ["onehot", "steep", "flat", "extreme"])
def test_softmax_regimes(M, D, regime):
    """Saturating probabilities (one key gets 2^pb - 1: the clamp and the third digit of pn are used),
    the same with the largest Ms and the smallest Ss of the 32-bit index form, a flat softmax (Ms = 0:
    every p = 65534) and all-(-128) operands (maximal scores)."""
    rng = np.random.default_rng(M + D + len(regime))
    H, Hkv, pos, max_seq = 4, 2, 70, 128
    kc = rng.integers(-128, 128, (Hkv, max_seq, D)).astype(np.int8)
    vc = rng.integers(-128, 128, (Hkv, max_seq, D)).astype(np.int8)
    q = rng.integers(-128, 128, (M, H * D))
    Ms, Ss, Mo, So = (1 << 31) + 12345, 20, (1 << 31) - 1, 40
    if regime == "flat":
        Ms = 0
    elif regime == "steep":
        Ms, Ss = (1 << 31) - 1, 32
    elif regime == "extreme":
        kc[:] = -128
        vc[:] = -128
        q[:] = -128
        Ms, Ss = 1 << 20, 24
    for pb in (15, 8):
        got = gpu_attention(q, kc, vc, pos, H, Hkv, D, Ms, Ss, Mo, So, pb)
        want = O.attention_c(q, kc, vc, pos, H, Hkv, D, Ms, Ss, Mo, So, pb)
        assert np.array_equal(got, want), pb


@pytest.mark.parametrize("M,H,Hkv,D,pos,max_seq", [(520, 14, 2, 64, 500, 1024),    # eight waves, two workgroups per CU
                                                   (600, 14, 2, 64, 400, 1024),    # four waves
                                                   (384, 16, 8, 128, 1730, 2176),  # 34 tiles: seven in LDS, the last again
                                                   (250, 24, 8, 128, 300, 640), (234, 24, 8, 128, 300, 640)])
def test_waves_per_workgroup(M, H, Hkv, D, pos, max_seq):
    """Both sides of the rule for four or eight waves, and four waves with more tiles than LDS keeps."""
    test_attention_matches_oracle(M, H, Hkv, D, pos, max_seq)
