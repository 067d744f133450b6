"""Registers and scratch of the built kernels (the code objects' own metadata, no GPU): the kernels of the
decode and prompt paths keep nothing in scratch, and the eight-wave workgroups of the fused launches fit a
compute unit twice."""
from __future__ import annotations

import re
import struct

import pytest

from llaccel_amd import _lib

msgpack = pytest.importorskip("msgpack")

NT_AMDGPU_METADATA = 32


def _code_objects(blob: bytes):
    """The gfx950 ELF images of the library's offload bundles (one bundle per source file)."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    for m in re.finditer(magic, blob):
        at = m.end()
        (n,) = struct.unpack_from("<Q", blob, at)
        at += 8
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", blob, at)
            triple = blob[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" in triple and size:
                yield blob[m.start() + off:m.start() + off + size]


def _metadata(elf: bytes):
    """The kernels' metadata maps from the ELF's AMDGPU note."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entsize, num = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(num):
        kind, = struct.unpack_from("<I", elf, shoff + i * entsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * entsize + 24)
        if kind != 7:  # SHT_NOTE
            continue
        at = off
        while at < off + size:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, at)
            desc = at + 12 + (namesz + 3) // 4 * 4
            if ntype == NT_AMDGPU_METADATA:
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            at = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    if not _lib.LIB_PATH.exists():
        pytest.skip("library not built")
    got = {k[".name"]: k for e in _code_objects(_lib.LIB_PATH.read_bytes()) for k in _metadata(e)}
    assert len(got) > 100
    return got


def _named(kernels, name):
    hit = {n: k for n, k in kernels.items() if re.search(rf"\d{name}(I|E|P|v)", n)}
    assert hit, name
    return hit


@pytest.mark.parametrize("name", ["attn_in_kernel", "mlp_in_kernel", "norm_gemv_kernel", "dec_mlp_kernel",
                                  "dec_logits_kernel", "attention_tiled", "attention_rowhead", "attention_row_fused",
                                  "linear_gemv", "linear_gemv1", "norm_rope_quant_kernel", "rmsnorm_quant_kernel"])
def test_no_scratch(kernels, name):
    for n, k in _named(kernels, name).items():
        assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_spill_count"] == 0, n


def test_eight_wave_workgroups_fit_twice(kernels):
    """At most 128 vector registers: four waves per SIMD, two workgroups of 512 threads per compute unit."""
    for name in ("attn_in_kernel", "mlp_in_kernel", "norm_gemv_kernel"):
        for n, k in _named(kernels, name).items():
            if k[".max_flat_workgroup_size"] <= 512:
                assert k[".vgpr_count"] <= 128, (n, k[".vgpr_count"])


def test_gemm_tiles_without_scratch(kernels):
    """linear_mfma below the 256 x 256 tile: a vector register or an argument more sends the 64 x 128 instances to scratch."""
    for n, k in _named(kernels, "linear_mfma").items():
        if "ILi256E" not in n and "ELi256ELi256E" not in n:
            assert k[".private_segment_fixed_size"] == 0, n
