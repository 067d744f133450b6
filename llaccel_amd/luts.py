"""LUTs of the integer datapath (same names and definitions as the reference's
python/llaccel/luts.py:18-29, docs/NUMERICS.md "SiLU"/"Attention"):

  SIG[j]  = round(sigmoid(-8 + j/16) * 65536), j = 0..256, capped at 65535
  EXPI[i] = round(exp(-i) * 65535),           i = 0..15
  EXPF[f] = round(exp(-f/256) * 65535),       f = 0..255

Python's round (half to even) on doubles.  `write_hip_tables()` regenerates
`csrc/luts.inc`, the committed copy the HIP kernels compile in as __constant__ data.  The HIP
copy of SIG carries one trailing zero (258 entries, 129 whole dwords) so kernels can stage it in
LDS with 4-byte loads; the interpolation reads entries 0..256 only.
"""
from __future__ import annotations

import math
from pathlib import Path

import numpy as np

INC = Path(__file__).resolve().parent / "csrc" / "luts.inc"


def sigmoid_lut() -> np.ndarray:
    return np.array([min(65535, round(65536.0 / (1.0 + math.exp(8.0 - j / 16.0)))) for j in range(257)], np.uint16)


def exp_int_lut() -> np.ndarray:
    return np.array([round(65535 * math.exp(-i)) for i in range(16)], np.uint16)


def exp_frac_lut() -> np.ndarray:
    return np.array([round(65535 * math.exp(-f / 256.0)) for f in range(256)], np.uint16)


def hip_tables_text() -> str:
    lines = ["// GENERATED by llaccel_amd/luts.py -- do not edit.", ""]
    sig_padded = np.append(sigmoid_lut(), np.uint16(0))
    for name, arr in (("kSig", sig_padded), ("kExpI", exp_int_lut()), ("kExpF", exp_frac_lut())):
        lines.append(f"static __constant__ constexpr uint16_t {name}[{len(arr)}] = {{")
        for i in range(0, len(arr), 16):
            lines.append("    " + ", ".join(f"{int(v)}" for v in arr[i:i + 16]) + ",")
        lines.append("};")
        lines.append("")
    return "\n".join(lines)


def write_hip_tables(path: Path = INC) -> None:
    Path(path).write_text(hip_tables_text())


if __name__ == "__main__":
    write_hip_tables()
    print("wrote", INC)
