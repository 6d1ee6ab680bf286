"""The legacy encode's division by the scale and its code step (csrc/lrq_legacy.hip, the MFMA
encode) against the reference's (low_rank_extraction_fuse_compression_quantization.py:165-166,
torch form: `(x - o) / s`, bf16, then round and clamp), exhaustively on the host
(tests/legacy_code_check.c):

* the code forms: at 1 bit one compare of the fp32 quotient with -(0.5 + 2^-9); at 2, 4 and 8
  bits the clamped bits of bf16(q) + 1.5 * 2^23; both equal clamp(rint(bf16(q))) + 2^(b-1) for
  every fp32 quotient but NaN;
* the quotient: for every finite bf16 numerator and every bf16 scale with
  2^-100 <= |s| <= 2^100, the two-term product a r1 + a r2, 1/s = r1 + r2 in bf16, gives the IEEE
  quotient's code at 1, 2, 4 and 8 bits (magnitudes of 2^118 |s| and more are divided).

The check fails for a threshold of -0.5, a bias of 2^23, or a quotient of the first term alone."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).resolve().parent


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_code_step_forms_give_the_reference_codes(tmp_path):
    exe = tmp_path / "legacy_code_check"
    subprocess.run(["gcc", "-O2", "-fopenmp", "-ffp-contract=off", "-o", str(exe), str(HERE / "legacy_code_check.c"),
                    "-lm"], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=600).stdout.split()
    checked, bad1, bad2, bad4, bad8, pairs, e1, e2, e4, e8 = map(int, out)
    assert checked == 2 ** 32 - 2 * (2 ** 23 - 1)  # every bit pattern but the NaNs
    assert (bad1, bad2, bad4, bad8) == (0, 0, 0, 0)
    # two-term quotients.  Scales: the 200 binades 2^-100 .. 2^99 (128 each) and 2^100, both signs; numerators: the
    # 65280 finite bf16 values
    assert pairs == 2 * (200 * 128 + 1) * 65280
    assert (e1, e2, e4, e8) == (0, 0, 0, 0)


def _bf16(f: np.ndarray) -> np.ndarray:
    """fp32 rounded to bf16 (nearest even), as fp32."""
    u = f.astype(np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000
    return u.astype(np.uint32).view(np.float32)


def test_two_term_quotient_gives_the_reference_codes():
    """The same without a compiler, at scales from the smallest to the largest served: 1/s as two bf16 terms r1 + r2, a r1 (exact) and then a r2
    added with one fp32 rounding (at 1 bit the threshold 0.5 + 2^-9 enters with a r1, and the sign is
    the code): its code is the IEEE quotient's for every pair of bf16 mantissas and signs at every
    exponent difference that can reach a code boundary (|q| from 2^-4 to 2^9; beyond, both clamp)."""
    man = np.arange(128, 256, dtype=np.float32)
    a0 = np.concatenate([man, -man])[:, None]
    for es in (-107, -100, -93, -60, -31, -7, 0, 3, 24, 55, 92):  # (times 128 .. 255: 2^-100 .. 2^100)
        for sg in (1.0, -1.0):
            s = (sg * man * 2.0 ** es).astype(np.float32)[None, :]
            rc = (np.float32(1.0) / s).astype(np.float32)
            r1 = _bf16(rc)
            r2 = _bf16(rc - r1)
            for ea in range(-5, 10):
                a = (a0 * np.float32(2.0) ** (es + ea)).astype(np.float32)
                q = (a / s).astype(np.float32)
                p1, p2 = a.astype(np.float64) * r1.astype(np.float64), a.astype(np.float64) * r2.astype(np.float64)
                t = (p1 + p2).astype(np.float32)
                for bits in (2, 4, 8):
                    half = 1 << (bits - 1)
                    ref = np.clip(np.rint(_bf16(q)), -half, half - 1)
                    assert np.array_equal(np.clip(np.rint(_bf16(t)), -half, half - 1), ref), (es, ea, bits)
                one = ((p1 + (0.5 + 2.0 ** -9)).astype(np.float32).astype(np.float64) + p2).astype(np.float32)
                ref = np.clip(np.rint(_bf16(q)), -1, 0) + 1
                assert np.array_equal((~np.signbit(one)).astype(np.float32), ref), (es, ea, 1)
