"""The two-float quantization of the layout kernels (``qa_round_f32x2`` in
``qa_common.h``) against the reference's float64 quotient, compiled for the
host: it decides right or asks for the double form, also where the float32
quotient overflows."""

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="no hipcc")
def test_two_float_quantization_is_exact(tmp_path):
    exe = tmp_path / "quantize_f32x2"
    subprocess.run([HIPCC, "-O2", "-std=c++17",
                    f"-I{ROOT / 'quantanything_amd' / 'csrc'}",
                    str(ROOT / "tests" / "native" / "quantize_f32x2.cpp"),
                    "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe), "2000000"], capture_output=True,
                         text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "mismatches 0" in out.stdout
