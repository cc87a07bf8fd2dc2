"""Kernels that synchronise with a bare ``s_barrier`` (not ``__syncthreads``,
which would wait for every direct load in flight) wait for their LDS writes
first: the barrier itself waits for no memory, so a write still on its way
would be read too early by another wave. Checked in the assembly compiled
from each source, on the CPU."""

import re
import shutil
import subprocess

import pytest

from quantanything_amd import build

pytestmark = pytest.mark.skipif(shutil.which(build.HIPCC) is None,
                                reason="no hipcc")


def _kernels(src, tmp_path):
    """Each kernel's instructions, in the order of the listing."""
    out = tmp_path / "k.s"
    subprocess.run([build.HIPCC, *build.COMMON, *build.DEVICE_FLAGS,
                    "--cuda-device-only", "-S", str(build.CSRC / src), "-o",
                    str(out)], check=True, capture_output=True)
    kernels, cur = {}, None
    for line in out.read_text().splitlines():
        label = re.match(r"^(_Z\w+):", line)
        if label:
            cur = kernels.setdefault(label.group(1), [])
        text = line.split(";")[0].strip()
        if cur is not None and text and not text.startswith("."):
            cur.append(text)
    return kernels


@pytest.mark.parametrize("src", ["qa_gemm_narrow.hip", "qa_narrow_chain.hip"])
def test_lds_writes_are_waited_for(tmp_path, src):
    barriers = 0
    for name, ins in _kernels(src, tmp_path).items():
        for at, text in enumerate(ins):
            if not text.startswith("s_barrier"):
                continue
            barriers += 1
            for back in reversed(ins[:at]):
                if back.startswith("s_waitcnt") and "lgkmcnt(0)" in back:
                    break
                assert not back.startswith("ds_write"), \
                    f"{name}: {back} still in flight at a barrier"
    assert barriers > 0


def test_ring_reads_are_waited_for(tmp_path):
    """A barrier of the staged GEMM's ring leaves no fragment read in flight
    but those of the last step (MT + NT of them): the stage of the step
    before is refilled right after it."""
    barriers = 0
    for name, ins in _kernels("qa_gemm_stage.hip", tmp_path).items():
        bm, bn, wm, wn = map(int, re.search(
            r"k_gemm_stageILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E", name).groups())
        reads = bm // wm // 16 + bn // wn // 16
        for at, text in enumerate(ins):
            if not text.startswith("s_barrier"):
                continue
            barriers += 1
            for back in reversed(ins[:at]):
                wait = re.match(r"s_waitcnt.*lgkmcnt\((\d+)\)", back)
                if wait:
                    assert int(wait.group(1)) <= reads, name
                    break
                assert not back.startswith("ds_"), \
                    f"{name}: {back} not waited for at a barrier"
    assert barriers > 0
