"""What the compiler reports for kernels whose speed rests on it: no register of the loss kernels lives in scratch memory."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def resources(source, tmp_path):
    """{mangled kernel name: {remark: value}} of csrc/<source>, compiled with the package's own flags."""
    from picotron_amd import build
    if shutil.which(build._hipcc()) is None:
        pytest.skip("no hipcc")
    out = subprocess.run([build._hipcc(), *build.FLAGS, "-c", os.path.join(build.CSRC, source), "-o", str(tmp_path / "out.o"),
                          "-Rpass-analysis=kernel-resource-usage"], capture_output=True, text=True, timeout=600, check=True).stderr
    kernels, now = {}, None
    for key, value in re.findall(r"remark: (?:\S+:\d+:\d+: )?\s*([A-Za-z ]+?)(?: \[[^\]]*\])?: (\S+) \[-Rpass", out):
        if key == "Function Name":
            now = kernels.setdefault(value, {})
        else:
            now[key] = int(value) if value.isdigit() else value
    return kernels


def test_loss_kernels_keep_the_row_in_registers(tmp_path):
    kernels = resources("loss.hip", tmp_path)
    assert sum("ce_one_pass_kernel" in name for name in kernels) == 22
    for name, r in kernels.items():
        assert r["ScratchSize"] == 0 and r["VGPRs Spill"] == 0, (name, r)
