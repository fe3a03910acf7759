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


def test_attention_kernels_fit_a_cu_as_often_as_their_plans_count_on(tmp_path):
    """Registers: waves per SIMD x 4 SIMDs hold the workgroups of a CU (LDS is asserted where the tiles are laid out), and
    none of them are in scratch.  Eight waves have a CU to themselves at head_dim 128 and with split keys, and in dQ; the
    four waves of dQ at head_dim 128 do as well."""
    per_cu = {}
    for source in ("attn_fwd.hip", "attn_bwd.hip"):
        for name, r in resources(source, tmp_path).items():
            assert r["ScratchSize"] == 0 and r["VGPRs Spill"] == 0, (name, r)
            numbers = [int(n) for n in re.findall(r"L[ib](\d+)E", name)]
            if "attn_fwd_kernel" in name:
                D, _, NW, _, KS, _ = numbers
                want = 1 if NW == 8 and (D == 128 or KS == 2) else 2
            elif "attn_bwd_dq_kernel" in name:
                D, NW, _, _, KS, _ = numbers
                want = 2 if NW == 4 and D == 64 else 1
            elif "dkdv_kernel" in name:
                NW, want = (4, 2) if "_d64" in name else (8, 1)
            else:
                continue
            assert r["Occupancy"] * 4 >= want * NW, (name, r)
            per_cu[name] = want
    assert len(per_cu) == 12 + 24 + 4


@pytest.mark.parametrize("B,Hq,Hkv,S,D", [(1, 20, 20, 2500, 128), (1, 20, 20, 3000, 128), (1, 32, 32, 4000, 64), (1, 16, 16, 8000, 64)])
def test_launches_that_fill_the_gpu_run_whole(B, Hq, Hkv, S, D):
    """Attention launches that every piece length slows down, by 1 to 16 %, ask for no scratch memory: neither the forward
    nor dQ and dK/dV are cut."""
    import ctypes
    import math

    import torch
    from picotron_amd import _lib, ops
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    q, k = (torch.empty(B, h, S, D, dtype=torch.bfloat16) for h in (Hq, Hkv))
    d = ops._desc(q, k, k, q, 1 / math.sqrt(D), True, 0)
    assert _lib.lib().pico_attn_fwd_workspace_bytes(ctypes.byref(d), 1) == 0
    assert _lib.lib().pico_attn_bwd_workspace_bytes(ctypes.byref(d), 1) == 0
