"""What the compiler makes of kernels whose speed or safety rests on it: registers, scratch memory, and the requests that go to LDS
without passing the registers."""
import functools
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@functools.lru_cache(maxsize=None)
def compiled(path):
    """({mangled kernel name: {remark: value}}, device assembly) of a source, compiled with the package's own flags."""
    from picotron_amd import build
    if shutil.which(build._hipcc()) is None:
        pytest.skip("no hipcc")
    res = subprocess.run([build._hipcc(), *build.FLAGS, f"-I{build.CSRC}", "--cuda-device-only", "-S", path, "-o", "-", build.RESOURCES],
                         capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stderr
    return build.kernel_resources(res.stderr), res.stdout


def csrc(source):
    from picotron_amd import build
    return os.path.join(build.CSRC, source)


def resources(source):
    return compiled(csrc(source))[0]


def test_loss_kernels_keep_the_row_in_registers():
    kernels = resources("loss.hip")
    assert sum("ce_one_pass_kernel" in name for name in kernels) == 22
    for name, r in kernels.items():
        assert r["ScratchSize"] == 0 and r["VGPRs Spill"] == 0, (name, r)


def test_attention_kernels_fit_a_cu_as_often_as_their_plans_count_on():
    """Registers: waves per SIMD x 4 SIMDs hold the workgroups of a CU (LDS is asserted where the tiles are laid out), and
    none of them are in scratch.  Eight waves have a CU to themselves at head_dim 128 and with split keys, and in dQ."""
    per_cu = {}
    for source in ("attn_fwd.hip", "attn_bwd.hip"):
        for name, r in resources(source).items():
            assert r["ScratchSize"] == 0 and r["VGPRs Spill"] == 0, (name, r)
            numbers = [int(n) for n in re.findall(r"L[ib](\d+)E", name)]
            if "attn_fwd_kernel" in name:
                D, _, NW, _, KS, _ = numbers
                want = 1 if NW == 8 and (D == 128 or KS == 2) else 2
            elif "attn_bwd_dq_kernel" in name:
                D, NW, _, _, KS, _ = numbers
                want = 2 if NW == 4 else 1
            elif "dkdv_kernel" in name:
                NW, want = (4, 2) if "_d64" in name else (8, 1)
            elif "dkdv_few_kernel" in name:
                NW, want = 8, 1
            else:
                assert "_kernel" in name and not re.search("dkdv|dq|attn_fwd", name) or "join" in name, name
                continue
            assert r["Occupancy"] * 4 >= want * NW, (name, r)
            per_cu[name] = want
    assert len(per_cu) == 12 + 24 + 5


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


@pytest.mark.parametrize("Hq,S,dkdv_pieces", [(16, 4096, 272), (12, 5888, 288)])
def test_dq_of_four_waves_at_head_dim_64_runs_whole(Hq, S, dkdv_pieces):
    """It is never faster in pieces (B2 H8 S4096 64.1 us, cut 71.1).  With one key head the scratch memory that dQ's pieces would ask for is
    larger than that of dK/dV's (four key waves, 2 x 32 x 64 floats each), which is what the call asks for."""
    import ctypes

    import torch
    from picotron_amd import _lib, ops
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    q, k = (torch.empty(1, h, S, 64, dtype=torch.bfloat16) for h in (Hq, 1))
    d = ops._desc(q, k, k, q, 0.125, True, 0)
    assert _lib.lib().pico_attn_bwd_workspace_bytes(ctypes.byref(d), 1) == dkdv_pieces * 4 * 2 * 32 * 64 * 4


def test_kernels_that_make_requests_have_no_scratch_and_no_lds_of_their_own(tmp_path):
    """A spill counts among the memory operations of which product_mid and product_large wait for all but the newest few, and the
    requests' places in LDS are counted from 0: the build refuses both.  A workgroup of the products has a CU to itself, two
    waves per SIMD.  The kernels that the build looks at are those with requests in their code."""
    from picotron_amd import build
    for source, count in (("product_mid.hip", 79), ("product_large.hip", 30), ("attn_fwd.hip", 12), ("attn_bwd.hip", 29)):
        kernels, assembly = compiled(csrc(source))
        looked_at = {name for name in kernels if re.search(build.REQUESTING[source], name)}
        assert len(looked_at) == count
        for name, r in kernels.items():
            body = assembly[assembly.index(f"\n{name}:"):]
            requests = " lds\n" in body[:body.index("s_endpgm")] or " lds\n" in body[:body.index(".Lfunc_end")]
            assert not requests or name in looked_at, name
            if name in looked_at:
                assert r["ScratchSize"] == 0 and r["VGPRs Spill"] == 0 and r["LDS Size"] == 0, (name, r)
                assert not source.startswith("product") or r["Occupancy"] >= 2, (name, r)
    both = tmp_path / "both.hip"
    both.write_text('''#include <hip/hip_runtime.h>
extern "C" __global__ __launch_bounds__(1024) void spilling_kernel(const float* x, float* y) {
  float v[200];
#pragma unroll
  for (int i = 0; i < 200; ++i) v[i] = x[i * 1024 + threadIdx.x];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 200; ++i) y[(i * 7 % 200) * 1024 + threadIdx.x] = v[i] * v[(i * 13 + 5) % 200];
}
extern "C" __global__ void static_kernel(const float* x, float* y) {
  __shared__ float lds[64];
  lds[threadIdx.x] = x[threadIdx.x];
  __syncthreads();
  y[threadIdx.x] = lds[63 - threadIdx.x];
}
''')
    remarks = subprocess.run([build._hipcc(), *build.FLAGS, "--cuda-device-only", "-c", str(both), "-o", str(tmp_path / "o"), build.RESOURCES],
                             capture_output=True, text=True, timeout=600).stderr
    spilling, static = (remarks[remarks.index(f"Function Name: {name}") - 60:] for name in ("spilling_kernel", "static_kernel"))
    with pytest.raises(RuntimeError, match="spilling_kernel keeps registers in scratch"):
        build.check_requesting("product_mid.hip", spilling)
    with pytest.raises(RuntimeError, match="static_kernel has LDS of its own"):
        build.check_requesting("product_mid.hip", static)
    with pytest.raises(RuntimeError, match="no such kernel"):
        build.check_requesting("product_mid.hip", "")


@pytest.mark.parametrize("source", ["product_mid.hip", "product_large.hip", "attn_fwd.hip", "attn_bwd.hip"])
def test_requests_find_their_aim_in_m0(source):
    """m0 is written by nothing but the statement that aims a request, in the same straight run of code, and one instruction at least
    lies between the two (the hardware asks for one, and the compiler does not look into the statements)."""
    lines = [l.split(";")[0].strip() for l in compiled(csrc(source))[1].splitlines()]
    lines = [l for l in lines if l and not l.startswith((".", "//", "#"))]
    requests, aimed = 0, None                       # instructions since m0 was written; None: not in this run of code
    for line in lines:
        if "pico_wait_" in line:                    # (a wait that goes round by itself: entered from above only, and m0 stays)
            continue
        if line.endswith(":"):
            aimed = None
            continue
        if re.search(r"\bm0\b", line):
            assert line.startswith("s_add_u32 m0,"), line
            assert aimed is None or aimed < 0, line  # (the aim before has been used)
            aimed = 0
            continue
        if line.startswith("buffer_load") and line.endswith(" lds"):
            assert aimed is not None and aimed >= 1, line
            requests, aimed = requests + 1, -1
        elif aimed is not None and aimed >= 0:
            aimed = None if line.startswith(("s_cbranch", "s_branch", "s_setpc", "s_endpgm")) else aimed + 1
    assert requests > 100


def test_the_compiler_keeps_nothing_in_m0_across_a_request(tmp_path):
    """A value that the compiler has in m0 before a request is written there again after it (never run: compiled only)."""
    source = tmp_path / "around.hip"
    source.write_text('''#include "attn_common.h"
using namespace pico;
extern "C" __global__ void whole(uint64_t base, uint32_t bytes, uint32_t to) {
  const u32x4 window = request_window(base, bytes);
  __builtin_amdgcn_s_sendmsg(1, 40);
  request16_to<16>(to, window, threadIdx.x * 16);
  __builtin_amdgcn_s_sendmsg(1, 40);
}
extern "C" __global__ void parted(uint64_t base, uint32_t bytes, uint32_t to) {
  const u32x4 window = request_window(base, bytes);
  __builtin_amdgcn_s_sendmsg(1, 40);
  const uint32_t aim = aim_request<16>(to);
  asm volatile("s_nop 0");
  request16(aim, window, threadIdx.x * 16);
  __builtin_amdgcn_s_sendmsg(1, 40);
}
''')
    assembly = compiled(str(source))[1]
    for name in ("whole", "parted"):
        body = assembly[assembly.index(f"\n{name}:"):]
        seen = re.findall(r"s_mov_b32 m0, 40|s_sendmsg|s_add_u32 m0|offen lds", body[:body.index("s_endpgm")])
        assert seen == ["s_mov_b32 m0, 40", "s_sendmsg", "s_add_u32 m0", "offen lds", "s_mov_b32 m0, 40", "s_sendmsg"], (name, seen)


def test_streaming_optimizer_kernels_store_past_the_caches():
    """Every vector store of the AdamW kernels for arrays larger than the caches carries the streaming hint, and none of the others does;
    of the loads all but the gradient's do."""
    _, text = compiled(csrc("optim.hip"))
    seen = 0
    for name, body in re.findall(r"^(_Z\w*adamw\w*):\s*;.*?$(.*?)s_endpgm", text, flags=re.S | re.M):
        streams = re.search(r"kernelILb([01])E", name).group(1) == "1"
        loads, stores = (re.findall(r"^\s*global_%s_dwordx[24] .*$" % what, body, flags=re.M) for what in ("load", "store"))
        assert loads and stores, name
        assert all((" nt" in line) == streams for line in stores), name
        assert sum(" nt" in line for line in loads) == (3 * len(loads) // 4 if streams else 0), name
        seen += 1
    assert seen == 24   # one and many tensors, streaming or not, six combinations of types


def test_the_kernel_of_two_roles_fits_a_cu():
    """Eight waves share a CU, with no register in scratch memory and no LDS of their own (its requests count from 0)."""
    kernels = compiled(csrc("attn_bwd_roles.hip"))[0]
    assert len(kernels) == 1
    for name, r in kernels.items():
        assert "attn_bwd_roles_kernel" in name and r["Occupancy"] >= 2
        assert r["ScratchSize"] == 0 and r["VGPRs Spill"] == 0 and r["LDS Size"] == 0, (name, r)
