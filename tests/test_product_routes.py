"""Which projections' products may leave torch, decided from the operands' metadata alone.  The operands are tensors over
addresses that nothing follows, made through DLPack with a device that need not exist, so this runs without a GPU; in a
process of its own, which is told that the device runtime is up."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

OPERANDS = '''
import ctypes
import torch
torch.cuda._lazy_init = lambda: None
i64 = ctypes.c_int64


class DLTensor(ctypes.Structure):
    _fields_ = [("data", ctypes.c_void_p), ("device_type", ctypes.c_int32), ("device_id", ctypes.c_int32), ("ndim", ctypes.c_int32),
                ("code", ctypes.c_uint8), ("bits", ctypes.c_uint8), ("lanes", ctypes.c_uint16), ("shape", ctypes.POINTER(i64)),
                ("strides", ctypes.POINTER(i64)), ("offset", ctypes.c_uint64), ("context", ctypes.c_void_p), ("deleter", ctypes.c_void_p)]


capsule = ctypes.pythonapi.PyCapsule_New
capsule.restype, capsule.argtypes = ctypes.py_object, [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]
kept = []


def operand(rows, cols, pitch=None, device=0, address=1 << 20):
    """A bf16 [rows, cols] matrix with `pitch` elements between rows."""
    ROCM, BFLOAT = 10, 4
    shape, strides = (i64 * 2)(rows, cols), (i64 * 2)(pitch or cols, 1)
    t = DLTensor(address, ROCM, device, 2, BFLOAT, 16, 1, shape, strides, 0, None, None)
    kept.append((t, shape, strides))
    return torch.utils.dlpack.from_dlpack(capsule(ctypes.addressof(t), b"dltensor", None))


def message(call, *args):
    try:
        call(*args)
    except RuntimeError as e:
        return str(e)
    return "no error"


from picotron_amd import _lib
host = _lib.host()
'''


def run(body):
    from picotron_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    res = subprocess.run([sys.executable, "-c", OPERANDS + body], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout + res.stderr


def test_operands_on_two_devices_are_refused():
    """As nn.Linear refuses them, in the forward and in both gradients, whichever route their sizes would have taken."""
    run('''
for rows, wide in ((512, 576), (4096, 2048)):
    x, w = operand(rows, 576), operand(wide, 576, device=1)
    dy = operand(rows, wide)
    for what in (message(host.linear, x, w), message(host.fused_linear, x, w, [w]), message(host.product, x, w, "NT"),
                 message(host.product, dy, w, "NN"), message(host.product, operand(rows, wide, device=1), x, "TN")):
        assert "same device" in what, what
''')
