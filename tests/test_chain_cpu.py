"""Which runs of commands the chain launch refuses, checked without a GPU.

m3_hip_launch_chain plans a run on the host and touches its device handle
only for a run that it takes, so the refusals can be called with a handle of
zeroed memory. A run over tensors without elements is refused, whatever axis
is the empty one and however the other operand broadcasts over it: the
commands then run one by one, each with nothing to do. Each case runs in a
process of its own, so that a fault on the host fails its case alone.
"""
import subprocess
import sys

import pytest

from conftest import ROOT

CHILD = r"""
import ctypes
import importlib.util
import os
import sys

spec = importlib.util.spec_from_file_location(
    "m3c_amd", os.path.join(sys.argv[1], "m3.c_amd", "__init__.py"))
m3 = importlib.util.module_from_spec(spec)
sys.modules["m3c_amd"] = m3
spec.loader.exec_module(m3)
shapes = eval(sys.argv[2])
_, hip = m3.load()


class View(ctypes.Structure):
    _fields_ = [("base", ctypes.c_void_p), ("byte_offset", ctypes.c_uint64),
                ("element_count", ctypes.c_uint64),
                ("shape", ctypes.c_uint64 * 8),
                ("byte_strides", ctypes.c_uint64 * 8),
                ("rank", ctypes.c_uint32), ("dtype", ctypes.c_uint32)]


class Command(ctypes.Structure):
    _fields_ = [("kind", ctypes.c_uint32), ("op", ctypes.c_uint32),
                ("link", ctypes.c_uint32), ("left", View), ("right", View),
                ("output", View)]


def view(base, shape):
    v = View(base=base, rank=len(shape))
    count = 1
    for axis in reversed(range(len(shape))):
        v.shape[axis] = shape[axis]
        v.byte_strides[axis] = 4 * count
        count *= shape[axis]
    v.element_count = count
    return v


space, other = shapes
commands = (Command * 2)()
for k in range(2):
    commands[k].kind = 0
    commands[k].op = k
    commands[k].left = view(0x10000 + 0x1000 * k, space)
    commands[k].right = view(0x20000 + 0x1000 * k, other)
    commands[k].output = view(0x11000 + 0x1000 * k, space)
device = (ctypes.c_uint8 * 8192)()
taken = ctypes.c_int(7)
message = ctypes.create_string_buffer(256)
hip.m3_hip_launch_chain.argtypes = [
    ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint32,
    ctypes.POINTER(ctypes.c_int), ctypes.c_char_p, ctypes.c_size_t]
code = hip.m3_hip_launch_chain(device, commands, 2, ctypes.byref(taken),
                               message, 256)
assert code == 0, message.value
assert taken.value == 0
print("refused")
"""


@pytest.mark.parametrize("space,other", [
    ((0,), (0,)), ((0,), (1,)), ((0, 3), (1, 3)), ((0, 3), (3,)),
    ((0, 3), (0, 1)), ((3, 0), (3, 1)), ((3, 0), (1, 0)), ((3, 0), (0,)),
    ((2, 0, 5), (2, 1, 1)), ((2, 0, 5), (1, 0, 1)), ((2, 0, 5), (5,)),
    ((4, 2, 0), (2, 1)), ((4, 2, 0), (4, 1, 1)), ((0, 2, 4), (0, 1, 1))])
def test_empty_runs_are_refused(space, other):
    result = subprocess.run(
        [sys.executable, "-c", CHILD, ROOT, repr((space, other))],
        capture_output=True, text=True, timeout=120)
    assert result.returncode == 0, (result.returncode, result.stderr)
    assert result.stdout.strip() == "refused"
