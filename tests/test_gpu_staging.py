"""Host copies through the device's pinned staging memory (GPU).

Copies of 257 bytes to 128 KiB to the device, and of up to 256 KiB or 1 to 4
MiB from it, go through staging memory, reads in chunks; others, those of
middle sizes behind a runtime copy or in a long row, and those with timing on
take other paths. Sizes at the edges of the paths and chunks, at any byte
offset, in rows, and from several threads over one device.
"""
import ctypes
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

from conftest import m3

pytestmark = pytest.mark.gpu

KIB = 1 << 10
MIB = 1 << 20


class Device:
    def __init__(self, arena_bytes):
        _, self.hip = m3.load()
        vp, sz = ctypes.c_void_p, ctypes.c_size_t
        self.hip.m3_hip_arena_reserve.argtypes = [vp, sz, ctypes.POINTER(vp),
                                                  ctypes.c_char_p, sz]
        self.hip.m3_hip_arena_release.argtypes = [vp, vp]
        for name in ("m3_hip_copy_h2d", "m3_hip_copy_d2h"):
            getattr(self.hip, name).argtypes = [vp, vp, vp, sz,
                                                ctypes.c_char_p, sz]
        self.device = vp()
        self.base = vp()
        message = ctypes.create_string_buffer(256)
        assert self.hip.m3_hip_device_open(0, ctypes.byref(self.device),
                                           message, 256) == 0
        self.hip.m3_hip_host_waits.argtypes = [
            vp, ctypes.POINTER(ctypes.c_uint64)]
        assert self.hip.m3_hip_arena_reserve(
            self.device, arena_bytes, ctypes.byref(self.base), message,
            256) == 0

    def write(self, offset, array):
        message = ctypes.create_string_buffer(256)
        assert self.hip.m3_hip_copy_h2d(
            self.device, self.base.value + offset,
            array.ctypes.data, array.nbytes, message, 256) == 0, message.value

    def read(self, offset, count):
        out = np.empty(count, np.uint8)
        message = ctypes.create_string_buffer(256)
        assert self.hip.m3_hip_copy_d2h(
            self.device, out.ctypes.data, self.base.value + offset, count,
            message, 256) == 0, message.value
        return out

    def host_waits(self):
        waits = ctypes.c_uint64(0)
        assert self.hip.m3_hip_host_waits(self.device,
                                          ctypes.byref(waits)) == 0
        return waits.value

    def close(self):
        self.hip.m3_hip_arena_release(self.device, self.base)
        self.hip.m3_hip_device_close(self.device)


@pytest.fixture()
def device(gpu):
    opened = Device(16 * MIB)
    yield opened
    opened.close()


@pytest.mark.parametrize("count", [
    1, 8, 15, 16, 17, 31, 255, 256, 257, 1000, 4096, 32 * KIB, 32 * KIB + 1,
    128 * KIB, 128 * KIB + 1, 192 * KIB, 256 * KIB - 1, 256 * KIB, 256 * KIB + 1,
    512 * KIB, 512 * KIB + 4, 700001, MIB - 65, MIB - 1, MIB, 3 * MIB + 7, 4 * MIB, 4 * MIB + 1])
@pytest.mark.parametrize("offset", [0, 1, 2, 4, 6, 8, 15])
def test_copy_sizes(device, count, offset):
    rng = np.random.default_rng(count + offset)
    room = count + 64
    before = rng.integers(0, 256, room, np.uint8)
    data = rng.integers(0, 256, count, np.uint8)
    device.write(0, before)
    device.write(offset, data)
    expected = before.copy()
    expected[offset:offset + count] = data
    assert np.array_equal(device.read(0, room), expected)
    assert np.array_equal(device.read(offset, count), data)


def test_many_writes_in_order(device):
    """Writes one after the other, overlapping and reusing the staging
    memory, take effect in order."""
    rng = np.random.default_rng(5)
    expected = np.zeros(2 * MIB, np.uint8)
    device.write(0, expected)
    for k in range(200):
        count = int(rng.integers(1, 300 * KIB))
        offset = int(rng.integers(0, 2 * MIB - count))
        data = np.full(count, k & 255, np.uint8)
        device.write(offset, data)
        data[:] = 77  # the caller's buffer is free when the call returns
        expected[offset:offset + count] = k & 255
    assert np.array_equal(device.read(0, 2 * MIB), expected)


@pytest.mark.parametrize("count", [32 * KIB, 96 * KIB, 128 * KIB, 256 * KIB])
def test_rows_of_copies(device, count):
    """Uniform rows, longer than those that stay staged, with runtime copies
    and small ones between: every copy whole, in order."""
    rng = np.random.default_rng(count)
    data = rng.integers(0, 256, (40, count), np.uint8)
    for k in range(40):
        device.write((k & 3) * count, data[k])
        if k % 17 == 16:
            device.write(8 * MIB, data[0][:100])
            device.write(9 * MIB, np.resize(data[0], 600 * KIB))
        assert np.array_equal(device.read((k & 3) * count, count), data[k])
    for k in range(40):
        device.write((k & 15) * count, data[k])
    for k in range(24, 40):
        assert np.array_equal(device.read((k & 15) * count, count), data[k])


def allocations():
    _, hip = m3.load()
    count = ctypes.c_uint64(0)
    hip.m3_hip_allocation_count.argtypes = [ctypes.POINTER(ctypes.c_uint64)]
    assert hip.m3_hip_allocation_count(ctypes.byref(count)) == 0
    return count.value


def test_handles_share_staging_memory(gpu):
    """Handles opened, used and closed in turn, and several open at once:
    after the first copies of the process no copy allocates, and closing one
    handle leaves the others' copies whole."""
    rng = np.random.default_rng(11)
    data = rng.integers(0, 256, 4 * MIB, np.uint8)

    def use(opened):
        for count in (1000, 96 * KIB, 192 * KIB):
            opened.write(16, data[:count])
            assert np.array_equal(opened.read(16, count), data[:count])
        opened.write(0, data[:2 * MIB])
        assert np.array_equal(opened.read(0, 2 * MIB), data[:2 * MIB])

    first = Device(5 * MIB)
    use(first)
    first.close()
    opened = Device(5 * MIB)
    before = allocations()
    use(opened)
    assert allocations() == before
    several = [Device(5 * MIB) for _ in range(6)]
    before = allocations()
    for one in several + [opened]:
        use(one)
    assert allocations() == before
    while several:
        several.pop(0).close()
        for one in several + [opened]:
            use(one)
    assert allocations() == before
    opened.close()


def test_staging_is_taken(gpu):
    """In a process of its own: the copies meant for the staging memory take
    it (one allocation, at the first of them), and the others do not."""
    code = """
import sys
sys.path.insert(0, %r)
import numpy as np
import test_gpu_staging as t
device = t.Device(5 * t.MIB)
def made(call):
    before = t.allocations()
    call()
    return t.allocations() - before
zeros = np.zeros(4 * t.MIB + 1, np.uint8)
assert made(lambda: device.write(0, zeros[:256])) == 0
assert made(lambda: device.write(0, zeros[:128 * t.KIB + 1])) == 0
assert made(lambda: device.read(0, 4 * t.MIB + 1)) == 0
assert made(lambda: device.read(0, 512 * t.KIB)) == 0
assert made(lambda: device.%s) == 1
assert made(lambda: device.write(0, zeros[:128 * t.KIB])) == 0
assert made(lambda: device.read(0, 4 * t.MIB)) == 0
device.close()
print("taken")
"""
    here = os.path.dirname(os.path.abspath(__file__))
    for first in ("read(0, 1)", "write(0, zeros[:257])", "read(0, t.MIB)"):
        result = subprocess.run([sys.executable, "-c", code % (here, first)],
                                capture_output=True, text=True, timeout=100)
        assert result.returncode == 0, result.stderr
        assert "taken" in result.stdout


def test_threads_copy_through_one_device(device):
    failures = []
    before = device.host_waits()

    def work(index):
        rng = np.random.default_rng(index)
        base = index * 4 * MIB
        for _ in range(40):
            count = int(rng.integers(257, 600 * KIB))
            data = rng.integers(0, 256, count, np.uint8)
            device.write(base, data)
            if not np.array_equal(device.read(base, count), data):
                failures.append((index, count))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert not failures
    # every copy of more than 256 bytes waits once, and every wait is counted
    assert device.host_waits() - before == 4 * 40 * 2
