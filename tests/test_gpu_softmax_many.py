"""Softmax over more rows than the device has room for at once (GPU).

Tensors of few rows run kernels that spread a row over more lanes: rows of
257..1,024 columns up to eight rows per CU, rows of 2,049..65,536 columns up
to one per CU. The tests of those widths elsewhere have a handful of rows;
here the row counts come from the device's CUs, so that the kernels for many
rows run: every row class, aligned and ragged, F32 and 16-bit, with special
rows at every place of a wave, in place, uneven row starts, rounding ties,
segments whose exponentials are formed twice, and workgroups that take
several rows in turn. Checked against the oracle bit for bit.
"""
import ctypes
import os

import numpy as np
import pytest

from conftest import m3
from harness import HipFixture, ViewSpec, as_bytes, subnormal_tie_rows
from test_gpu_parity import lane_row_logits
from test_gpu_softmax_wide import (compare, source_of, unstaged_rows,
                                   wide_rows)

pytestmark = pytest.mark.gpu

# the widest rows of each class of many long rows: even ones and ragged ones
CLASSES = [4096, 8192, 12288, 16384, 20480, 24576, 32768, 49152, 65536]
WIDE = [w for c, cut in zip(CLASSES, [1, 3, 2, 5, 1, 6, 3, 2, 1])
        for w in (c, c - cut)]


@pytest.fixture(scope="module")
def hip(gpu):
    fixture = HipFixture()
    yield fixture
    fixture.close()


@pytest.fixture(scope="module")
def compute_units(gpu):
    _, lib = m3.load()
    device = ctypes.c_void_p()
    message = ctypes.create_string_buffer(256)
    units = ctypes.c_uint32(0)
    assert lib.m3_hip_device_open(0, ctypes.byref(device), message, 256) == 0
    lib.m3_hip_device_properties.argtypes = [
        ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p,
        ctypes.POINTER(ctypes.c_uint32), ctypes.c_char_p, ctypes.c_size_t]
    assert lib.m3_hip_device_properties(device, None, 0, None,
                                        ctypes.byref(units), message,
                                        256) == 0
    lib.m3_hip_device_close(device)
    return units.value


def run(hip, logits, dtypes, name):
    shape = logits.shape
    compare(hip, [source_of(logits, dtypes[0]),
                  np.zeros(logits.size * m3.DTYPE_SIZES[dtypes[1]],
                           np.uint8)],
            [ViewSpec(0, dtypes[0], shape), ViewSpec(1, dtypes[1], shape)],
            "%s %s %s" % (name, shape, dtypes))


def repeated(block, rows):
    """`rows` rows that cycle through those of `block`, the whole cycle one
    row on from one time to the next."""
    index = np.arange(rows)
    return block[(index + index // len(block)) % len(block)]


@pytest.mark.parametrize("dtypes", [(m3.F32, m3.F32), (m3.F16, m3.F16),
                                    (m3.BF16, m3.BF16), (m3.BF16, m3.F32),
                                    (m3.F32, m3.BF16), (m3.F16, m3.F32)])
@pytest.mark.parametrize("width", [260, 511, 512, 700, 1020, 1024])
def test_many_lane_rows(hip, compute_units, width, dtypes):
    rng = np.random.default_rng(81000 + width + 8 * dtypes[0] + dtypes[1])
    rows = 8 * compute_units + 5
    run(hip, lane_row_logits(rng, rows, width), dtypes, "many lane rows")


@pytest.mark.parametrize("dtype", [m3.F32, m3.BF16])
@pytest.mark.parametrize("width", [300, 512, 1000, 1024])
def test_many_lane_rows_layouts(hip, compute_units, width, dtype):
    rng = np.random.default_rng(82000 + width + dtype)
    outer = 4 * compute_units + 1
    rows = 2 * outer
    size = m3.DTYPE_SIZES[dtype]
    logits = lane_row_logits(rng, rows, width)
    source = source_of(logits, dtype)
    out = np.zeros(rows * width * size, np.uint8)
    compare(hip, [source, out],
            [ViewSpec(0, dtype, (2, outer, width),
                      (width * size, 2 * width * size, size)),
             ViewSpec(1, dtype, (2, outer, width))],
            "many lane rows uneven %d dtype %d" % (width, dtype))
    compare(hip, [source], [ViewSpec(0, dtype, (rows, width)),
                            ViewSpec(0, dtype, (rows, width))],
            "many lane rows in place %d dtype %d" % (width, dtype))


@pytest.mark.parametrize("dtypes", [(m3.F32, m3.F32), (m3.BF16, m3.F16)])
@pytest.mark.parametrize("width", WIDE)
def test_many_wide_rows(hip, compute_units, width, dtypes):
    rng = np.random.default_rng(83000 + width + dtypes[0])
    rows = compute_units + 3
    run(hip, repeated(wide_rows(rng, 24, width), rows), dtypes,
        "many wide rows")


@pytest.mark.parametrize("width", [4096, 12288, 24573])
def test_many_wide_rows_in_place(hip, compute_units, width):
    rng = np.random.default_rng(84000 + width)
    rows = compute_units + 1
    logits = np.ascontiguousarray(repeated(wide_rows(rng, 24, width), rows))
    compare(hip, [as_bytes(logits)], [ViewSpec(0, m3.F32, (rows, width)),
                                      ViewSpec(0, m3.F32, (rows, width))],
            "many wide rows in place %d" % width)


def test_many_wide_rows_subnormal_ties(hip, compute_units):
    rng = np.random.default_rng(85000)
    rows = compute_units + 8
    run(hip, repeated(subnormal_tie_rows(rng, 24, 8192), rows),
        (m3.F32, m3.F32), "many wide rows, ties")


@pytest.mark.parametrize("width,near", [(4096, 2200), (12286, 3600),
                                        (16384, 3600), (24576, 3600),
                                        (32768, 3600), (49152, 3600)])
def test_many_wide_rows_unstaged_segments(hip, compute_units, width, near):
    """Rows with more segments near a power of two than the kernel keeps
    exponentials of."""
    rng = np.random.default_rng(86000 + width)
    rows = compute_units + 1
    run(hip, repeated(unstaged_rows(rng, 12, width, near), rows),
        (m3.F32, m3.F32), "many wide rows, unstaged")


@pytest.fixture(scope="module")
def hip_capped(gpu):
    """At most 37 workgroups per long-row launch."""
    saved = os.environ.get("M3_HIP_SOFTMAX_WIDE_GRID")
    os.environ["M3_HIP_SOFTMAX_WIDE_GRID"] = "37"
    try:
        fixture = HipFixture()
    finally:
        if saved is None:
            del os.environ["M3_HIP_SOFTMAX_WIDE_GRID"]
        else:
            os.environ["M3_HIP_SOFTMAX_WIDE_GRID"] = saved
    yield fixture
    fixture.close()


@pytest.mark.parametrize("dtypes", [(m3.F32, m3.F32), (m3.BF16, m3.F32)])
@pytest.mark.parametrize("width", WIDE[:14:2] + WIDE[1:15:4])
def test_many_wide_rows_several_per_workgroup(hip_capped, compute_units,
                                              width, dtypes):
    rng = np.random.default_rng(87000 + width + dtypes[0])
    rows = compute_units + 40
    run(hip_capped, repeated(wide_rows(rng, 24, width), rows), dtypes,
        "many wide rows, 37 workgroups")
