"""Softmax rows of any width and alignment, every kernel class (GPU).

Rows move in four-column accesses at any alignment; the lane that holds a
row's end reads its last four columns and moves them into place. The widths
are the edges of the kernels' classes (64, 128, 256, 512, 1024, 2048 and the
long-row classes up to 65,536, the streamed kernel beyond), one to three
columns past and short of a multiple of four, and those where the two halves
of a row of 1,025 to 2,048 columns change length. Each is checked against
the oracle bit for bit, with -inf tails, +inf entries and all -inf rows.
"""
import sys

import numpy as np
import pytest

from conftest import m3
from harness import HipFixture, ViewSpec, as_bytes, run_oracle

pytestmark = pytest.mark.gpu

SHORT = [1, 2, 3, 4, 5, 6, 7, 63, 64, 65, 127, 128, 129, 130, 255, 256]
LANE = [257, 258, 259, 320, 511, 512, 513, 575, 577, 1022, 1023, 1024]
HALVES = [1025, 1026, 1088, 1089, 1151, 1152, 1153, 1281, 1408, 1409, 1663,
          1921, 2045, 2047, 2048]
LONG = [2049, 2051, 4095, 4097, 8190, 8193, 12289, 16383, 16385, 20479,
        20481, 24577, 32767, 32769, 40000, 49151, 49153, 65533, 65536, 65537]
DTYPES = [(m3.F32, m3.F32), (m3.F16, m3.F16), (m3.BF16, m3.BF16),
          (m3.BF16, m3.F32), (m3.F32, m3.F16)]


@pytest.fixture(scope="module")
def hip(gpu):
    fixture = HipFixture()
    yield fixture
    fixture.close()


def compare(hip, storages, views, name):
    print("gpu case", name, flush=True, file=sys.stderr)
    status, got, message = hip.run(m3.OP_SOFTMAX, storages, views)
    ostatus, expected = run_oracle(m3.OP_SOFTMAX, storages, views)
    assert status == ostatus, (name, m3.status_name(status), message)
    for index, (a, b) in enumerate(zip(got, expected)):
        if bytes(a) != bytes(b):
            diff = np.flatnonzero(a != b)
            raise AssertionError("%s: storage %d differs at %d bytes, first "
                                 "at byte %d" % (name, index, diff.size,
                                                 diff[0]))


def logits_of(rng, rows, width):
    logits = (rng.standard_normal((rows, width)) * 3).astype(np.float32)
    for r in range(rows):
        kind = r % 7
        if kind == 1:  # a -inf tail that starts anywhere
            logits[r, 1 + int(rng.integers(0, width)):] = -np.inf
        elif kind == 2:
            logits[r, :] = -np.inf
        elif kind == 3:  # +inf entries, the last column among them
            logits[r, ::3] = np.inf
            logits[r, width - 1] = np.inf
        elif kind == 4:  # the maximum alone in the last column
            logits[r, width - 1] = 40.0
        elif kind == 5:  # only the last column is not -inf
            logits[r, : width - 1] = -np.inf
    return logits


def elements(logits, dtype):
    if dtype == m3.F16:
        return logits.astype(np.float16).view(np.uint16)
    if dtype == m3.BF16:
        return (logits.view(np.uint32) >> 16).astype(np.uint16)
    return logits


@pytest.mark.parametrize("dtypes", DTYPES)
@pytest.mark.parametrize("width", SHORT + LANE + HALVES + LONG)
def test_softmax_row_widths(hip, width, dtypes):
    """Contiguous rows, every row's start at another alignment when the
    width is odd; rows that do not fill the last wave."""
    rng = np.random.default_rng(41000 + width * 8 + dtypes[0])
    rows = 43 if width <= 256 else 23 if width <= 2048 else 8
    source = elements(logits_of(rng, rows, width), dtypes[0])
    out = np.zeros(rows * width * m3.DTYPE_SIZES[dtypes[1]], np.uint8)
    compare(hip, [as_bytes(source), out],
            [ViewSpec(0, dtypes[0], (rows, width)),
             ViewSpec(1, dtypes[1], (rows, width))],
            "rows %s w=%d" % (dtypes, width))


@pytest.mark.parametrize("dtypes", DTYPES)
@pytest.mark.parametrize("width", [7, 66, 129, 256, 259, 512, 1023, 1024,
                                   1090, 2048, 2050, 4096, 16386])
def test_softmax_row_alignments(hip, width, dtypes):
    """Input and output that start one to three elements past a 16-byte
    boundary (guard elements around the output stay as they are), padded
    rows, uneven outer axes, and in place."""
    rng = np.random.default_rng(43000 + width * 8 + dtypes[0])
    rows = 12
    sizes = [m3.DTYPE_SIZES[d] for d in dtypes]
    source = elements(logits_of(rng, rows, width), dtypes[0])
    count = rows * width
    for shift in (1, 2, 3):
        moved = np.zeros(count + 8, source.dtype)
        moved[shift:shift + count] = source.ravel()
        out = np.full((count + 8) * sizes[1], 0xA5, np.uint8)
        compare(hip, [as_bytes(moved), out],
                [ViewSpec(0, dtypes[0], (rows, width), None,
                          shift * sizes[0]),
                 ViewSpec(1, dtypes[1], (rows, width), None,
                          (4 - shift) * sizes[1])],
                "rows shifted %d %s w=%d" % (shift, dtypes, width))
    out = np.zeros(count * sizes[1], np.uint8)
    padded = np.zeros((rows, width + 3), source.dtype)
    padded[:, :width] = source
    compare(hip, [as_bytes(padded), out],
            [ViewSpec(0, dtypes[0], (rows, width),
                      ((width + 3) * sizes[0], sizes[0])),
             ViewSpec(1, dtypes[1], (rows, width))],
            "rows padded %s w=%d" % (dtypes, width))
    compare(hip, [as_bytes(source), out],
            [ViewSpec(0, dtypes[0], (4, 3, width),
                      (width * sizes[0], 4 * width * sizes[0], sizes[0])),
             ViewSpec(1, dtypes[1], (4, 3, width))],
            "rows uneven %s w=%d" % (dtypes, width))
    if dtypes[0] == dtypes[1]:
        compare(hip, [as_bytes(source)],
                [ViewSpec(0, dtypes[0], (rows, width)),
                 ViewSpec(0, dtypes[0], (rows, width))],
                "rows in place %s w=%d" % (dtypes, width))


@pytest.mark.parametrize("dtypes", [(m3.F32, m3.F32), (m3.BF16, m3.F32)])
@pytest.mark.parametrize("width,rows", [
    (257, 2049), (511, 2049), (513, 2049), (1021, 2049), (2049, 257),
    (4097, 257), (8193, 300), (16385, 257)])
def test_softmax_many_rows(hip, width, rows, dtypes):
    """More rows than the layouts for a few rows take: the same widths in
    the other layouts, with rows of every kind at every place of a wave."""
    rng = np.random.default_rng(45000 + width)
    source = elements(logits_of(rng, rows, width), dtypes[0])
    out = np.zeros(rows * width * m3.DTYPE_SIZES[dtypes[1]], np.uint8)
    compare(hip, [as_bytes(source), out],
            [ViewSpec(0, dtypes[0], (rows, width)),
             ViewSpec(1, dtypes[1], (rows, width))],
            "many rows %s w=%d rows=%d" % (dtypes, width, rows))
