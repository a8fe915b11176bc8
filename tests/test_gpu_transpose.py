"""COPY and CAST of permuted views through transposing tiles (GPU).

An input whose unit-stride axis is not the output's innermost one runs a
64 x 128 tile kernel when both axes have at least 16 elements and fill enough
of their tiles, else the general kernel. The extents are the edges of the tiles and of the rule, and
one to three elements past a multiple of four; the views are transposes
with outer axes before, between and after, padded, broadcast and offset.
Checked against the oracle bit for bit, NaN payloads included.
"""
import sys

import numpy as np
import pytest

from conftest import m3
from harness import HipFixture, ViewSpec, as_bytes, run_oracle

pytestmark = pytest.mark.gpu

PAIRS = [(s, d) for s in (m3.F32, m3.F16, m3.BF16, m3.I32)
         for d in (m3.F32, m3.F16, m3.BF16, m3.I32)]


@pytest.fixture(scope="module")
def hip(gpu):
    fixture = HipFixture()
    yield fixture
    fixture.close()


def compare(hip, src, dst, source, view, shape, name, offset=0):
    print("gpu case", name, flush=True, file=sys.stderr)
    kind = m3.OP_COPY if src == dst else m3.OP_CAST
    size = m3.DTYPE_SIZES[dst]
    out = np.full((int(np.prod(shape)) + 8) * size, 0xA5, np.uint8)
    storages = [as_bytes(source), out]
    views = [view, ViewSpec(1, dst, shape, None, offset * size)]
    status, got, message = hip.run(kind, storages, views)
    ostatus, expected = run_oracle(kind, storages, views)
    assert status == ostatus == m3.OK, (name, m3.status_name(status), message)
    for a, b in zip(got, expected):
        if bytes(a) != bytes(b):
            diff = np.flatnonzero(a != b)
            raise AssertionError("%s differs at %d bytes, first at byte %d"
                                 % (name, diff.size, diff[0]))


def source_of(rng, src, dst, count):
    if src == m3.I32:
        return rng.integers(-2 ** 31, 2 ** 31, count).astype(np.int32)
    values = (rng.standard_normal(count) * 100).astype(np.float32)
    if src == m3.F16:
        bits = values.astype(np.float16).view(np.uint16)
    elif src == m3.BF16:
        bits = (values.view(np.uint32) >> 16).astype(np.uint16)
    else:
        bits = values.view(np.uint32)
    if dst != m3.I32:  # every bit pattern: NaN payloads, infinities, tiny
        picks = rng.integers(0, count, count // 4)
        bits[picks] = rng.integers(0, 1 << (8 * m3.DTYPE_SIZES[src]),
                                   picks.size)
    return bits


@pytest.mark.parametrize("src,dst", PAIRS)
@pytest.mark.parametrize("length,channels", [
    (16, 16), (15, 64), (64, 15), (17, 18), (63, 65), (64, 128), (65, 127),
    (127, 66), (129, 67), (130, 64), (257, 131), (16, 64), (64, 16), (16, 48),
    (24, 24), (24, 32), (32, 40), (40, 32), (30, 43), (16, 65), (160, 16)])
def test_transposed(hip, src, dst, length, channels):
    rng = np.random.default_rng(51000 + length * 7 + channels)
    size = m3.DTYPE_SIZES[src]
    source = source_of(rng, src, dst, 2 * length * channels)
    strides = (length * channels * size, size, channels * size)
    compare(hip, src, dst, source,
            ViewSpec(0, src, (2, channels, length), strides),
            (2, channels, length),
            "%d->%d [2,%d,%d]" % (src, dst, channels, length))


@pytest.mark.parametrize("src,dst", [(m3.F32, m3.F32), (m3.F16, m3.F16),
                                     (m3.BF16, m3.F32), (m3.F32, m3.BF16)])
def test_transposed_layouts(hip, src, dst):
    rng = np.random.default_rng(52000 + 4 * src + dst)
    size = m3.DTYPE_SIZES[src]
    source = source_of(rng, src, dst, 3 * 5 * 70 * 90 + 64)
    # memory [3][70][5][90]: views (a, d, c, b) and (c, d, a, b)
    a, b, c, d = 3, 70, 5, 90
    sa, sb, sc, sd = b * c * d * size, c * d * size, d * size, size
    for shape, strides, name in [
            ((a, d, c, b), (sa, sd, sc, sb), "outer axis between"),
            ((c, d, a, b), (sc, sd, sa, sb), "uneven outer axes"),
            ((d, a, c, b), (sd, sa, sc, sb), "unit axis first"),
            ((2, d, b), (0, sd, sb), "broadcast outer axis"),
            ((d, b), (sd, sb + 3 * size), "padded rows")]:
        compare(hip, src, dst, source, ViewSpec(0, src, shape, strides),
                shape, "%s %d->%d" % (name, src, dst))
    # input and output one to three elements past a boundary
    for shift in (1, 2, 3):
        compare(hip, src, dst, source,
                ViewSpec(0, src, (d, b), (sd, sb), shift * size), (d, b),
                "shifted %d %d->%d" % (shift, src, dst), 4 - shift)
