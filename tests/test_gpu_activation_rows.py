"""SNAKE1D, TANH and GATED_SILU at odd lengths, alignments and row pitches
(GPU), bit for bit against the oracle.

Tensors with fewer elements than the device has lanes (about: 393,216 to
917,504 on one MI355X) run one element per lane; the vector kernels take four
consecutive elements per lane at any alignment. A Snake1d group that a channel's end cuts uses two alphas; a
GATED_SILU group that a row's end cuts reads its elements one by one when
gate and up are rows of a wider tensor.
"""
import sys

import numpy as np
import pytest

from conftest import m3
from harness import HipFixture, ViewSpec, as_bytes, run_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip(gpu):
    fixture = HipFixture()
    yield fixture
    fixture.close()


def compare(hip, kind, storages, views, name):
    print("gpu case", name, flush=True, file=sys.stderr)
    status, got, message = hip.run(kind, storages, views)
    ostatus, expected = run_oracle(kind, storages, views)
    assert status == ostatus == m3.OK, (name, m3.status_name(status), message)
    for index, (a, b) in enumerate(zip(got, expected)):
        if bytes(a) != bytes(b):
            diff = np.flatnonzero(a != b)
            raise AssertionError("%s: storage %d differs at %d bytes, first "
                                 "at byte %d" % (name, index, diff.size,
                                                 diff[0]))


def special(rng, values):
    """A few infinities, NaN, zeros and large magnitudes among values."""
    picks = rng.integers(0, values.size, max(1, values.size // 97))
    values.ravel()[picks] = rng.choice(
        np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, 1e30, -3e4, 1e-40],
                 np.float32), picks.size)
    return values


@pytest.mark.parametrize("batch,channels,length", [
    (1, 1, 4), (1, 3, 4), (2, 5, 5), (2, 7, 6), (1, 64, 7), (3, 9, 63),
    (2, 33, 65), (2, 3, 1021), (1, 2, 4098), (2, 5, 3), (2, 5, 1),
    (2, 66, 3001), (1, 99001, 4), (2, 40009, 5), (2, 30011, 7),
    (3, 131, 1023), (1, 3, 150001)])
def test_snake1d_lengths(hip, batch, channels, length):
    rng = np.random.default_rng(61000 + channels * 31 + length)
    shape = (batch, channels, length)
    x = special(rng, (rng.standard_normal(shape) * 4).astype(np.float32))
    alpha = (rng.random(channels) * 40 + 0.1).astype(np.float32)
    alpha[0] = 200.0  # large angles
    for shift in (0, 1, 3):
        moved = np.zeros(x.size + 8, np.float32)
        moved[shift:shift + x.size] = x.ravel()
        out = np.full((x.size + 8) * 4, 0xA5, np.uint8)
        compare(hip, m3.OP_SNAKE1D, [as_bytes(moved), as_bytes(alpha), out],
                [ViewSpec(0, m3.F32, shape, None, 4 * shift),
                 ViewSpec(1, m3.F32, (1, channels, 1)),
                 ViewSpec(2, m3.F32, shape, None, 4 * ((3 * shift) % 4))],
                "snake1d %s shift %d" % (shape, shift))


@pytest.mark.parametrize("count", [1, 3, 4, 5, 1023, 4097, 393215, 393216,
                                   700003])
@pytest.mark.parametrize("shift", [1, 2, 3])
def test_tanh_alignments(hip, count, shift):
    rng = np.random.default_rng(62000 + count + shift)
    x = special(rng, (rng.standard_normal(count + 8) * 3).astype(np.float32))
    out = np.full((count + 8) * 4, 0xA5, np.uint8)
    compare(hip, m3.OP_TANH, [as_bytes(x), out],
            [ViewSpec(0, m3.F32, (count,), None, 4 * shift),
             ViewSpec(1, m3.F32, (count,), None, 4 * (4 - shift))],
            "tanh %d shift %d" % (count, shift))


@pytest.mark.parametrize("dtype", [m3.F32, m3.F16, m3.BF16])
@pytest.mark.parametrize("count", [5, 4099, 393215, 393217, 524289, 786435])
def test_gated_silu_alignments(hip, dtype, count):
    """Contiguous operands at different alignments, on both sides of the
    sizes from which the vector kernels run."""
    rng = np.random.default_rng(64000 + count)
    size = m3.DTYPE_SIZES[dtype]
    values = special(rng, (rng.standard_normal(2 * count + 8) * 4).astype(
        np.float32))
    if dtype == m3.F16:
        with np.errstate(over="ignore"):
            values = values.astype(np.float16).view(np.uint16)
    elif dtype == m3.BF16:
        values = (values.view(np.uint32) >> 16).astype(np.uint16)
    for shift in (0, 1, 3):
        out = np.full((count + 8) * size, 0xA5, np.uint8)
        compare(hip, m3.OP_GATED_SILU, [as_bytes(values), out],
                [ViewSpec(0, dtype, (count,), None, shift * size),
                 ViewSpec(0, dtype, (count,), None,
                          (count + 2 * shift) * size),
                 ViewSpec(1, dtype, (count,), None, shift * size)],
                "gated_silu %d shift %d dtype %d" % (count, shift, dtype))


@pytest.mark.parametrize("dtype", [m3.F32, m3.F16, m3.BF16])
@pytest.mark.parametrize("rows,width", [(1, 9), (3, 4), (5, 5), (7, 6),
                                        (9, 7), (2, 63), (33, 65), (5, 1023),
                                        (17, 3), (4, 1024), (131075, 4),
                                        (240001, 4), (200003, 5),
                                        (150001, 7), (1021, 1023)])
def test_gated_silu_rows(hip, dtype, rows, width):
    """Both halves of one tensor's rows, and one operand contiguous while
    the other lies in padded rows; every start one element off. The larger
    tensors have enough elements for the kernel of rows, the others run the
    general one."""
    rng = np.random.default_rng(63000 + rows * 17 + width)
    size = m3.DTYPE_SIZES[dtype]

    def values(count):
        v = special(rng, (rng.standard_normal(count) * 4).astype(np.float32))
        if dtype == m3.F16:
            with np.errstate(over="ignore"):
                return v.astype(np.float16).view(np.uint16)
        if dtype == m3.BF16:
            return (v.view(np.uint32) >> 16).astype(np.uint16)
        return v

    pitch = 2 * width + 1
    both = values(rows * pitch + 4)
    flat = values(rows * width + 4)
    strides = (pitch * size, size)
    shape = (rows, width)
    out = np.full((rows * width + 4) * size, 0xA5, np.uint8)
    gate = ViewSpec(0, dtype, shape, strides, size)
    for up, name in [
            (ViewSpec(0, dtype, shape, strides, (1 + width) * size), "both"),
            (ViewSpec(1, dtype, shape, None, 3 * size), "flat up"),
            (ViewSpec(1, dtype, shape, (0, size), size), "broadcast up")]:
        compare(hip, m3.OP_GATED_SILU, [as_bytes(both), as_bytes(flat), out],
                [gate, up, ViewSpec(2, dtype, shape, None, size)],
                "gated_silu %s %s dtype %d" % (name, shape, dtype))
    compare(hip, m3.OP_GATED_SILU, [as_bytes(both), as_bytes(flat), out],
            [ViewSpec(1, dtype, shape, None, size), gate,
             ViewSpec(2, dtype, shape)],
            "gated_silu flat gate %s dtype %d" % (shape, dtype))
