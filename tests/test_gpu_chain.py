"""Command lists whose consecutive elementwise commands run as one launch
(GPU).

A binary operation or float cast over the output of the command before it
joins that command's launch (m3_hip_launch_chain), and TANH joins the
SNAKE1D before it. Every list here is compared, storage by storage, with the
oracle run command by command: random operations, links on either side,
dtypes, broadcasts of every class, special values, and lists in which an
output overlaps another operand, where the commands must stay apart.
"""
import sys

import numpy as np
import pytest

from conftest import m3
from harness import HipFixture, ViewSpec, as_bytes, run_oracle

pytestmark = pytest.mark.gpu

BINARY = [m3.OP_ADD, m3.OP_MUL, m3.OP_SUB, m3.OP_DIV]
FLOATS = [m3.F32, m3.F16, m3.BF16]


@pytest.fixture(scope="module")
def hip(gpu):
    fixture = HipFixture()
    yield fixture
    fixture.close()


def check(hip, arrays, commands, name):
    """`commands`: (kind, [ViewSpec]) in order over `arrays`."""
    print("gpu case", name, flush=True, file=sys.stderr)
    storages = [as_bytes(a).copy() for a in arrays]
    expected = storages
    for kind, specs in commands:
        status, expected = run_oracle(kind, expected, specs)
        assert status == m3.OK, name
    handles = hip.upload(storages)
    status, message = hip.execute([(kind, hip.views(handles, specs))
                                   for kind, specs in commands])
    assert status == m3.OK, (name, message)
    got = hip.download(handles, [np.empty_like(s) for s in storages])
    for index, (a, b) in enumerate(zip(got, expected)):
        if bytes(a) != bytes(b):
            diff = np.flatnonzero(a != b)
            raise AssertionError("%s: storage %d differs at %d bytes, first "
                                 "at byte %d" % (name, index, diff.size,
                                                 diff[0]))


def values(rng, dtype, count):
    x = (rng.standard_normal(count) * 3).astype(np.float32)
    picks = rng.integers(0, count, max(1, count // 61))
    x[picks] = rng.choice(np.array([np.inf, -np.inf, 0.0, -0.0, 1e30, 1e-39],
                                   np.float32), picks.size)
    if dtype == m3.F32:
        bits = x.view(np.uint32)
        nan, span = 0x7F800000, 1 << 23
    elif dtype == m3.F16:
        with np.errstate(over="ignore"):
            bits = x.astype(np.float16).view(np.uint16)
        nan, span = 0x7C00, 1 << 10
    else:
        bits = (x.view(np.uint32) >> 16).astype(np.uint16)
        nan, span = 0x7F80, 1 << 7
    picks = rng.integers(0, count, max(1, count // 83))
    bits[picks] = (nan + rng.integers(1, span, picks.size)).astype(bits.dtype)
    return bits


def operand(rng, arrays, dtype, shape, kind):
    """A new array read as a broadcast of class `kind` over `shape`."""
    b, c, n = shape
    size = m3.DTYPE_SIZES[dtype]
    dims = {"full": shape, "inner": (n,), "row": (c, 1), "scalar": (1,),
            "batch": (b, 1, 1), "plane": (c, n), "strided": shape}[kind]
    count = int(np.prod(dims))
    shift = int(rng.integers(0, 4))
    arrays.append(values(rng, dtype, count + 8))
    strides = None
    if kind == "strided":  # memory [b][n][c]: no chain takes it
        strides = (n * c * size, size, c * size)
    return ViewSpec(len(arrays) - 1, dtype, dims, strides, shift * size)


def output(arrays, dtype, shape, shift):
    size = m3.DTYPE_SIZES[dtype]
    arrays.append(np.full((int(np.prod(shape)) + 8) * size, 0xA5, np.uint8))
    return ViewSpec(len(arrays) - 1, dtype, shape, None, shift * size)


@pytest.mark.parametrize("shape", [(1, 1, 3), (1, 1, 4), (2, 3, 5),
                                   (3, 4, 64), (2, 7, 63), (1, 5, 1026),
                                   (2, 33, 257), (4, 100, 8), (2, 50, 3)])
@pytest.mark.parametrize("seed", range(12))
def test_random_chains(hip, shape, seed):
    rng = np.random.default_rng(71000 + 100 * seed + sum(shape))
    one_dtype = FLOATS[seed % 3] if seed % 2 else None
    kinds = ["full", "inner", "row", "scalar", "batch", "plane"]
    if seed % 4 == 3:
        kinds.append("strided")
    arrays = []
    commands = []
    last = operand(rng, arrays, one_dtype or FLOATS[int(rng.integers(3))],
                   shape, "full")
    for _ in range(int(rng.integers(2, 6))):
        dtype = one_dtype or FLOATS[int(rng.integers(3))]
        out = output(arrays, dtype, shape, int(rng.integers(0, 4)))
        if commands and dtype != last.dtype and rng.random() < 0.5:
            commands.append((m3.OP_CAST, [last, out]))
        else:
            other = operand(rng, arrays,
                            one_dtype or FLOATS[int(rng.integers(3))], shape,
                            kinds[int(rng.integers(len(kinds)))])
            pair = [last, other] if rng.random() < 0.5 else [other, last]
            commands.append((BINARY[int(rng.integers(4))], pair + [out]))
        last = out
    check(hip, arrays, commands, "chain %s seed %d" % (shape, seed))


def test_overlapping_lists(hip):
    """Lists in which one launch would read what it has already written."""
    rng = np.random.default_rng(72000)
    shape = (4, 8, 33)
    count = int(np.prod(shape))

    def spec(index, dims=shape, offset=0):
        return ViewSpec(index, m3.F32, dims, None, offset)

    def arrays(n):
        return [values(rng, m3.F32, count + 64) for _ in range(n)]

    # the second command squares the link; broadcasts the first output; and
    # overwrites the first operand, which a third command reads again
    check(hip, arrays(3), [
        (m3.OP_MUL, [spec(0), spec(1), spec(2)]),
        (m3.OP_MUL, [spec(2), spec(2), spec(0)])], "both operands linked")
    check(hip, arrays(4), [
        (m3.OP_ADD, [spec(0), spec(1), spec(2)]),
        (m3.OP_MUL, [spec(2), spec(2, (1, 8, 33)), spec(3)])],
        "output broadcast into the next")
    check(hip, arrays(3), [
        (m3.OP_ADD, [spec(0), spec(1), spec(2)]),
        (m3.OP_MUL, [spec(2), spec(1), spec(0)]),
        (m3.OP_ADD, [spec(0), spec(2), spec(1)])], "operands overwritten")
    check(hip, arrays(2), [
        (m3.OP_ADD, [spec(0), spec(1), spec(0)]),
        (m3.OP_MUL, [spec(0), spec(1), spec(0)]),
        (m3.OP_SUB, [spec(0), spec(1), spec(1)])], "in place")
    # outputs in one storage: apart, and a third one element into the first
    wide = values(rng, m3.F32, 2 * count + 64)
    check(hip, arrays(2) + [wide], [
        (m3.OP_ADD, [spec(0), spec(1), spec(2)]),
        (m3.OP_MUL, [spec(2), spec(1), spec(2, shape, 4 * count)])],
        "outputs side by side")
    check(hip, arrays(2) + [wide] + arrays(1), [
        (m3.OP_ADD, [spec(0), spec(1), spec(2)]),
        (m3.OP_MUL, [spec(2), spec(1), spec(3)]),
        (m3.OP_SUB, [spec(3), spec(0), spec(2, shape, 4 * count - 4)])],
        "outputs that meet")
    # the chain's value broadcast from a view that the second output covers
    check(hip, arrays(3), [
        (m3.OP_ADD, [spec(0, (8, 33)), spec(1), spec(2)]),
        (m3.OP_MUL, [spec(2), spec(1), spec(0)])], "value overwritten")


def test_chain_before_a_failing_check(hip):
    """The commands before a softmax over a NaN they produced have run, it
    and the chain after it have not."""
    shape = (4, 16)
    x = np.ones(64, np.float32)
    x[5] = np.nan
    one = np.ones(1, np.float32)
    arrays = [x, one] + [np.full(64, -9.0, np.float32) for _ in range(5)]
    full = [ViewSpec(i, m3.F32, shape) for i in range(7)]
    scalar = ViewSpec(1, m3.F32, (1,))
    handles = hip.upload([as_bytes(a).copy() for a in arrays])
    status, message = hip.execute([
        (kind, hip.views(handles, specs)) for kind, specs in [
            (m3.OP_MUL, [full[0], scalar, full[2]]),
            (m3.OP_ADD, [full[2], scalar, full[3]]),
            (m3.OP_SOFTMAX, [full[3], full[4]]),
            (m3.OP_MUL, [full[4], scalar, full[5]]),
            (m3.OP_ADD, [full[5], scalar, full[6]])]])
    assert status == m3.OUT_OF_RANGE, message
    got = hip.download(handles, [np.empty_like(as_bytes(a)) for a in arrays])
    got = [g.view(np.float32) for g in got]
    assert got[2][0] == 1.0 and np.isnan(got[2][5])
    assert got[3][0] == 2.0 and np.isnan(got[3][5])
    for k in (4, 5, 6):
        assert np.all(got[k] == -9.0)


@pytest.mark.parametrize("shape", [(1, 3, 4), (2, 5, 5), (2, 7, 63),
                                   (3, 2, 1026), (2, 5, 3)])
def test_snake1d_tanh(hip, shape):
    rng = np.random.default_rng(73000 + sum(shape))
    count = int(np.prod(shape))
    x = values(rng, m3.F32, count)
    alpha = (rng.random(shape[1]) * 3 + 0.1).astype(np.float32)
    room = [np.full(4 * (count + 8), 0xA5, np.uint8) for _ in range(2)]
    x_view = ViewSpec(0, m3.F32, shape)
    a_view = ViewSpec(1, m3.F32, (1, shape[1], 1))
    for shift in (0, 1):
        y = ViewSpec(2, m3.F32, shape, None, 4 * shift)
        wave = ViewSpec(3, m3.F32, shape, None, 12 * shift)
        check(hip, [x, alpha] + room,
              [(m3.OP_SNAKE1D, [x_view, a_view, y]),
               (m3.OP_TANH, [y, wave])], "snake1d tanh %s" % (shape,))
    check(hip, [x, alpha] + room,
          [(m3.OP_SNAKE1D, [x_view, a_view, x_view]),
           (m3.OP_TANH, [x_view, ViewSpec(2, m3.F32, shape)])],
          "snake1d in place, tanh %s" % (shape,))
    check(hip, [x, alpha] + room,
          [(m3.OP_SNAKE1D, [x_view, a_view, ViewSpec(2, m3.F32, shape)]),
           (m3.OP_TANH, [ViewSpec(2, m3.F32, shape), x_view])],
          "snake1d, tanh over its input %s" % (shape,))


@pytest.mark.parametrize("shape,dims", [((3, 0), (3, 1)), ((0, 4), (1, 4)),
                                        ((2, 0, 5), (2, 1, 1)),
                                        ((0, 3), (3,))])
def test_lists_over_empty_tensors(hip, shape, dims):
    """An empty run inside a list does nothing, and the commands around it
    run."""
    rng = np.random.default_rng(8)
    empty = np.zeros(0, np.uint8)
    other = values(rng, m3.F32, 16)
    x, s = values(rng, m3.F32, 24), values(rng, m3.F32, 24)
    arrays = [empty, other, empty.copy(), empty.copy(), x, s,
              np.zeros(24, np.float32), np.zeros(24, np.float32)]
    e = [ViewSpec(i, m3.F32, shape) for i in (0, 2, 3)]
    o = ViewSpec(1, m3.F32, dims)
    full = [ViewSpec(i, m3.F32, (24,)) for i in (4, 5, 6, 7)]
    check(hip, arrays,
          [(m3.OP_MUL, [full[0], full[1], full[2]]),
           (m3.OP_MUL, [e[0], o, e[1]]), (m3.OP_ADD, [e[1], o, e[2]]),
           (m3.OP_ADD, [full[2], full[1], full[3]])],
          "empty %s %s" % (shape, dims))
