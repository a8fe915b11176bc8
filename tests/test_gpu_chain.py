"""Command lists whose consecutive elementwise commands run as one launch
(GPU).

A binary operation or float cast over the output of the command before it
joins that command's launch (m3_hip_launch_chain), and TANH joins the
SNAKE1D before it. Every list here is compared, storage by storage, with the
oracle run command by command: random operations, links on either side,
dtypes, broadcasts of every class, special values, and lists in which an
output overlaps another operand, where the commands must stay apart.
"""
import ctypes
import sys

import numpy as np
import pytest

from conftest import m3
from harness import (HipFixture, HipScanFixture, ViewSpec, as_bytes,
                     run_oracle)

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


def launches(nodes, shape):
    """The kernels, by launches, of one run of a session over `nodes`:
    (kind, out dtype, operand names), "x" the input, "c" a constant of
    shape's last axis, "s" a Snake1d alpha, and a number the value of that
    node."""
    rng = np.random.default_rng(9)
    graph = m3.Graph()
    values = {"x": graph.add_value(m3.INPUT, m3.F32, shape)}
    for name, dims in (("c", (shape[-1],)), ("s", (1, shape[1], 1))):
        if any(name in inputs for _, _, inputs in nodes):
            values[name] = graph.add_value(m3.CONSTANT, m3.F32, dims)
            graph.set_constant(values[name],
                               (rng.random(dims) + 0.5).astype(np.float32))
    for k, (kind, dtype, inputs) in enumerate(nodes):
        values[k] = graph.add_value(m3.OUTPUT, dtype, shape)
        graph.add_node(kind, [values[v] for v in inputs], [values[k]])
    session = m3.Session(graph)
    graph.free()
    session.write(values["x"],
                  rng.standard_normal(shape).astype(np.float32))
    session.run()
    session.timing_reset()
    session.timing_enable(True)
    session.run()
    kernels = session.timing_read()
    session.timing_enable(False)
    session.free()
    return {name: count for name, (count, _) in kernels.items()}


def test_chains_are_taken(gpu, monkeypatch):
    """Runs that a kernel takes are one launch, and others are not (in
    sessions that leave the commands as they are: M3_HIP_FUSION=0)."""
    monkeypatch.setenv("M3_HIP_FUSION", "0")
    shape = (2, 16, 1000)
    mul, cast = m3.OP_MUL, m3.OP_CAST
    assert launches([(mul, m3.F32, ["x", "c"]), (cast, m3.BF16, [0])],
                    shape) == {"m3_chain": 1}
    assert launches([(mul, m3.F32, ["x", "c"]), (cast, m3.F16, [0]),
                     (cast, m3.F32, [1])], shape) == {"m3_chain": 1}
    assert launches([(m3.OP_SNAKE1D, m3.F32, ["x", "s"]),
                     (m3.OP_TANH, m3.F32, [0])],
                    shape) == {"m3_snake1d_tanh": 1}
    # the second command reads something else than the first one's output
    apart = launches([(mul, m3.F32, ["x", "c"]), (cast, m3.BF16, ["x"])],
                     shape)
    assert "m3_chain" not in apart and sum(apart.values()) == 2


def test_overlapping_runs_are_refused(gpu):
    """m3_hip_launch_chain over one device: taken with outputs apart, and
    refused, with nothing launched, when an output overlaps another output
    or an operand."""
    _, hip_lib = m3.load()

    class Command(ctypes.Structure):
        _fields_ = [("kind", ctypes.c_uint32), ("op", ctypes.c_uint32),
                    ("link", ctypes.c_uint32), ("left", m3.HipView),
                    ("right", m3.HipView), ("output", m3.HipView)]

    hip_lib.m3_hip_launch_chain.argtypes = [
        ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint32,
        ctypes.POINTER(ctypes.c_int), ctypes.c_char_p, ctypes.c_size_t]
    device = HipScanFixture()
    try:
        count = 1000
        at = [device.upload(np.zeros(count, np.float32)) for _ in range(5)]

        def view(address):
            return device.view(address, m3.F32, (count,))

        def taken(x, y, first, z, second):
            commands = (Command * 2)()
            commands[0] = Command(0, 0, 0, view(x), view(y), view(first))
            commands[1] = Command(0, 1, 0, view(first), view(z),
                                  view(second))
            result = ctypes.c_int(7)
            assert hip_lib.m3_hip_launch_chain(
                device.device, commands, 2, ctypes.byref(result),
                device.message, 256) == 0, device.message.value
            return result.value

        a, b, c, d, e = at
        assert taken(a, b, c, d, e) == 1
        assert taken(a, a, c, a, e) == 1
        assert taken(a, b, a, d, e) == 0  # in place
        assert taken(a, b, c, d, c) == 0  # both outputs one
        assert taken(a, b, c, d, a) == 0  # over what the first reads
        assert taken(a, b, c, d, d + 4 * (count - 1)) == 0  # one element
        assert taken(a, b, c, c + 4, e) == 0  # reads a part of the link
    finally:
        device.close()


@pytest.mark.parametrize("src,dst", [(m3.F16, m3.F32), (m3.BF16, m3.F32),
                                     (m3.F16, m3.BF16), (m3.BF16, m3.F16)])
def test_every_16bit_value(hip, src, dst):
    """All 65,536 patterns of a 16-bit float through the chain kernel's
    widening, rounding and NaN rules: converted, then converted back."""
    patterns = np.arange(1 << 16, dtype=np.uint32).astype(np.uint16)
    size = m3.DTYPE_SIZES[dst]
    shape = (1 << 16,)
    check(hip, [patterns, np.zeros(size << 16, np.uint8),
                np.zeros(1 << 16, np.uint16)],
          [(m3.OP_CAST, [ViewSpec(0, src, shape), ViewSpec(1, dst, shape)]),
           (m3.OP_CAST, [ViewSpec(1, dst, shape), ViewSpec(2, src, shape)])],
          "every value %d->%d" % (src, dst))
