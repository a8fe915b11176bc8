"""Workloads of the m3 HIP execution provider, measured through its public API.

Two ways of calling the library appear, as its users have them:
  * command lists over device storage (include/m3_backend.h): storages and
    views are made once, each pass hands their commands to
    m3_command_executor_execute, and the results stay on the device for the
    next list;
  * graph sessions (include/m3.h): each pass writes the input from host
    memory, runs the compiled graph and reads the output back.

Results are bit-exact with the reference CPU provider, whatever the kernel:
every tolerance is "exact".
"""
import ctypes
import importlib.util
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    if "m3c_amd" in sys.modules:
        return sys.modules["m3c_amd"]
    spec = importlib.util.spec_from_file_location(
        "m3c_amd", os.path.join(ROOT, "m3.c_amd", "__init__.py"))
    module = importlib.util.module_from_spec(spec)
    sys.modules["m3c_amd"] = module
    spec.loader.exec_module(module)
    return module


m3 = _package()

DTYPES = {"f32": m3.F32, "f16": m3.F16, "bf16": m3.BF16}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZES = {"f32": 4, "f16": 2, "bf16": 2}

# The largest drawn tensor, in elements: no drawn case moves more than the
# long-row softmax listed below.
MOST_ELEMENTS = 1 << 25


def listed():
    return [
        # One guided Euler step of the flow solver: six one-command lists
        # and three one-element host writes on a short latent. The smallest
        # calls: launches and host work.
        {"name": "flow_step", "path": "flow", "length": 1024,
         "channels": 128},
        # The attention weights of one decoded token, a whole session call:
        # scores in, scale + mask + softmax, weights out.
        {"name": "attention_decode", "path": "attention", "heads": 16,
         "queries": 1, "keys": 1501},
        # The 30-step guided Euler solve as one graph: latent in, latent out.
        {"name": "euler_graph", "path": "euler", "batch": 2, "length": 1024,
         "channels": 128, "steps": 30},
        # Causal attention scores of a prefill, the benchmark's headline.
        {"name": "softmax_prefill", "path": "softmax", "batch": 16,
         "rows": 1024, "width": 1024, "dtype": "f32", "out": "f32",
         "causal": True},
        # The same for a prompt of no round length, in 16 bits.
        {"name": "softmax_ragged", "path": "softmax", "batch": 16,
         "rows": 777, "width": 777, "dtype": "bf16", "out": "bf16",
         "causal": True},
        # Long rows, the benchmark's [4096, 16384]: the largest call.
        {"name": "softmax_long", "path": "softmax", "batch": 1,
         "rows": 4096, "width": 16384, "dtype": "f32", "out": "f32",
         "causal": False},
        # Sampling: a few rows over a vocabulary of odd size.
        {"name": "softmax_vocab", "path": "softmax", "batch": 1, "rows": 32,
         "width": 32003, "dtype": "f32", "out": "f32", "causal": False},
        # A norm's weight over hidden states, kept in 16 bits and widened
        # again (the benchmark's MUL shape).
        {"name": "weight_scale", "path": "weight", "batch": 8,
         "length": 1024, "channels": 1536, "half": "bf16"},
        # Per-channel scale and bias of an audio feature map of odd length.
        {"name": "channel_affine", "path": "channel", "batch": 2,
         "channels": 512, "length": 24001, "dtype": "f32"},
        # Hidden states to channels-first: a permuted view made contiguous.
        {"name": "to_channels", "path": "permute", "batch": 2,
         "length": 8191, "channels": 512, "dtype": "f32", "out": "f32"},
        # The vocoder's activations: Snake1d over its feature map, tanh.
        {"name": "vocoder_activations", "path": "vocoder", "batch": 2,
         "channels": 192, "length": 60001},
        # The gate of a gated MLP.
        {"name": "mlp_gate", "path": "gate", "rows": 3001, "width": 3072,
         "dtype": "bf16", "packed": False},
    ]


def _log(rng, low, high):
    """A whole number in [low, high], spread over its logarithm."""
    value = low * (high / low) ** rng.random()
    return max(low, min(high, int(round(value))))


def _size(rng, low, high):
    """_log, or (one time in three) a multiple of 64 or 8 near it: prompts,
    clips and vocabularies have any length, model widths round ones."""
    value = _log(rng, low, high)
    kind = rng.randrange(6)
    step = 64 if kind == 0 else 8 if kind == 1 else 1
    return max(low, min(high, (value + step - 1) // step * step))


def draw(rng):
    path = rng.choice(["flow", "attention", "euler", "softmax", "softmax",
                       "softmax", "long", "long", "weight", "channel",
                       "channel", "permute", "permute", "vocoder", "vocoder",
                       "gate"])
    floats = ("f32", "f16", "bf16")
    if path == "flow":
        return {"path": path, "length": _size(rng, 32, 8192),
                "channels": _size(rng, 32, 256)}
    if path == "attention":
        queries = rng.choice([1, 1, _size(rng, 2, 96)])
        return {"path": path, "heads": rng.choice([8, 12, 16, 24, 32]),
                "queries": queries, "keys": _size(rng, 32, 4096)}
    if path == "euler":
        return {"path": path, "batch": rng.choice([1, 2]),
                "length": _size(rng, 64, 2048),
                "channels": 8 * _log(rng, 8, 32),
                "steps": rng.choice([10, 20, 30])}
    if path == "softmax":
        width = _size(rng, 33, 2048)
        batch = _size(rng, 1, 64)
        rows = min(_size(rng, 1, 2048),
                   max(1, MOST_ELEMENTS // (batch * width)))
        dtype = rng.choice(floats)
        return {"path": path, "batch": batch, "rows": rows, "width": width,
                "dtype": dtype, "out": rng.choice([dtype, "f32"]),
                "causal": rng.random() < 0.5}
    if path == "long":
        width = _size(rng, 2049, 65536)
        rows = min(_size(rng, 1, 4096), max(1, MOST_ELEMENTS // width))
        dtype = rng.choice(("f32", "f32", "bf16"))
        return {"path": "softmax", "batch": 1, "rows": rows, "width": width,
                "dtype": dtype, "out": "f32", "causal": False}
    if path == "weight":
        channels = _size(rng, 64, 4096)
        return {"path": path, "batch": rng.choice([1, 2, 4, 8]),
                "length": min(_size(rng, 16, 2048),
                              MOST_ELEMENTS // (8 * channels)),
                "channels": channels, "half": rng.choice(floats[1:])}
    if path == "channel":
        channels = _size(rng, 16, 1024)
        batch = rng.choice([1, 2])
        return {"path": path, "batch": batch, "channels": channels,
                "length": min(_size(rng, 100, 200000),
                              MOST_ELEMENTS // (batch * channels)),
                "dtype": rng.choice(floats)}
    if path == "permute":
        channels = _size(rng, 32, 2048)
        batch = rng.choice([1, 2, 4])
        dtype = rng.choice(floats)
        return {"path": path, "batch": batch,
                "length": min(_size(rng, 50, 50000),
                              MOST_ELEMENTS // (batch * channels)),
                "channels": channels, "dtype": dtype,
                "out": rng.choice([dtype, dtype, "f32"])}
    if path == "vocoder":
        channels = _size(rng, 16, 1536)
        batch = rng.choice([1, 2])
        return {"path": path, "batch": batch, "channels": channels,
                "length": min(_size(rng, 200, 200000),
                              MOST_ELEMENTS // (batch * channels))}
    width = _size(rng, 256, 8192)
    return {"path": "gate", "rows": min(_size(rng, 1, 8192),
                                        MOST_ELEMENTS // (2 * width)),
            "width": width, "dtype": rng.choice(floats),
            "packed": rng.random() < 0.3}


# ---- inputs -----------------------------------------------------------------


def _inputs(case, seed):
    """The case's inputs as CUDA tensors, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, generator=g, device="cuda") * scale

    path = case["path"]
    if path == "flow":
        return {"velocity": normal(2, case["length"], case["channels"]),
                "latent": normal(1, case["length"], case["channels"])}
    if path == "attention":
        scores = normal(case["heads"], case["queries"], case["keys"],
                        scale=8.0)
        # each query sees the keys up to its own position
        position = torch.arange(case["keys"], device="cuda")
        last = (torch.arange(case["queries"], device="cuda") +
                case["keys"] - case["queries"])
        mask = torch.where(position[None, :] > last[:, None],
                           float("-inf"), 0.0)
        return {"scores": scores, "mask": mask.float()}
    if path == "euler":
        shape = (case["batch"], case["length"], case["channels"])
        return {"x": normal(*shape),
                "vu": [normal(*shape) for _ in range(case["steps"])],
                "vc": [normal(*shape) for _ in range(case["steps"])]}
    if path == "softmax":
        x = normal(case["batch"], case["rows"], case["width"], scale=3.0)
        if case["causal"]:
            hidden = torch.ones(case["rows"], case["width"], device="cuda",
                                dtype=torch.bool)
            x.masked_fill_(torch.triu(hidden, 1), float("-inf"))
        return {"x": x.to(TORCH[case["dtype"]])}
    if path == "weight":
        shape = (case["batch"], case["length"], case["channels"])
        return {"x": normal(*shape), "c": normal(case["channels"])}
    if path == "channel":
        dtype = TORCH[case["dtype"]]
        return {"x": normal(case["batch"], case["channels"],
                            case["length"]).to(dtype),
                "scale": (1.0 + normal(case["channels"], 1,
                                       scale=0.1)).to(dtype),
                "bias": normal(case["channels"], 1, scale=0.5).to(dtype)}
    if path == "permute":
        return {"x": normal(case["batch"], case["length"],
                            case["channels"]).to(TORCH[case["dtype"]])}
    if path == "vocoder":
        alpha = torch.rand(1, case["channels"], 1, generator=g,
                           device="cuda") * 1.9 + 0.1
        return {"x": normal(case["batch"], case["channels"],
                            case["length"]), "alpha": alpha}
    dtype = TORCH[case["dtype"]]
    if case["packed"]:
        return {"both": normal(case["rows"], 2 * case["width"],
                               scale=2.0).to(dtype)}
    return {"gate": normal(case["rows"], case["width"], scale=2.0).to(dtype),
            "up": normal(case["rows"], case["width"]).to(dtype)}


def _host(tensor):
    """The tensor's elements in host memory (16-bit ones as uint16)."""
    tensor = tensor.contiguous()
    if tensor.element_size() == 2:
        tensor = tensor.view(torch.int16)
    return np.ascontiguousarray(tensor.cpu().numpy())


# ---- command lists over device storage ---------------------------------------


class _Backend:
    """The program's HIP backend and command executor."""

    def __init__(self):
        self.lib, _ = m3.load()
        self.lib.m3_command_executor_init.argtypes = [ctypes.c_void_p,
                                                      ctypes.c_void_p]
        self.lib.m3_command_executor_execute.restype = ctypes.c_int
        self.lib.m3_command_executor_execute.argtypes = [
            ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t,
            ctypes.c_void_p]
        self.handle = ctypes.c_void_p()
        error = m3.Error()
        m3.check(self.lib.m3_backend_create_hip(ctypes.byref(self.handle),
                                                ctypes.byref(error)), error)
        self.executor = (ctypes.c_uint8 * 64)()
        self.lib.m3_command_executor_init(self.executor, self.handle)


_BACKEND = None


def _backend():
    global _BACKEND
    if _BACKEND is None:
        _BACKEND = _Backend()
    return _BACKEND


class _DeviceArray:
    """A storage's memory for torch; keeps the storages alive."""

    def __init__(self, owner, pointer, shape, dtype):
        self.owner = owner
        self.__cuda_array_interface__ = {
            "shape": tuple(shape), "strides": None, "version": 2,
            "typestr": "<f4" if dtype == "f32" else "<i2",
            "data": (pointer, False)}


class _Buffers:
    """Storages on the program's backend, freed together."""

    def __init__(self):
        self.backend = _backend()
        self.lib = self.backend.lib
        self.storages = {}

    def allocate(self, name, byte_count):
        storage = ctypes.c_void_p()
        error = m3.Error()
        m3.check(self.lib.m3_storage_allocate(
            self.backend.handle, byte_count, 256, ctypes.byref(storage),
            ctypes.byref(error)), error)
        self.storages[name] = storage

    def write(self, name, array, byte_offset=0):
        error = m3.Error()
        m3.check(self.lib.m3_storage_write(
            self.storages[name], byte_offset,
            array.ctypes.data_as(ctypes.c_void_p), array.nbytes,
            ctypes.byref(error)), error)

    def upload(self, name, tensor):
        array = _host(tensor)
        self.allocate(name, array.nbytes)
        self.write(name, array)

    def view(self, name, dtype, shape, byte_offset=0, byte_strides=None):
        view = m3.TensorView()
        dims = (ctypes.c_uint64 * 8)(*shape)
        error = m3.Error()
        if byte_strides is None:
            status = self.lib.m3_tensor_view_contiguous(
                ctypes.byref(view), self.storages[name], DTYPES[dtype],
                len(shape), dims, byte_offset, ctypes.byref(error))
        else:
            strides = (ctypes.c_size_t * 8)(*byte_strides)
            status = self.lib.m3_tensor_view_strided(
                ctypes.byref(view), self.storages[name], DTYPES[dtype],
                len(shape), dims, strides, byte_offset, ctypes.byref(error))
        m3.check(status, error)
        return view

    def tensor(self, name, dtype, shape):
        """The storage as a CUDA tensor."""
        pointer = self.lib.m3_storage_device_data(self.storages[name])
        tensor = torch.as_tensor(_DeviceArray(self, pointer, shape, dtype),
                                 device="cuda")
        return tensor if dtype == "f32" else tensor.view(TORCH[dtype])

    def __del__(self):
        for storage in self.storages.values():
            self.lib.m3_storage_free(storage)


class _List:
    """One command list: (kind, views) in order, run as one call."""

    def __init__(self, buffers, *commands):
        self.buffers = buffers
        self.views = [views for _, views in commands]
        self.array = (m3.Command * len(commands))()
        for command, (kind, views) in zip(self.array, commands):
            command.kind = kind
            for i, view in enumerate(views):
                command.descriptor.views[i] = ctypes.pointer(view)
        self.error = m3.Error()
        self.arguments = (buffers.backend.executor,
                          ctypes.addressof(self.array), len(commands),
                          ctypes.addressof(self.error))

    def run(self):
        execute = self.buffers.lib.m3_command_executor_execute
        m3.check(execute(*self.arguments), self.error)


class _FlowStep:
    """One Euler step with classifier-free guidance, as the flow solver
    issues it: v = u + s (c - u), next = x + dt v, the scalars rewritten
    from the host between one-command lists."""

    def __init__(self, case, seed):
        data = _inputs(case, seed)
        b = _Buffers()
        shape = (1, case["length"], case["channels"])
        half = 4 * case["length"] * case["channels"]
        b.upload("velocity", data["velocity"])
        b.upload("latent", data["latent"])
        b.allocate("arith", half)
        b.allocate("next", half)
        b.allocate("scalar", 4)
        cond = b.view("velocity", "f32", shape)
        uncond = b.view("velocity", "f32", shape, half)
        latent = b.view("latent", "f32", shape)
        arith = b.view("arith", "f32", shape)
        following = b.view("next", "f32", shape)
        scalar = b.view("scalar", "f32", (1,))
        self.buffers = b
        self.scalars = [np.array([v], np.float32)
                        for v in (-1.0, 3.0, 1.0 / 30.0)]
        self.lists = [
            _List(b, (m3.OP_MUL, [uncond, scalar, arith])),
            _List(b, (m3.OP_ADD, [cond, arith, arith])),
            _List(b, (m3.OP_MUL, [arith, scalar, arith])),
            _List(b, (m3.OP_ADD, [uncond, arith, arith])),
            _List(b, (m3.OP_MUL, [arith, scalar, arith])),
            _List(b, (m3.OP_ADD, [latent, arith, following]))]
        self.outputs = {"next": b.tensor("next", "f32", shape)}

    def run(self):
        for i, commands in enumerate(self.lists):
            if i % 2 == 0:
                self.buffers.write("scalar", self.scalars[i // 2])
            commands.run()
        return self.outputs


class _DeviceList:
    """A case that is one command list; its outputs stay on the device."""

    def __init__(self, case, seed):
        data = _inputs(case, seed)
        b = _Buffers()
        self.outputs = {}
        self.buffers = b
        for name, tensor in data.items():
            b.upload(name, tensor)
        data = {name: tuple(t.shape) for name, t in data.items()}
        commands = getattr(self, "_" + case["path"])(case, data)
        self.list = _List(b, *commands)

    def _output(self, name, dtype, shape):
        count = int(np.prod(shape))
        self.buffers.allocate(name, count * SIZES[dtype])
        self.outputs[name] = self.buffers.tensor(name, dtype, shape)
        return self.buffers.view(name, dtype, shape)

    def _softmax(self, case, shapes):
        x = self.buffers.view("x", case["dtype"], shapes["x"])
        p = self._output("p", case["out"], shapes["x"])
        return [(m3.OP_SOFTMAX, [x, p])]

    def _weight(self, case, shapes):
        x = self.buffers.view("x", "f32", shapes["x"])
        c = self.buffers.view("c", "f32", shapes["c"])
        y = self._output("y", "f32", shapes["x"])
        half = self._output("half", case["half"], shapes["x"])
        wide = self._output("wide", "f32", shapes["x"])
        return [(m3.OP_MUL, [x, c, y]), (m3.OP_CAST, [y, half]),
                (m3.OP_CAST, [half, wide])]

    def _channel(self, case, shapes):
        dtype = case["dtype"]
        x = self.buffers.view("x", dtype, shapes["x"])
        scale = self.buffers.view("scale", dtype, shapes["scale"])
        bias = self.buffers.view("bias", dtype, shapes["bias"])
        scaled = self._output("scaled", dtype, shapes["x"])
        y = self._output("y", dtype, shapes["x"])
        return [(m3.OP_MUL, [x, scale, scaled]),
                (m3.OP_ADD, [scaled, bias, y])]

    def _permute(self, case, shapes):
        batch, length, channels = shapes["x"]
        size = SIZES[case["dtype"]]
        x = self.buffers.view("x", case["dtype"], (batch, channels, length),
                              0, (length * channels * size, size,
                                  channels * size))
        y = self._output("y", case["out"], (batch, channels, length))
        kind = m3.OP_COPY if case["dtype"] == case["out"] else m3.OP_CAST
        return [(kind, [x, y])]

    def _vocoder(self, case, shapes):
        x = self.buffers.view("x", "f32", shapes["x"])
        alpha = self.buffers.view("alpha", "f32", shapes["alpha"])
        y = self._output("y", "f32", shapes["x"])
        wave = self._output("wave", "f32", shapes["x"])
        return [(m3.OP_SNAKE1D, [x, alpha, y]), (m3.OP_TANH, [y, wave])]

    def _gate(self, case, shapes):
        dtype = case["dtype"]
        shape = (case["rows"], case["width"])
        if case["packed"]:
            # both halves of one projection's output
            size = SIZES[dtype]
            strides = (2 * case["width"] * size, size)
            gate = self.buffers.view("both", dtype, shape, 0, strides)
            up = self.buffers.view("both", dtype, shape,
                                   case["width"] * size, strides)
        else:
            gate = self.buffers.view("gate", dtype, shape)
            up = self.buffers.view("up", dtype, shape)
        return [(m3.OP_GATED_SILU, [gate, up,
                                    self._output("y", dtype, shape)])]

    def run(self):
        self.list.run()
        return self.outputs


# ---- graph sessions ----------------------------------------------------------


class _Attention:
    """scores * scale + mask, then softmax, as one graph session."""

    def __init__(self, case, seed):
        data = _inputs(case, seed)
        self.input = _host(data["scores"])
        mask = _host(data["mask"])
        shape = self.input.shape
        graph = m3.Graph()
        self.scores = graph.add_value(m3.INPUT, m3.F32, shape)
        scale = graph.add_value(m3.CONSTANT, m3.F32, (1,))
        hidden = graph.add_value(m3.CONSTANT, m3.F32, mask.shape)
        graph.set_constant(scale, np.array([0.125], np.float32))
        graph.set_constant(hidden, mask)
        scaled = graph.add_value(m3.TEMPORARY, m3.F32, shape)
        logits = graph.add_value(m3.TEMPORARY, m3.F32, shape)
        self.weights = graph.add_value(m3.OUTPUT, m3.F32, shape)
        graph.add_node(m3.OP_MUL, [self.scores, scale], [scaled])
        graph.add_node(m3.OP_ADD, [scaled, hidden], [logits])
        graph.add_node(m3.OP_SOFTMAX, [logits], [self.weights])
        self.session = m3.Session(graph)
        graph.free()
        self.output = np.empty(shape, np.float32)

    def run(self):
        self.session.write(self.scores, self.input)
        self.session.run()
        return {"weights": self.session.read(self.weights, self.output)}


class _Euler:
    """All steps of a guided Euler solve as one graph session."""

    def __init__(self, case, seed):
        data = _inputs(case, seed)
        self.input = _host(data["x"])
        shape = self.input.shape
        graph = m3.Graph()
        current = self.x = graph.add_value(m3.INPUT, m3.F32, shape)
        scalars = []
        for value in (-1.0, 3.0, 1.0 / case["steps"]):
            scalars.append(graph.add_value(m3.CONSTANT, m3.F32, (1,)))
            graph.set_constant(scalars[-1], np.array([value], np.float32))
        minus_one, scale, dt = scalars
        for k in range(case["steps"]):
            vu = graph.add_value(m3.CONSTANT, m3.F32, shape)
            vc = graph.add_value(m3.CONSTANT, m3.F32, shape)
            graph.set_constant(vu, _host(data["vu"][k]))
            graph.set_constant(vc, _host(data["vc"][k]))
            t = [graph.add_value(m3.TEMPORARY, m3.F32, shape)
                 for _ in range(5)]
            role = (m3.OUTPUT if k == case["steps"] - 1 else m3.TEMPORARY)
            following = graph.add_value(role, m3.F32, shape)
            graph.add_node(m3.OP_MUL, [vu, minus_one], [t[0]])
            graph.add_node(m3.OP_ADD, [vc, t[0]], [t[1]])
            graph.add_node(m3.OP_MUL, [t[1], scale], [t[2]])
            graph.add_node(m3.OP_ADD, [vu, t[2]], [t[3]])
            graph.add_node(m3.OP_MUL, [t[3], dt], [t[4]])
            graph.add_node(m3.OP_ADD, [current, t[4]], [following])
            current = following
        self.latent = current
        self.session = m3.Session(graph)
        graph.free()
        self.output = np.empty(shape, np.float32)

    def run(self):
        self.session.write(self.x, self.input)
        self.session.run()
        return {"latent": self.session.read(self.latent, self.output)}


_STATES = {"flow": _FlowStep, "attention": _Attention, "euler": _Euler}


def prepare(case, seed):
    return _STATES.get(case["path"], _DeviceList)(case, seed)


def run(state):
    return state.run()


# ---- what a pass cannot do without -------------------------------------------


def work(case):
    path = case["path"]
    if path == "flow":
        n = case["length"] * case["channels"]
        return {"bytes": 4 * 4 * n, "flops": 6 * n}
    if path == "attention":
        n = case["heads"] * case["queries"] * case["keys"]
        mask = case["queries"] * case["keys"]
        return {"bytes": 4 * (2 * n + mask), "flops": 6 * n}
    if path == "euler":
        n = case["batch"] * case["length"] * case["channels"]
        return {"bytes": 4 * n * (2 * case["steps"] + 2),
                "flops": 6 * n * case["steps"]}
    if path == "softmax":
        n = case["batch"] * case["rows"] * case["width"]
        return {"bytes": n * (SIZES[case["dtype"]] + SIZES[case["out"]]),
                "flops": 4 * n}
    if path == "weight":
        n = case["batch"] * case["length"] * case["channels"]
        return {"bytes": n * (4 + 4 + 2 + 4) + 4 * case["channels"],
                "flops": 3 * n}
    if path == "channel":
        n = case["batch"] * case["channels"] * case["length"]
        return {"bytes": SIZES[case["dtype"]] * (3 * n +
                                                 2 * case["channels"]),
                "flops": 2 * n}
    if path == "permute":
        n = case["batch"] * case["length"] * case["channels"]
        return {"bytes": n * (SIZES[case["dtype"]] + SIZES[case["out"]]),
                "flops": 0}
    if path == "vocoder":
        n = case["batch"] * case["channels"] * case["length"]
        return {"bytes": 4 * (3 * n + case["channels"]), "flops": 60 * n}
    n = case["rows"] * case["width"]
    return {"bytes": 3 * n * SIZES[case["dtype"]], "flops": 12 * n}


def tolerance(case):
    del case
    return "exact"


# ---- the same in 64 bits ------------------------------------------------------


def exact(case, seed):
    data = _inputs(case, seed)
    path = case["path"]

    def wide(tensor):
        return tensor.double()

    if path == "flow":
        cond, uncond = wide(data["velocity"])
        v = uncond + 3.0 * (cond - uncond)
        return {"next": wide(data["latent"]) + v / 30.0}
    if path == "attention":
        logits = wide(data["scores"]) * 0.125 + wide(data["mask"])
        return {"weights": torch.softmax(logits, -1)}
    if path == "euler":
        x = wide(data["x"])
        for vu, vc in zip(data["vu"], data["vc"]):
            u = wide(vu)
            x = x + (u + 3.0 * (wide(vc) - u)) / case["steps"]
        return {"latent": x}
    if path == "softmax":
        return {"p": torch.softmax(wide(data["x"]), -1)}
    if path == "weight":
        y = wide(data["x"]) * wide(data["c"])
        return {"y": y, "half": y, "wide": y}
    if path == "channel":
        scaled = wide(data["x"]) * wide(data["scale"])
        return {"scaled": scaled, "y": scaled + wide(data["bias"])}
    if path == "permute":
        return {"y": wide(data["x"]).transpose(1, 2)}
    if path == "vocoder":
        x, alpha = wide(data["x"]), wide(data["alpha"])
        # the op's epsilon, the F32 value with the bits 0x3089705f
        y = x + torch.sin(alpha * x) ** 2 / (alpha + float.fromhex(
            "0x1.12e0bep-30"))
        return {"y": y, "wave": torch.tanh(y)}
    if case["packed"]:
        gate, up = wide(data["both"]).split(case["width"], -1)
    else:
        gate, up = wide(data["gate"]), wide(data["up"])
    return {"y": torch.nn.functional.silu(gate) * up}
