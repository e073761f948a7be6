"""The work this engine is used for, as measurable cases.

Seven kinds of work, each through the entry points a user's program calls:

* ``forward``  a network's inference on the tape machine, the way it is served: the batch on the host (bound
               with Let, or written into the machine's own buffer) or already on the device, the weights resident,
               the result on the host after RunAll.  The networks are the repository's three: the MLP, the convnet
               and the Tiny-YOLO-v2-shaped stack.
* ``train``    a training step on the tape machine: forward, every gradient and the solver's update of the
               resident weights, a new batch uploaded by each step.  The convnet of the reference's example, and
               a stack of convolution + batch normalisation + rectifier + pooling in front of one dense layer.
* ``chain``    elementwise operators on tensors in device memory, as one segment of commands with a
               row-broadcast bias, or call by call through the engine's methods.
* ``matmul``   one product through Engine.MatMul, operands as they lie or transposed, both float types.
* ``bmm``      many equal products as one strided-batched command.

Every program here waits for its result (RunAll, DoWork and sync do that), as a user's has to.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from gorgonia_amd import device as D
from gorgonia_amd import graph as G
from gorgonia_amd.configs import YOLO_CHANNELS
from gorgonia_amd.engine import Engine

DTYPES = {"f32": (np.float32, torch.float32, 0, 4), "f64": (np.float64, torch.float64, 1, 8)}
BLOCKS = (3, 16, 32, 64, 128)     # channels of the batch-normalised training stack
CLASSES = 10


def listed():
    return [
        # one request at a time: what a single row costs is launches and waits
        {"name": "mlp_forward_1", "op": "forward", "net": "mlp", "batch": 1, "size": 0, "dtype": "f32", "feed": "let"},
        # the benchmark's own step: the batch is on the device, only the 128 x 10 result leaves it
        {"name": "convnet_forward_128", "op": "forward", "net": "convnet", "batch": 128, "size": 28, "dtype": "f32", "feed": "resident"},
        # a detector's throughput setting: 16.6 MB of images a step, the loader writes them where the machine reads them
        {"name": "yolo_forward_8", "op": "forward", "net": "yolo", "batch": 8, "size": 416, "dtype": "f32", "feed": "borrowed"},
        # and its latency setting: one camera frame, bound with Let
        {"name": "yolo_forward_1", "op": "forward", "net": "yolo", "batch": 1, "size": 416, "dtype": "f32", "feed": "let"},
        # the example's training step, in the float type the benchmark trains in
        {"name": "convnet_train_128", "op": "train", "net": "convnet", "batch": 128, "size": 28, "dtype": "f32", "solver": "rmsprop"},
        # the same in float64, the type the reference's example starts with, at a batch no tile divides
        {"name": "convnet_train_f64_50", "op": "train", "net": "convnet", "batch": 50, "size": 28, "dtype": "f64", "solver": "rmsprop"},
        # a network with batch statistics: large images, few channels
        {"name": "blocks_train_8", "op": "train", "net": "blocks", "batch": 8, "size": 208, "dtype": "f32", "solver": "adam"},
        # the elementwise chain on 64 MiB tensors: bandwidth
        {"name": "chain_4096x4096", "op": "chain", "rows": 4096, "cols": 4096, "dtype": "f32", "act": "sigmoid", "via": "commands"},
        # five engine calls and a wait on a tensor that fits one corner of the chip: host time and launches
        {"name": "chain_small", "op": "chain", "rows": 73, "cols": 137, "dtype": "f32", "act": "sigmoid", "via": "engine"},
        # large and square
        {"name": "matmul_4096", "op": "matmul", "m": 4096, "n": 4096, "k": 4096, "dtype": "f32", "ta": False, "tb": False},
        # ragged, float64, the left operand a transposed view (a weight gradient's form)
        {"name": "matmul_f64_ragged", "op": "matmul", "m": 777, "n": 1543, "k": 1021, "dtype": "f64", "ta": True, "tb": False},
        # a batch of middling products
        {"name": "bmm_64x512", "op": "bmm", "batch": 64, "m": 512, "n": 512, "k": 512, "dtype": "f32", "tb": False},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["forward", "forward", "train", "chain", "matmul", "bmm"])
    if op == "forward":
        net = rng.choice(["mlp", "convnet", "yolo"])
        c = {"op": op, "net": net, "feed": rng.choice(["let", "borrowed", "resident"])}
        if net == "mlp":
            c.update(batch=_log(rng, 1, 4096), size=0, dtype=rng.choice(["f32", "f32", "f64"]))
        elif net == "convnet":
            dt = rng.choice(["f32", "f32", "f64"])
            c.update(batch=_log(rng, 1, 1024 if dt == "f32" else 256), size=28, dtype=dt)
        else:
            c.update(batch=rng.randint(1, 8), size=32 * rng.randint(7, 13), dtype="f32")
        return c
    if op == "train":
        solver = rng.choice(["rmsprop", "adam", "vanilla"])
        if rng.random() < 0.5:
            return {"op": op, "net": "blocks", "batch": rng.randint(1, 8), "size": rng.randint(48, 208), "dtype": "f32", "solver": solver}
        dt = rng.choice(["f32", "f32", "f64"])
        return {"op": op, "net": "convnet", "batch": _log(rng, 8, 384 if dt == "f32" else 96), "size": 28, "dtype": dt, "solver": solver}
    if op == "chain":
        dt = rng.choice(["f32", "f32", "f64"])
        n = _log(rng, 1000, (1 << 24) if dt == "f32" else (1 << 23))
        cols = _log(rng, 10, min(n, 8192))
        return {"op": op, "rows": max(2, n // cols), "cols": cols, "dtype": dt, "act": rng.choice(["sigmoid", "tanh", "exp", "square"]),
                "via": rng.choice(["commands", "engine"])}
    dt = rng.choice(["f32", "f32", "f64"])
    if op == "matmul":
        top = 4096 if dt == "f32" else 2048
        return {"op": op, "m": _log(rng, 16, top), "n": _log(rng, 16, top), "k": _log(rng, 16, top), "dtype": dt,
                "ta": rng.random() < 0.3, "tb": rng.random() < 0.3}
    top = 512 if dt == "f32" else 256
    return {"op": op, "batch": _log(rng, 2, 64), "m": _log(rng, 16, top), "n": _log(rng, 16, top), "k": _log(rng, 16, top), "dtype": dt,
            "tb": rng.random() < 0.4}


# ---- inputs ----------------------------------------------------------------------------------------------------


class _Owner:
    """The library objects whose memory a program looks into.  Gives the memory back when the program and the last
    view of it are gone."""

    def __init__(self, machine=None, engine=None, context=None):
        self.machine, self.engine, self.context = machine, engine, context
        self.pointers = []

    def __del__(self):
        if self.machine is not None:
            self.machine.Close()
        if self.engine is not None:
            self.engine.Close()
            self.engine.destroy()
        if self.context is not None:
            for p in self.pointers:
                self.context.free(p)
            self.context.close()


class _Memory:
    """Memory the library owns, for torch.as_tensor and numpy.asarray (no copy); the view keeps the owner."""

    def __init__(self, owner, address, shape, dtype, host=False):
        self.owner = owner
        said = {"data": (int(address), False), "shape": tuple(int(s) for s in shape), "typestr": np.dtype(dtype).str, "strides": None}
        if host:
            self.__array_interface__ = dict(said, version=3)
        else:
            self.__cuda_array_interface__ = dict(said, version=2)


def _view(owner, address, shape, dtype):
    return torch.as_tensor(_Memory(owner, address, shape, dtype), device="cuda")


class _Gen:
    """Seeded inputs, made on the GPU."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) * 7919 + 17)
        self.dtype = DTYPES[dtype][1]

    def uniform(self, shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device="cuda", dtype=self.dtype) * (hi - lo) + lo

    def normal(self, shape, std=1.0, mean=0.0):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=self.dtype) * std + mean

    def weights(self, *shape):
        fan_in = shape[0] if len(shape) == 2 else shape[1] * shape[2] * shape[3]
        return self.normal(shape, math.sqrt(2.0 / fan_in))


def _host(t):
    return t.cpu().numpy()


class _State:
    """What a program keeps between passes."""


# ---- forward ---------------------------------------------------------------------------------------------------


def _layers(c, r, g, x):
    """The network's result node, its weights resident."""
    def par(t):
        return G.NewTensor(g, _host(t), resident=True)

    b = c["batch"]
    if c["net"] == "mlp":
        h = x
        for i, (k, n) in enumerate(((784, 300), (300, 100), (100, 10))):
            lim = math.sqrt(6.0 / (k + n))
            h = G.BroadcastAdd(G.Mul(h, par(r.uniform((k, n), -lim, lim))), par(r.uniform((1, n), -0.1, 0.1))) if b > 1 else \
                G.Add(G.Mul(h, par(r.uniform((k, n), -lim, lim))), par(r.uniform((1, n), -0.1, 0.1)))
            if i < 2:
                h = G.Rectify(h)
        return G.SoftMax(h)
    if c["net"] == "convnet":
        h = x
        for cin, cout in ((1, 32), (32, 64), (64, 128)):
            h = G.Rectify(G.Conv2d(h, par(r.weights(cout, cin, 3, 3)), (3, 3), (1, 1), (1, 1), (1, 1)))
            h = G.MaxPool2D(h, (2, 2), (0, 0), (2, 2))
        h = G.Rectify(G.Mul(G.Reshape(h, (b, 1152)), par(r.weights(1152, 625))))
        return G.SoftMax(G.Mul(h, par(r.weights(625, CLASSES))))
    h = x
    for i in range(7):
        cin, cout = YOLO_CHANNELS[i], YOLO_CHANNELS[i + 1]
        h = G.Conv2d(h, par(r.weights(cout, cin, 3, 3)), (3, 3), (1, 1), (1, 1), (1, 1))
        mean, var = par(r.normal((cout,), 0.1)), par(r.uniform((cout,), 0.5, 1.5))
        gamma, beta = par(r.uniform((cout,), 0.5, 1.5)), par(r.normal((cout,), 0.1))
        h = G.LeakyRelu(G.BatchNorm(h, gamma, beta, mean, var, 1e-5), 0.1)
        if i < 5:
            h = G.MaxPool2D(h, (2, 2), (0, 0), (2, 2))
        elif i == 5:
            h = G.MaxPool2D(h, (2, 2), (1, 0, 1, 0), (1, 1))
    return G.Conv2d(h, par(r.weights(425, 1024, 1, 1)), (1, 1), (0, 0), (1, 1), (1, 1))


def _input_shape(c):
    b, s = c["batch"], c["size"]
    return {"mlp": (b, 784), "convnet": (b, 1, s, s), "yolo": (b, 3, s, s), "blocks": (b, 3, s, s)}[c["net"]]


def _prepare_forward(c, seed):
    s, r = _State(), _Gen(seed, c["dtype"])
    s.batch = _host(r.uniform(_input_shape(c)))
    s.feed = c["feed"]
    s.graph = G.NewGraph()
    s.x = G.NewTensor(s.graph, s.batch, resident=s.feed == "resident")
    if s.feed == "borrowed":
        G.LetBorrowed(s.x)
    out = _layers(c, r, s.graph, s.x)
    # a detector's result is used where the machine wrote it; the classifiers' few values are copied out
    s.borrowed_out = G.ReadBorrowed(out) if c["net"] == "yolo" else None
    s.out = None if s.borrowed_out is not None else G.Read(out)
    s.machine = G.NewTapeMachine(s.graph, graph_replay="measured", fuse_activations=True)
    s.owner = _Owner(machine=s.machine)
    if s.feed == "borrowed":
        s.machine.input(s.x)[...] = s.batch   # the loader's part
    if s.borrowed_out is not None:
        lent = s.machine.value(s.borrowed_out)
        s.out = np.asarray(_Memory(s.owner, lent.ctypes.data, lent.shape, lent.dtype, host=True))
    return s


def _run_forward(s):
    if s.feed == "let":
        G.Let(s.x, s.batch)
    s.machine.RunAll()
    return s.out


# ---- train -----------------------------------------------------------------------------------------------------

CONV = dict(kernelShape=(3, 3), pad=(1, 1), stride=(1, 1), dilation=(1, 1))


def _prepare_train(c, seed):
    s, r = _State(), _Gen(seed, c["dtype"])
    np_dt = DTYPES[c["dtype"]][0]
    b, size = c["batch"], c["size"]
    s.batch = _host(r.uniform(_input_shape(c)))
    s.labels = np.zeros((b, CLASSES), np_dt)
    s.labels[np.arange(b), _host(torch.randint(0, CLASSES, (b,), generator=r.g, device="cuda"))] = 1.0
    s.graph = g = G.NewGraph()
    s.x, s.y = G.NewTensor(g, s.batch), G.NewTensor(g, s.labels)
    chans = (1, 32, 64, 128) if c["net"] == "convnet" else BLOCKS
    norm = c["net"] == "blocks"
    weights, saved, h, hw = [], [], s.x, size

    def par(t):
        return G.NewTensor(g, t if isinstance(t, np.ndarray) else _host(t), resident=True)

    stats = []
    for cin, cout in zip(chans, chans[1:]):
        w = par(r.weights(cout, cin, 3, 3))
        z = G.Conv2d(h, w, (3, 3), (1, 1), (1, 1), (1, 1))
        n = z
        st = None
        if norm:
            st = [par(np.zeros(cout, np_dt)), par(np.ones(cout, np_dt)), par(np.zeros(cout, np_dt)), par(np.zeros(cout, np_dt))]
            stats += st[:2]
            n = G.BatchNormTrain(z, *st)
        a = G.Rectify(n)
        saved.append((h, z, n, a, st))
        h = G.MaxPool2D(a, (2, 2), (0, 0), (2, 2))
        weights.append(w)
        hw //= 2
    flat = G.Reshape(h, (b, chans[-1] * hw * hw))
    f = flat
    if not norm:   # the example's hidden dense layer
        weights.append(par(r.weights(chans[-1] * hw * hw, 625)))
        z3 = G.Mul(flat, weights[-1])
        f = G.Rectify(z3)
    weights.append(par(r.weights(f.Shape()[1], CLASSES)))
    out = G.SoftMax(G.Mul(f, weights[-1]))
    s.out = G.Read(out)
    scale = G.NewScalar(g, -1.0 / (b * CLASSES), dtype=np_dt)
    up = G.SoftMaxDiff(out, G.HadamardProd(s.y, scale))
    grads = [G.Mul(f, up, transA=True)]
    up = G.Mul(up, weights[-1], transB=True)
    if not norm:
        up = G.RectifyDiff(z3, up)
        grads.insert(0, G.Mul(flat, up, transA=True))
        up = G.Mul(up, weights[-2], transB=True)
    grad = G.Reshape(up, h.Shape())
    for i in range(len(saved) - 1, -1, -1):
        x_in, z, n, a, st = saved[i]
        dz = G.RectifyDiff(n, G.MaxPool2DDiff(a, grad, (2, 2), (0, 0), (2, 2)))
        if norm:
            dz = G.BatchNormDiff(z, dz, st[2], st[3])
        grads.insert(0, G.Conv2dDiffFilter(x_in, dz, **CONV))
        if i:
            grad = G.Conv2dDiffImage(dz, weights[i], x_in.Shape(), **CONV)
    s.step, s.corrections, keep = 0, None, list(weights) + stats
    if c["solver"] == "adam":
        s.corrections = G.NewTensor(g, G.AdamCorrections(1, dtype=np_dt))
    for w, dw in zip(weights, grads):
        caches = [par(np.zeros(w.Shape(), np_dt)) for _ in range({"vanilla": 0, "rmsprop": 1, "adam": 2}[c["solver"]])]
        keep += caches
        opts = {"rmsprop": dict(eta=1e-3, l2reg=1e-6, clip=5.0), "adam": dict(eta=1e-4, corrections=s.corrections),
                "vanilla": dict(eta=1e-2)}[c["solver"]]
        G.SolverStep(c["solver"], w, dw, caches, **opts)
    s.np_dt = np_dt
    s.machine = G.NewTapeMachine(g, graph_replay="measured", fuse_activations=True)
    s.owner, s.keep, s.held = _Owner(machine=s.machine), keep, None
    return s


def _run_train(s):
    G.Let(s.x, s.batch)
    G.Let(s.y, s.labels)
    s.step += 1
    if s.corrections is not None:
        G.Let(s.corrections, G.AdamCorrections(s.step, dtype=s.np_dt))
    s.machine.RunAll()
    if s.held is None:   # the resident weights, running statistics and solver caches keep their places on the device
        s.held = [_view(s.owner, s.machine.register_address(n), n.Shape(), s.np_dt) for n in s.keep]
    return [s.out] + s.held


# ---- chain, products -------------------------------------------------------------------------------------------


def _prepare_chain(c, seed):
    s, r = _State(), _Gen(seed, c["dtype"])
    np_dt, _, code, item = DTYPES[c["dtype"]]
    rows, cols = c["rows"], c["cols"]
    n = rows * cols
    s.act, s.via = c["act"], c["via"]
    shape = (rows, cols)
    values = {"x": r.uniform(shape, -4, 4), "y": r.uniform(shape, -4, 4),
              "b": r.uniform((1, cols) if s.via == "commands" else shape, -4, 4), "two": r.uniform((1,), 2, 2)}
    if s.via == "commands":
        s.context = D.Context(0, 0)
        own = _Owner(context=s.context)
        p = {}
        for k in ("x", "y", "b", "two", "z", "t", "p"):
            shp = tuple(values[k].shape) if k in values else shape
            p[k] = s.context.malloc(int(np.prod(shp)) * item)
            own.pointers.append(p[k])
            if k in values:
                _view(own, p[k], shp, np_dt).copy_(values[k])
        s.commands = [D.cmd_bin("mul", "vv", p["x"], p["y"], n, dtype=code, dst=p["z"]),
                      D.cmd_bcast("add", p["z"], p["z"], p["b"], rows, cols, 1, dtype=code),
                      D.cmd_unary(s.act, p["z"], n, dtype=code),
                      D.cmd_unary("tanh", p["z"], n, dtype=code, dst=p["t"]),
                      D.cmd_bin("pow", "vs", p["z"], p["two"], n, dtype=code, dst=p["p"])]
        s.outs = [_view(own, p[k], shape, np_dt) for k in ("z", "t", "p")]
        return s
    s.engine = Engine()
    own = _Owner(engine=s.engine)
    s.engine.Init(0, 6 * n * item + 4096)
    for k in ("x", "y", "b"):
        t = s.engine.new_tensor(shape, np_dt)
        _view(own, t.mem, shape, np_dt).copy_(values[k])
        setattr(s, k, t)
    s.two = s.engine.new_tensor((), np_dt)
    _view(own, s.two.mem, (1,), np_dt).copy_(values["two"])
    s.z, s.t, s.p = (s.engine.new_tensor(shape, np_dt) for _ in range(3))
    s.outs = [_view(own, t.mem, shape, np_dt) for t in (s.z, s.t, s.p)]
    return s


def _run_chain(s):
    if s.via == "commands":
        s.context.submit(s.commands)
        s.context.sync()
        return s.outs
    e = s.engine
    e.Mul(s.x, s.y, reuse=s.z)
    e.Add(s.z, s.b, unsafe=True)
    e.Unary(s.act, s.z)
    e.Unary("tanh", s.z, dst=s.t)
    e.PowScalar(s.z, s.two, True, reuse=s.p)
    e.DoWork()
    return s.outs


def _prepare_matmul(c, seed):
    s, r = _State(), _Gen(seed, c["dtype"])
    np_dt, _, _, item = DTYPES[c["dtype"]]
    m, n, k = c["m"], c["n"], c["k"]
    s.engine = Engine()
    own = _Owner(engine=s.engine)
    s.engine.Init(0, (m * k + k * n + m * n) * item + 4096)

    def operand(rows, cols, transposed):
        stored = (cols, rows) if transposed else (rows, cols)
        t = s.engine.new_tensor(stored, np_dt)
        _view(own, t.mem, stored, np_dt).copy_(r.normal(stored))
        return t.T() if transposed else t

    s.a, s.b = operand(m, k, c["ta"]), operand(k, n, c["tb"])
    s.c = s.engine.new_tensor((m, n), np_dt)
    s.out = _view(own, s.c.mem, (m, n), np_dt)
    return s


def _run_matmul(s):
    s.engine.MatMul(s.a, s.b, s.c)
    s.engine.DoWork()
    return s.out


def _prepare_bmm(c, seed):
    s, r = _State(), _Gen(seed, c["dtype"])
    np_dt, _, code, item = DTYPES[c["dtype"]]
    b, m, n, k = c["batch"], c["m"], c["n"], c["k"]
    s.context = D.Context(0, 0)
    own = _Owner(context=s.context)
    own.pointers = pa, pb, pc = [s.context.malloc(b * q * item) for q in (m * k, k * n, m * n)]
    for p, shp in ((pa, (b, m, k)), (pb, (b, n, k) if c["tb"] else (b, k, n))):
        _view(own, p, shp, np_dt).copy_(r.normal(shp))
    s.commands = [D.cmd_gemm(pa, pb, pc, m, n, k, trans_b=c["tb"], batch=b, stride_a=m * k, stride_b=k * n, stride_c=m * n, dtype=code)]
    s.out = _view(own, pc, (b, m, n), np_dt)
    return s


def _run_bmm(s):
    s.context.submit(s.commands)
    s.context.sync()
    return s.out


PREPARE = {"forward": _prepare_forward, "train": _prepare_train, "chain": _prepare_chain, "matmul": _prepare_matmul, "bmm": _prepare_bmm}
RUN = {"forward": _run_forward, "train": _run_train, "chain": _run_chain, "matmul": _run_matmul, "bmm": _run_bmm}


def prepare(case, seed):
    s = PREPARE[case["op"]](case, seed)
    s.op = case["op"]
    torch.cuda.synchronize()   # the inputs were written on torch's stream, the library works on its own
    return s


def run(state):
    return RUN[state.op](state)


# ---- what a pass cannot do without -----------------------------------------------------------------------------


def _network(c):
    """(weights, flops of the forward products, flops of the first layer's products, values of input, of output)."""
    b, net, s = c["batch"], c["net"], c["size"]
    if net == "mlp":
        dense = ((784, 300), (300, 100), (100, 10))
        return sum(k * n + n for k, n in dense), sum(2 * b * k * n for k, n in dense), 0, b * 784, b * 10
    chans = {"convnet": (1, 32, 64, 128), "yolo": YOLO_CHANNELS, "blocks": BLOCKS}[net]
    w = fl = first = 0
    for i, (cin, cout) in enumerate(zip(chans, chans[1:])):
        w += cin * cout * 9
        f = 2 * b * s * s * cin * cout * 9
        first = first or f
        fl += f
        if net != "yolo" or i < 5:
            s //= 2
    if net == "yolo":
        return w + 1024 * 425, fl + 2 * b * s * s * 1024 * 425, first, b * 3 * c["size"] ** 2, b * 425 * s * s
    feat = chans[-1] * s * s
    dense = ((feat, 625), (625, CLASSES)) if net == "convnet" else ((feat, CLASSES),)
    w += sum(k * n for k, n in dense)
    fl += sum(2 * b * k * n for k, n in dense)
    return w, fl, first, b * chans[0] * c["size"] ** 2, b * CLASSES


def work(case):
    item = DTYPES[case["dtype"]][3]
    op = case["op"]
    if op == "forward":
        w, fl, _, x, y = _network(case)
        return {"bytes": item * (w + x + y), "flops": fl}
    if op == "train":
        # each product once forward, once for each of its two gradients (the first layer has none for its image);
        # weights and solver caches are read and written
        w, fl, first, x, y = _network(case)
        held = w * (1 + {"vanilla": 0, "rmsprop": 1, "adam": 2}[case["solver"]])
        return {"bytes": item * (2 * held + x + 2 * y), "flops": 3 * fl - first}
    if op == "chain":
        n = case["rows"] * case["cols"]
        small = case["cols"] if case["via"] == "commands" else n
        return {"bytes": item * (5 * n + small), "flops": 5 * n}
    b = case.get("batch", 1)
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": b * item * (m * k + k * n + m * n), "flops": 2 * b * m * n * k}


def tolerance(case):
    single = case["dtype"] == "f32"
    if case["op"] == "chain":   # a few units in the last place
        return {"rel": 5e-7, "max": 3e-6} if single else {"rel": 1e-15, "max": 1e-14}
    if case["op"] == "train":
        # Where a rectifier's input or a pooling window's two largest values lie within rounding of each other, another
        # order of summing sends a gradient element the other way: a few of some million elements, which is up to the
        # root of their share (1e-3) of a filter gradient, twice that of the squared gradients the solvers keep, and
        # a tenth of the few values the element reaches.
        return {"rel": 2e-3, "max": 0.3} if single else {"rel": 1e-10, "max": 1e-7}
    return {"rel": 1e-5, "max": 3e-4} if single else {"rel": 1e-13, "max": 1e-11}
