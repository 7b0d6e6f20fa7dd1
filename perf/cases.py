"""Performance cases of the library: what its users have it do, through its
public entry points, from the smallest calls to the largest.

Four kinds of work, each a dict of plain values:

  train      steps of an MLP through the C ABI of include/volta_train.h, each
             on the next minibatch of a dataset -- in device memory
             (volta_train_step_device) or in host memory (volta_train_step /
             volta_train_step_labels, the reference library's own entry
             points) -- then the loss and the weights, as a program does that
             trains for a while, logs and saves.
  infer      volta_train_infer on a model made by volta_infer_model_create
             (what a `volta-hip compile` library runs): host rows in, host
             rows out.
  graph      Backend::execute_terminal of the runtime's MLP graph on device
             tensors, its tables built once.
  optimizer  Backend::apply_gradients over a model's parameter tensors.

Sizes of the named training cases are the benchmark's (bench.py WORKLOADS);
the ragged ones have generic sizes (784 inputs and 10 classes, and round
decimal widths).  A training pass is 50 steps, the benchmark configurations'
run length, or 10 where a step is long.
"""
import ctypes as C
import math

import numpy as np
import torch

from volta_amd import load_hip
from volta_amd.abi import MlpSpec, Trainer, fptr, iptr
from volta_amd.backend import Graph, HipBackend, RtOptimizer, build_execution_plan, config, lower_model_to_graph

WIDE = "512-1024-1024-512-256-1"


def train(name, sizes, act, opt, loss, batch, lr, steps=50, feed="device", layernorm=False, dropout=0.0, clip=0.0):
    return {"name": name, "kind": "train", "sizes": sizes, "act": act, "opt": opt, "loss": loss, "batch": batch,
            "lr": lr, "steps": steps, "feed": feed, "layernorm": layernorm, "dropout": dropout, "clip": clip}


def listed():
    return [
        # the smallest benchmark model, driven as a program linked against the
        # reference's library drives it: host arrays, one call per step
        train("train_small_host_b64", "256-512-512-256-1", "relu", "sgd", "mse", 64, 0.01, feed="host"),
        # the headline regression model: latency and launch count
        train("train_wide_adam_b64", WIDE, "relu", "adam", "mse", 64, 1e-3),
        # the largest B=64 model: memory traffic of the optimizer state
        train("train_2048_adamw_b64", "512-2048-2048-512-1", "gelu", "adamw", "mse", 64, 1e-3),
        # the batch sweep's middle, where products and traffic balance
        train("train_wide_silu_b256", WIDE, "silu", "sgd", "mse", 256, 0.01),
        # the batch sweep's end: matrix products on a part of the chip
        train("train_wide_silu_b1024", WIDE, "silu", "sgd", "mse", 1024, 0.01),
        # an image classifier of 784 inputs at a batch of 100: no size is a
        # multiple of a tile
        train("train_784_10_b100", "784-300-100-10", "relu", "adam", "ce", 100, 1e-3),
        # the wide classifier: bound by the matrix cores
        train("train_4096_ce_b4096", "1024-4096-4096-1024-10", "relu", "adagrad", "ce", 4096, 1e-3, steps=10),
        # a large classifier with round decimal widths and 100 classes
        train("train_3000_ce_b2000", "1500-3000-3000-1000-100", "gelu", "adamw", "ce", 2000, 1e-3, steps=10),
        # every codegen extra at once, on the headline model
        train("train_extras_b64", WIDE, "relu", "adam", "mse", 64, 1e-3, layernorm=True, dropout=0.2, clip=1.0),
        # one request of a serving program
        {"name": "infer_1_row", "kind": "infer", "sizes": WIDE, "act": "relu", "rows": 1},
        # the runtime's graph of the wide classifier on a full batch
        {"name": "graph_4096_rows", "kind": "graph", "sizes": "1024-4096-4096-1024-10", "act": "relu", "rows": 4096},
        # one optimizer update of the wide classifier's parameters
        {"name": "optimizer_adam_25m", "kind": "optimizer", "sizes": "1024-4096-4096-1024-10", "opt": "adam"},
    ]


# The most work of a drawn case: under the largest listed one (5.8e12 flops,
# 7.6e9 bytes), since ragged sizes may run at a lower rate.
MOST_FLOPS, MOST_BYTES = 2.5e12, 3e9


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A layer width, log-uniform: half multiples of 64, the rest round decimals or any number."""
    w, style = _log_int(rng, lo, hi), rng.random()
    if style < 0.5 and w >= 32:
        return max(64, (w + 32) // 64 * 64)
    if style < 0.75 and w >= 20:
        return w // 100 * 100 if w >= 200 else w // 10 * 10
    return w


def _rows(rng):
    """A batch, log-uniform from 1 to 4096: half powers of two, the rest any number."""
    return 2 ** rng.randint(0, 12) if rng.random() < 0.5 else _log_int(rng, 1, 4096)


def draw(rng):
    """One more case of the listed ranges."""
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
            return c


def _draw(rng):
    kind = rng.choice(["train"] * 6 + ["infer", "graph", "graph", "optimizer"])
    hidden = [_width(rng, 16, 4096) for _ in range(rng.randint(1, 4))]
    first = _width(rng, 4, 2048)
    if kind == "train":
        loss = rng.choice(["mse", "ce"])
        last = rng.choice([1, 1, _log_int(rng, 2, 64)]) if loss == "mse" else rng.choice([10, 100, _log_int(rng, 2, 1000)])
        sizes = "-".join(str(s) for s in [first] + hidden + [last])
        extras = rng.random() < 0.2
        opt = rng.choice(["sgd", "adam", "adam", "adamw", "adagrad"])
        # a step that stays stable at any width
        lr = {"sgd": 0.01, "adagrad": 0.01}.get(opt, 1e-3) * min(1.0, 256.0 / max(hidden))
        c = train("", sizes, rng.choice(["relu", "relu", "relu", "gelu", "silu", "tanh", "sigmoid", "leaky_relu"]), opt,
                  loss, _rows(rng), lr, feed=rng.choice(["device", "device", "host"]),
                  layernorm=extras and rng.random() < 0.6, dropout=0.2 if extras and rng.random() < 0.6 else 0.0,
                  clip=1.0 if extras and rng.random() < 0.4 else 0.0)
        del c["name"]
        if work(c)["flops"] > 1e12:
            c["steps"] = 10
        return c
    sizes = "-".join(str(s) for s in [first] + hidden + [rng.choice([1, 10, 100])])
    if kind == "optimizer":
        return {"kind": kind, "sizes": sizes, "opt": rng.choice(["sgd", "adam", "adamw", "rmsprop", "adagrad", "lars"])}
    return {"kind": kind, "sizes": sizes, "act": "relu" if kind == "infer" else rng.choice(["relu", "sigmoid"]),
            "rows": _rows(rng)}


def _sizes(case):
    return [int(s) for s in case["sizes"].split("-")]


# ---------------------------------------------------------------------------
# Inputs, from the seed alone (on the GPU, so that making them is quick).
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _weights(g, sizes):
    """He-uniform W_i; zero biases."""
    ws = [(2 * torch.rand(r, c, generator=g, device="cuda") - 1) * math.sqrt(6.0 / r) for r, c in zip(sizes, sizes[1:])]
    return ws, [torch.zeros(c, device="cuda") for c in sizes[1:]]


def _dataset(case, g):
    """X [steps*B x L0] ~ N(0,1) and its targets: N(0,1), or uniform class labels."""
    sizes, rows = _sizes(case), case["steps"] * case["batch"]
    X = _normal(g, rows, sizes[0])
    if case["loss"] == "ce":
        return X, torch.randint(0, sizes[-1], (rows,), generator=g, device="cuda", dtype=torch.int32)
    return X, _normal(g, rows, sizes[-1])


RESUMED = 1000  # steps the optimizer state has behind it


def _opt_state(case, g):
    """The optimizer's state of a resumed run: first moments of W_i and b_i, then the second moments (Adagrad's sums)."""
    def like(f):
        sizes = _sizes(case)
        return [f(r, c) for r, c in zip(sizes, sizes[1:])], [f(c) for c in sizes[1:]]
    second = 1.0 if case["opt"] == "adagrad" else 1e-4
    return like(lambda *s: 1e-3 * _normal(g, *s)), like(lambda *s: second * (0.5 + torch.rand(*s, generator=g, device="cuda")))


def _graph_names(sizes):
    """The parameter names lower_model_to_graph gives (layers of one shape share them), with their shapes."""
    shapes = {}
    for r, c in zip(sizes, sizes[1:]):
        shapes["weight_%d_%d" % (r, c)] = (r, c)
        shapes["bias_%d" % c] = (1, c)
    return shapes


def _graph_inputs(case, g):
    sizes = _sizes(case)
    t = {"x": _normal(g, case["rows"], sizes[0])}
    for name, (r, c) in _graph_names(sizes).items():
        t[name] = 0.1 * _normal(g, r, c) if r == 1 else (2 * torch.rand(r, c, generator=g, device="cuda") - 1) * math.sqrt(6.0 / r)
    return t


def _tensors(case, g):
    """Parameter tensors [W_0, b_0, ...] and their gradients."""
    sizes, ps = _sizes(case), []
    for w in _weights(g, sizes)[0]:
        ps += [w, 0.1 * _normal(g, w.shape[1])]
    return ps, [1e-2 * torch.randn(p.shape, generator=g, device="cuda") for p in ps]


def _opt_config(case):
    lr = 0.01 if case["opt"] in ("sgd", "adagrad", "lars") else 1e-3
    return config(case["opt"], lr, weight_decay=0.01, momentum=0.9 if case["opt"] in ("rmsprop", "lars") else 0.0)


# ---------------------------------------------------------------------------
# What a program has in hand before the call, and the call.
# ---------------------------------------------------------------------------
class _Mirror:
    """A view of the library's host mirror of W_i or b_i; keeps its handle alive."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__array_interface__ = {"data": (C.cast(ptr, C.c_void_p).value, False), "shape": shape, "typestr": "<f4",
                                    "version": 3}


def _trainer(case, g):
    spec = MlpSpec(_sizes(case), case["act"], case["opt"], case["loss"], clip_grad=case["clip"],
                   dropout_p=case["dropout"], layernorm=case["layernorm"])
    t = Trainer(load_hip(), spec, case["batch"])
    ws, bs = _weights(g, spec.sizes)
    t.set_all_params([w.cpu().numpy() for w in ws], [b.cpu().numpy() for b in bs])
    # resume as from a checkpoint: an empty state divides every gradient by
    # its own size, and the first steps would be the signs of rounding errors
    (mw, mb), (vw, vb) = _opt_state(case, g)
    parts = []
    for i in range(len(ws)):
        parts += {"sgd": [], "adagrad": [vw[i], vb[i]]}.get(case["opt"], [mw[i], mb[i], vw[i], vb[i]])
    for b in bs[:-1] if case["layernorm"] else []:
        parts += [torch.ones_like(b), b]
    if parts:
        t.set_state(torch.cat([x.reshape(-1) for x in parts]).cpu().numpy(), RESUMED)
    return t


def prepare(case, seed):
    g = _gen(seed)
    kind, sizes = case["kind"], _sizes(case)
    lib = load_hip().lib
    if kind == "train":
        t = _trainer(case, g)
        X, Y = _dataset(case, g)
        n, B = len(sizes) - 1, case["batch"]
        yrow = 1 if case["loss"] == "ce" else sizes[-1]
        wo, bo = (C.POINTER(C.c_float) * n)(), (C.POINTER(C.c_float) * n)()
        lib.volta_train_get_params(t.h, wo, bo)
        out = {"w": [np.asarray(_Mirror(t, wo[i], s)) for i, s in enumerate(t.spec.shapes())],
               "b": [np.asarray(_Mirror(t, bo[i], (s[1],))) for i, s in enumerate(t.spec.shapes())]}
        lr = C.c_float(case["lr"])
        if case["feed"] == "device":
            fn = lib.volta_train_step_device
            calls = [(t.h, C.c_void_p(X.data_ptr() + 4 * i * B * sizes[0]), C.c_void_p(Y.data_ptr() + 4 * i * B * yrow), lr)
                     for i in range(case["steps"])]
        else:
            X, Y = X.cpu().numpy(), Y.reshape(case["steps"] * B, yrow).cpu().numpy()
            fn, yp = (lib.volta_train_step_labels, iptr) if case["loss"] == "ce" else (lib.volta_train_step, fptr)
            calls = [(t.h, fptr(X[i * B:]), yp(Y[i * B:]), lr) for i in range(case["steps"])]
        return {"kind": kind, "trainer": t, "lib": lib, "data": (X, Y), "fn": fn, "calls": calls, "ptrs": (wo, bo),
                "out": out}
    if kind == "infer":
        ws, bs = _weights(g, sizes)
        flat = torch.cat([t.reshape(-1) for p in zip(ws, bs) for t in p]).cpu().numpy()
        h = lib.volta_infer_model_create(len(sizes), (C.c_int32 * len(sizes))(*sizes), 0, fptr(flat))
        if not h:
            raise RuntimeError(load_hip().last_error())
        return {"kind": kind, "model": Trainer(load_hip(), MlpSpec(sizes, "relu"), 1, handle=h),
                "x": _normal(g, case["rows"], sizes[0]).cpu().numpy()}
    if kind == "graph":
        tensors = _graph_inputs(case, g)
        graph = Graph()
        x = graph.add_op("input", name="x")
        graph.add_op("output", lower_model_to_graph(graph, sizes, case["act"], x, False))
        for name, v in tensors.items():
            graph.bind_input_shape(name, v.shape)
        out = torch.empty(case["rows"], sizes[-1], device="cuda")
        call = HipBackend().graphs.prepare(graph, build_execution_plan(graph), None,
                                           {k: v.data_ptr() for k, v in tensors.items()}, out.data_ptr(), out.numel())
        return {"kind": kind, "call": call, "tensors": tensors, "out": out}
    ps, gs = _tensors(case, g)
    opt = RtOptimizer(lib, [p.numel() for p in ps])
    return {"kind": kind, "opt": opt, "cfg": _opt_config(case), "params": ps, "grads": gs,
            "pp": [p.data_ptr() for p in ps], "gp": [x.data_ptr() for x in gs]}


def run(state):
    kind = state["kind"]
    if kind == "train":
        fn, lib, t = state["fn"], state["lib"], state["trainer"]
        for args in state["calls"]:
            fn(*args)
        loss = t.loss()
        lib.volta_train_get_params(t.h, *state["ptrs"])
        return {"loss": loss, **state["out"]}
    if kind == "infer":
        return state["model"].infer(state["x"])
    if kind == "graph":
        state["call"]()
        return state["out"]
    state["opt"].apply(state["cfg"], state["pp"], state["gp"])
    return state["params"]


# ---------------------------------------------------------------------------
# Work, tolerance, and the same results in 64 bits.
# ---------------------------------------------------------------------------
def work(case):
    sizes = _sizes(case)
    pairs = list(zip(sizes, sizes[1:]))
    W = sum(r * c for r, c in pairs)
    P = W + sum(sizes[1:])
    kind = case["kind"]
    if kind == "train":
        B, n = case["batch"], case["steps"]
        io = 4.0 * B * (sizes[0] + (1 if case["loss"] == "ce" else sizes[-1]))
        # a step reads and writes the parameters and their state; the weights are read once at the end
        state = {"sgd": 1, "adagrad": 2}.get(case["opt"], 3)
        return {"bytes": n * (io + 8.0 * state * P) + 4.0 * P,
                "flops": n * (6.0 * B * W - 2.0 * B * sizes[0] * sizes[1])}
    if kind in ("infer", "graph"):
        return {"bytes": 4.0 * (case["rows"] * (sizes[0] + sizes[-1]) + P), "flops": 2.0 * case["rows"] * W}
    per = {"sgd": 12, "adam": 28, "adamw": 28, "rmsprop": 28}.get(case["opt"], 20)
    return {"bytes": float(per * P), "flops": 10.0 * P}


def tolerance(case):
    """About four times what another order of the fp32 sums changes.  A training pass is mostly within 1e-4 of the 64-bit
    result; where a ReLU's input lies within rounding of zero one element changes sides and the steps after it follow, and
    a bias (zero at the start, so all of it is accumulated gradient) has differed by 2e-3 to 2e-2."""
    kind = case["kind"]
    if kind == "optimizer":
        return {"rel": 1e-6, "max": 1e-5}
    if kind in ("infer", "graph"):
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 1e-2, "max": 0.5}


def _act(kind, x):
    """f(x) and f'(x)."""
    if kind == "relu":
        return x.clamp_min(0), (x > 0).to(x.dtype)
    if kind == "leaky_relu":
        return torch.where(x > 0, x, 0.01 * x), torch.where(x > 0, 1.0, 0.01).to(x.dtype)
    if kind == "sigmoid":
        y = torch.sigmoid(x)
        return y, y * (1 - y)
    if kind == "tanh":
        y = torch.tanh(x)
        return y, 1 - y * y
    if kind == "silu":
        s = torch.sigmoid(x)
        return x * s, s * (1 + x * (1 - s))
    c, k = 0.7978845608, 0.044715
    t = torch.tanh(c * (x + k * x * x * x))
    return 0.5 * x * (1 + t), 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * c * (1 + 3 * k * x * x)


class _Lcg:
    """The dropout stream s -> A s + C (mod 2^64), drawn a block at a time."""

    A, C = 6364136223846793005, 1442695040888963407

    def __init__(self, seed):
        self.s = np.uint64(seed)

    def draws(self, count):
        a, c = np.empty(count, np.uint64), np.empty(count, np.uint64)
        with np.errstate(over="ignore"):
            a[0], c[0] = self.A, self.C
            have = 1
            while have < count:  # the maps of have+1 .. 2*have draws, from those of 1 .. have
                m = min(have, count - have)
                a[have:have + m] = a[:m] * a[have - 1]
                c[have:have + m] = a[:m] * c[have - 1] + c[:m]
                have += m
            s = a * self.s + c
        self.s = s[-1]
        return (s >> np.uint64(33)).astype(np.float32) / np.float32(2147483648.0)


def _exact_train(case, seed):
    g, sizes, B, n = _gen(seed), _sizes(case), case["batch"], len(_sizes(case)) - 1
    ws, bs = _weights(g, sizes)
    (mw, mb), (vw, vb) = ([[x.double() for x in part] for part in moment] for moment in _opt_state(case, g))
    X, Y = _dataset(case, g)
    w, b = [x.double() for x in ws], [x.double() for x in bs]
    f32 = lambda v: float(np.float32(v))  # noqa: E731  (the constants the library is given)
    lr, b1, b2, eps, wd = f32(case["lr"]), f32(0.9), f32(0.999), f32(1e-8), f32(0.01) if case["opt"] == "adamw" else 0.0
    gamma, beta = [torch.ones_like(x) for x in b[:-1]], [torch.zeros_like(x) for x in b[:-1]]
    p, stream = f32(case["dropout"]), _Lcg(12345678)
    scale = float(np.float32(1.0) / (np.float32(1.0) - np.float32(case["dropout"])))
    extras = case["layernorm"] or p > 0
    loss = None
    for s in range(case["steps"]):
        a, der, keep, inv = [X[s * B:(s + 1) * B].double()], [], [], []
        for i in range(n):
            z = a[i] @ w[i] + b[i]
            if i == n - 1:
                a.append(z)
                break
            y, d = _act(case["act"], z)
            if case["layernorm"]:
                mu = y.mean(1, keepdim=True)
                inv.append(1 / torch.sqrt(((y - mu) ** 2).mean(1, keepdim=True) + f32(1e-5)))
                y = (y - mu) * inv[i] * gamma[i] + beta[i]
            if p > 0:
                k = torch.from_numpy(stream.draws(y.numel()) >= np.float32(p)).to(y.device).reshape(y.shape)
                keep.append(k.double() * scale)
                y = y * keep[i]
            # sigmoid and tanh take the layer's output for their derivative, as the generated step does
            if extras and case["act"] == "sigmoid":
                d = y * (1 - y)
            elif extras and case["act"] == "tanh":
                d = 1 - y * y
            der.append(d)
            a.append(y)
        y, z = Y[s * B:(s + 1) * B], a[n]
        if case["loss"] == "ce":
            lp = torch.log_softmax(z, 1)
            hot = torch.nn.functional.one_hot(y.long(), sizes[-1]).double()
            loss, d = -(lp * hot).sum() / B, (lp.exp() - hot) / B
        else:
            e = z - y.double()
            loss, d = (e * e).mean(), 2 * e / e.numel()
        delta, db = [None] * n, [None] * n
        for i in range(n - 1, -1, -1):
            if i < n - 1:
                if case["layernorm"]:
                    xh = (a[i + 1] - beta[i]) / (gamma[i] + f32(1e-12))
                    dg, dbe, dx = (d * xh).sum(0), d.sum(0), d * gamma[i]
                    d = inv[i] * (dx - dx.mean(1, keepdim=True) - xh * (dx * xh).mean(1, keepdim=True))
                    gamma[i], beta[i] = gamma[i] - lr * dg, beta[i] - lr * dbe
                if p > 0:
                    d = d * keep[i]
                d = d * der[i]
            delta[i], db[i] = d, d.sum(0)
            if i:
                d = d @ w[i].T
        if case["clip"] > 0:
            norm = math.sqrt(sum(float((x * x).sum()) for x in delta))
            if norm > case["clip"]:
                delta = [x * (case["clip"] / norm) for x in delta]
        for i in range(n):
            for x, m, v, grad, decay in ((w, mw, vw, a[i].T @ delta[i], wd), (b, mb, vb, db[i], 0.0)):
                if case["opt"] == "sgd":
                    x[i] = x[i] - lr * grad
                elif case["opt"] == "adagrad":
                    v[i] = v[i] + grad * grad
                    x[i] = x[i] - lr * grad / (v[i].sqrt() + eps)
                else:
                    m[i] = b1 * m[i] + (1 - b1) * grad
                    v[i] = b2 * v[i] + (1 - b2) * grad * grad
                    mh, vh = m[i] / (1 - b1 ** (RESUMED + s + 1)), v[i] / (1 - b2 ** (RESUMED + s + 1))
                    x[i] = x[i] - lr * (mh / (vh.sqrt() + eps) + decay * x[i])
    return {"loss": float(loss), "w": w, "b": b}


def _exact_optimizer(case, seed):
    ps, gs = _tensors(case, _gen(seed))
    c, out = _opt_config(case), []
    for p, g in zip(ps, gs):
        p, g = p.double(), g.double()
        if case["opt"] == "sgd":
            p = p - c.lr * g
        elif case["opt"] in ("adam", "adamw"):  # the first step: m / bias1 = g, v / bias2 = g^2
            p = p - c.lr * (g / (g.abs() + c.epsilon) + (c.weight_decay * p if case["opt"] == "adamw" else 0.0))
        else:
            d = g + c.weight_decay * p
            if case["opt"] == "lars":
                np_, ng = float(p.norm()), float(g.norm())
                local = c.lr * c.trust_coeff * np_ / (ng + c.weight_decay * np_ + c.epsilon) if np_ > 0 and ng > 0 else c.lr
                p = p - local * d
            else:
                s = d * d * (1 - c.alpha if case["opt"] == "rmsprop" else 1.0)
                p = p - c.lr * d / (s.sqrt() + c.epsilon)
        out.append(p)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "optimizer":
        return _exact_optimizer(case, seed)
    g, sizes = _gen(seed), _sizes(case)
    if kind == "infer":
        ws, bs = _weights(g, sizes)
        x = _normal(g, case["rows"], sizes[0]).double()
    else:
        t = _graph_inputs(case, g)
        x = t["x"].double()
        ws = [t["weight_%d_%d" % p] for p in zip(sizes, sizes[1:])]
        bs = [t["bias_%d" % c] for c in sizes[1:]]
    for i, (w, b) in enumerate(zip(ws, bs)):
        x = x @ w.double() + b.double().reshape(1, -1)
        if i < len(ws) - 1:
            x = _act(case["act"], x)[0]
    return x.cpu().numpy() if kind == "infer" else x
