"""The work that programs on this backend do, as cases that can be timed and compared.

Every pass goes through the public surface: ``raven_amd.nx_backend.Backend`` (one call per Nx
primitive), ``raven_amd.nx_frontend.Nx`` (the frontend's lowering to those primitives) and
``raven_amd.kaun_gpt2`` (Kaun's GPT-2 over the frontend). The kinds of work:

    mlp          a training step of a small classifier: forward, backward, update (Kaun / Rune)
    conv         a convolution layer, forward and backward: windows, products, folds (Kaun)
    embedding    a token table, forward (gather) and backward (scatter-add)
    gpt2         Kaun's GPT-2 small, bfloat16: a prompt's logits, issued call by call in the
                 deferred mode or replayed as a recorded graph
    matmul       batched products, every operand layout a forward and a backward pass has
    decode       a few activations times a weight matrix, what a decoding step is made of
    elementwise  permuted and broadcast operands, scalars, a narrowing cast, integers, a select
    reduce       statistics over rows and over columns
    sampling     probabilities, their order and their running sum over a vocabulary
    fft          filtering in the frequency domain: rows of a signal, or images
    solve        linear systems: Cholesky with two substitutions, or QR with one

Inputs are made on the GPU from the seed; results are torch tensors over the backend's storage.
"""

from __future__ import annotations

import math

import torch

from raven_amd import dtype as dt
from raven_amd import kaun_gpt2 as gpt2
from raven_amd.nx_backend import Backend
from raven_amd.nx_frontend import Nx

TORCH = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32,
         "float64": torch.float64, "int32": torch.int32, "bool": torch.uint8,
         "complex64": torch.complex64}
TYPESTR = {"float16": "<f2", "bfloat16": "<i2", "float32": "<f4", "float64": "<f8", "int32": "<i4",
           "bool": "|u1", "complex64": "<c8"}
LEARNING_RATE = 0.05


# ── contexts and the exchange of tensors with torch ─────────────────────────────────────────────

_CONTEXTS: dict = {}


def _context(deferred: bool = False) -> Nx:
    """A program has one context; the deferred mode is switched on once, when it is made."""
    nx = _CONTEXTS.get(deferred)
    if nx is None:
        backend = Backend()
        backend.set_deferred(deferred)
        nx = _CONTEXTS[deferred] = Nx(backend)
    return nx


class _Interface:
    """A backend tensor as torch takes it: the storage stays the backend's and lives as long as
    the torch tensor that is made from this."""

    def __init__(self, t):
        v, name = t.view, t.dtype.name
        size = t.dtype.itemsize
        self.tensor = t
        self.__cuda_array_interface__ = {
            "shape": v.shape, "strides": tuple([s * size for s in v.strides]), "typestr": TYPESTR[name],
            "data": (t.buffer.ptr + v.offset * size, False), "version": 2}


def _torch(t):
    x = torch.as_tensor(_Interface(t), device="cuda")
    return x.view(torch.bfloat16) if t.dtype is dt.bfloat16 else x


def _tensor(nx: Nx, x: torch.Tensor, dtype=None):
    """A backend tensor with the values of a torch tensor (complete once prepare() has waited)."""
    dtype = dtype or dt.BY_NAME[str(x.dtype).removeprefix("torch.")]
    t = nx.B.buffer(dtype, tuple(x.shape))
    _torch(t).copy_(x)
    return t


class _Draws:
    """The inputs of one seed, drawn on the GPU in a fixed order."""

    def __init__(self, nx: Nx, seed: int):
        self.nx = nx
        self.g = torch.Generator("cuda").manual_seed(seed)

    def raw(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std

    def normal(self, dtype, *shape, std=1.0):
        return _tensor(self.nx, self.raw(*shape, std=std).to(TORCH[dtype]))

    def integers(self, low, high, *shape):
        return _tensor(self.nx, torch.randint(low, high, shape, generator=self.g, device="cuda",
                                              dtype=torch.int32))


# ── the cases ───────────────────────────────────────────────────────────────────────────────────

def listed():
    return [
        # The smallest calls: some forty launches over a few kilobytes each (an MNIST-sized classifier).
        {"name": "mlp_step", "kind": "mlp", "batch": 32, "inputs": 784, "hidden": 128, "classes": 10},
        # A layer in the middle of a small image classifier, 3 x 3 windows of 28 x 28 maps.
        {"name": "conv_layer", "kind": "conv", "batch": 32, "channels": 32, "filters": 64, "size": 28,
         "kernel": 3, "stride": 1},
        # GPT-2 small's token table over a batch of 8 x 1024 tokens; most rows of the gradient stay zero.
        {"name": "embedding", "kind": "embedding", "tokens": 8192, "vocab": 50257, "dim": 768},
        # A short prompt issued call by call: the host's share of a forward shows.
        {"name": "gpt2_prompt", "kind": "gpt2", "batch": 1, "seq": 48, "how": "calls"},
        # The whole context window for eight sequences, as a serving program replays it.
        {"name": "gpt2_batch", "kind": "gpt2", "batch": 8, "seq": 1024, "how": "replay"},
        # The largest product of the benchmark.
        {"name": "matmul_batched", "kind": "matmul", "dtype": "bfloat16", "batch": 16, "m": 4096, "k": 4096,
         "n": 4096, "ta": False, "tb": False},
        # The benchmark's decoding product: bound by reading the weights.
        {"name": "decode", "kind": "decode", "dtype": "bfloat16", "m": 8, "k": 4096, "n": 16384},
        # The benchmark's headline step.
        {"name": "elementwise", "kind": "elementwise", "b": 64, "m": 512, "n": 512},
        # Statistics of a table whose rows are no whole number of vectors or tiles.
        {"name": "reduce_ragged", "kind": "reduce", "rows": 6000, "cols": 5001},
        # Nucleus sampling for a batch of sequences over GPT-2's vocabulary.
        {"name": "sampling", "kind": "sampling", "rows": 64, "cols": 50257},
        # Frames of a signal, filtered in the frequency domain.
        {"name": "fft_filter", "kind": "fft", "form": "rows", "rows": 8192, "n": 2048},
        # Regression with a few hundred unknowns, a handful of targets.
        {"name": "solve", "kind": "solve", "method": "cholesky", "dtype": "float32", "batch": 1, "n": 512,
         "nrhs": 16},
    ]


def _log(rng, low, high):
    """A whole number between low and high, spread over its logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(sorted(KINDS))
    case = {"kind": kind}
    if kind == "mlp":
        case.update(batch=_log(rng, 8, 2048), inputs=_log(rng, 16, 1024), hidden=_log(rng, 16, 1024),
                    classes=rng.randint(2, 100))
    elif kind == "conv":
        case.update(batch=rng.randint(1, 32), channels=_log(rng, 1, 64), filters=_log(rng, 8, 64),
                    size=rng.randint(8, 64), kernel=rng.choice([3, 3, 3, 5]), stride=rng.choice([1, 1, 2]))
    elif kind == "embedding":
        case.update(tokens=_log(rng, 32, 16384), vocab=_log(rng, 256, 50257), dim=_log(rng, 32, 1024))
    elif kind == "gpt2":
        seq = _log(rng, 16, 1024)
        case.update(batch=rng.randint(1, max(1, min(8, 4096 // seq))), seq=seq,
                    how=rng.choice(["calls", "replay"]))
    elif kind == "matmul":
        case.update(dtype=rng.choice(["float32", "bfloat16", "float16"]), batch=_log(rng, 1, 16),
                    m=_log(rng, 32, 2048), k=_log(rng, 32, 2048), n=_log(rng, 32, 2048),
                    ta=rng.random() < 0.25, tb=rng.random() < 0.25)
    elif kind == "decode":
        case.update(dtype=rng.choice(["bfloat16", "float16", "float32"]), m=rng.randint(1, 16),
                    k=_log(rng, 256, 16384), n=_log(rng, 256, 16384))
    elif kind == "elementwise":
        case.update(b=_log(rng, 1, 64), m=_log(rng, 8, 512), n=_log(rng, 8, 512))
    elif kind == "reduce":
        case.update(rows=_log(rng, 16, 8192), cols=_log(rng, 16, 8192))
    elif kind == "sampling":
        case.update(rows=_log(rng, 1, 64), cols=_log(rng, 256, 50257))
    elif kind == "fft":
        form = rng.choice(["rows", "rows", "image"])
        # half of the lengths are powers of two, the others what a signal or an image happens to have
        n = 2 ** rng.randint(6, 13) if rng.random() < 0.5 else _log(rng, 50, 5000)
        if form == "rows":
            case.update(form=form, rows=_log(rng, 1, max(1, (1 << 24) // n)), n=n)
        else:
            n = min(n, 2048)
            case.update(form=form, rows=_log(rng, 1, max(1, (1 << 22) // (n * n))), n=n)
    else:
        n = _log(rng, 16, 1024)
        case.update(method=rng.choice(["cholesky", "cholesky", "qr"]), dtype=rng.choice(["float32", "float64"]),
                    batch=_log(rng, 1, max(1, (1 << 20) // (n * n))), n=n, nrhs=_log(rng, 1, 64))
    return case


def prepare(case, seed):
    kind = case["kind"]
    nx = _context(deferred=kind == "gpt2")
    nx.B.synchronize()  # storage given back may still be in use by the context's stream
    make, do = KINDS[kind]
    state = make(case, nx, _Draws(nx, seed))
    torch.cuda.synchronize()
    if kind == "gpt2" and case["how"] == "replay":
        state = _Recorded(*state)
    return do, state


def run(state):
    return state[0](state[1])


# ── mlp: logits = max(x w1 + b1, 0) w2 + b2, mean cross entropy against one-hot targets ─────────

def _prepare_mlp(c, nx, d):
    b, i, h, k = c["batch"], c["inputs"], c["hidden"], c["classes"]
    x = d.normal("float32", b, i)
    labels = torch.randint(0, k, (b,), generator=d.g, device="cuda")
    onehot = _tensor(nx, torch.nn.functional.one_hot(labels, k).float())
    params = [d.normal("float32", i, h, std=1 / math.sqrt(i)), _tensor(nx, torch.zeros(h, device="cuda")),
              d.normal("float32", h, k, std=1 / math.sqrt(h)), _tensor(nx, torch.zeros(k, device="cuda"))]
    return nx, x, onehot, params, [_torch(p) for p in params]


def _run_mlp(state):
    nx, x, onehot, params, updated = state
    w1, b1, w2, b2 = params
    binary, n = nx.B.binary, float(x.shape[0])
    z = nx.add(nx.matmul(x, w1), b1)
    h = nx._binop("max", z, nx.scalar_like(z, 0.0))
    logits = nx.add(nx.matmul(h, w2), b2)
    # the loss as logits - log(sum(exp)) picked by the targets
    shifted = nx.sub(logits, nx.max(logits, [1], keepdims=True))
    e = nx.exp(shifted)
    total = nx.sum(e, [1], keepdims=True)
    log_p = nx.sub(shifted, nx.B.unary("log", total))
    loss = nx.mul_s(nx.sum(binary("mul", onehot, log_p), [0, 1]), -1.0 / n)
    # the transposed steps
    g = nx.mul_s(nx.sub(nx.div(e, total), onehot), 1.0 / n)
    grads = [None] * 4
    grads[2] = nx.matmul(nx.transpose(h), g)
    grads[3] = nx.sum(g, [0])
    dh = nx.matmul(g, nx.transpose(w2))
    zero = nx.scalar_like(z, 0.0)
    positive = nx.B.compare("cmplt", nx.broadcast_to(z.shape, zero), z)
    dz = nx.where(positive, dh, zero)
    grads[0] = nx.matmul(nx.transpose(x), dz)
    grads[1] = nx.sum(dz, [0])
    for p, grad in zip(params, grads):
        nx.B.assign(p, nx.sub(p, nx.mul_s(grad, LEARNING_RATE)))
    return updated, _torch(loss)


# ── conv: y = max(w * windows(x) + b, 0) and the gradients of x, w and b ────────────────────────

def _conv_geometry(c):
    k, s = c["kernel"], c["stride"]
    pad = (k - 1) // 2
    out = (c["size"] + 2 * pad - k) // s + 1
    return [[k, k], [s, s], [1, 1], [(pad, pad), (pad, pad)]], out


def _prepare_conv(c, nx, d):
    taps = c["channels"] * c["kernel"] ** 2
    geometry, out = _conv_geometry(c)
    x = d.normal("float32", c["batch"], c["channels"], c["size"], c["size"])
    w = d.normal("float32", c["filters"], taps, std=1 / math.sqrt(taps))
    b = d.normal("float32", c["filters"], 1, std=0.1)
    g = d.normal("float32", c["batch"], c["filters"], out * out)
    return nx, geometry, x, w, b, g


def _run_conv(state):
    nx, geometry, x, w, b, g = state
    B = nx.B
    batch, channels, size, _ = x.shape
    filters, taps = w.shape
    cols = B.unfold(x, *geometry)
    cols = nx.reshape((batch, taps, cols.shape[-1]), cols)
    wide = nx.broadcast_to((batch, filters, taps), w)
    z = nx.add(nx.matmul(wide, cols), b)
    zero = nx.scalar_like(z, 0.0)
    y = nx._binop("max", z, zero)
    dz = nx.where(B.compare("cmplt", nx.broadcast_to(z.shape, zero), z), g, zero)
    dw = nx.sum(nx.matmul(dz, nx.swapaxes(1, 2, cols)), [0])
    db = nx.sum(dz, [0, 2])
    dcols = nx.matmul(nx.swapaxes(1, 2, wide), dz)
    dx = B.fold(nx.reshape((batch, channels, taps // channels, cols.shape[-1]), dcols), [size, size], *geometry)
    return _torch(y), _torch(dw), _torch(db), _torch(dx)


# ── embedding ───────────────────────────────────────────────────────────────────────────────────

def _prepare_embedding(c, nx, d):
    table = d.normal("float32", c["vocab"], c["dim"], std=0.02)
    ids = d.integers(0, c["vocab"], c["tokens"])
    return nx, table, ids, d.normal("float32", c["tokens"], c["dim"])


def _run_embedding(state):
    nx, table, ids, g = state
    rows = nx.take(table, ids, axis=0)
    index = nx.broadcast_to(g.shape, nx.reshape((g.shape[0], 1), ids))
    zeros = nx.B.full(table.dtype, table.shape, 0.0)
    grad = nx.B.scatter("add", False, zeros, index, g, 0)
    return _torch(rows), _torch(grad)


# ── gpt2: Kaun's GPT-2 small over random weights ────────────────────────────────────────────────

def _prepare_gpt2(c, nx, d):
    cfg = gpt2.Config.small()
    e = cfg.n_embd

    def normal(*shape):
        return d.normal("bfloat16", *shape, std=0.02)

    def linear(i, o):
        return gpt2.Linear(normal(i, o), normal(o))

    def norm():
        return gpt2.LayerNorm(_tensor(nx, torch.ones(e, dtype=torch.bfloat16, device="cuda")),
                              _tensor(nx, torch.zeros(e, dtype=torch.bfloat16, device="cuda")))

    blocks = [gpt2.Block(norm(), gpt2.Attention(*(linear(e, e) for _ in range(4))), norm(),
                         linear(e, cfg.n_inner), linear(cfg.n_inner, e)) for _ in range(cfg.n_layer)]
    params = gpt2.Params(normal(cfg.vocab_size, e), normal(cfg.n_positions, e), blocks, norm())
    ids = d.integers(0, cfg.vocab_size, c["batch"], c["seq"])
    return nx, gpt2.Gpt2(nx, cfg), params, ids


class _Recorded:
    """A forward recorded once for its shape; every pass copies its ids in and replays it."""

    def __init__(self, nx, model, params, ids):
        self.nx, self.params, self.ids = nx, params, ids
        self.slot = nx.B.copy(ids)
        model.logits(params, self.slot)  # every entry point runs once before it is recorded
        nx.B.synchronize()
        nx.B.capture_begin()
        try:
            self.logits = model.logits(params, self.slot)
        finally:
            self.graph = nx.B.capture_end()
        self.result = _torch(self.logits)

    def __del__(self):
        if getattr(self, "graph", None) is not None:
            self.graph.destroy()


def _run_gpt2(state):
    if isinstance(state, _Recorded):
        state.nx.B.assign(state.slot, state.ids)
        state.graph.launch()
        return state.result
    nx, model, params, ids = state
    return _torch(model.logits(params, ids))


# ── matmul and decode ───────────────────────────────────────────────────────────────────────────

def _prepare_matmul(c, nx, d):
    def operand(rows, cols, transposed):
        shape = (c["batch"], cols, rows) if transposed else (c["batch"], rows, cols)
        t = d.normal(c["dtype"], *shape, std=0.02)
        return nx.swapaxes(1, 2, t) if transposed else t

    return nx, operand(c["m"], c["k"], c["ta"]), operand(c["k"], c["n"], c["tb"])


def _run_matmul(state):
    nx, a, b = state
    return _torch(nx.matmul(a, b))


def _prepare_decode(c, nx, d):
    return nx, d.normal(c["dtype"], c["m"], c["k"], std=0.02), d.normal(c["dtype"], c["k"], c["n"], std=0.02)


_run_decode = _run_matmul


# ── elementwise: a is read through a permuted view, b is broadcast ──────────────────────────────

def _prepare_elementwise(c, nx, d):
    b, m, n = c["b"], c["m"], c["n"]
    return (nx, nx.B.permute(d.normal("float32", b, n, m), (0, 2, 1)), d.normal("float32", 1, m, 1),
            nx.B.permute(d.integers(-1000, 1001, b, n, m), (0, 2, 1)), d.integers(-1000, 1001, 1, m, 1))


def _run_elementwise(state):
    nx, a, b, ai, bi = state
    scaled = nx.mul_s(nx.add(a, b), 0.5)
    half = nx.cast(dt.float16, scaled)
    greater = nx.B.compare("cmplt", nx.broadcast_to(ai.shape, bi), ai)
    out = (scaled, half, nx.add(ai, bi), nx.mul(ai, bi), nx.where(greater, ai, bi))
    return [_torch(t) for t in out]


# ── reduce ──────────────────────────────────────────────────────────────────────────────────────

def _prepare_reduce(c, nx, d):
    return nx, d.normal("float32", c["rows"], c["cols"]), d.integers(-1000, 1001, c["rows"], c["cols"])


def _run_reduce(state):
    nx, x, xi = state
    out = []
    for axis in (1, 0):
        out += [nx.sum(x, [axis]), nx.max(x, [axis]), nx.B.argmax(x, axis), nx.sum(xi, [axis])]
    return [_torch(t) for t in out]


# ── sampling ────────────────────────────────────────────────────────────────────────────────────

def _prepare_sampling(c, nx, d):
    return nx, d.normal("float32", c["rows"], c["cols"], std=2.0)


def _run_sampling(state):
    nx, logits = state
    p = nx.softmax(logits)
    order = nx.B.argsort(logits, 1, True)
    ranked = nx.B.gather(p, order, 1)
    return _torch(order), _torch(ranked), _torch(nx.B.associative_scan(1, "sum", ranked))


# ── fft ─────────────────────────────────────────────────────────────────────────────────────────

def _prepare_fft(c, nx, d):
    n, r = c["n"], c["rows"]
    if c["form"] == "rows":
        x = d.normal("float32", r, n)
        spectrum = torch.complex(d.raw(1, n // 2 + 1), d.raw(1, n // 2 + 1))
    else:
        x = _tensor(nx, torch.complex(d.raw(r, n, n), d.raw(r, n, n)))
        spectrum = torch.complex(d.raw(1, n, n), d.raw(1, n, n))
    return nx, c["form"], x, _tensor(nx, spectrum)


def _run_fft(state):
    nx, form, x, spectrum = state
    n = x.shape[-1]
    if form == "rows":
        y = nx.B.irfft(nx.mul(nx.B.rfft(x, dt.complex64, [1]), spectrum), dt.float32, [1], [n])
        return _torch(nx.mul_s(y, 1.0 / n))
    y = nx.B.ifft(nx.mul(nx.B.fft(x, [1, 2]), spectrum), [1, 2])
    return _torch(nx.mul_s(y, 1.0 / (n * n)))


# ── solve ───────────────────────────────────────────────────────────────────────────────────────

def _prepare_solve(c, nx, d):
    b, n = c["batch"], c["n"]
    a = d.raw(b, n, n).double()
    if c["method"] == "cholesky":  # the normal matrix of a regression with a ridge
        a = a @ a.transpose(1, 2).contiguous() + n * torch.eye(n, device="cuda", dtype=torch.float64)
    else:
        a = a + math.sqrt(n) * 2 * torch.eye(n, device="cuda", dtype=torch.float64)
    return nx, c["method"], _tensor(nx, a.to(TORCH[c["dtype"]])), d.normal(c["dtype"], b, n, c["nrhs"])


def _run_solve(state):
    nx, method, a, rhs = state
    B = nx.B
    if method == "cholesky":
        factor = B.cholesky(a)
        y = B.triangular_solve(factor, rhs, upper=False, transpose=False, unit_diag=False)
        return _torch(factor), _torch(B.triangular_solve(factor, y, upper=False, transpose=True, unit_diag=False))
    q, r = B.qr(a)
    x = B.triangular_solve(r, nx.matmul(nx.swapaxes(1, 2, q), rhs), upper=True, transpose=False, unit_diag=False)
    return _torch(q), _torch(r), _torch(x)


KINDS = {
    "mlp": (_prepare_mlp, _run_mlp), "conv": (_prepare_conv, _run_conv),
    "embedding": (_prepare_embedding, _run_embedding), "gpt2": (_prepare_gpt2, _run_gpt2),
    "matmul": (_prepare_matmul, _run_matmul), "decode": (_prepare_decode, _run_decode),
    "elementwise": (_prepare_elementwise, _run_elementwise), "reduce": (_prepare_reduce, _run_reduce),
    "sampling": (_prepare_sampling, _run_sampling), "fft": (_prepare_fft, _run_fft),
    "solve": (_prepare_solve, _run_solve),
}


# ── what a pass cannot do without, and how close two correct results are ────────────────────────

def work(case):
    c, kind = case, case["kind"]
    size = {"float16": 2, "bfloat16": 2, "float32": 4, "float64": 8}.get(c.get("dtype"), 4)
    if kind == "mlp":
        b, i, h, k = c["batch"], c["inputs"], c["hidden"], c["classes"]
        return {"bytes": 4 * (b * (i + k) + 2 * (i * h + h + h * k + k)),
                "flops": 2 * b * (2 * i * h + 3 * h * k)}
    if kind == "conv":
        taps, out = c["channels"] * c["kernel"] ** 2, _conv_geometry(c)[1] ** 2
        return {"bytes": 4 * (2 * c["batch"] * c["channels"] * c["size"] ** 2 + 2 * c["filters"] * (taps + 1)
                              + 2 * c["batch"] * c["filters"] * out),
                "flops": 3 * 2 * c["batch"] * c["filters"] * taps * out}
    if kind == "embedding":
        return {"bytes": 4 * (3 * c["tokens"] * c["dim"] + c["tokens"] + c["vocab"] * c["dim"]),
                "flops": c["tokens"] * c["dim"]}
    if kind == "gpt2":
        cfg, t = gpt2.Config.small(), c["batch"] * c["seq"]
        e, v = cfg.n_embd, cfg.vocab_size
        weights = cfg.n_layer * (4 * e * e + 2 * e * cfg.n_inner) + v * e
        return {"bytes": 2 * (weights + t * v),
                "flops": 2 * t * weights + cfg.n_layer * 4 * t * (c["seq"] + 1) / 2 * e}
    if kind == "matmul":
        b, m, k, n = c["batch"], c["m"], c["k"], c["n"]
        return {"bytes": size * b * (m * k + k * n + m * n), "flops": 2 * b * m * k * n}
    if kind == "decode":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": size * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    if kind == "elementwise":
        # in: both operands; out: two of four bytes and one of two, three of four
        return {"bytes": c["b"] * c["m"] * c["n"] * (8 + 6 + 12), "flops": 7 * c["b"] * c["m"] * c["n"]}
    if kind == "reduce":
        return {"bytes": 8 * c["rows"] * c["cols"] + 16 * (c["rows"] + c["cols"]), "flops": 8 * c["rows"] * c["cols"]}
    if kind == "sampling":
        return {"bytes": 16 * c["rows"] * c["cols"], "flops": 5 * c["rows"] * c["cols"]}
    if kind == "fft":
        n, r = c["n"], c["rows"]
        if c["form"] == "rows":
            return {"bytes": 8 * r * n + 4 * n, "flops": 5 * r * n * math.log2(n) + 3 * r * n}
        return {"bytes": 16 * r * n * n + 8 * n * n, "flops": 20 * r * n * n * math.log2(n) + 6 * r * n * n}
    n, b, m = c["n"], c["batch"], c["nrhs"]
    if c["method"] == "cholesky":
        return {"bytes": size * b * (2 * n * n + 2 * n * m), "flops": b * (n ** 3 / 3 + 2 * n * n * m)}
    return {"bytes": size * b * (3 * n * n + 2 * n * m), "flops": b * (8 * n ** 3 / 3 + 3 * n * n * m)}


def tolerance(case):
    """About four times what each path was seen to be off from the same pass in float64 (gpt2: the
    fused pass from the primitives one by one, whose roundings fall elsewhere)."""
    kind, dtype = case["kind"], case.get("dtype")
    if kind == "elementwise":
        return "exact"  # one rounding per operation, the rest whole numbers
    if kind == "gpt2":
        return {"rel": 2.5e-2, "max": 0.3}  # seen: 1.2e-2, 0.072
    if kind in ("matmul", "decode"):
        # seen: 1.7e-3 and 2.1e-4, the rounding of the result; 6e-7, a float32 sum of a thousand terms
        return {"bfloat16": {"rel": 4e-3, "max": 1.6e-2}, "float16": {"rel": 8e-4, "max": 2e-3},
                "float32": {"rel": 3e-6}}[dtype]
    if kind == "solve":
        return {"rel": 1e-14} if dtype == "float64" else {"rel": 4e-7}  # seen: 2e-15, 6e-8
    return {"rel": {"mlp": 1e-6, "conv": 3e-6, "embedding": 1e-6, "reduce": 1e-6, "sampling": 5e-7, "fft": 4e-7}[kind]}
