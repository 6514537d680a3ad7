"""Performance cases: the gradient evaluations that programs on this package run, over the range of sizes they run them at.

Every case is one of the package's benchmark programs (``autograd_amd.configs``) or example programs at some size, in
one of the two ways a program evaluates a derivative: eagerly, where every pass goes through the tracer, the tape and
the backward pass, or replayed from a recorded graph (``capture``), as a training loop on fixed shapes does.

  tanh     derivatives of an elementwise formula to some order (the plotted tanh example, config 1)
  lse      gradient of sum(logsumexp(A*b + c)) with respect to A, b and c (config 2)
  mlp      log-softmax classifier: gradient of its loss, or its predictions alone (config 3)
  adam     the neural-net example: a few Adam steps on minibatches, parameters flattened and unflattened on the way
  rnn      gradient of a tanh recurrent net's log likelihood over all its time steps (config 4)
  rosen    Hessian-vector product of the Rosenbrock function, reverse-over-reverse or forward-over-reverse (config 5)
  convnet  gradient of the LeNet-style convolution stack (the convnet example)

``listed()`` gives named cases, ``draw(rng)`` others from the same ranges; ``prepare`` makes a case's inputs on the GPU
from a seed, ``run`` makes one pass, ``work`` counts what a pass cannot do without, ``tolerance`` says how far the
results of two correct evaluations at one precision may lie apart.
"""

import math

import torch

import autograd_amd as ag
import autograd_amd.numpy as np
from autograd_amd import configs
from autograd_amd.misc.flatten import flatten
from autograd_amd.misc.optimizers import adam
from autograd_amd.numpy.devarray import DevArray
from autograd_amd.scipy.signal import convolve
from autograd_amd.scipy.special import logsumexp

_TORCH = {"float32": torch.float32, "float64": torch.float64}


def listed():
    return [
        # 200 points of a plot (examples/tanh.py): nothing but the latency of a call
        dict(name="tanh_plot", kind="tanh", n=200, dtype="float64", order=2, replay=False),
        # config 1 at its own size, third derivative: long chains of elementwise rules
        dict(name="tanh_order3", kind="tanh", n=4194304, dtype="float64", order=3, replay=True),
        # config 2 at its own size: the headline benchmark, evaluated eagerly
        dict(name="lse_headline", kind="lse", rows=8192, cols=4096, dtype="float32", replay=False),
        # the same model on a matrix whose extents divide nothing, double precision, in a loop on fixed shapes
        dict(name="lse_ragged", kind="lse", rows=3001, cols=1999, dtype="float64", replay=True),
        # config 3 at its own size, as a training loop replays it
        dict(name="mlp", kind="mlp", batch=1024, sizes="784,1024,1024,10", dtype="float32", what="grad", replay=True),
        # a classifier with wide layers and many classes: the largest contractions
        dict(name="mlp_wide", kind="mlp", batch=4096, sizes="2048,4096,4096,1000", dtype="float32", what="grad", replay=False),
        # examples/neural_net.py with its layer sizes, batch size and precision: optimizer steps on minibatches
        dict(name="mlp_adam", kind="adam", batch=256, sizes="784,200,100,10", dtype="float64", steps=4),
        # config 4 at its own size, replayed: a long chain of small dependent steps
        dict(name="rnn", kind="rnn", steps=64, batch=256, inputs=128, state=512, outputs=128, dtype="float32", replay=True),
        # examples/rnn.py with its state size and precision, evaluated eagerly: a tape of small operations
        dict(name="rnn_example", kind="rnn", steps=30, batch=35, inputs=128, state=40, outputs=128, dtype="float64", replay=False),
        # config 5 at its own size, evaluated eagerly
        dict(name="rosen_hvp", kind="rosen", n=16777216, dtype="float64", way="hvp_rev", replay=False),
        # the forward-over-reverse product on an odd number of unknowns, inside a solver's loop
        dict(name="rosen_jvp", kind="rosen", n=1000003, dtype="float32", way="hvp_fwd", replay=True),
        # the convnet example's layers and precision
        dict(name="convnet", kind="convnet", batch=256, dtype="float64", replay=True),
    ]


def _between(rng, low, high):
    """A whole number, spread over the logarithm of the range."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("tanh", "lse", "mlp", "adam", "rnn", "rosen", "convnet"))
    dtype, replay = rng.choice(("float32", "float64")), rng.random() < 0.5
    if kind == "tanh":
        # (the formula's third derivative overflows single precision over this range)
        order = rng.randint(1, 3 if dtype == "float64" else 2)
        return dict(kind=kind, n=_between(rng, 100, 1 << 24), dtype=dtype, order=order, replay=replay)
    if kind == "lse":
        rows = _between(rng, 16, 16384)
        cols = _between(rng, 8, min(32768, (1 << 25) // rows))
        return dict(kind=kind, rows=rows, cols=cols, dtype=dtype, replay=replay)
    if kind == "mlp":
        sizes = [_between(rng, 32, 4096)] + [_between(rng, 64, 4096) for _ in range(rng.randint(1, 3))]
        sizes.append(rng.choice((2, 10, 100, _between(rng, 2, 1000))))
        most = int(1e11 / sum(m * n for m, n in zip(sizes, sizes[1:]))) // (1 if dtype == "float32" else 4)
        return dict(kind=kind, batch=_between(rng, 16, min(4096, max(most, 16))), sizes=",".join(map(str, sizes)), dtype=dtype,
                    what=rng.choice(("grad", "grad", "predict")), replay=replay)
    if kind == "adam":
        sizes = [_between(rng, 16, 1024), _between(rng, 16, 1024), _between(rng, 16, 256), 10]
        return dict(kind=kind, batch=_between(rng, 16, 1024), sizes=",".join(map(str, sizes)), dtype=dtype, steps=rng.randint(2, 5))
    if kind == "rnn":
        vocabulary = _between(rng, 16, 128)
        return dict(kind=kind, steps=_between(rng, 6, 64 if replay else 32), batch=_between(rng, 8, 256), inputs=vocabulary,
                    state=_between(rng, 24, 512), outputs=vocabulary, dtype=dtype, replay=replay)
    if kind == "rosen":
        return dict(kind=kind, n=_between(rng, 1000, 1 << 24), dtype=dtype, way=rng.choice(("hvp_rev", "hvp_fwd")), replay=replay)
    return dict(kind=kind, batch=_between(rng, 16, 512), dtype=dtype, replay=replay)


# --------------------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------------------
class _Source:
    """Seeded draws made on the GPU."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.dtype = _TORCH[dtype]

    def normal(self, *shape, scale=1.0):
        return DevArray(torch.randn(shape, generator=self.g, device="cuda", dtype=self.dtype) * scale)

    def uniform(self, low, high, *shape):
        return DevArray(torch.rand(shape, generator=self.g, device="cuda", dtype=self.dtype) * (high - low) + low)

    def one_hot(self, classes, *shape):
        ids = torch.randint(classes, shape, generator=self.g, device="cuda")
        return DevArray(torch.nn.functional.one_hot(ids, classes).to(self.dtype))

    def layers(self, sizes):
        return [(self.normal(m, n, scale=1 / math.sqrt(m)), self.normal(n, scale=0.1)) for m, n in zip(sizes, sizes[1:])]


def _sizes(case):
    return [int(s) for s in case["sizes"].split(",")]


def _tanh(case, src):
    return configs.tanh_program(configs.device_backend())[f"d{case['order']}"], (src.uniform(-7.0, 7.0, case["n"]),)


def _lse(case, src):
    rows, cols = case["rows"], case["cols"]
    inputs = (src.normal(rows, cols), src.uniform(0.5, 1.5, cols), src.normal(rows))
    return configs.bcast_program(configs.device_backend())["grad"], inputs


def _predict(params, inputs):
    """A dense log-softmax classifier (examples/neural_net.py:28-36)."""
    for W, b in params:
        outputs = np.dot(inputs, W) + b
        inputs = np.tanh(outputs)
    return outputs - logsumexp(outputs, axis=1, keepdims=True)


def _mlp(case, src):
    sizes = _sizes(case)
    params, X, T = src.layers(sizes), src.normal(case["batch"], sizes[0]), src.one_hot(sizes[-1], case["batch"])
    if case["what"] == "predict":
        return _predict, (params, X)
    return configs.mlp_program(configs.device_backend())["grad"], (params, X, T)


def _adam(case, src):
    """examples/neural_net.py:38-110: minus the log posterior of a minibatch, minimised by Adam."""
    sizes, batch, batches = _sizes(case), case["batch"], 3
    params = src.layers(sizes)
    X, T = src.normal(batches * batch, sizes[0]), src.one_hot(sizes[-1], batches * batch)

    def objective(params, i):
        rows = slice(i % batches * batch, (i % batches + 1) * batch)
        flat, _ = flatten(params)
        return 0.01 * np.dot(flat, flat) - np.sum(_predict(params, X[rows]) * T[rows])

    gradient = ag.grad(objective)
    return (lambda params: adam(gradient, params, step_size=0.001, num_iters=case["steps"])), (params,)


def _rnn(case, src):
    steps, batch, inputs, state, outputs = (case[k] for k in ("steps", "batch", "inputs", "state", "outputs"))
    params = {
        "init hiddens": src.normal(1, state, scale=0.1),
        "change": src.normal(inputs + state + 1, state, scale=1 / math.sqrt(state)),
        "predict": src.normal(state + 1, outputs, scale=1 / math.sqrt(state)),
    }
    data = src.one_hot(inputs, steps, batch), src.one_hot(outputs, steps, batch)
    return configs.rnn_program(configs.device_backend())["grad"], (params,) + data


def _rosen(case, src):
    return configs.rosen_program(configs.device_backend())[case["way"]], (src.uniform(-2.0, 2.0, case["n"]), src.normal(case["n"]))


def _convnet(case, src):
    def layer(*shape):
        return src.normal(*shape, scale=1 / math.sqrt(math.prod(shape) / shape[1]))

    params = {"c1": layer(1, 6, 5, 5), "b1": src.normal(1, 6, 1, 1, scale=0.1), "c2": layer(6, 16, 5, 5), "b2": src.normal(1, 16, 1, 1, scale=0.1)}
    for k, (W, b) in zip("345", src.layers([256, 120, 84, 10])):
        params["w" + k], params["b" + k] = W, b
    X, T = src.uniform(0.0, 1.0, case["batch"], 1, 28, 28), src.one_hot(10, case["batch"])
    return configs.convnet_program(configs.device_backend(), convolve)["grad"], (params, X, T)


_KINDS = {"tanh": _tanh, "lse": _lse, "mlp": _mlp, "adam": _adam, "rnn": _rnn, "rosen": _rosen, "convnet": _convnet}


def prepare(case, seed):
    """The function that a program evaluates over and over, and its arguments on the GPU."""
    function, args = _KINDS[case["kind"]](case, _Source(seed, case["dtype"]))
    return (ag.capture(function, *args) if case.get("replay") else function), args


# --------------------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------------------
def _tensors(result):
    if isinstance(result, (list, tuple)):
        return [_tensors(r) for r in result]
    if isinstance(result, dict):
        return {k: _tensors(r) for k, r in result.items()}
    return result._t


def run(state):
    function, args = state
    return _tensors(function(*args))


# --------------------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------------------
def _dense(batch, sizes):
    """Parameters, and multiply-adds of one forward pass, of dense layers."""
    pairs = list(zip(sizes, sizes[1:]))
    return sum((m + 1) * n for m, n in pairs), batch * sum(m * n for m, n in pairs), batch * sizes[0] * sizes[1]


def work(case):
    """Bytes: inputs read once and results written once.  Flops: contractions (the input needs no cotangent) and a
    rough count of elementwise arithmetic where there is no contraction."""
    kind, size = case["kind"], 4 if case["dtype"] == "float32" else 8
    if kind == "tanh":
        return {"bytes": 2 * size * case["n"], "flops": 20 * case["order"] * case["n"]}
    if kind == "lse":
        rows, cols = case["rows"], case["cols"]
        return {"bytes": 2 * size * (rows * cols + rows + cols), "flops": 10 * rows * cols}
    if kind == "mlp":
        sizes, batch = _sizes(case), case["batch"]
        weights, forward, first = _dense(batch, sizes)
        if case["what"] == "predict":
            return {"bytes": size * (weights + batch * (sizes[0] + sizes[-1])), "flops": 2 * forward}
        return {"bytes": size * (2 * weights + batch * (sizes[0] + sizes[-1])), "flops": 2 * (3 * forward - first)}
    if kind == "adam":
        sizes, batch, steps = _sizes(case), case["batch"], case["steps"]
        weights, forward, first = _dense(batch, sizes)
        # the update is double precision whatever the point's type: state and parameters read and written
        return {"bytes": steps * (48 * weights + size * batch * (sizes[0] + sizes[-1])), "flops": steps * 2 * (3 * forward - first)}
    if kind == "rnn":
        steps, batch, inputs, state, outputs = (case[k] for k in ("steps", "batch", "inputs", "state", "outputs"))
        weights = state + (inputs + state + 1) * state + (state + 1) * outputs
        step = batch * state * (2 * (inputs + state + 1) + state) + 3 * batch * (state + 1) * outputs
        return {"bytes": size * (2 * weights + steps * batch * (inputs + outputs)), "flops": 2 * steps * step}
    if kind == "rosen":
        return {"bytes": 3 * size * case["n"], "flops": 20 * case["n"]}
    batch = case["batch"]
    conv1, conv2 = 24 * 24 * 6 * 25, 8 * 8 * 16 * 6 * 25
    weights, forward, _ = _dense(batch, [256, 120, 84, 10])
    return {"bytes": size * (2 * (weights + 156 + 2416) + batch * (784 + 10)), "flops": 2 * (batch * (2 * conv1 + 3 * conv2) + 3 * forward)}


# About four times what a pass was measured to differ by: in single precision from the same pass in double precision, in
# double precision from the derivative's closed form (tanh) or from that figure in units of roundoff (sums in another order
# differ by less).  The tanh formula's higher derivatives cancel; in single precision a pooling window whose two largest
# entries nearly tie may pick either, and its whole cotangent goes there.
_REL = {
    "float32": {"tanh": 6e-6, "lse": 2e-6, "mlp": 6e-6, "adam": 6e-6, "rnn": 6e-6, "rosen": 3e-7, "convnet": 1.5e-2},
    "float64": {"tanh": 5e-14, "lse": 3e-15, "mlp": 1.2e-14, "adam": 1.2e-14, "rnn": 1.2e-14, "rosen": 5e-16, "convnet": 1.2e-14},
}


def tolerance(case):
    return {"rel": _REL[case["dtype"]][case["kind"]]}
