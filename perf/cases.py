"""The workloads this framework is timed on: what a user's program does with it once a task is scheduled.

A program registers its operator (or takes a registered one), asks for the shipped config of the task and
falls back to the default one, builds the plan and then calls the plan on device tensors:

    config = lookup(key) or Config([], None)
    plan, bufs = schedule_with_config(key, config)
    func = flextensor_amd.build(plan, bufs, "rocm")
    func(a, b, c)

Scheduling, compiling and building happen once, the call is what repeats; a pass is one call. The listed cases
are the layers the shipped log was tuned for (through the registered task) and layers nobody tuned, which run
on the default config; the drawn ones are further sizes of every operator, odd ones among them.
"""
import math

import torch

import flextensor_amd
from flextensor_amd import nn
from flextensor_amd.scheduler import schedule_with_config
from flextensor_amd.task import TASK_TABLE, Task, register_task
from flextensor_amd.te import placeholder
from flextensor_amd.tuned import lookup
from flextensor_amd.utils import Config


def listed():
    return [
        # the fp32 matrix product of the benchmark: a dense layer of 1024 features over 1024 rows
        dict(name="gemm_1024", op="gemm", m=1024, k=1024, n=1024, trans_b=False),
        # a product whose extents are no multiples of anything: row counts and vocabularies as they come
        dict(name="gemm_odd", op="gemm", m=1000, k=1531, n=777, trans_b=False),
        # few rows against a large weight matrix: a dense layer at the batch size of serving, bound by the
        # stream of the weights
        dict(name="gemm_few_rows", op="gemm", m=32, k=4096, n=4096, trans_b=False),
        # many small products at once, the right operand stored transposed: similarity of 197 positions with
        # 197 positions in 64 features, one product per head and image
        dict(name="batch_gemm_heads", op="batch_gemm", b=96, m=197, k=64, n=197, trans_b=True),
        # the smallest call of the benchmark: one image, an early 3x3 layer; launches count
        dict(name="conv_1x64x56x56", op="conv2d", b=1, c=64, h=56, w=56, o=64, r=3, stride=1, pad=1, bias=False,
             table="baseline0"),
        # an ordinary 3x3 layer at batch 8
        dict(name="conv_8x256x14x14", op="conv2d", b=8, c=256, h=14, w=14, o=512, r=3, stride=1, pad=1, bias=False,
             table="baseline1"),
        # a downsampling layer with a bias on an odd image, nobody tuned it
        dict(name="conv_16x128x57x57_s2", op="conv2d", b=16, c=128, h=57, w=57, o=256, r=3, stride=2, pad=1,
             bias=True),
        # a pointwise layer with a bias on an odd image at a small batch, nobody tuned it
        dict(name="conv_2x240x35x35_1x1", op="conv2d", b=2, c=240, h=35, w=35, o=160, r=1, stride=1, pad=0,
             bias=True),
        # depthwise layer of the benchmark, bound by memory
        dict(name="depthwise_8x512x28x28", op="depthwise", b=8, c=512, h=28, w=28, r=3, stride=1, pad=1, bias=False),
        # depthwise layer on an odd image with a bias and rows that are no whole vectors, nobody tuned it
        dict(name="depthwise_16x144x57x57", op="depthwise", b=16, c=144, h=57, w=57, r=3, stride=1, pad=1,
             bias=True),
        # the largest product of the benchmark: int8 operands, exact int32 sums
        dict(name="gemm_i8_4096", op="gemm_int8", m=4096, k=4096, n=4096),
        # a quantised product of odd extents
        dict(name="gemm_i8_odd", op="gemm_int8", m=1000, k=1531, n=777),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A further size of one of the operators, over the range its listed cases stand for: on the default
    config unless the draw meets a tuned task."""
    op = rng.choice(["gemm", "gemm", "gemm_few_rows", "batch_gemm", "conv3", "conv3", "conv1", "depthwise",
                     "gemm_int8", "gemm_int8"])
    if op in ("gemm", "gemm_int8"):
        while True:
            m, k, n = (_log_int(rng, 64, 4096) for _ in range(3))
            if 2 * m * k * n <= (7e9 if op == "gemm" else 6e10):
                break
        if rng.random() < 0.5:                      # whole vectors as often as not
            m, k, n = (max(64, int(round(x / 16.0)) * 16) for x in (m, k, n))
        if op == "gemm_int8":
            return dict(op=op, m=m, k=k, n=n)
        return dict(op=op, m=m, k=k, n=n, trans_b=rng.random() < 0.3)
    if op == "gemm_few_rows":
        return dict(op="gemm", m=rng.randint(8, 64), k=_log_int(rng, 512, 4096), n=_log_int(rng, 512, 4096),
                    trans_b=rng.random() < 0.3)
    if op == "batch_gemm":
        while True:
            b, m, n = rng.randint(8, 128), _log_int(rng, 32, 512), _log_int(rng, 32, 512)
            k = rng.choice([32, 48, 64, 80, 96, 128, _log_int(rng, 32, 512)])
            if 2 * b * m * k * n <= 7e9:
                break
        return dict(op=op, b=b, m=m, k=k, n=n, trans_b=rng.random() < 0.5)
    if op == "depthwise":
        while True:
            b, c, h, w = rng.randint(1, 32), rng.randint(16, 512), rng.randint(7, 112), rng.randint(7, 112)
            if b * c * h * w <= 1.2e7:
                break
        r = rng.choice([3, 3, 5])
        return dict(op=op, b=b, c=c, h=h, w=w, r=r, stride=rng.choice([1, 1, 2]), pad=r // 2,
                    bias=rng.random() < 0.5)
    r = 3 if op == "conv3" else 1
    while True:
        b, c, o = rng.randint(1, 16), _log_int(rng, 16, 512), _log_int(rng, 16, 512)
        h, stride = _log_int(rng, 7, 112), rng.choice([1, 1, 2])
        w = h if rng.random() < 0.7 else _log_int(rng, 7, 112)
        if 2.0 * b * c * o * r * r * (h // stride) * (w // stride) <= 7e9:
            break
    return dict(op="conv2d", b=b, c=c, h=h, w=w, o=o, r=r, stride=stride, pad=r // 2, bias=rng.random() < 0.5)


# ---- the operator definitions a user's program registers: shapes -> (ops, bufs) ----------------------------

def _gemm(m, k, n, trans_b):
    a, b = placeholder((m, k), name="A"), placeholder((n, k) if trans_b else (k, n), name="B")
    c = nn.gemm(a, b, transposeB=bool(trans_b))
    return [c.op], [a, b, c]


def _batch_gemm(nb, m, k, n, trans_b):
    a, b = placeholder((nb, m, k), name="A"), placeholder((nb, n, k) if trans_b else (nb, k, n), name="B")
    c = nn.batch_gemm(a, b, transposeB=bool(trans_b))
    return [c.op], [a, b, c]


def _gemm_int8(m, k, n):
    a, b = placeholder((m, k), dtype="int8", name="A"), placeholder((n, k), dtype="int8", name="B")
    c = nn.gemm_int8(a, b)
    return [c.op], [a, b, c]


def _conv2d(b, c, h, w, o, r, stride, pad, bias):
    x, wt = placeholder((b, c, h, w), name="X"), placeholder((o, c, r, r), name="W")
    bs = placeholder((o,), name="bias") if bias else None
    y = nn.conv2d_nchw(x, wt, bs, stride=stride, padding=pad)
    return [y.op], [x, wt] + ([bs] if bias else []) + [y]


def _depthwise(b, c, h, w, r, stride, pad, bias):
    x, wt = placeholder((b, c, h, w), name="X"), placeholder((c, 1, r, r), name="W")
    bs = placeholder((c,), name="bias") if bias else None
    y = nn.depthwise_conv2d_nchw(x, wt, bs, stride=stride, padding=pad)
    return [y.op], [x, wt] + ([bs] if bias else []) + [y]


_BUILDERS = {
    "gemm": (_gemm, ("m", "k", "n", "trans_b")),
    "batch_gemm": (_batch_gemm, ("b", "m", "k", "n", "trans_b")),
    "gemm_int8": (_gemm_int8, ("m", "k", "n")),
    "conv2d": (_conv2d, ("b", "c", "h", "w", "o", "r", "stride", "pad", "bias")),
    "depthwise": (_depthwise, ("b", "c", "h", "w", "r", "stride", "pad", "bias")),
}


def _task_key(case):
    """Key of the registered task of these sizes where the framework has a tuned one; otherwise the key of a
    task registered here for the user's own layer."""
    op = case["op"]
    key = None
    if op == "gemm" and not case["trans_b"]:
        key = Task("gemm", "gemm", None, (case["m"], case["k"], case["n"]), "rocm", 0).key
    elif op == "gemm_int8":
        key = Task("gemm", "gemm_int8", None, (case["m"], case["k"], case["n"]), "rocm", 0).key
    elif op == "conv2d" and case.get("table"):
        key = Task("conv2d", case["table"], None, (case["b"], case["c"], case["h"], case["w"], case["o"], case["r"],
                                                   case["stride"], case["pad"], 1, 1), "rocm", 0).key
    elif op == "depthwise" and not case["bias"]:
        key = Task("conv2d", "depthwise", None, (case["b"], case["c"], case["h"], case["w"], 1, case["r"],
                                                 case["stride"], case["pad"], 1), "rocm", 0).key
    if key is not None and key in TASK_TABLE and lookup(key) is not None:
        return key
    builder, names = _BUILDERS[op]
    task = Task(op, "user_layer", builder, tuple(case[n] for n in names), "rocm", 0)
    register_task(task)
    return task.key


def prepare(case, seed):
    key = _task_key(case)
    plan, bufs = schedule_with_config(key, lookup(key) or Config([], None))
    func = flextensor_amd.build(plan, bufs, "rocm")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))

    def normal(shape, scale=1.0):
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * scale

    def quantised(shape):
        return (torch.randn(shape, generator=gen, device="cuda") * 32).round().clamp(-128, 127).to(torch.int8)

    shapes = [tuple(int(e) for e in b.shape) for b in bufs]
    op = case["op"]
    if op == "gemm_int8":
        # activations and weights after symmetric quantisation: bell-shaped over the int8 range
        inputs = [quantised(shapes[0]), quantised(shapes[1])]
    elif op in ("gemm", "batch_gemm"):
        inputs = [normal(shapes[0]), normal(shapes[1], case["k"] ** -0.5)]
    else:
        # an image behind a rectifier, weights at the scale that keeps the variance, a small bias
        fan_in = case["r"] * case["r"] * (case["c"] if op == "conv2d" else 1)
        inputs = [normal(shapes[0]).clamp_(min=0), normal(shapes[1], (2.0 / fan_in) ** 0.5)]
        if case["bias"]:
            inputs.append(normal(shapes[2], 0.1))
    out = torch.empty(shapes[-1], device="cuda", dtype=torch.int32 if op == "gemm_int8" else torch.float32)
    return func, tuple(inputs) + (out,)


def run(state):
    func, tensors = state
    func(*tensors)
    return tensors[-1]


def _out_hw(case):
    return tuple((case[d] + 2 * case["pad"] - case["r"]) // case["stride"] + 1 for d in "hw")


def work(case):
    op = case["op"]
    if op in ("gemm", "gemm_int8", "batch_gemm"):
        b, m, k, n = case.get("b", 1), case["m"], case["k"], case["n"]
        size = 1 if op == "gemm_int8" else 4
        return {"bytes": b * (size * (m * k + k * n) + 4 * m * n), "flops": 2 * b * m * k * n}
    p, q = _out_hw(case)
    b, c, r = case["b"], case["c"], case["r"]
    o = case["o"] if op == "conv2d" else c
    reduce = r * r * (c if op == "conv2d" else 1)
    floats = b * c * case["h"] * case["w"] + o * reduce + (o if case["bias"] else 0) + b * o * p * q
    return {"bytes": 4 * floats, "flops": 2 * b * o * p * q * reduce}


def tolerance(case):
    if case["op"] == "gemm_int8":
        return "exact"                  # integer sums: every order gives the same numbers
    # four times what separates the kernels from the same sums in float64 (worst of the listed and a dozen drawn
    # cases): depthwise rel 5.1e-8, max 5.1e-7 (9 taps; 25 at most are drawn); the others rel 1.15e-6, max
    # 6.9e-6 at k = 4096
    if case["op"] == "depthwise":
        return {"rel": 3e-7, "max": 3e-6}
    return {"rel": 5e-6, "max": 3e-5}
