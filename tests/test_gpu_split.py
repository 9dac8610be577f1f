"""Products in bf16 parts (pipeline depths 9 to 11) at the sizes where their parts have edges, against sums in float64, and
the numbers that have no such parts.

Bound: a product of two numbers in three parts is off by up to 2^-24 of itself, the large sum is rounded once for every
16 or 32 of K (six times for every 16 where a wavefront has four blocks), each time by up to 2^-24 of what it holds;
for the K of these cases (up to 1023) that is below 1e-5 of the largest result whatever the order."""
import numpy as np
import pytest

from test_gpu_direct import conv_of, gemm_of, rel, run

pytestmark = pytest.mark.gpu
TOL = 1e-5


def split_plan(func, args, tile, mfma, groups, depth, xcd=1, by_image=False):
    """The plan of the operator's contraction on tiles of (wavefronts, MFMA tiles each) along M and along N."""
    from flextensor_amd.scheduler import flatten_graph, schedule_with_config_ops
    from flextensor_amd.templates import gfx950
    from flextensor_amd.utils import Config, ceil_div
    ops, bufs = func(*args)
    configs = []
    for op in flatten_graph(ops)[0]:
        cfg = gfx950._empty_config()
        if op.kind in gfx950.GEMM_KINDS:
            (wm, rm, wn, rn), view = tile, gfx950.GemmView(op)
            view = view.by_image() if by_image else view
            cfg["spatial"] = [[ceil_div(view.M, mfma * wm * rm), wm, rm, mfma], [ceil_div(view.N, mfma * wn * rn), wn, rn, mfma]]
            cfg["reduce"], cfg["unroll"] = [[groups, ceil_div(view.K, 32 * groups), 32]], [[depth, 1]]
            cfg["fuse"], cfg["reorder"] = [[4]], [[xcd, 1 if groups > 1 else 0, 0] + ([2] if by_image else [])]
        configs.append(cfg)
    plan, bufs = schedule_with_config_ops(ops, bufs, Config(configs, None))
    assert plan.specs[-1].template == gfx950.SPLIT_DEPTHS[depth][0] and plan.specs[-1].defines["SPLIT"] == 1
    return plan, bufs


# (wavefronts, MFMA tiles each) along M and N, MFMA edge, groups, depth
GEMM_KERNELS = [((2, 2, 4, 1), 16, 1, 9), ((4, 1, 2, 2), 16, 2, 10), ((2, 1, 2, 1), 16, 4, 9), ((2, 1, 2, 1), 32, 2, 10),
                ((2, 2, 4, 1), 32, 1, 9), ((1, 1, 4, 1), 16, 1, 10), ((1, 2, 1, 2), 32, 4, 11), ((1, 1, 1, 1), 32, 2, 11),
                ((1, 2, 1, 1), 32, 4, 11), ((1, 1, 2, 2), 32, 2, 11)]


@pytest.mark.parametrize("kernel", GEMM_KERNELS)
@pytest.mark.parametrize("shape,trans_b", [
    ((1, 16, 1, 16), False), ((1, 17, 33, 19), False),              # one k; K that ends inside a vector
    ((1, 130, 321, 135), False), ((1, 65, 96, 129), True),          # edges along M and N; whole steps, rows of B^T
    ((1, 70, 90, 45), True), ((1, 64, 1023, 64), False),            # groups with fewer steps than others
    ((6, 23, 651, 1), False), ((1, 70, 330, 2), False), ((3, 100, 320, 1), False),      # rows of B of one load and less
    ((3, 40, 70, 37), False), ((2, 37, 100, 41), True),             # batches, whose rows end where the next product's begin
])
def test_gemm(shape, trans_b, kernel):
    from flextensor_amd.measure import seeded_inputs
    plan, bufs = split_plan(gemm_of(trans_b), shape, *kernel)
    a, b = seeded_inputs(bufs, seed=sum(shape))
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert rel(run(plan, bufs, [a, b]), np.matmul(a64, np.swapaxes(b64, -1, -2) if trans_b else b64)) <= TOL


@pytest.mark.parametrize("kernel", [((2, 1, 2, 1), 16, 2, 10), ((2, 2, 4, 1), 32, 1, 9), ((4, 1, 2, 2), 16, 1, 9),
                                    ((1, 2, 1, 2), 32, 4, 11), ((1, 1, 1, 1), 32, 2, 11), ((1, 1, 1, 3), 32, 4, 11)])
@pytest.mark.parametrize("shape,bias", [
    # padding on every side, windows of 1 to 25 taps, strides, dilation, channel groups, a window that covers the image
    ((2, 5, 9, 7, 19, 3, 1, 1, 1, 1), True), ((1, 16, 14, 14, 33, 3, 2, 1, 1, 1), False), ((3, 37, 8, 11, 20, 1, 1, 0, 1, 1), True),
    ((2, 24, 13, 13, 24, 3, 1, 2, 2, 2), False), ((1, 3, 15, 15, 40, 5, 1, 2, 1, 1), True), ((5, 32, 3, 3, 17, 3, 1, 0, 1, 1), True),
    ((2, 64, 7, 7, 70, 1, 2, 0, 1, 1), False), ((3, 32, 8, 8, 64, 1, 1, 0, 1, 1), False),
    # windows whose last rows are padding for every pixel, and lie behind the image's end
    ((1, 8, 5, 5, 40, 3, 1, 6, 6, 1), False), ((1, 20, 10, 10, 33, 3, 1, 12, 12, 1), True), ((1, 40, 1, 1, 70, 5, 1, 2, 1, 1), False)])
def test_conv2d(oracle, shape, bias, kernel):
    from flextensor_amd.measure import seeded_inputs
    plan, bufs = split_plan(conv_of(bias), shape, *kernel)
    host = seeded_inputs(bufs, seed=sum(shape))
    ref = oracle.conv2d_nchw_c(host[0], host[1], *shape[6:])
    if bias:
        ref = oracle.bias_add_nchw_np(ref, host[2])
    assert rel(run(plan, bufs, host), ref) <= TOL


@pytest.mark.parametrize("kernel", [((2, 2, 4, 1), 16, 2, 9), ((1, 1, 1, 1), 32, 2, 11)])
@pytest.mark.parametrize("xcd", [0, 1])
def test_image_by_image_and_order_of_the_workgroups(oracle, kernel, xcd):
    from flextensor_amd.measure import seeded_inputs
    shape = (3, 40, 9, 11, 70, 1, 1, 0, 1, 1)
    plan, bufs = split_plan(conv_of(True), shape, *kernel, xcd=xcd, by_image=True)
    assert plan.specs[-1].defines["IMAGES"] == 3 and plan.specs[-1].defines["XCD_REMAP"] == xcd
    host = seeded_inputs(bufs, seed=7)
    ref = oracle.bias_add_nchw_np(oracle.conv2d_nchw_c(host[0], host[1], *shape[6:]), host[2])
    assert rel(run(plan, bufs, host), ref) <= TOL


# factors of the two operands: numbers of every size that float32 holds, results that no sum of scaled parts holds
NUMBERS = {"small": (1e-34, 1e10), "denormal": (1e-41, 1e38), "large": (7e37, 1e-3), "large sums": (1e15, 1e15), "zero": (0.0, 1.0)}
# factors along k of (weights or A, columns of B), and along the columns: an ordinary number hides none that is below 2^-110
MIXED = {"columns": ((1e20, 1e20), (1.0, 1.0), (1.0, 2.0 ** -120)), "small terms": ((1.0, 2.0 ** -120), (0.0, 2.0 ** 100), (1.0, 1.0)),
         "terms of two sizes": ((2.0 ** -118, 2.0 ** 60), (2.0 ** 70, 2.0 ** -124), (1.0, 1.0)),
         "denormal terms": ((2.0 ** 90, 1.0), (2.0 ** -140, 2.0 ** -45), (1.0, 1.0))}


def in_turn(factors, count):
    return np.resize(np.asarray(factors), count)


@pytest.mark.parametrize("kernel", [((2, 2, 4, 1), 16, 2, 10), ((2, 1, 2, 1), 32, 1, 9), ((1, 2, 1, 2), 32, 4, 11), ((1, 1, 1, 1), 32, 2, 11)])
@pytest.mark.parametrize("what", sorted(NUMBERS) + sorted(MIXED) + ["infinite", "nan", "scattered"])
@pytest.mark.parametrize("func,args", [(gemm_of(False), (1, 100, 150, 90)), (gemm_of(True), (1, 100, 150, 90)),
                                       (conv_of(False), (2, 20, 13, 11, 70, 3, 1, 1, 1, 1))])
def test_numbers_without_three_parts(func, args, what, kernel):
    """Operands of one size, at both ends of the range; ordinary numbers beside those whose low parts bf16 does not hold, in
    neighbouring columns, along k where the other operand is zero, and scattered; single infinities and NaNs. Every result that float32
    holds is off by no more than TOL of the sum of its own products' magnitudes, the others are the infinities and NaNs
    that the products give."""
    import torch
    from flextensor_amd.measure import seeded_inputs
    plan, bufs = split_plan(func, args, *kernel)
    conv, trans_b = len(args) == 10, bool(func(*args)[0][0].attrs.get("transposeB"))
    host = [x.astype(np.float64) for x in seeded_inputs(bufs, seed=11)]
    if what in NUMBERS:
        host = [x * s for x, s in zip(host, NUMBERS[what])]
    elif what in MIXED:
        fa, fb, fn = MIXED[what]
        if conv:            # the weights' k are channels, columns are pixels: every other one of a row of the image
            host[1] *= in_turn(fa, 20)[:, None, None]
            host[0] *= in_turn(fb, 20)[:, None, None] * in_turn(fn, 11)
        else:
            host[0] *= in_turn(fa, 150)
            host[1] *= (in_turn(fb, 150)[:, None] * in_turn(fn, 90)).T if trans_b else in_turn(fb, 150)[:, None] * in_turn(fn, 90)
    elif what == "scattered":
        host[0].ravel()[::7] *= 1e-36
        host[1].ravel()[::11] *= 1e30           # 11 divides no row: every column has them at k of its own
    host = [x.astype(np.float32) for x in host]
    if what in ("infinite", "nan"):
        host[0].ravel()[host[0].size // 2] = np.inf if what == "infinite" else np.nan
    x, y = [torch.from_numpy(h).double() for h in host]

    def product(x, y):
        if conv:
            return torch.stack([y.reshape(70, -1) @ c for c in torch.nn.functional.unfold(x, 3, padding=1)]).reshape(bufs[-1].shape).numpy()
        return (x @ (y.T if trans_b else y)).numpy()

    with np.errstate(all="ignore"):
        held, most = product(x, y).astype(np.float32).astype(np.float64), product(x.abs(), y.abs())
    out = run(plan, bufs, host).astype(np.float64)
    finite = np.isfinite(held)
    assert np.array_equal(out[~finite], held[~finite], equal_nan=True)
    # and half of the least float32 number for each group of K that is rounded to one
    assert np.all(np.abs(out[finite] - held[finite]) <= TOL * most[finite] + 2.0 ** -147)


@pytest.mark.parametrize("shape,trans_b,kernel", [
    ((1, 128, 2304, 128), False, ((2, 2, 4, 1), 16, 1, 9)), ((1, 300, 1300, 200), True, ((2, 2, 4, 1), 32, 1, 9)),
    # four blocks of a wavefront share one set of accumulators: with K divided by at least twice the default's groups
    ((1, 1000, 1531, 777), False, ((1, 2, 1, 2), 32, 4, 11)), ((1, 700, 2000, 900), True, ((1, 2, 1, 2), 32, 4, 11)),
    ((1, 1024, 1024, 1024), False, ((1, 2, 1, 2), 32, 8, 11)), ((1, 320, 4096, 520), False, ((1, 1, 1, 2), 32, 8, 11))])
def test_more_exact_than_fp32_products(shape, trans_b, kernel, monkeypatch):
    """Nearer to float64 than the kernel the default takes where products are fp32; bell-shaped operands of both signs."""
    from flextensor_amd.scheduler import schedule_with_config_ops
    from flextensor_amd.templates import gfx950
    from flextensor_amd.utils import Config
    func = gemm_of(trans_b)
    plan, bufs = split_plan(func, shape, *kernel)
    monkeypatch.setattr(gfx950, "_or_split", lambda view, cfg, call: cfg)
    other, _ = schedule_with_config_ops(*func(*shape), Config([], None))
    spec = other.specs[-1]
    assert "SPLIT" not in spec.defines and (kernel[0] != (1, 2, 1, 2) or kernel[2] >= 2 * spec.defines.get("WAVES_K", 1))
    rng = np.random.default_rng(5)
    a, b = (rng.standard_normal([int(e) for e in x.shape]).astype(np.float32) for x in bufs[:2])
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    ref = a64 @ (b64.T if trans_b else b64)
    mine, theirs = (np.linalg.norm(run(p, bufs, [a, b]) - ref) for p in (plan, other))
    assert mine < theirs


@pytest.mark.parametrize("func,args,kernel", [
    (gemm_of(True), (1, 1500, 1000, 3001), ((2, 2, 4, 1), 32, 1, 9)), (gemm_of(False), (1, 1000, 1531, 777), ((1, 2, 1, 2), 32, 4, 11)),
    (gemm_of(False), (1, 1500, 1000, 3001), ((4, 1, 2, 1), 32, 2, 9)), (conv_of(False), (16, 128, 57, 57, 256, 3, 2, 1, 1, 1), ((4, 1, 2, 1), 32, 1, 9))])
def test_infinities_do_not_slow_a_call_down_by_much(func, args, kernel):
    """With an infinity in every row of A (the weights) all products are made again, by fp32 MFMAs, which are 2.7 times as
    long as the bf16 ones: at most four times an ordinary call (measured 1.5 to 2.6 times)."""
    import torch
    from flextensor_amd.plan import build
    plan, bufs = split_plan(func, args, *kernel)
    call = build(plan, bufs, "rocm")
    data = [torch.randn([int(e) for e in x.shape], device="cuda") for x in bufs]

    def shortest():
        times = []
        for _ in range(8):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(30):
                call(*data)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    ordinary = shortest()
    rows = data[1 if len(args) == 10 else 0]
    rows.view(rows.shape[0], -1)[:, 3] = float("inf")
    assert shortest() <= 4 * ordinary
    call.close()


def test_several_streams_and_capture():
    """The plan owns no workspace: calls on two streams at once, and replays of a captured graph, each against the eager result."""
    import torch
    from flextensor_amd.measure import seeded_inputs
    from flextensor_amd.plan import build
    plan, bufs = split_plan(gemm_of(False), (1, 200, 300, 150), (2, 2, 4, 1), 16, 2, 10)
    assert not plan.specs[-1].workspace
    func = build(plan, bufs, "rocm")
    sets = [[torch.from_numpy(x).cuda() for x in seeded_inputs(bufs, seed=s)] + [torch.zeros(200, 150, device="cuda")] for s in (1, 2)]
    eager = []
    for s in sets:
        func(*s)
        eager.append(s[2].clone())
        s[2].zero_()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in sets]
    for stream, s in zip(streams, sets):
        with torch.cuda.stream(stream):
            for _ in range(10):
                func(*s)
    torch.cuda.synchronize()
    assert all(torch.equal(s[2], e) for s, e in zip(sets, eager))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        func(*sets[0])
    for _ in range(3):
        sets[0][2].zero_()
        func(*sets[1])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(sets[0][2], eager[0]) and torch.equal(sets[1][2], eager[1])
    func.close()
