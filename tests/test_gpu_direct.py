"""Tiles whose operands go straight into registers (direct_f32.hip), at the sizes where their parts have edges, against
the CPU oracle: max|diff| / max|ref| <= 1e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-5
VARIANTS = (1,)


def direct_plan(func, args, tile, groups, ahead, variant, xcd=1):
    """The plan of the operator's contraction on tiles of (wavefronts, MFMA tiles each) along M and along N, K divided
    among ``groups`` of wavefronts, ``ahead`` k steps on their way."""
    from flextensor_amd.scheduler import flatten_graph, schedule_with_config_ops
    from flextensor_amd.templates import gfx950
    from flextensor_amd.utils import Config, ceil_div
    ops, bufs = func(*args)
    lst, _ = flatten_graph(ops)
    configs = []
    for op in lst:
        cfg = gfx950._empty_config()
        if op.kind in gfx950.GEMM_KINDS:
            (wm, rm, wn, rn), view = tile, gfx950.GemmView(op)
            cfg["spatial"] = [[ceil_div(view.M, 16 * wm * rm), wm, rm, 16], [ceil_div(view.N, 16 * wn * rn), wn, rn, 16]]
            cfg["reduce"], cfg["unroll"] = [[groups, ceil_div(view.K, 32 * groups), 32]], [[ahead, 1]]
            cfg["fuse"], cfg["reorder"] = [[4]], [[xcd, 1 if groups > 1 else 0, 0, variant]]
        configs.append(cfg)
    plan, bufs = schedule_with_config_ops(ops, bufs, Config(configs, None))
    assert [s.template for s in plan.specs] == ["direct_f32.hip"]
    return plan, bufs


def run(plan, bufs, host):
    import torch
    from flextensor_amd.plan import build
    func = build(plan, bufs, "rocm")
    out = torch.full(bufs[-1].shape, -77.0, dtype=torch.float32, device="cuda")
    func(*[torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in host], out)
    torch.cuda.synchronize()
    func.close()
    return out.cpu().numpy()


def rel(a, b):
    return float(np.max(np.abs(a.astype(np.float64) - b)) / np.max(np.abs(b)))


def gemm_of(trans_b):
    def func(nb, m, k, n):
        from flextensor_amd import nn
        from flextensor_amd.te import placeholder
        lead = (nb,) if nb > 1 else ()
        a, b = placeholder(lead + (m, k), name="A"), placeholder(lead + ((n, k) if trans_b else (k, n)), name="B")
        c = (nn.batch_gemm if nb > 1 else nn.gemm)(a, b, transposeB=trans_b)
        return [c.op], [a, b, c]
    return func


def conv_of(bias):
    def func(nb, c, h, w, o, k, stride, pad, dil, groups):
        from flextensor_amd import nn
        from flextensor_amd.te import placeholder
        x, wt = placeholder((nb, c, h, w), name="X"), placeholder((o, c // groups, k, k), name="W")
        bs = placeholder((o,), name="bias") if bias else None
        y = nn.conv2d_nchw(x, wt, bs, stride=stride, padding=pad, dilation=dil, groups=groups)
        return [y.op], [x, wt] + ([bs] if bias else []) + [y]
    return func


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("shape,trans_b,tile,groups,ahead", [
    # edges of the tile along M and N; K that ends with a step, inside one, inside a lane's eight and inside its vectors
    ((1, 16, 32, 16), False, (1, 1, 1, 1), 1, 2), ((1, 17, 33, 19), False, (1, 1, 1, 2), 2, 2),
    ((1, 33, 63, 130), False, (1, 2, 1, 2), 2, 4), ((1, 65, 129, 67), False, (1, 1, 1, 4), 4, 1),
    ((1, 50, 321, 70), True, (1, 3, 1, 3), 8, 2), ((1, 31, 90, 45), True, (1, 4, 1, 4), 1, 1),
    # groups of wavefronts with fewer steps than others and with none
    ((1, 130, 1023, 61), False, (1, 2, 1, 1), 16, 2), ((1, 64, 288, 64), False, (1, 2, 1, 4), 8, 1),
    # several wavefronts side by side; batches, whose rows end where the next product's begin
    ((3, 40, 95, 37), False, (2, 2, 1, 4), 2, 1), ((3, 37, 100, 41), True, (1, 2, 2, 1), 1, 2),
    ((2, 100, 70, 150), False, (1, 3, 2, 4), 2, 1),
])
def test_gemm(oracle, shape, trans_b, tile, groups, ahead, variant):
    from flextensor_amd.measure import seeded_inputs
    plan, bufs = direct_plan(gemm_of(trans_b), shape, tile, groups, ahead, variant)
    a, b = seeded_inputs(bufs, seed=sum(shape))
    out = run(plan, bufs, [a, b])
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert rel(out, np.matmul(a64, np.swapaxes(b64, -1, -2) if trans_b else b64)) <= TOL


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("shape,bias,tile,groups,ahead", [
    # padding on every side, windows of 1 to 25 taps, strides, dilation, channel groups, a window that covers the image
    ((2, 5, 9, 7, 19, 3, 1, 1, 1, 1), True, (1, 1, 1, 1), 2, 2), ((1, 16, 14, 14, 33, 3, 2, 1, 1, 1), False, (1, 2, 1, 2), 4, 2),
    ((3, 37, 8, 11, 20, 1, 1, 0, 1, 1), True, (2, 1, 1, 4), 1, 2), ((2, 24, 13, 13, 24, 3, 1, 2, 2, 2), False, (1, 1, 2, 3), 2, 1),
    ((4, 8, 6, 6, 16, 2, 2, 0, 1, 1), False, (1, 1, 1, 1), 1, 1), ((1, 3, 15, 15, 40, 5, 1, 2, 1, 1), True, (1, 3, 1, 1), 1, 2),
    ((5, 32, 3, 3, 17, 3, 1, 0, 1, 1), True, (1, 4, 1, 4), 8, 1), ((2, 64, 7, 7, 32, 1, 2, 0, 1, 1), False, (1, 2, 1, 4), 2, 1),
])
def test_conv2d(oracle, shape, bias, tile, groups, ahead, variant):
    from flextensor_amd.measure import seeded_inputs
    plan, bufs = direct_plan(conv_of(bias), shape, tile, groups, ahead, variant)
    host = seeded_inputs(bufs, seed=sum(shape))
    ref = oracle.conv2d_nchw_c(host[0], host[1], *shape[6:])
    if bias:
        ref = oracle.bias_add_nchw_np(ref, host[2])
    assert rel(run(plan, bufs, host), ref) <= TOL


@pytest.mark.parametrize("shape,func", [
    ((1, 34, 2149, 1917), gemm_of(False)), ((13, 77, 8, 8, 130, 3, 1, 1, 1, 1), conv_of(False))])
def test_defaults_take_the_tiles_without_lds(oracle, shape, func):
    """Few rows, few pixels: the default plan is one of these, and right; a call on another stream runs there."""
    import torch
    from flextensor_amd.plan import build
    from flextensor_amd.measure import seeded_inputs
    from flextensor_amd.scheduler import schedule_with_config_ops
    from flextensor_amd.utils import Config
    ops, bufs = func(*shape)
    plan, bufs = schedule_with_config_ops(ops, bufs, Config([], None))
    assert [s.template for s in plan.specs] == ["direct_f32.hip"] and not plan.specs[0].workspace
    host = seeded_inputs(bufs, seed=3)
    ref = (np.matmul(host[0].astype(np.float64), host[1].astype(np.float64)) if len(shape) == 4
           else oracle.conv2d_nchw_c(host[0], host[1], *shape[6:]))
    assert rel(run(plan, bufs, host), ref) <= TOL
    # the stream is busy for milliseconds before it writes the operands: a launch elsewhere would read zeros
    func = build(plan, bufs, "rocm")
    busy = torch.randn(2048, 2048, device="cuda")
    new = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in host]
    tensors = [torch.zeros_like(a) for a in new] + [torch.zeros(bufs[-1].shape, device="cuda")]
    stream = torch.cuda.Stream()
    busy @ busy
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(20):
            busy @ busy
        for a, b in zip(tensors, new):
            a.copy_(b)
        func(*tensors)
        got = tensors[-1].clone()
    torch.cuda.synchronize()
    func.close()
    assert rel(got.cpu().numpy(), ref) <= TOL


@pytest.mark.parametrize("xcd", [0, 1])
def test_order_of_the_workgroups(oracle, xcd):
    """The first number of the reorder entry: workgroups in order, or renumbered by XCD. 15 tiles in three batches."""
    from flextensor_amd.measure import seeded_inputs
    plan, bufs = direct_plan(gemm_of(False), (3, 40, 64, 70), (1, 1, 1, 1), 1, 2, 1, xcd)
    assert plan.specs[0].defines["XCD_REMAP"] == xcd and plan.specs[0].grid[0] == 45
    a, b = seeded_inputs(bufs, seed=xcd)
    assert rel(run(plan, bufs, [a, b]), np.matmul(a.astype(np.float64), b.astype(np.float64))) <= TOL
