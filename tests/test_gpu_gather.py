"""The gathered operand where K tiles cut windows: padding bits and scalar or per-lane taps, against the CPU oracle:
max|diff| / max|ref| <= 1e-5."""
import numpy as np
import pytest

from test_gpu_direct import conv_of, rel, run

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.mark.parametrize("tile,bk,depth,groups", [
    ((4, 1, 4, 1, 16), 32, 8, 1),         # a wavefront's 64 elements are one row of the tile: scalars
    ((4, 2, 4, 1, 16), 32, 3, 1),         # the same through registers
    ((4, 1, 2, 1, 16), 32, 3, 2),         # two rows, K divided
    ((1, 1, 1, 1, 16), 16, 2, 4),         # four rows, one pixel a thread
    ((2, 1, 2, 1, 16), 32, 5, 1),         # two rows, straight into LDS
    ((1, 2, 4, 4, 16), 32, 3, 1),         # all wavefronts load from one row: its number is known when compiled
    ((1, 1, 1, 8, 16), 16, 2, 2),         # rows of two elements a thread
])
@pytest.mark.parametrize("shape,bias", [
    ((2, 24, 9, 7, 19, 3, 1, 1, 1, 1), True),       # columns and rows that end inside the tile
    ((3, 9, 13, 11, 40, 5, 2, 2, 1, 1), False),     # 25 taps
    ((1, 64, 8, 8, 70, 2, 2, 0, 1, 1), False),      # nothing to mask
    ((2, 48, 10, 10, 32, 3, 1, 2, 2, 2), True),     # dilation, channel groups
    ((2, 11, 12, 12, 16, 7, 1, 3, 1, 1), False),    # 49 taps: more than a word's bits
])
def test_gather(oracle, shape, bias, tile, bk, depth, groups):
    from flextensor_amd.measure import seeded_inputs
    from flextensor_amd.scheduler import flatten_graph, schedule_with_config_ops
    from flextensor_amd.templates import gfx950
    from flextensor_amd.utils import Config, ceil_div
    ops, bufs = conv_of(bias)(*shape)
    configs = []
    for op in flatten_graph(ops)[0]:
        cfg = gfx950._empty_config()
        if op.kind == "conv2d_nchw":
            (wm, rm, wn, rn, mf), view = tile, gfx950.GemmView(op)
            cfg["spatial"] = [[ceil_div(view.M, mf * wm * rm), wm, rm, mf], [ceil_div(view.N, mf * wn * rn), wn, rn, mf]]
            cfg["reduce"], cfg["unroll"] = [[groups, ceil_div(view.K, bk * groups), bk]], [[depth, 1]]
            cfg["fuse"], cfg["reorder"] = [[4]], [[1, 1 if groups > 1 else 0, 0]]
        configs.append(cfg)
    plan, bufs = schedule_with_config_ops(ops, bufs, Config(configs, None))
    assert plan.specs[-1].template == "igemm_f32.hip"
    host = seeded_inputs(bufs, seed=sum(shape))
    ref = oracle.conv2d_nchw_c(host[0], host[1], *shape[6:])
    if bias:
        ref = oracle.bias_add_nchw_np(ref, host[2])
    assert rel(run(plan, bufs, host), ref) <= TOL
