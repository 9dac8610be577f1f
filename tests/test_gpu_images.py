"""1x1 layers image by image, against the CPU oracle: max|diff| / max|ref| <= 1e-5."""
import numpy as np
import pytest

from test_gpu_direct import conv_of, rel, run

pytestmark = pytest.mark.gpu
TOL = 1e-5


def image_plan(shape, bias, tile, bk, depth, groups):
    from flextensor_amd.scheduler import flatten_graph, schedule_with_config_ops
    from flextensor_amd.templates import gfx950
    from flextensor_amd.utils import Config, ceil_div
    ops, bufs = conv_of(bias)(*shape)
    configs = []
    for op in flatten_graph(ops)[0]:
        cfg = gfx950._empty_config()
        if op.kind == "conv2d_nchw":
            (wm, rm, wn, rn, mf), view = tile, gfx950.GemmView(op).by_image()
            cfg["spatial"] = [[ceil_div(view.M, mf * wm * rm), wm, rm, mf], [ceil_div(view.N, mf * wn * rn), wn, rn, mf]]
            cfg["reduce"], cfg["unroll"] = [[groups, ceil_div(view.K, bk * groups), bk]], [[depth, 1]]
            cfg["fuse"], cfg["reorder"] = [[4]], [[1, 1 if groups > 1 else 0, 0, 2]]
        configs.append(cfg)
    return schedule_with_config_ops(ops, bufs, Config(configs, None))


@pytest.mark.parametrize("tile,bk,depth,groups", [
    ((2, 1, 4, 1, 16), 64, 8, 1), ((1, 1, 4, 1, 16), 32, 3, 2), ((2, 1, 2, 1, 16), 32, 5, 1), ((1, 1, 1, 1, 16), 16, 2, 4)])
@pytest.mark.parametrize("shape,bias", [
    ((3, 60, 9, 7, 35, 1, 1, 0, 1, 1), True),       # 63 pixels: rows that are no whole vectors, K that ends inside a tile
    ((2, 125, 5, 13, 17, 1, 1, 0, 1, 1), False),    # 65 pixels, K no multiple of 4: the next image's rows lie behind K
    ((5, 64, 16, 8, 64, 1, 1, 0, 1, 1), True),      # whole tiles
    ((1, 61, 3, 1, 16, 1, 1, 0, 1, 1), True),       # one image of fewer pixels than a vector
])
def test_by_image(oracle, shape, bias, tile, bk, depth, groups):
    from flextensor_amd.measure import seeded_inputs
    plan, bufs = image_plan(shape, bias, tile, bk, depth, groups)
    assert plan.specs[-1].defines["IMAGES"] == shape[0]
    host = seeded_inputs(bufs, seed=sum(shape))
    host[0][-1, :, 0, 0] = np.nan                   # stays in its image and pixel
    ref = oracle.conv2d_nchw_c(np.nan_to_num(host[0]), host[1], *shape[6:])
    if bias:
        ref = oracle.bias_add_nchw_np(ref, host[2])
    out = run(plan, bufs, host)
    assert np.isnan(out[-1, :, 0, 0]).all() and np.isnan(out).sum() == shape[4]
    assert rel(np.where(np.isnan(out), ref, out), ref) <= TOL


def test_defaults_and_what_is_refused(oracle):
    from flextensor_amd.measure import seeded_inputs
    from flextensor_amd.scheduler import schedule_with_config_ops
    from flextensor_amd.templates import gfx950
    from flextensor_amd.utils import Config
    shape = (2, 240, 35, 35, 160, 1, 1, 0, 1, 1)
    ops, bufs = conv_of(True)(*shape)
    plan, _ = schedule_with_config_ops(ops, bufs, Config([], None))
    assert plan.specs[-1].defines["IMAGES"] == 2
    host = seeded_inputs(bufs, seed=1)
    ref = oracle.bias_add_nchw_np(oracle.conv2d_nchw_c(host[0], host[1], 1, 0, 1, 1), host[2])
    assert rel(run(plan, bufs, host), ref) <= TOL
    for other in ((2, 8, 14, 14, 8, 3, 1, 1, 1, 1), (2, 8, 14, 14, 8, 1, 2, 0, 1, 1), (2, 8, 14, 14, 8, 1, 1, 0, 1, 2)):
        ops, bufs = conv_of(False)(*other)
        op = bufs[-1].op
        cfg = gfx950.untuned_config(op)
        assert len(cfg["reorder"][0]) == 3 or cfg["reorder"][0][3] != 2
        cfg["reorder"] = [[1, 0, 0, 2]]
        with pytest.raises(gfx950.InvalidConfig):
            gfx950.lower(op, cfg, None, "out", ["x", "w"])
