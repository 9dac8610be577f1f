"""Workgroups renumbered by XCD, at counts that 8 divides and at others: fp32 against sums in float64
(max|diff| / max|ref| <= 1e-5), int8 exactly."""
import numpy as np
import pytest

from test_gpu_direct import conv_of, gemm_of, rel, run

TOL = 1e-5


def plan_of(ops_bufs, kind, tile, bk, parts=1):
    """One wavefront per workgroup and one MFMA block per wavefront; the count of tiles, parts of K included."""
    from flextensor_amd.scheduler import flatten_graph, schedule_with_config_ops
    from flextensor_amd.templates import gfx950
    from flextensor_amd.utils import Config, ceil_div
    ops, bufs = ops_bufs
    configs = []
    for op in flatten_graph(ops)[0]:
        cfg = gfx950._empty_config()
        if op.kind == kind:
            view = gfx950.GemmView(op)
            cfg["spatial"] = [[ceil_div(view.M, tile), 1, 1, tile], [ceil_div(view.N, tile), 1, 1, tile]]
            cfg["reduce"], cfg["unroll"] = [[parts, ceil_div(view.K, bk * parts), bk]], [[2, 1]]
            cfg["fuse"], cfg["reorder"] = [[4]], [[1, 0, 0]]
        configs.append(cfg)
    plan, bufs = schedule_with_config_ops(ops, bufs, Config(configs, None))
    return plan, bufs, plan.specs[-1].grid[0]


ORDER_C = """
int order(int bid, int count, int mode) {
    enum { TILES_N = 1, SPLITK = 1, CG = 1 };
    const int TILES_M = count, MODE = mode;
    (void)MODE;
    %s
    return bid;
}
"""


@pytest.fixture(scope="module")
def orders(tmp_path_factory):
    """{template: its renumbering, compiled for the host}: the lines between #if XCD_REMAP and #endif that turn blockIdx.x
    into a tile (K streaming's, which renumbers whole units, aside)."""
    import ctypes
    import re
    import subprocess
    from flextensor_amd.templates import gfx950
    out = {}
    for template in ("igemm_f32.hip", "gemm_i8.hip", "direct_f32.hip"):
        source = gfx950.template_source(template)
        (lines,) = [x for x in re.findall(r"#if XCD_REMAP\n(.*?)#endif", source, re.S) if "nblk" in x]
        if "int nblk" not in lines:
            lines = re.search(r"const int nblk = [^;]*;", source).group(0) + lines
        folder = tmp_path_factory.mktemp("order")
        (folder / "order.c").write_text(ORDER_C % lines)
        subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(folder / "order.so"), str(folder / "order.c")])
        out[template] = ctypes.CDLL(str(folder / "order.so")).order
    return out


@pytest.mark.parametrize("template", ["igemm_f32.hip", "gemm_i8.hip", "direct_f32.hip"])
@pytest.mark.parametrize("count", list(range(1, 40)) + [196, 255, 256, 257, 263, 1023, 4095])
def test_every_tile_once_and_neighbours_together(orders, template, count):
    """The kernels' renumbering: a permutation that gives XCD x (workgroups x, x + 8, ...) consecutive tiles. Only a
    gathered operand (MODE 1 of igemm_f32.hip) whose grid is ragged and resident at once stays in order."""
    for mode in (0, 1, 2):
        tiles = [orders[template](b, count, mode) for b in range(count)]
        if template == "igemm_f32.hip" and mode == 1 and count % 8 and count <= 256:
            assert tiles == list(range(count))
            continue
        assert sorted(tiles) == list(range(count))
        for x in range(min(8, count)):
            assert np.all(np.diff(tiles[x::8]) == 1)


@pytest.mark.gpu
@pytest.mark.parametrize("nb,tm,tn", [(1, 1, 1), (1, 1, 7), (1, 2, 4), (1, 3, 3), (1, 5, 3), (3, 3, 19), (1, 16, 16), (1, 1, 257)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_gemm(nb, tm, tn, trans_b):
    from flextensor_amd.measure import seeded_inputs
    plan, bufs, grid = plan_of(gemm_of(trans_b)(nb, tm * 16 - 3, 48, tn * 16 - 5), "batch_gemm" if nb > 1 else "gemm", 16, 16)
    assert grid == nb * tm * tn
    a, b = seeded_inputs(bufs, seed=grid)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert rel(run(plan, bufs, [a, b]), np.matmul(a64, np.swapaxes(b64, -1, -2) if trans_b else b64)) <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("shape,tiles", [
    ((1, 16, 9, 12, 20, 3, 1, 1, 1, 1), 14),            # a gathered operand, resident at once: in order
    ((1, 16, 32, 32, 60, 3, 1, 1, 1, 1), 256),
    ((1, 16, 27, 60, 40, 3, 1, 1, 1, 1), 306),          # more than one a unit: renumbered
    ((2, 32, 23, 59, 30, 1, 1, 0, 1, 2), 340),          # groups, pixels of two images in a tile
])
def test_conv2d(oracle, shape, tiles):
    from flextensor_amd.measure import seeded_inputs
    plan, bufs, grid = plan_of(conv_of(False)(*shape), "conv2d_nchw", 16, 16)
    assert grid == tiles
    host = seeded_inputs(bufs, seed=sum(shape))
    assert rel(run(plan, bufs, host), oracle.conv2d_nchw_c(host[0], host[1], *shape[6:])) <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("tm,tn,parts", [(1, 1, 1), (1, 7, 1), (3, 3, 1), (4, 4, 1), (5, 3, 2), (7, 37, 1)])
def test_gemm_int8(tm, tn, parts):
    import torch
    from flextensor_amd import nn
    from flextensor_amd.measure import seeded_inputs
    from flextensor_amd.plan import build
    from flextensor_amd.te import placeholder
    a, b = placeholder((tm * 16 - 3, 256), dtype="int8"), placeholder((tn * 16 - 5, 256), dtype="int8")
    c = nn.gemm_int8(a, b)
    plan, bufs, grid = plan_of(([c.op], [a, b, c]), "gemm_int8", 16, 64, parts)
    assert grid == tm * tn * parts
    x, y = seeded_inputs(bufs, seed=grid)
    func = build(plan, bufs, "rocm")
    out = torch.full(bufs[-1].shape, -77, dtype=torch.int32, device="cuda")
    func(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda(), out)
    torch.cuda.synchronize()
    func.close()
    assert np.array_equal(out.cpu().numpy(), x.astype(np.int32) @ y.astype(np.int32).T)
