"""Sizes at which the kernels' tiles, vectors and dispatch rules have their edges, on the default plans,
against the CPU oracle: int32 results are identical, fp32 within max|diff| / max|ref| <= 1e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def build_default(func, category, args):
    from flextensor_amd.plan import build as build_plan
    from flextensor_amd.scheduler import schedule_with_config
    from flextensor_amd.task import Task, register
    from flextensor_amd.utils import Config
    register(func, category, "edges", args, "rocm", 0)
    s, bufs = schedule_with_config(Task(category, "edges", None, args, "rocm", 0).key, Config([], None))
    return build_plan(s, bufs, "rocm"), bufs


def gemm_of(trans_b, batch=0):
    """fp32 GEMM task function (M, K, N) -> (ops, bufs), B stored [N][K] with ``trans_b``."""
    def func(m, k, n):
        from flextensor_amd import nn
        from flextensor_amd.te import placeholder
        lead = (batch,) if batch else ()
        a, b = placeholder(lead + (m, k), name="A"), placeholder(lead + ((n, k) if trans_b else (k, n)), name="B")
        c = (nn.batch_gemm if batch else nn.gemm)(a, b, transposeB=trans_b)
        return [c.op], [a, b, c]
    return func


def build_config(func, args, config):
    from flextensor_amd.plan import build as build_plan
    from flextensor_amd.scheduler import schedule_with_config_ops
    from flextensor_amd.utils import Config
    ops, bufs = func(*args)
    s, bufs = schedule_with_config_ops(ops, bufs, Config([config] if config else [], None))
    return build_plan(s, bufs, "rocm"), bufs


def gemm_config(m, k, n, wm, wn, rep, mfma, bk, depth, groups=1):
    cd = lambda a, b: -(-a // b)
    return dict(spatial=[[cd(m, wm * rep * mfma), wm, rep, mfma], [cd(n, wn * rep * mfma), wn, rep, mfma]],
                reduce=[[groups, cd(k, groups * bk), bk]], unroll=[[depth, 1]], fuse=[[4]],
                reorder=[[1, 1 if groups > 1 else 0, 0]], inline=[], merge=[], special=[])


def close(got, want):
    """The fp32 bound of the product's own gate: max|diff| / max|ref| <= 1e-5."""
    return float(np.max(np.abs(got - want)) / np.max(np.abs(want))) <= 1e-5


def placed(array, offset=0):
    """A contiguous device tensor of ``array`` that begins ``offset`` elements behind an allocation's start."""
    import torch
    flat = torch.empty(array.size + offset, dtype=torch.from_numpy(array).dtype, device="cuda")
    t = flat[offset:].view(array.shape)
    t.copy_(torch.from_numpy(array))
    return t


@pytest.mark.parametrize("m,k,n", [
    (1, 1, 1), (5, 3, 2), (33, 15, 70), (33, 17, 70), (70, 61, 33), (64, 66, 64), (65, 127, 63), (40, 129, 300),
    (130, 255, 131), (130, 260, 131), (129, 1027, 257), (700, 390, 1100),      # 128x128 tiles through registers
    (64, 2080, 192), (32, 1000, 32), (520, 144, 514), (1030, 112, 1026)])
def test_int8_rows_at_any_byte(oracle, m, k, n):
    """K of every alignment (16-byte rows straight into LDS, dword-aligned rows, rows that begin at any byte),
    tails inside a 16-byte chunk, and operands that begin at an odd address themselves (copied where the rows are whole
    dwords) or at a dword that begins no 16 bytes."""
    import torch
    from flextensor_amd.task import gemm_int8
    f, _ = build_default(gemm_int8, "gemm", (m, k, n))
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    a, b = [rng.integers(-128, 128, size=s, dtype=np.int8) for s in ((m, k), (n, k))]
    want = oracle.gemm_i8_c(a, b)
    for oa, ob in ((0, 0), (1, 3), (2, 1), (4, 8)):
        c = torch.full((m, n), -7, dtype=torch.int32, device="cuda")
        f(placed(a, oa), placed(b, ob), c)
        assert np.array_equal(c.cpu().numpy(), want), (oa, ob)


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("m,k,n", [
    (1, 1, 1), (5, 3, 2), (3, 5, 4), (17, 33, 19), (64, 30, 65), (33, 17, 70), (130, 130, 258), (127, 129, 126),
    (30, 999, 611), (201, 77, 131), (513, 67, 259), (1030, 35, 1027)])
def test_fp32_rows_of_any_length(oracle, m, k, n, trans_b):
    """Default plans at extents that are no multiples of a vector, a tile or a k block."""
    import torch
    rng = np.random.default_rng(m + 3 * k + 7 * n)
    a, b = [rng.uniform(-1, 1, s).astype(np.float32) for s in ((m, k), (k, n))]
    f, _ = build_config(gemm_of(trans_b), (m, k, n), None)
    c = torch.full((m, n), -7.0, device="cuda")
    f(placed(a, 1), placed(np.ascontiguousarray(b.T) if trans_b else b, 3), c)
    assert close(c.cpu().numpy(), oracle.gemm_f32_c(a, b))


@pytest.mark.parametrize("depth,bk,mfma,groups", [(1, 16, 16, 1), (2, 16, 32, 2), (3, 32, 16, 1), (4, 16, 16, 1), (5, 32, 16, 1),
                                                  (5, 32, 32, 2), (6, 32, 16, 1), (7, 32, 16, 1), (8, 32, 16, 1), (8, 32, 32, 1)])
@pytest.mark.parametrize("k", [61, 62, 63, 109, 127])
@pytest.mark.parametrize("trans_b", [False, True])
def test_what_a_row_takes_from_the_next_one_does_not_count(depth, bk, mfma, groups, k, trans_b):
    """The last vector of a row along K runs into the next row on every pipeline: an infinity or a NaN that
    begins that row must not reach the row before it (0 * inf is not 0)."""
    import torch
    m, n = 70, 66
    rng = np.random.default_rng(k)
    a, b = [rng.uniform(-1, 1, s).astype(np.float32) for s in ((m, k), (k, n))]
    want = a.astype(np.float64) @ b.astype(np.float64)
    a[5, :3] = [np.inf, np.nan, np.inf]
    f, _ = build_config(gemm_of(trans_b), (m, k, n), gemm_config(m, k, n, 2, 2, 1, mfma, bk, depth, groups))
    for spoil_b in (False, True) if trans_b else (False,):
        bb = b.copy()
        if spoil_b:
            bb[:3, 9] = [np.nan, np.inf, np.inf]
        c = torch.full((m, n), -7.0, device="cuda")
        f(placed(a), placed(np.ascontiguousarray(bb.T) if trans_b else bb), c)
        got = c.cpu().numpy()
        rows, cols = np.arange(m) != 5, np.arange(n) != (9 if spoil_b else -1)
        assert not np.isfinite(got[5]).any()
        assert close(got[rows][:, cols], want[rows][:, cols]), (depth, k, spoil_b)


@pytest.mark.parametrize("b,m,k,n,trans_b", [(3, 49, 33, 50, True), (5, 17, 31, 18, False), (70, 197, 64, 31, True),
                                             (9, 128, 129, 127, False)])
def test_batched_products_of_odd_extents(b, m, k, n, trans_b):
    import torch
    rng = np.random.default_rng(b + m)
    x, y = [rng.uniform(-1, 1, s).astype(np.float32) for s in ((b, m, k), (b, k, n))]
    f, _ = build_config(gemm_of(trans_b, batch=b), (m, k, n), None)
    c = torch.full((b, m, n), -7.0, device="cuda")
    f(placed(x), placed(np.ascontiguousarray(y.transpose(0, 2, 1)) if trans_b else y), c)
    assert close(c.cpu().numpy(), np.matmul(x.astype(np.float64), y.astype(np.float64)))


@pytest.mark.parametrize("m,k,groups", [(1, 257, 2), (3, 259, 4), (1, 385, 2)])
def test_int8_tiles_wholly_behind_k(oracle, m, k, groups):
    """K divided so that the last group's last tiles lie behind K altogether, over operands of few rows: the
    tile's scalar offset would be beyond the buffer."""
    import torch
    from flextensor_amd.task import gemm_int8
    n, bk = 33, 128
    config = dict(spatial=[[1, 1, 1, 16], [3, 1, 1, 16]], reduce=[[groups, -(-k // (groups * bk)), bk]], unroll=[[2, 1]],
                  fuse=[[4]], reorder=[[1, 1, 0]], inline=[], merge=[], special=[])
    f, _ = build_config(gemm_int8, (m, k, n), config)
    rng = np.random.default_rng(k)
    a, b = [rng.integers(-128, 128, size=s, dtype=np.int8) for s in ((m, k), (n, k))]
    c = torch.full((m, n), -7, dtype=torch.int32, device="cuda")
    f(placed(a), placed(b), c)
    assert np.array_equal(c.cpu().numpy(), oracle.gemm_i8_c(a, b))


@pytest.mark.parametrize("depth", [3, 5, 8])
@pytest.mark.parametrize("trans_b", [False, True])
def test_fp32_tiles_wholly_behind_k(oracle, depth, trans_b):
    import torch
    m, k, n, groups, bk = 1, 416, 64, 4, 32        # 13 tiles of K for 4 groups of 4
    cfg = gemm_config(m, k, n, 1, 1, 1, 16, bk, depth, groups)
    cfg["spatial"] = [[1, 1, 1, 16], [1, 1, 4, 16]]
    f, _ = build_config(gemm_of(trans_b), (m, k, n), cfg)
    rng = np.random.default_rng(k)
    a, b = [rng.uniform(-1, 1, s).astype(np.float32) for s in ((m, k), (k, n))]
    c = torch.full((m, n), -7.0, device="cuda")
    f(placed(a), placed(np.ascontiguousarray(b.T) if trans_b else b), c)
    assert close(c.cpu().numpy(), oracle.gemm_f32_c(a, b))


# ---- convolutions on the default plan ----------------------------------------------------------------------

@pytest.mark.parametrize("args", [
    # b, c, h, w, o, r, stride, padding, dilation, groups
    (1, 1, 5, 5, 1, 3, 1, 1, 1, 1), (2, 3, 9, 7, 5, 1, 1, 0, 1, 1), (1, 17, 6, 6, 33, 1, 1, 0, 1, 1), (3, 16, 7, 7, 17, 3, 1, 1, 1, 1),
    (4, 64, 7, 7, 64, 3, 2, 1, 1, 1), (9, 78, 8, 8, 69, 3, 2, 1, 1, 1),       # K over wavefront groups, tiles behind K
    (2, 223, 13, 15, 56, 3, 1, 1, 1, 1), (11, 152, 7, 17, 30, 3, 2, 1, 1, 1),
    (8, 130, 29, 31, 130, 3, 1, 1, 1, 1), (16, 129, 33, 33, 255, 3, 2, 1, 1, 1),    # whole windows, ragged K and edges
    (5, 33, 57, 61, 150, 1, 1, 0, 1, 1), (10, 17, 94, 94, 67, 1, 1, 0, 1, 1), (4, 139, 41, 12, 235, 1, 2, 0, 1, 1),
    (2, 12, 15, 17, 20, 5, 1, 2, 1, 1), (2, 24, 15, 17, 36, 3, 1, 2, 2, 2), (1, 3, 40, 40, 24, 7, 2, 3, 1, 1)])
def test_convolutions_of_any_extent(oracle, args):
    """Default plans: pixels and windows, strides, dilation and groups, K that no K tile divides; the image lies
    between NaN so that a gather from beyond it would show."""
    import torch
    from flextensor_amd.task import conv2d
    b, c, h, w, o, r, st, pd, dl, gr = args
    rng = np.random.default_rng(sum(args))
    x, wt = rng.standard_normal((b, c, h, w)).astype(np.float32), rng.standard_normal((o, c // gr, r, r)).astype(np.float32)
    f, bufs = build_default(conv2d, "conv2d", args)
    flat = torch.full((x.size + 64,), float("nan"), device="cuda")
    flat[33:33 + x.size] = torch.from_numpy(x).cuda().flatten()
    y = torch.full(tuple(int(e) for e in bufs[-1].shape), -7.0, device="cuda")
    f(flat[33:33 + x.size].view(x.shape), placed(wt, 1), y)
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(wt).double(), None, st, pd, dl, gr).numpy()
    assert close(y.cpu().numpy(), want)


# ---- depthwise rows of any length --------------------------------------------------------------------------

@pytest.mark.parametrize("args", [
    # b, c, h, w, factor, r, stride, padding, dilation
    (2, 5, 57, 57, 1, 3, 1, 1, 1), (1, 3, 7, 7, 1, 3, 1, 1, 1), (2, 4, 9, 10, 1, 5, 1, 2, 1), (2, 4, 11, 13, 1, 3, 2, 1, 1),
    (1, 6, 14, 14, 2, 3, 1, 1, 1), (2, 3, 12, 17, 1, 5, 2, 2, 1), (1, 2, 13, 15, 1, 3, 1, 2, 2), (3, 4, 6, 5, 1, 3, 1, 0, 1),
    (1, 4, 30, 31, 1, 4, 3, 1, 1), (2, 2, 8, 6, 1, 5, 1, 4, 1),
    # images of a few bytes, smaller than a patch row's vectors
    (1, 1, 1, 3, 1, 3, 1, 2, 1), (1, 1, 1, 5, 1, 7, 1, 3, 1), (1, 1, 1, 1, 1, 5, 1, 4, 1), (1, 1, 2, 2, 1, 5, 2, 5, 1)])
def test_depthwise_rows_of_any_length(oracle, args):
    """Row lengths, strides and paddings whose rows are no whole vectors; the image is surrounded by NaN so that
    an element from beyond a row's or the tensor's end would show."""
    import torch
    from flextensor_amd.task import depthwise_conv2d
    b, c, h, w, fa, r, st, pd, dl = args
    rng = np.random.default_rng(sum(args))
    x, wt = rng.standard_normal((b, c, h, w)).astype(np.float32), rng.standard_normal((c, fa, r, r)).astype(np.float32)
    want = oracle.depthwise_nchw_c(x, wt, st, pd, dl)
    f, _ = build_default(depthwise_conv2d, "conv2d", args)
    flat = torch.full((x.size + 64,), float("nan"), device="cuda")
    flat[33:33 + x.size] = torch.from_numpy(x).cuda().flatten()
    y = torch.full((want.size + 64,), -7.0, device="cuda")
    f(flat[33:33 + x.size].view(x.shape), placed(wt, 1), y[31:31 + want.size].view(want.shape))
    got = y.cpu().numpy()
    assert close(got[31:31 + want.size].reshape(want.shape), want)
    assert (got[:31] == -7).all() and (got[31 + want.size:] == -7).all()


# ---- the native call ----------------------------------------------------------------------------------------

def test_a_plan_refuses_what_it_does_not_take():
    import torch
    f, _ = build_config(gemm_of(False), (16, 8, 12), None)
    a, b, c = torch.randn(16, 8, device="cuda"), torch.randn(8, 12, device="cuda"), torch.empty(16, 12, device="cuda")
    f(a, b, c)
    assert torch.allclose(c, a @ b, atol=1e-4)
    for bad in ((a, b), (a, b, c, c), (a.t(), b, c), (a.double(), b, c), (a.cpu(), b, c), (torch.randn(8, 16, device="cuda").t(), b, c),
                (a, torch.randn(8, 24, device="cuda")[:, ::2], c)):
        with pytest.raises(ValueError):
            f(*bad)
    f(torch.nn.Parameter(a), b, c)


def test_a_plan_called_by_threads_on_streams():
    import threading
    import torch
    f, _ = build_config(gemm_of(False), (96, 64, 80), None)
    sets = [[torch.randn(96, 64, device="cuda"), torch.randn(64, 80, device="cuda"), torch.empty(96, 80, device="cuda")] for _ in range(4)]
    streams = [torch.cuda.Stream() for _ in sets]
    torch.cuda.synchronize()

    def work(ts, stream):
        with torch.cuda.stream(stream):
            for _ in range(200):
                f(*ts)

    threads = [threading.Thread(target=work, args=p) for p in zip(sets, streams)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for a, b, c in sets:
        assert torch.allclose(c, a @ b, atol=1e-4)


@pytest.mark.parametrize("native", [True, False])
def test_a_call_runs_on_the_current_stream(native):
    """Each stream is busy for milliseconds before it writes the operand the call reads: a launch on any other
    stream would read the operand as it was, and its result would be taken before it is there."""
    import threading
    import torch
    f, _ = build_config(gemm_of(False), (96, 64, 80), None)
    if not native:
        f._native = None
    busy = torch.randn(2048, 2048, device="cuda")
    sets = [[torch.randn(96, 64, device="cuda"), torch.randn(64, 80, device="cuda"),
             torch.zeros(96, 64, device="cuda"), torch.zeros(96, 80, device="cuda")] for _ in range(3)]
    streams, results = [torch.cuda.Stream() for _ in sets], [None] * len(sets)
    busy @ busy
    torch.cuda.synchronize()

    def work(i):
        new, b, a, c = sets[i]
        with torch.cuda.stream(streams[i]):
            for _ in range(20):
                busy @ busy
            a.copy_(new)
            f(a, b, c)
            results[i] = c.clone()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sets))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for (new, b, a, c), got in zip(sets, results):
        want = new.double() @ b.double()
        assert close(got.cpu().numpy(), want.cpu().numpy())


@pytest.mark.parametrize("n", [15, 22])
def test_a_plan_of_many_operators(n):
    """More buffers and launches than a call keeps on its stack: the native call and the general one agree, and with
    the product in float64 to n stages of |fl(xW) - xW| <= K u |x||W| (2-norms; W orthogonal, | |W| | <= sqrt(K))."""
    import torch
    from test_host_scheduler import chain_of_gemms
    m, k = 20, 24
    f, _ = build_config(lambda: chain_of_gemms(n, m, k), (), None)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    ws = [np.linalg.qr(rng.standard_normal((k, k)))[0].astype(np.float32) for _ in range(n)]
    tensors = [placed(a) for a in [x] + ws]
    outs = [torch.full((m, k), -7.0, device="cuda") for _ in range(2)]
    assert f._native(*tensors, outs[0]) is True
    f._native = None
    f(*tensors, outs[1])
    assert torch.equal(outs[0], outs[1])
    want = x.astype(np.float64)
    for w in ws:
        want = want @ w
    assert np.linalg.norm(outs[0].cpu().numpy() - want) <= n * k * k ** 0.5 * 2.0 ** -24 * np.linalg.norm(want)
