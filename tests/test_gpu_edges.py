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
    tails inside a 16-byte chunk, and operands that begin at an odd address themselves."""
    import torch
    from flextensor_amd.task import gemm_int8
    f, _ = build_default(gemm_int8, "gemm", (m, k, n))
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    a, b = [rng.integers(-128, 128, size=s, dtype=np.int8) for s in ((m, k), (n, k))]
    want = oracle.gemm_i8_c(a, b)
    for oa, ob in ((0, 0), (1, 3), (2, 1)) if k % 4 else ((0, 0),):
        c = torch.full((m, n), -7, dtype=torch.int32, device="cuda")
        f(placed(a, oa), placed(b, ob), c)
        assert np.array_equal(c.cpu().numpy(), want), (oa, ob)
