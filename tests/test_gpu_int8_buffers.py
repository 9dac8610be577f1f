"""int8 tiles straight into three LDS buffers, and tiles two ahead in registers: sums of products, exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(m, k, n, tile_m, tile_n, bk, depth, parts=1, in_wg=1, shift=0):
    import torch
    from flextensor_amd import nn
    from flextensor_amd.plan import build
    from flextensor_amd.scheduler import schedule_with_config_ops
    from flextensor_amd.te import placeholder
    from flextensor_amd.templates import gfx950
    from flextensor_amd.utils import Config, ceil_div
    a, b = placeholder((m, k), dtype="int8"), placeholder((n, k), dtype="int8")
    c = nn.gemm_int8(a, b)
    cfg = gfx950._empty_config()
    cfg["spatial"] = [[ceil_div(m, tile_m[0] * tile_m[1] * 16)] + list(tile_m) + [16],
                      [ceil_div(n, tile_n[0] * tile_n[1] * 16)] + list(tile_n) + [16]]
    cfg["reduce"], cfg["unroll"] = [[parts, ceil_div(k, bk * parts), bk]], [[depth, 1]]
    cfg["fuse"], cfg["reorder"] = [[4]], [[1, in_wg if parts > 1 else 0, 0]]
    plan, bufs = schedule_with_config_ops([c.op], [a, b, c], Config([cfg], None))
    rng = np.random.default_rng(m * k + n)
    x, y = [rng.integers(-128, 128, shape, dtype=np.int8) for shape in ((m, k), (n, k))]
    func = build(plan, bufs, "rocm")
    out = torch.full((m, n), -77, dtype=torch.int32, device="cuda")

    def at(host, byte):
        """The operand ``byte`` bytes into an allocation, with ones around it."""
        room = torch.ones(host.size + 64, dtype=torch.int8, device="cuda")
        room[byte:byte + host.size] = torch.from_numpy(host).cuda().reshape(-1)
        return room[byte:byte + host.size].reshape(host.shape)
    func(at(x, shift), at(y, 3 * shift), out)
    torch.cuda.synchronize()
    func.close()
    # |sums| <= 4096 * 2^14 < 2^53: exact in float64
    assert np.array_equal(out.cpu().numpy(), np.rint(x.astype(np.float64) @ y.astype(np.float64).T).astype(np.int64))
    return plan


@pytest.mark.parametrize("tile_m,tile_n,bk,parts,in_wg", [
    ((2, 1), (2, 1), 128, 1, 1), ((2, 1), (2, 2), 256, 2, 1), ((4, 1), (2, 2), 128, 1, 1), ((4, 1), (2, 2), 128, 2, 0),
    ((2, 2), (4, 2), 128, 1, 1), ((4, 2), (2, 4), 128, 1, 1), ((1, 1), (4, 1), 256, 1, 1)])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 7])
def test_three_buffers(tile_m, tile_n, bk, parts, in_wg, steps):
    m, n = tile_m[0] * tile_m[1] * 32 - 3, tile_n[0] * tile_n[1] * 16 + 5
    plan = run(m, steps * bk * parts - 48, n, tile_m, tile_n, bk, 9, parts, in_wg)       # the last step is partly zeros
    assert plan.specs[-1].defines["STAGES"] == 3 and plan.specs[-1].defines["DTL"] == 1


@pytest.mark.parametrize("tile_m,tile_n,bk", [((2, 1), (2, 1), 128), ((2, 1), (2, 1), 256), ((2, 1), (2, 2), 128), ((1, 1), (4, 1), 256),
                                              ((4, 1), (2, 2), 128), ((2, 2), (4, 2), 128), ((4, 2), (2, 4), 128)])
@pytest.mark.parametrize("k,shift", [(124, 0), (260, 4), (380, 0), (388, 8), (516, 12), (1276, 4)])
def test_rows_of_whole_dwords_in_three_buffers(tile_m, tile_n, bk, k, shift):
    """K ends after one, two or three dwords of a chunk; operands begin at any dword."""
    m, n = tile_m[0] * tile_m[1] * 32 - 3, tile_n[0] * tile_n[1] * 16 + 5
    assert run(m, k, n, tile_m, tile_n, bk, 9, shift=shift).specs[-1].defines["STAGES"] == 3


@pytest.mark.parametrize("k", [516, 900, 1276])
@pytest.mark.parametrize("in_wg", [0, 1])
def test_rows_of_whole_dwords_with_k_divided(k, in_wg):
    run(61, k, 69, (2, 1), (2, 1), 128, 9, 2, in_wg)


@pytest.mark.parametrize("k", [1, 127, 129, 258, 1531])
@pytest.mark.parametrize("depth", [3, 4])
def test_eight_wavefronts_through_registers(k, depth):
    run(70, k, 131, (4, 1), (2, 2), 128, depth)


@pytest.mark.parametrize("k", [3329, 3455, 3458])
def test_small_tiles_three_ahead(k):
    run(35, k, 131, (2, 1), (2, 2), 128, 4)


def test_default_takes_the_third_buffer():
    """Where K is long and a unit holds the larger workgroups; not where they would run one at a time."""
    from flextensor_amd import nn
    from flextensor_amd.te import placeholder
    from flextensor_amd.templates import gfx950

    def depth(m, k, n):
        a, b = placeholder((m, k), dtype="int8"), placeholder((n, k), dtype="int8")
        return gfx950.untuned_config(nn.gemm_int8(a, b).op)["unroll"][0][0]
    assert depth(1152, 3808, 512) == 9 and depth(1152, 3804, 512) == 9 and depth(1152, 112, 512) == 6 and depth(1152, 3801, 512) == 3
    assert depth(1251, 4045, 361) == 4 and depth(1086, 2893, 290) == 5
