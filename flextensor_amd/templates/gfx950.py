"""gfx950 (MI355X) kernel templates: schedule space and config -> kernel.

Where the reference turns a config dict into TVM schedule primitives
(flextensor/templates/cuda.py:390-661 for GPUs, templates/cpu.py:316-518 for
CPUs), this module turns the same dict into the ``-D`` constants of a
hand-written HIP kernel template plus launch geometry. Nothing here touches a
device: lowering is pure Python and can be unit-tested on a CPU.

Operator kinds and the template each one lowers to:

  gemm                   igemm_f32.hip  MODE 0 (MODE 2 for transposeB)
  conv2d_nchw            igemm_f32.hip  MODE 1 (implicit GEMM, padding folded
                                         into the gather; or PAD=0 over a
                                         materialised padded tensor)
                         Products in bf16 parts are the second kernel of igemm_f32.hip and of direct_f32.hip: pipeline
                         depths 9 to 11, chosen by the defaults, not searched
  both and batch_gemm    direct_f32.hip (operands straight into registers, no LDS tiles: fourth number of the
                                         reorder entry 1; chosen by the defaults, not searched)
  conv2d_nchw, 1x1       igemm_f32.hip  MODE 0 per image where the fourth number of the reorder entry is 2 (the same)
  gemm_int8              gemm_i8.hip
  depthwise_conv2d_nchw  depthwise_f32.hip (direct; also what conv2d_nchw builds
                                         for one input channel per group)
  zero_pad2d             elementwise.hip   (only when not inlined)

Meaning of the config keys: see flextensor_amd/space.py.
"""
import copy
import json
import os

from ..space import (Space, SplitSpace, TileSplitSpace, LaneTileSpace, UnrollSpace, EnumSpace)
from ..utils import ceil_div

_HERE = os.path.dirname(os.path.abspath(__file__))

LDS_BYTES = 160 * 1024        # per workgroup on gfx950
MAX_ACC_REGS = 256            # accumulation VGPRs per lane
MAX_THREADS = 1024
NUM_XCD = 8
NUM_CUS = 256                 # compute units of one MI355X


class InvalidConfig(ValueError):
    """The config does not describe a kernel this template can build."""


_SOURCES = {}


def template_source(name):
    if name not in _SOURCES:
        with open(os.path.join(_HERE, name), "r") as f:
            _SOURCES[name] = f.read()
    return _SOURCES[name]


class KernelSpec(object):
    """One kernel of a plan, fully determined on the host.

    template     file name of the HIP source
    kernel       extern "C" symbol
    defines      dict of -D constants
    grid, block  launch geometry
    args         list of argument descriptors: ("buf", name) for a device
                 buffer bound by the plan, ("i32", value) / ("i64", value) /
                 ("u32", value) for scalars
    align        dict buffer name -> bytes its address has to be a multiple of, where that is
                 more than its type's size
    """

    def __init__(self, template, kernel, defines, grid, block, args, lds_bytes=0, note="",
                 workspace=None, align=None):
        self.align = dict(align or {})
        # name -> (shape, dtype) of zero-initialised device buffers the plan
        # owns and the kernel leaves zeroed where it relies on zeros
        self.workspace = dict(workspace or {})
        self.template = template
        self.kernel = kernel
        self.defines = dict(defines)
        self.grid = tuple(grid)
        self.block = tuple(block)
        self.args = list(args)
        self.lds_bytes = lds_bytes
        self.note = note

    def options(self):
        return ["-DFT_%s=%s" % (k, v) for k, v in sorted(self.defines.items())]

    def source(self):
        return template_source(self.template)

    def __repr__(self):
        return "KernelSpec(%s %s grid=%s block=%s)" % (self.kernel, self.defines, self.grid, self.block)


# --------------------------------------------------------------------------
# GEMM view of an operator
# --------------------------------------------------------------------------

def _conv_steps(attrs):
    """Stride, padding and dilation constants of a convolution, rows (H) and columns (W)
    apart: the operator definitions take pairs (flextensor/nn/ops.py:448-459)."""
    return dict(CSTRH=attrs["stride"][0], CSTRW=attrs["stride"][1], CPADH=attrs["padding"][0],
                CPADW=attrs["padding"][1], CDILH=attrs["dilation"][0], CDILW=attrs["dilation"][1])


class GemmView(object):
    """M, N, K and addressing mode of a contraction-shaped operator."""

    def __init__(self, op, col_inlined=False):
        kind = op.kind
        self.kind = kind
        self.conv = None
        self.groups = 1
        self.images = 0             # > 0: as many images, one at a time (by_image)
        self.pixels = None          # of one image, for layers that can be taken so
        self.trans_a = False
        if kind == "gemm":
            self.trans_a = bool(op.attrs.get("transposeA"))     # A stored [K][M] (ops.py:1093-1100)
            self.M, self.N = op.axis[0].extent, op.axis[1].extent
            self.K = op.reduce_axis[0].extent
            self.mode = 2 if op.attrs.get("transposeB") else 0
            self.dtype = "float32"
        elif kind == "batch_gemm":
            # one GEMM per batch entry: the batch index is the group index of the kernel
            self.groups = op.axis[0].extent
            self.trans_a = bool(op.attrs.get("transposeA"))
            self.M, self.N = op.axis[1].extent, op.axis[2].extent
            self.K = op.reduce_axis[0].extent
            self.mode = 2 if op.attrs.get("transposeB") else 0
            self.dtype = "float32"
        elif kind == "gemm_int8":
            self.M, self.N = op.axis[0].extent, op.axis[1].extent
            self.K = op.reduce_axis[0].extent
            self.mode = 0
            self.dtype = "int8"
        elif kind == "conv2d_nchw":
            a = op.attrs
            b, kout, p, q = [x.extent for x in op.axis]
            c = op.reduce_axis[0].extent
            s = op.reduce_axis[1].extent  # rw
            r = op.reduce_axis[2].extent  # rh
            _, _, h, w = a["in_shape"]
            groups = a["groups"]
            # one GEMM per group: c is already the per-group channel count
            self.M, self.N, self.K = kout // groups, b * p * q, c * r * s
            self.mode = 1
            self.dtype = "float32"
            self.groups = groups
            self.conv = dict(CB=b, CG=groups, CC=c * groups, CH=h, CW=w, CR=r, CS=s, CP=p, CQ=q,
                             **_conv_steps(a))
            # one image, 1x1 kernel, stride 1, no padding: O [K][H*W] = W [K][C] x X [C][H*W] in the
            # tensors' own layouts, a plain GEMM whose B rows load as 16-byte vectors
            as_matrix = (groups == 1 and r == 1 and s == 1 and tuple(a["stride"]) == (1, 1)
                         and tuple(a["padding"]) == (0, 0))
            self.pointwise = b == 1 and as_matrix
            if as_matrix:
                self.pixels = (b, p * q)
        elif kind == "col_gemm":
            # the GEMM stage of an im2col convolution: one [Mg,K] x [K,N] product per group.
            # With the column matrix read through (inlined) it is the implicit GEMM over the
            # image; otherwise a batch of plain GEMMs over the stored columns.
            a = op.attrs
            groups = op.axis[0].extent
            self.M, self.N = op.axis[1].extent, op.axis[2].extent
            self.K = op.reduce_axis[0].extent
            self.groups = groups
            self.dtype = "float32"
            b, cin, h, w = a["in_shape"]
            r, sw = a["kernel"]
            p, q = a["out_hw"]
            self.conv = dict(CB=b, CG=groups, CC=cin, CH=h, CW=w, CR=r, CS=sw, CP=p, CQ=q, **_conv_steps(a))
            self.mode = 1 if col_inlined else 0
        else:
            raise InvalidConfig("operator kind %s has no GEMM view" % kind)
        # K as the kernels iterate it: fp32 pads the tail up to a multiple of
        # 16 (int8: 64) with zero-filling loads unless it already is a multiple
        # of 8.
        if min(self.M, self.N, self.K) < 1:
            raise InvalidConfig("empty operator: M, N, K = %d, %d, %d" % (self.M, self.N, self.K))
        if self.dtype == "int8":
            self.KP_options = [ceil_div(self.K, 64) * 64]
        else:
            self.KP = ceil_div(self.K, 16) * 16
            self.KP_options = [self.KP]
            if self.K % 8 == 0 and self.K % 16 != 0:
                # e.g. K = 72: unpadded for 32x32x2 tiles of 8 or 72, padded to 80 for 16x16x4
                self.KP_options.insert(0, self.K)
            if not any(kp % 32 == 0 or kp % 48 == 0 or kp % 72 == 0 for kp in self.KP_options):
                # an awkward K (400 = 16 channels x 5x5) only divides into LDS tiles of 8 or 16: every
                # tile is a round trip to memory, 25 in a row. Up to an eighth of zero padding (the load
                # predicates supply it) buys tiles of 32 .. 144: 416, 432, 448 for K = 400
                wider = {ceil_div(self.K, bk) * bk for bk in (32, 48, 64, 72, 144)}
                self.KP_options += sorted(kp for kp in wider if kp > self.KP and kp * 8 <= self.K * 9)
            return
        self.KP = self.KP_options[-1]


    def by_image(self):
        """The same 1x1 layer image by image: O_i [K][H*W] = W [K][C] x X_i [C][H*W], a batch of GEMMs with one A."""
        view = copy.copy(self)
        view.images, view.N = self.pixels
        view.groups, view.mode, view.conv = view.images, 0, None
        return view


GEMM_KINDS = ("gemm", "gemm_int8", "conv2d_nchw", "batch_gemm", "col_gemm")

F32_BK = (8, 16, 32, 48, 64, 72, 128, 144)   # 72/144: whole 3x3 windows per LDS tile
I8_BK = (64, 128, 256)


def _gemm_space(view):
    space = Space()
    i8 = view.dtype == "int8"
    reps = (1, 2, 3, 4, 5, 6, 7, 8)
    space.add_subspace("split_m_0", TileSplitSpace(view.M, reps=reps), "spatial")
    space.add_subspace("split_n_1", TileSplitSpace(view.N, reps=reps), "spatial")
    bks = I8_BK if i8 else F32_BK
    max_split = 16

    def keep(e):
        return e[2] in bks and e[0] <= max_split

    rs = SplitSpace(3, view.KP_options[0], keep=keep)
    for other in view.KP_options[1:]:
        extra = SplitSpace(3, other, keep=keep)
        rs.static_entities = rs.static_entities + extra.static_entities
        rs._index = {tuple(e): i for i, e in enumerate(rs.static_entities)}
        rs.size = len(rs.static_entities)
    if rs.size == 0:
        raise InvalidConfig("K=%d has no admissible LDS tile extent" % view.K)
    space.add_subspace("split_k_0", rs, "reduce")
    space.add_subspace("unroll", UnrollSpace([1, 2, 3, 4, 5, 6, 7, 8] + list(I8_BUFFERS if i8 else ()), explicit=True,
                                               extra=() if i8 else [[8, 2], [8, 4], [8, 6], [8, 8]]),
                       "unroll")
    space.add_subspace("group_m", EnumSpace([[1], [2], [4], [8], [16]]), "fuse")
    # [xcd remap, K partitions inside the workgroup (1) or across workgroups (0)]
    # the third number: balanced K streaming with that many workgroups per compute unit (fp32 only)
    space.add_subspace("xcd_remap", EnumSpace([[1, 0, 0], [0, 0, 0], [1, 1, 0], [0, 1, 0]] if i8 else
                                            [[1, 0, 0], [0, 0, 0], [1, 1, 0], [0, 1, 0], [1, 0, 1], [1, 0, 2]]),
                       "reorder")
    return space


def _depthwise_space(op):
    space = Space()
    b, c, p, q = [x.extent for x in op.axis]
    space.add_subspace("split_b_0", LaneTileSpace(b, [1]), "spatial")
    space.add_subspace("split_c_1", LaneTileSpace(c, [1]), "spatial")
    space.add_subspace("split_h_2", LaneTileSpace(p, [1, 2, 4, 7, 8, 14]), "spatial")
    space.add_subspace("split_w_3", LaneTileSpace(q, [1, 2, 4]), "spatial")
    space.add_subspace("waves", EnumSpace([[1], [2], [4], [8]]), "fuse")
    return space


def generate_space(op):
    """Schedule space of one operator for gfx950."""
    if op.kind in GEMM_KINDS:
        return _gemm_space(GemmView(op))
    if op.kind == "depthwise_conv2d_nchw":
        return _depthwise_space(op)
    if op.kind in ("zero_pad2d", "bias_add_nchw", "bias_add_ghw", "im2col_nchw", "col2img_nchw"):
        return Space()
    raise InvalidConfig("no gfx950 template for operator kind %s" % op.kind)


# --------------------------------------------------------------------------
# special (task-level enumerated) knobs
# --------------------------------------------------------------------------

SPECIAL_DEFAULTS = {
    # fp32: [APAD, BPAD] in floats; APAD -1 = unpadded, XOR-swizzled A tile;
    # BPAD -1 = the padding that spreads the k-groups of one MFMA operand read
    # over disjoint banks (4 floats for 16x16x4, 8 for 32x32x2).
    # int8: [PAD bytes / 4, unused]
    # the default admits every pipeline depth (tiles straight into LDS need unpadded A rows), so
    # that an operator search under the graph level's defaults can reach them
    "lds_pad": [-1, -1],
    "nt_store": [0],
    "halo_shfl": [0],
    "lds_planes": [0],
    "lane_items": [1],
    "row_exchange": [0],
    # depthwise with several kernels per input channel: 1 = a lane computes its patch for all of them
    "kernel_fuse": [1],
    # 1x1 convolution, stride 1, no padding, one image: 1 = the GEMM addressing mode (the image is
    # the B matrix as it lies in memory, rows load as 16-byte vectors), 0 = the gather of the general case
    "image_as_matrix": [1],
    # K streaming: 1 = the arrival count and the look at the counter are a device-scope
    # release / acquire (what the memory model asks for; costs an L2 write-back and invalidate per
    # hand-off, +4.5 % on the 8x256x14x14 benchmark layer), 0 = relaxed device-scope atomics behind
    # an explicit wait for the slot stores (the measured trade-off the shipped entries use). Not in
    # the searched knobs: a task opts in with set_specific_space("sk_fenced", "enum", [[1]])
    "sk_fenced": [0],
}

# unroll entity [[depth, 1]] -> (LDS stages, prefetch distance in tiles);
# depth 5 = two stages with the fragment-prefetch pipeline (int8 GEMM)
# depth -> (LDS buffers, global prefetch distance); 5 = int8: MFMA fragment prefetch, fp32: tiles
# loaded straight into LDS; int8 only:
# 6 = tiles loaded straight into LDS (no staging registers), 7 = 6 with MFMA fragment prefetch,
# 8 = 7 with the main loop's instruction order written out (fragment reads and tile loads issued
# one at a time between the MFMAs);
# fp32: 6 and 7 = 5 with three and four LDS buffers (two and three tiles requested ahead)
# fp32: 9 and 10 = products in bf16 parts (the second kernel of igemm_f32.hip), one and two k steps ahead; 11 = the same
# with every wavefront on its own (the second kernel of direct_f32.hip)
SPLIT_DEPTHS = {9: ("igemm_f32.hip", 1), 10: ("igemm_f32.hip", 2), 11: ("direct_f32.hip", 0)}
# int8: 9 = 6 with three LDS buffers (two tiles requested ahead). Four and six were timed beside it on 38 sizes: 1.02
# and 1.12 times its time in the geometric mean, so there are no depths for them.
I8_BUFFERS = {9: 3}
PIPELINE = {1: (1, 1), 2: (2, 1), 3: (2, 2), 4: (2, 3), 5: (2, 1), 6: (2, 1), 7: (2, 1), 8: (2, 1)}


def special_knobs(kind):
    """Enumerated knobs a task of this operator kind carries by default; they
    are attached with Task.set_specific_space and searched at graph level."""
    if kind == "pointwise_conv2d_nchw":
        # a 1x1 / stride 1 / unpadded convolution over one image (the task tells: the operator kind
        # is conv2d_nchw like any other convolution's)
        return {"lds_pad": [[-1, -1], [4, -1], [4, 8], [4, 4], [0, 0], [8, -1], [-1, 0]],
                "image_as_matrix": [[1], [0]]}
    if kind in ("gemm", "conv2d_nchw", "batch_gemm", "col_gemm"):
        return {"lds_pad": [[-1, -1], [4, -1], [4, 8], [4, 4], [0, 0], [8, -1], [-1, 0]]}
    if kind == "gemm_int8":
        return {"lds_pad": [[-1, 0], [4, 0], [0, 0], [8, 0]],
                "nt_store": [[0], [1], [2], [3], [4], [5], [6], [7]]}
    if kind == "depthwise_conv2d_nchw":
        return {"nt_store": [[0], [1], [2], [3]], "halo_shfl": [[0], [1]], "lds_planes": [[0], [1], [2], [4], [8]],
                "lane_items": [[1], [2], [3], [4], [6], [8]], "row_exchange": [[0], [1], [2], [3], [4]],
                "kernel_fuse": [[1], [0]]}
    return {}


def _special(graph_special, name):
    if graph_special and name in graph_special:
        return list(graph_special[name])
    return list(SPECIAL_DEFAULTS[name])


# --------------------------------------------------------------------------
# lowering
# --------------------------------------------------------------------------

def _one(config, key, n, what):
    lst = config.get(key) or []
    if len(lst) != n:
        raise InvalidConfig("%s: expected %d '%s' entries, got %d" % (what, n, key, len(lst)))
    return lst


def _lower_gemm(op, config, special, out_name, in_names, materialized_pad=False, bias_name=None,
                through=(), merged_out=None):
    view = GemmView(op, col_inlined="im2col_nchw" in through)
    if getattr(view, "pointwise", False) and int(_special(special, "image_as_matrix")[0]) \
            and bias_name is None and merged_out is None:
        view.mode = 0        # A = weight [K][C], B = image [C][H*W], C = output [K][H*W]
    if bias_name is not None and view.mode != 1 and op.kind != "col_gemm":
        raise InvalidConfig("only the convolution has a bias epilogue")
    if merged_out is not None and not (op.kind == "col_gemm" and merged_out == "col2img_nchw"):
        raise InvalidConfig("stage %s cannot run in the stores of %s" % (merged_out, op.kind))
    if merged_out is not None and view.mode != 1 and view.conv["CB"] != 1:
        # for one image [groups][M][P*Q] is NCHW already; a batch interleaves the images
        raise InvalidConfig("col2img merges into the GEMM that reads the image itself")
    sp = _one(config, "spatial", 2, op.kind)
    rd = _one(config, "reduce", 1, op.kind)
    (gm, wm, rm, mfm), (gn, wn, rn, mfn) = [list(map(int, x)) for x in sp]
    splitk, kiters, bk = [int(x) for x in rd[0]]
    depth = int((config.get("unroll") or [[2, 1]])[0][0])
    split = view.dtype != "int8" and depth in SPLIT_DEPTHS
    buffers = I8_BUFFERS.get(depth, 0) if view.dtype == "int8" else 0
    if depth not in PIPELINE and not split and not buffers:
        raise InvalidConfig("pipeline depth %d is not available" % depth)
    stages, pd = PIPELINE.get(depth, (buffers or 2, 1))
    if view.dtype != "int8" and depth in (6, 7):
        stages = depth - 3        # fp32: 6 and 7 = tiles straight into LDS with three and four buffers
    # fp32 depth 8: as 5 (two buffers), and the first operands of the next tile are read from LDS
    # right behind the barrier, ahead of the last MFMAs of the current tile
    frag_prefetch = view.dtype != "int8" and depth == 8
    # with it, the second number of the unroll entry is the number of k blocks over which the
    # loads of the next tile are spread (1 = all in front of the tile's first MFMAs)
    load_spread = int((config.get("unroll") or [[2, 1]])[0][1]) if frag_prefetch else 1
    group_m = int((config.get("fuse") or [[4]])[0][0])
    ro = list((config.get("reorder") or [[1, 0]])[0]) + [0, 0, 0]
    xcd, in_wg, stream_k, direct = int(ro[0]), int(ro[1]), int(ro[2]), int(ro[3])
    if direct == 2:
        # the fourth number 2: a 1x1 layer image by image; one image without a bias is the plain GEMM already
        if view.pixels is None or merged_out is not None or not int(_special(special, "image_as_matrix")[0]):
            raise InvalidConfig("image by image: 1x1, stride 1, no padding, one group, and images read as matrices")
        view, direct = view if view.mode == 0 else view.by_image(), 0
    i8 = view.dtype == "int8"
    waves_k = 1
    if in_wg and splitk > 1:
        waves_k, splitk = splitk, 1

    if mfm != mfn or mfm not in (16, 32):
        raise InvalidConfig("MFMA edge must be 16 or 32 and equal on both axes")
    if min(wm, rm, wn, rn, splitk, kiters, bk, group_m) < 1:
        raise InvalidConfig("non-positive factor")
    nwaves = wm * wn * waves_k
    if nwaves * 64 > MAX_THREADS:
        raise InvalidConfig("more than 16 wavefronts per workgroup")
    bm, bn = wm * rm * mfm, wn * rn * mfn
    if gm != ceil_div(view.M, bm) or gn != ceil_div(view.N, bn):
        raise InvalidConfig("grid level does not match ceil(extent / tile)")
    nacc = rm * rn * (mfm * mfm // 64)
    if nacc > MAX_ACC_REGS:
        raise InvalidConfig("accumulators need %d registers per lane" % nacc)
    kp = splitk * waves_k * kiters * bk
    # the fewest whole tiles that cover K will do as well (zeros behind it): int8 always, fp32 up to a quarter more;
    # tiles without LDS multiply no zeros but give some groups of wavefronts fewer steps
    if kp not in view.KP_options and not (view.K <= kp < view.K + splitk * waves_k * bk
                                          and (i8 or direct or split or kp * 4 <= view.K * 5)):
        raise InvalidConfig("reduce split does not multiply to K, nor to the fewest whole tiles that cover it")
    nt = wm * wn * 64          # threads of one k-group
    D = dict(M=view.M, N=view.N, K=view.K, KP=kp, MFMA=mfm, WAVES_M=wm, WAVES_N=wn, REP_M=rm,
             REP_N=rn, BK=bk, STAGES=stages, GROUP_M=group_m, XCD_REMAP=xcd)

    if i8:
        if direct:
            raise InvalidConfig("operands straight into registers are an fp32 path")
        if stream_k:
            # the grid-level split (integer atomics: exact, any order) and the in-workgroup split
            # cover the int8 operator; the balanced K streaming protocol is an fp32 path
            raise InvalidConfig("int8 GEMM splits K across workgroups or wavefront groups, not by K streaming")
        mfma_k = 32 if mfm == 32 else 64
        if bk % mfma_k != 0:
            raise InvalidConfig("BK must be a multiple of the MFMA K extent")
        if depth >= 6 and view.K % (4 if buffers else 16) != 0:
            # a row's last chunk runs into the next row, and for K % 4 != 0 every chunk is cut out of five
            # dwords: both happen in registers, which the loads that write LDS directly pass by (three buffers:
            # a row's end is cut out of the fragments)
            raise InvalidConfig("int8 tiles straight into LDS need K to be a multiple of 16, of 4 with three buffers")
        pad = int(_special(special, "lds_pad")[0])
        pad = -1 if pad < 0 else pad * 4
        if pad >= 0 and pad % 16 != 0:
            raise InvalidConfig("int8 LDS padding must be a multiple of 16 bytes")
        if view.M * view.K >= 2 ** 31 or view.N * view.K >= 2 ** 31:
            raise InvalidConfig("operands of 2 GiB or more are not addressable by the buffer loads")
        if depth >= 6:
            if pad > 0 or (bm * bk // 16) % nt or (bn * bk // 16) % nt:
                raise InvalidConfig("direct-to-LDS tiles need unpadded rows and whole rounds of 16-byte chunks")
            if depth == 8:
                nm, nr, loads = rm * rn, rm + rn, (bm + bn) * bk // 16 // nt
                if (bk // mfma_k) % 2 or nm // 4 + nr > nm or nm // 4 + loads > nm:
                    raise InvalidConfig("the written-out schedule needs an even number of k-steps per tile "
                                        "and enough MFMAs per k-step to interleave with")
        elif (ceil_div(bm * bk // 16, nt) + ceil_div(bn * bk // 16, nt)) * 4 * pd > 160:
            raise InvalidConfig("global->LDS staging needs too many registers")
        lds = max(waves_k * stages * (bm + bn) * (bk + max(pad, 0)), (waves_k - 1) * nt * nacc * 4)
        if lds > LDS_BYTES:
            raise InvalidConfig("LDS tile needs %d bytes" % lds)
        # nt_store: bit 0 = non-temporal stores, bit 1 = transposed MFMA so that lanes store 128-bit rows,
        # bit 2 = the last tile multiplied block by block, every block stored as soon as it is complete
        store_mode = int(_special(special, "nt_store")[0])
        if store_mode & 2 and view.N % 4 != 0:
            raise InvalidConfig("128-bit C stores need N to be a multiple of 4")
        if store_mode & 4 and (depth != 7 or bk != 2 * mfma_k or kp // bk < 2 or splitk * waves_k != 1):
            raise InvalidConfig("early stores come with pipeline depth 7, two k-steps per tile, two tiles or more, "
                                "and an undivided K")
        D.update(PAD=pad, PD=pd, FRAGPF=1 if depth == 5 else 0, NT_STORE=store_mode & 1)
        if depth >= 6:
            D.update(DTL=1 if buffers else depth - 5)
        if store_mode & 2:
            D.update(CVEC=1)
        if store_mode & 4:
            D.update(EARLYST=1)
        specs = []
        if splitk > 1:
            # partial sums meet in C: zero it first (the fill writes zero bit patterns, whatever the type)
            D.update(SPLITK=splitk)
            nout = view.M * view.N
            specs.append(KernelSpec("elementwise.hip", "fill_zero_f32", {},
                                    (min(ceil_div(ceil_div(nout, 4), 256), 2048), 1, 1), (256, 1, 1),
                                    [("buf", out_name), ("i32", nout)], note="split-K zero fill"))
        if waves_k > 1:
            D.update(WAVES_K=waves_k)
        grid = (gm * gn * splitk, 1, 1)
        # rows of whole dwords are loaded as they lie, which takes operands that begin at a dword; for other K the
        # kernel shifts every chunk by the byte it begins at, the operand's own included
        align = {} if view.K % 4 else dict.fromkeys(in_names[:2], 4)
        specs.append(KernelSpec("gemm_i8.hip", "gemm_i8", D, grid, (nt * waves_k, 1, 1),
                                [("buf", in_names[0]), ("buf", in_names[1]), ("buf", out_name)], align=align))
        return specs

    if split:
        if bk != 32 or splitk > 1 or stream_k or direct:
            raise InvalidConfig("products in bf16 parts: k steps of 32, K divided inside the workgroup only")
        return _lower_split(op, view, D, depth, special, out_name, in_names, materialized_pad, bias_name, merged_out, waves_k)
    if direct:
        if mfm != 16 or bk != 32 or splitk > 1 or stream_k:
            raise InvalidConfig("operands straight into registers: 16x16 tiles, k steps of 32, K divided inside the "
                                "workgroup only")
        return _lower_direct(op, view, D, direct, depth, out_name, in_names, materialized_pad, bias_name, merged_out,
                             waves_k=waves_k)

    kblk = 4 * (64 // mfm)
    if bk % kblk != 0:
        raise InvalidConfig("BK must be a multiple of %d for this MFMA shape" % kblk)
    apad, bpad = [int(x) for x in _special(special, "lds_pad")[:2]]
    bpad_auto = bpad < 0
    if bpad < 0:
        bpad = 4 if mfm == 16 else 8
    if apad < -1 or (apad >= 0 and apad % 4 != 0) or bpad % 4 != 0:
        raise InvalidConfig("fp32 LDS padding must keep 16-byte alignment")
    # 16-byte loads at dword alignment: rows of any length (the kernel zeroes what a row's last vector along K
    # takes from the next row). Only an axis shorter than a vector goes one float at a time.
    av = 4 if (view.M if view.trans_a else view.K) >= 4 else 1      # vectors of a [K][M] operand run along M
    if view.mode == 0:
        bv = 4 if view.N >= 4 else 1
    elif view.mode == 2:
        bv = 4 if view.K >= 4 else 1
    else:
        bv = 1
    dtl = depth >= 5          # fp32: tiles loaded straight into LDS
    if dtl and view.trans_a and (bm % 64 or view.M % 4):
        raise InvalidConfig("direct-to-LDS tiles of a transposed A operand need tile rows of a multiple of 64 "
                            "and M a multiple of 4")
    if dtl:
        if view.mode == 0 and view.N >= 4 and bn % 64 == 0 and (bpad_auto or bpad == 0):
            bv, bpad = 4, 0   # B in 16-byte chunks too: unpadded rows, columns swizzled by k
        elif view.mode != 2:
            bv = 1            # B goes one float per lane
        if av != 4 or apad > 0 or (bm * bk // 4) % 64:
            raise InvalidConfig("direct-to-LDS tiles need 16-byte A chunks in whole wavefronts and unpadded A rows")
        if view.mode == 2 and (bv != 4 or (bn * bk // 4) % 64):
            raise InvalidConfig("direct-to-LDS tiles need 16-byte B chunks in whole wavefronts")
        if view.mode != 2 and bv == 1 and bn % 64:
            # B one float per lane: a wavefront writes 64 consecutive floats, so rows that are
            # not multiples of 64 floats land unpadded, in whole wavefronts per tile
            if bpad_auto:
                bpad = 0
            if bpad != 0 or (bn * bk) % 64:
                raise InvalidConfig("direct-to-LDS tiles with rows that are not multiples of 64 floats need "
                                    "unpadded B rows and whole wavefronts of floats per tile")
    sa = bk + max(apad, 0)
    if view.mode == 2:
        lds_b = bn * sa
    else:
        lds_b = bk * (bn + bpad)
    lds = max(waves_k * stages * 4 * (bm * sa + lds_b), (waves_k - 1) * nt * nacc * 4)
    if stream_k:
        lds += 16             # the arrival word of the K-streaming exchange
    if lds > LDS_BYTES:
        raise InvalidConfig("LDS tile needs %d bytes" % lds)
    # staging registers for the global->LDS copy must stay reasonable
    ea = ceil_div(bm * bk // av, nt)
    eb = ceil_div((bn * bk) // bv, nt)
    if not dtl and (ea * av + eb * bv) * pd > 160:
        raise InvalidConfig("global->LDS staging needs too many registers")
    if dtl and stages > 2 and ((bm * bk // av) % nt or ((bn * bk) // bv) % nt or (stages - 2) * (ea + eb) > 63):
        raise InvalidConfig("more than two direct-to-LDS buffers need whole rounds of loads per tile, "
                            "at most 63 of them in flight")
    # bytes behind the two buffer descriptors (A_BYTES / B_BYTES of the template) and of C: in MODE 1
    # B is the image itself, larger than K x N when the stride exceeds the kernel, and larger
    # still once the padding is materialised
    a_bytes = (1 if view.images else view.groups) * view.M * view.K * 4
    if view.mode == 1:
        cv = view.conv
        grow_h, grow_w = (2 * cv["CPADH"], 2 * cv["CPADW"]) if materialized_pad else (0, 0)
        b_bytes = cv["CB"] * cv["CC"] * (cv["CH"] + grow_h) * (cv["CW"] + grow_w) * 4
    else:
        b_bytes = view.groups * view.K * view.N * 4
    if max(a_bytes, b_bytes, view.groups * view.M * view.N * 4) >= 2 ** 31:
        raise InvalidConfig("operands of 2 GiB or more are not addressable by the buffer loads")
    D.update(MODE=view.mode, SPLITK=splitk, WAVES_K=waves_k, APAD=apad, BPAD=bpad, AV=av, BV=bv, PD=pd)
    if view.trans_a:
        D.update(TA=1)
    if dtl:
        D.update(DTL=1)
    if frag_prefetch:
        D.update(FPF=1)
        if load_spread < 1 or (load_spread > 1 and load_spread > bk // kblk - 1):
            raise InvalidConfig("the loads of the next tile spread over at most all but the last k block")
        if load_spread > 1:
            D.update(LSPREAD=load_spread)
    specs = []
    if view.mode == 1:
        conv = dict(view.conv)
        if materialized_pad:
            conv["CH"] += 2 * conv["CPADH"]
            conv["CW"] += 2 * conv["CPADW"]
            conv["CPADH"] = conv["CPADW"] = 0
        D.update(conv)
        if op.kind == "col_gemm" and merged_out is None:
            D.update(COLOUT=1)            # C stays [groups][M][N] for the col2img stage
        # A = weight, B = image
        a_name, b_name = in_names[1], in_names[0]
    else:
        a_name, b_name = in_names[0], in_names[1]
        if op.kind in ("col_gemm", "conv2d_nchw"):
            a_name, b_name = in_names[1], in_names[0]      # A = weight, B = stored columns / the image
        if view.images:
            D.update(MODE=1, IMAGES=view.images)
        elif view.groups > 1:
            D.update(CG=view.groups)      # batched GEMM
    if splitk > 1:
        nout = view.M * view.N * view.groups
        specs.append(KernelSpec("elementwise.hip", "fill_zero_f32", {},
                                (min(ceil_div(ceil_div(nout, 4), 256), 2048), 1, 1), (256, 1, 1),
                                [("buf", out_name), ("i32", nout)], note="split-K zero fill"))
    args = [("buf", a_name), ("buf", b_name), ("buf", out_name)]
    if bias_name is not None:
        D.update(HAS_BIAS=1)       # C = A*B + bias[row], added once whatever the K division
    workspace = {}
    if stream_k:
        # balanced K streaming: stream_k workgroups per compute unit share the
        # (tile, k-tile) units evenly; see the template for the protocol
        if stream_k < 0 or splitk != 1 or waves_k != 1:
            raise InvalidConfig("K streaming excludes the other K splits")
        units = gm * gn * view.groups * (kp // bk)
        per = ceil_div(units, NUM_CUS * stream_k)
        ngrid = ceil_div(units, per)
        if xcd:
            ngrid = ceil_div(ngrid, NUM_XCD) * NUM_XCD   # renumbering by XCD needs whole rounds
        D.update(SK_PER=per)
        if int(_special(special, "sk_fenced")[0]):
            D.update(SK_FENCED=1)
        grid = (ngrid, 1, 1)
        workspace = {out_name + "_parts": ((ngrid * 2 * nt * nacc,), "float32"),
                     out_name + "_count": ((gm * gn * view.groups,), "int32")}
        args += [("buf", out_name + "_parts"), ("buf", out_name + "_count")]
    else:
        grid = (gm * gn * splitk * view.groups, 1, 1)
    if bias_name is not None:
        args.append(("buf", bias_name))
    specs.append(KernelSpec("igemm_f32.hip", "igemm_f32", D, grid, (nt * waves_k, 1, 1), args,
                            workspace=workspace))
    return specs


def _lower_direct(op, view, D, direct, depth, out_name, in_names, materialized_pad, bias_name, merged_out, waves_k):
    """Tiles whose operands go straight into registers (direct_f32.hip)."""
    if direct != 1:
        raise InvalidConfig("no variant %d of the tiles without LDS" % direct)
    if view.trans_a or view.K < 32:
        raise InvalidConfig("operands straight into registers need a K of 32 and more and A stored [M][K]")
    waves, rm, rn = D["WAVES_M"] * D["WAVES_N"] * waves_k, D["REP_M"], D["REP_N"]
    if view.mode == 0 and rn not in (1, 2, 4):
        raise InvalidConfig("a lane's neighbouring columns are one load: 1, 2 or 4 blocks")
    if view.mode == 1 and view.conv["CR"] * view.conv["CS"] > 31:
        raise InvalidConfig("a pixel's valid taps are bits of a word")
    steps = ceil_div(view.K, 32)
    pd = min(depth, ceil_div(steps, waves_k))          # no group loads more steps ahead than it has
    regs = 4 * rm * rn + 8 * (rm + rn) * pd + rm + 2 * rn + 24
    if pd > 4 or regs > (256 if waves <= 8 else 128):
        raise InvalidConfig("the tile and its loads need %d registers per lane" % regs)
    # one after the other in the same LDS: the offsets of the gathered operand's k, the groups' partial sums
    if max(waves * rm * rn * 1024 if waves_k > 1 else 0, steps * 32 * 8 if view.mode == 1 else 0) + 16 > LDS_BYTES:
        raise InvalidConfig("partial sums or the offsets of a gathered operand need more than %d bytes" % LDS_BYTES)
    D = {k: D[k] for k in ("M", "N", "K", "WAVES_M", "WAVES_N", "REP_M", "REP_N", "GROUP_M", "XCD_REMAP")}
    D.update(MODE=view.mode, WAVES_K=waves_k, PD=pd)
    a_name, b_name = in_names[0], in_names[1]
    b_bytes = view.groups * view.K * view.N * 4
    if view.mode == 1:
        conv = dict(view.conv)
        if materialized_pad:
            conv["CH"] += 2 * conv["CPADH"]
            conv["CW"] += 2 * conv["CPADW"]
            conv["CPADH"] = conv["CPADW"] = 0
        D.update(conv)
        b_bytes = conv["CB"] * conv["CC"] * conv["CH"] * conv["CW"] * 4
        if op.kind == "col_gemm" and merged_out is None:
            D.update(COLOUT=1)
    elif view.groups > 1:
        D.update(CG=view.groups)
    if op.kind in ("col_gemm", "conv2d_nchw"):
        a_name, b_name = b_name, a_name          # A = weight, B = the image or the stored columns
    if max(view.groups * view.M * view.K * 4, b_bytes, view.groups * view.M * view.N * 4) >= 2 ** 31:
        raise InvalidConfig("operands of 2 GiB or more are not addressable by the buffer loads")
    args = [("buf", a_name), ("buf", b_name), ("buf", out_name)]
    if bias_name is not None:
        D.update(HAS_BIAS=1)
        args.append(("buf", bias_name))
    tiles = ceil_div(view.M, D["WAVES_M"] * rm * 16) * ceil_div(view.N, D["WAVES_N"] * rn * 16)
    return [KernelSpec("direct_f32.hip", "igemm_f32", D, (tiles * view.groups, 1, 1), (waves * 64, 1, 1), args)]


def _gathered_bytes(conv, ahead):
    """Bytes that the offsets of the gathered operand span: with LDS tiles (``ahead``) they count from before the padding."""
    return 4 * (conv["CB"] * conv["CC"] * conv["CH"] * conv["CW"] + (conv["CPADH"] * conv["CW"] + conv["CPADW"] if ahead else 0))


def _lower_split(op, view, D, depth, special, out_name, in_names, materialized_pad, bias_name, merged_out, waves_k):
    """Products in three bf16 parts (the second kernels of igemm_f32.hip and direct_f32.hip)."""
    template, ahead = SPLIT_DEPTHS[depth]
    if view.trans_a:
        raise InvalidConfig("products in bf16 parts need A stored [M][K]")
    if _special(special, "lds_pad") != SPECIAL_DEFAULTS["lds_pad"]:
        raise InvalidConfig("products in bf16 parts have an LDS layout of their own")
    if view.mode == 1 and (view.conv["CR"] * view.conv["CS"] > 31 or view.K > 16384):
        raise InvalidConfig("a pixel's valid taps are bits of a word, the offsets of the gathered operand's k a table")
    keys = ["M", "N", "K", "WAVES_M", "WAVES_N", "REP_M", "REP_N", "GROUP_M", "XCD_REMAP"]
    bm, bn = D["WAVES_M"] * D["REP_M"] * D["MFMA"], D["WAVES_N"] * D["REP_N"] * D["MFMA"]
    waves, blocks = D["WAVES_M"] * D["WAVES_N"] * waves_k, D["REP_M"] * D["REP_N"]
    sums = waves_k * bm * bn * 4 if waves_k > 1 else 0
    if depth == 11:
        if D["MFMA"] != 32 or blocks > 4 or blocks > 2 and waves_k < 4 or waves > 8 and blocks > 2:
            raise InvalidConfig("32x32 MFMAs, up to four of them a wavefront, more than two only where K is divided by four")
        if view.mode == 0 and D["REP_N"] not in (1, 2, 4) or view.mode == 1 and D["REP_N"] > 3:
            raise InvalidConfig("a lane's neighbouring columns are one load, loads in flight are counted to 63")
        rows = (D["REP_M"] + (D["REP_N"] if view.mode == 2 else 0)) * 32
        lds = waves * 2 * rows * 128 + (ceil_div(view.K, 32) * 256 if view.mode == 1 else 0)
    else:
        # 2 * blocks * NACC accumulators, the parts of a row of blocks and of a block, a thread's share of the tile
        regs = 2 * blocks * D["MFMA"] ** 2 // 64 + 12 * (D["REP_N"] + 1) + ceil_div((bm + bn) * 32 * ahead, waves // waves_k * 64) + 40
        if regs > (512 if waves <= 4 else 256 if waves <= 8 else 128):
            raise InvalidConfig("the tile and its loads need %d registers per lane" % regs)
        keys.append("MFMA")
        lds = waves_k * 2 * 192 * (bm + bn) + 16
    if max(lds, sums) > LDS_BYTES:
        raise InvalidConfig("LDS tiles or partial sums need %d bytes" % max(lds, sums))
    D = {k: D[k] for k in keys}
    D.update(SPLIT=1, MODE=view.mode, WAVES_K=waves_k)
    if ahead:
        D.update(PD=ahead)
    b_bytes = view.groups * view.K * view.N * 4
    a_name, b_name = in_names[0], in_names[1]
    if view.mode == 1:
        conv = dict(view.conv)
        if materialized_pad:
            conv["CH"] += 2 * conv["CPADH"]
            conv["CW"] += 2 * conv["CPADW"]
            conv["CPADH"] = conv["CPADW"] = 0
        D.update(conv)
        b_bytes = _gathered_bytes(conv, ahead)
        if op.kind == "col_gemm" and merged_out is None:
            D.update(COLOUT=1)
    elif view.images:
        D.update(IMAGES=view.images)
    elif view.groups > 1:
        D.update(CG=view.groups)
    if op.kind in ("col_gemm", "conv2d_nchw"):
        a_name, b_name = b_name, a_name          # A = weight, B = the image or the stored columns
    a_bytes = (1 if view.images else view.groups) * view.M * view.K * 4
    if max(a_bytes, b_bytes, view.groups * view.M * view.N * 4) >= 2 ** 31:
        raise InvalidConfig("operands of 2 GiB or more are not addressable by the buffer loads")
    args = [("buf", a_name), ("buf", b_name), ("buf", out_name)]
    if bias_name is not None:
        D.update(HAS_BIAS=1)
        args.append(("buf", bias_name))
    tiles = ceil_div(view.M, bm) * ceil_div(view.N, bn)
    return [KernelSpec(template, "igemm_f32", D, (tiles * view.groups, 1, 1), (waves * 64, 1, 1), args)]


def _lower_depthwise(op, config, special, out_name, in_names, materialized_pad=False, bias_name=None):
    sp = _one(config, "spatial", 4, op.kind)
    th, tw = int(sp[2][3]), int(sp[3][3])
    if int(sp[0][3]) != 1 or int(sp[1][3]) != 1:
        raise InvalidConfig("depthwise lanes own one batch entry and one channel")
    waves = int((config.get("fuse") or [[4]])[0][0])
    if waves < 1 or waves * 64 > MAX_THREADS:
        raise InvalidConfig("bad wavefront count")
    a = op.attrs
    b, cout, p, q = [x.extent for x in op.axis]
    s_ext = op.reduce_axis[0].extent  # rw
    r_ext = op.reduce_axis[1].extent  # rh
    _, c, h, w = a["in_shape"]
    if th < 1 or tw < 1 or th > p or tw > q:
        raise InvalidConfig("lane patch larger than the output plane")
    if int(sp[2][0]) != ceil_div(p, th) or int(sp[3][0]) != ceil_div(q, tw):
        raise InvalidConfig("grid level does not match ceil(extent / patch)")
    (st_h, st_w), (pad_h, pad_w), (dl_h, dl_w) = a["stride"], a["padding"], a["dilation"]   # rows, columns
    if materialized_pad:
        h, w, pad_h, pad_w = h + 2 * pad_h, w + 2 * pad_w, 0, 0
    ih_t = (th - 1) * st_h + (r_ext - 1) * dl_h + 1
    iw_t = (tw - 1) * st_w + (s_ext - 1) * dl_w + 1
    # the 128-bit input path requests every row of the patch before the first is used
    vec_rows = (tw == 4 and st_w <= 2 and w % 4 == 0 and q * st_w == w and pad_w + 4 * st_w <= iw_t)
    # kernel_fuse: with several kernels per input channel a lane computes its patch for all of them
    fm = a["factor"] if int(_special(special, "kernel_fuse")[0]) else 1
    # lane_items: patches per lane, all requested before the first is computed
    ipl = int(_special(special, "lane_items")[0])
    if ipl < 1 or ipl > 16:
        raise InvalidConfig("lane_items is 1 .. 16")
    if th * tw + ipl * (ih_t * iw_t + fm * r_ext * s_ext) > 220:
        raise InvalidConfig("lane patches need too many registers")
    if max(b * c * h * w, b * cout * p * q) * 4 >= 2 ** 31:
        raise InvalidConfig("tensors of 2 GiB or more are not addressable by the buffer accesses")
    nt = waves * 64
    items = b * (cout // fm) * ceil_div(p, th) * ceil_div(q, tw)
    ldsp = int(_special(special, "lds_planes")[0])
    nt_mode = int(_special(special, "nt_store")[0])     # bit 0: non-temporal stores, bit 1: non-temporal loads
    steps = dict(STRH=st_h, STRW=st_w, PADH=pad_h, PADW=pad_w, DILH=dl_h, DILW=dl_w)
    args = [("buf", in_names[0]), ("buf", in_names[1]), ("buf", out_name)]
    if bias_name is not None:
        # the bias stage merged into the kernel: added to every result in the store (ops.py:673-677)
        steps["HAS_BIAS"] = 1
        args.append(("buf", bias_name))
    if ldsp:
        # plane-staged variant: whole planes through LDS in copy order; the lane patch knobs do not apply
        if not (st_h == st_w == 1 and dl_h == dl_w == 1 and r_ext == 3 and s_ext == 3 and pad_h == pad_w == 1
                and p == h and q == w and w % 4 == 0 and a["factor"] == 1):
            raise InvalidConfig("plane staging needs a same-size 3x3 stride-1 pad-1 layer with rows of whole vectors")
        if ldsp < 0 or (ldsp * (h + 2) * (w + 8) + ldsp * 12) * 4 > LDS_BYTES:
            raise InvalidConfig("staged planes do not fit the LDS")
        D = dict(NT=nt, TH=th, TW=tw, NT_STORE=nt_mode & 1, NT_LOAD=nt_mode >> 1, SHFL=0, LDSP=ldsp,
                 CB=b, CC=c, CH=h, CW=w, CR=r_ext, CS=s_ext, FACT=1, CP=p, CQ=q, **steps)
        return [KernelSpec("depthwise_f32.hip", "depthwise_f32", D, (ceil_div(b * cout, ldsp), 1, 1),
                           (nt, 1, 1), args)]
    wx = int(_special(special, "row_exchange")[0])
    if wx:
        # row-exchange variant: a wavefront owns rpi * wx rows of one plane (rpi whole rows per load
        # instruction), loads each 16-byte chunk once and passes rows between lanes through its own
        # LDS window; the lane patch knobs do not apply
        if not (st_h == st_w == 1 and dl_h == dl_w == 1 and r_ext == 3 and s_ext == 3 and pad_h == pad_w == 1
                and p == h and q == w and w % 4 == 0 and a["factor"] == 1):
            raise InvalidConfig("row exchange needs a same-size 3x3 stride-1 pad-1 layer with rows of whole vectors")
        q4 = w // 4
        if wx < 1 or wx > 8 or 2 * q4 > 64:
            raise InvalidConfig("row exchange: 1 .. 8 chunks per lane, rows of at most 128 floats")
        # rows per instruction: as many as fit 64 lanes, fewer when that makes the spans tile the plane
        rpi_max = min(64 // q4, h)
        rpi = max([r for r in range(1, rpi_max + 1) if h % (r * wx) == 0] or [0])
        if rpi * 4 < rpi_max * 3:
            rpi = rpi_max         # too few lanes would carry work: ragged last span instead
        rows = rpi * wx
        if (waves * (rows + 2) * q4 + 64) * 16 > LDS_BYTES:      # 64 chunks of slack for the idle lanes' reads
            raise InvalidConfig("row-exchange windows do not fit the LDS")
        D = dict(NT=nt, TH=th, TW=tw, NT_STORE=nt_mode & 1, NT_LOAD=nt_mode >> 1, SHFL=0, WX=wx, WXR=rpi,
                 CB=b, CC=c, CH=h, CW=w, CR=r_ext, CS=s_ext, FACT=1, CP=p, CQ=q, **steps)
        return [KernelSpec("depthwise_f32.hip", "depthwise_f32", D,
                           (ceil_div(b * cout * ceil_div(h, rows), waves), 1, 1), (nt, 1, 1), args)]
    shfl = int(_special(special, "halo_shfl")[0])
    tiles_w = ceil_div(q, tw)
    if shfl:
        if not (vec_rows and st_w == 1 and s_ext == 3 and dl_w == 1 and pad_w == 1 and tiles_w <= 64):
            raise InvalidConfig("the shuffled halo needs the 128-bit input path of a 3-wide pad-1 layer")
        lanes = (64 // tiles_w) * tiles_w
        grid_x = ceil_div(ceil_div(items, lanes), waves * ipl)
    else:
        grid_x = ceil_div(items, nt * ipl)
    D = dict(NT=nt, TH=th, TW=tw, NT_STORE=nt_mode & 1, NT_LOAD=nt_mode >> 1, SHFL=shfl,
             CB=b, CC=c, CH=h, CW=w, CR=r_ext, CS=s_ext, FACT=a["factor"], CP=p, CQ=q, **steps)
    if ipl > 1:
        D.update(IPL=ipl)
    if fm > 1:
        D.update(MFUSE=1)
    return [KernelSpec("depthwise_f32.hip", "depthwise_f32", D, (grid_x, 1, 1), (nt, 1, 1), args)]


def _lower_pad(op, out_name, in_names):
    b, c, ph, pw = [x.extent for x in op.axis]
    pt, pb, pl, pr = op.attrs["padding"]          # rows above / below, columns left / right
    h, w = ph - pt - pb, pw - pl - pr
    D = dict(PADK=1, PB=b * c, CH=h, CW=w, PT=pt, PBOT=pb, PL=pl, PR=pr)
    n = b * c * ph * pw
    return [KernelSpec("elementwise.hip", "zero_pad2d_f32", D, (ceil_div(n, 256), 1, 1),
                       (256, 1, 1), [("buf", in_names[0]), ("buf", out_name)])]


def _lower_bias(op, out_name, in_names):
    if op.kind == "bias_add_ghw":
        # [groups][Mg][N] is one image of groups*Mg channels with N elements each
        g, mg, hw = [x.extent for x in op.axis]
        b, c, h, w = 1, g * mg, 1, hw
    else:
        b, c, h, w = [x.extent for x in op.axis]
    n = b * c * h * w
    return [KernelSpec("elementwise.hip", "bias_add_nchw_f32", {},
                       (min(ceil_div(n, 256), 4096), 1, 1), (256, 1, 1),
                       [("buf", in_names[0]), ("buf", in_names[1]), ("buf", out_name),
                        ("i32", n), ("i32", h * w), ("i32", c)])]


def _conv_defines(attrs, materialized_pad):
    b, cin, h, w = attrs["in_shape"]
    steps = _conv_steps(attrs)
    if materialized_pad:
        h, w = h + 2 * steps["CPADH"], w + 2 * steps["CPADW"]
        steps["CPADH"] = steps["CPADW"] = 0
    groups = attrs["groups"]
    return dict(COLK=1, CB=b, CG=groups, CC=cin, CH=h, CW=w, CR=attrs["kernel"][0], CS=attrs["kernel"][1],
                CP=attrs["out_hw"][0], CQ=attrs["out_hw"][1], MG=attrs["out_channel"] // groups, **steps)


def _lower_im2col(op, out_name, in_names, materialized_pad):
    g, k, n = [x.extent for x in op.axis]
    total = g * k * n
    return [KernelSpec("elementwise.hip", "im2col_nchw_f32", _conv_defines(op.attrs, materialized_pad),
                       (min(ceil_div(total, 256), 16384), 1, 1), (256, 1, 1),
                       [("buf", in_names[0]), ("buf", out_name)])]


def _lower_col2img(op, out_name, in_names):
    b, c, p, q = [x.extent for x in op.axis]
    g, mg, _ = op.input_tensors[0].shape
    # only the output geometry matters to this kernel; the image constants are placeholders
    D = dict(COLK=1, CB=b, CG=g, CC=g, CH=1, CW=1, CR=1, CS=1, CSTRH=1, CSTRW=1, CPADH=0, CPADW=0,
             CDILH=1, CDILW=1, CP=p, CQ=q, MG=mg)
    total = b * c * p * q
    return [KernelSpec("elementwise.hip", "col2img_nchw_f32", D,
                       (min(ceil_div(total, 256), 16384), 1, 1), (256, 1, 1),
                       [("buf", in_names[0]), ("buf", out_name)])]


def lower(op, config, special, out_name, in_names, materialized_pad=False, bias_name=None,
          through=(), merged_out=None):
    """Config of one operator -> list of KernelSpec (raises InvalidConfig).
    ``bias_name``: buffer of a per-channel bias merged into the epilogue;
    ``through``: kinds of the inlined producers the operator reads through;
    ``merged_out``: kind of a layout stage merged into the operator's stores."""
    if op.kind in GEMM_KINDS:
        return _lower_gemm(op, config, special, out_name, in_names, materialized_pad, bias_name,
                           through, merged_out)
    if merged_out is not None:
        raise InvalidConfig("operator kind %s takes no merged stage" % op.kind)
    if op.kind == "depthwise_conv2d_nchw":
        return _lower_depthwise(op, config, special, out_name, in_names, materialized_pad, bias_name)
    if bias_name is not None:
        raise InvalidConfig("operator kind %s has no bias epilogue" % op.kind)
    if op.kind == "im2col_nchw":
        return _lower_im2col(op, out_name, in_names, materialized_pad)
    if op.kind == "col2img_nchw":
        return _lower_col2img(op, out_name, in_names)
    if op.kind in ("bias_add_nchw", "bias_add_ghw"):
        return _lower_bias(op, out_name, in_names)
    if op.kind == "zero_pad2d":
        return _lower_pad(op, out_name, in_names)
    raise InvalidConfig("no gfx950 template for operator kind %s" % op.kind)


# --------------------------------------------------------------------------
# default (untuned) configs
# --------------------------------------------------------------------------

def _empty_config():
    return {k: [] for k in Space.valid_type_keys}


# tiles of the int8 default: (wavefronts, MFMA tiles per wavefront) along M and along N, 16x16x64 MFMAs
I8_TILES = (((2, 1), (2, 1)), ((2, 1), (2, 2)), ((4, 1), (2, 2)), ((2, 2), (4, 2)), ((4, 2), (2, 4)),
            ((4, 4), (4, 4)), ((1, 1), (4, 1)))


def _default_i8(view, padded=False):
    """Tile, K tile and K division of an int8 GEMM nobody tuned: the smallest predicted time over a few
    tiles that between them are within 3 % of the best measured one everywhere.

    The prediction, in clocks of one compute unit (2.3 GHz under this load): the busiest unit has n = tiles /
    256 of them; per byte of K a tile costs the longest of its matrix work, its LDS traffic (operand reads of
    all wavefronts, plus the tile's own bytes where they pass through registers) and its share of the L2's
    64 bytes per clock, plus a quarter of their sum because they do not overlap perfectly; but no tile is
    faster than its chain of k steps (230 clocks each, a barrier and an LDS round trip) behind the 1750
    clocks until the first operands are there, and only as many tiles run side by side as the LDS holds. The
    factors were fitted to 1 230 timings over 48 sizes (64 .. 4096 an axis, half of them no multiples
    of 16) of the kernels with two LDS buffers, among whose candidates the rule's pick was within 6 % of the best in
    the geometric mean: 64x3632x1376 4.8 us, 1712x1584x2080 13.6, 3488x176x80 2.6. With the third buffer and eight
    wavefronts on 64x64 tiles it is within 3.8 % of the best of 895 timings over 52 further sizes.
    """
    aligned = view.K % 16 == 0 and not padded        # tiles straight into LDS
    dwords = view.K % 4 == 0 and not padded          # into three buffers of it
    best = None
    for (wm, rm), (wn, rn) in I8_TILES:
        bm, bn = wm * rm * 16, wn * rn * 16
        if (bm >= 2 * view.M and bm > 32) or (bn >= 2 * view.N and bn > 32) or (bm > 128 and not aligned):
            continue
        tm, tn = ceil_div(view.M, bm), ceil_div(view.N, bn)
        tiles = tm * tn
        n = ceil_div(tiles, NUM_CUS)
        for bk in (128, 256):
            for groups in (1, 2, 4):
                # K of 64x64 tiles divided: 27 of 29 sizes 1.04 .. 1.29 times slower, the others have better tiles
                if groups > 1 and (tiles > 300 or view.K < bk * groups or bm == bn == 64) or groups * wm * wn > 16:
                    continue
                steps = ceil_div(view.K, bk * groups)
                if bm == bn == 64 and steps < 3 and n > 1:
                    wm, rm, wn, rn = 2, 2, 2, 2                # 297 .. 817 tiles: eight wavefronts 2 .. 7 % slower
                lds = groups * 2 * (bm + bn) * bk
                # A third LDS buffer: a tile's loads have two steps to land instead of one, which is what a step waits
                # for when its operands are not in the L2 yet (144 tiles of 64x64 at K = 3808: 15.8 -> 9.8 us; 216 of
                # 32x64 at K = 3536: 12.8 -> 8.3). Not where it leaves a compute unit with one workgroup at a time
                # out of several (425 tiles of 128x128 at 10 steps: 15.7 -> 17.3).
                third = dwords and steps > 2 and lds * 3 // 2 * min(n, 2) <= LDS_BYTES
                if third:
                    lds = lds * 3 // 2
                if lds > LDS_BYTES or ((aligned or third) and ((bm * bk // 16) % (wm * wn * 64)
                                                               or (bn * bk // 16) % (wm * wn * 64))):
                    continue
                if not (aligned or third) and (ceil_div(bm * bk // 16, wm * wn * 64)
                                               + ceil_div(bn * bk // 16, wm * wn * 64)) * 8 > 160:
                    continue          # staging registers
                mfma = bm * bn * 2 * 1.12 / 8192.0
                reads = 16 if bm == bn == 64 else wm * wn * (rm + rn)      # eight wavefronts of 64x64 hide what they read more
                lds_rw = (reads * 16 + (bm + bn) * (0.7 if aligned else 3.7)) * 0.96 / 128.0
                l2 = (bm + bn) * 0.68 / 64.0
                work = n * steps * bk * groups * (max(mfma, lds_rw, l2) + 0.23 * (mfma + lds_rw + l2))
                beside = max(1, min(LDS_BYTES // lds, 32 // (wm * wn * groups), n))
                chain = ceil_div(n, beside) * (steps * 230 + 1750 + (220 * rm * rn * (groups - 1)))
                clocks = max(work, chain) + n * bm * bn * 4 * 2.3 / 64.0
                if best is None or clocks < best[0]:
                    best = (clocks, [tm, wm, rm, 16], [tn, wn, rn, 16], [groups, steps, bk], third)
    cfg = _empty_config()
    _, tile_m, tile_n, reduce, third = best
    cfg["spatial"] = [tile_m, tile_n]
    cfg["reduce"] = [reduce]
    # Straight into LDS where rows are 16-byte aligned, with three buffers where they are whole dwords (1063x1844x486
    # 5.78 -> 4.69 us, 318x3700x534 5.56 -> 4.94). Otherwise two tiles ahead in registers (164 tiles of 64x64 at
    # K = 2050 8.0 -> 7.1 us against the fragment prefetch, 180 of 64x128 15.7 -> 11.5), for tiles of 32x32 from eight
    # steps on (72 at K = 2800: 5.70 -> 5.32; fewer steps: the same). Those of 32x64 keep the prefetch (188 at K = 2524:
    # 4.97 against 5.69) up to 25 steps; from about there on its steps take 370 ns instead of 250 at most sizes (why is
    # not known), and three tiles ahead is faster: of 47 sizes at K = 2800 .. 4057 the 14 of up to 25 steps take
    # 0.77 .. 1.05 of its time, half of them above 1, the 33 of more 0.75 .. 1.05, one above 1.02, 0.80 in the geometric
    # mean (1251x4045x361 14.1 -> 10.5 us).
    size = tile_m[1] * tile_m[2] * tile_n[1] * tile_n[2]
    ahead = size >= 16 or (size == 4 and reduce[1] >= 8)
    long = size == 8 and reduce[1] > 25
    cfg["unroll"] = [[9 if third else 6 if aligned else 3 if ahead else 4 if long else 5, 1]]
    cfg["fuse"] = [[4]]
    cfg["reorder"] = [[1, 1 if reduce[0] > 1 else 0, 0]]
    return cfg


# kernels of the fp32 default: (wavefronts, MFMA tiles per wavefront) along M and N, MFMA edge, K tile, pipeline depth
F32_KERNELS = (((1, 1), (1, 1), 16, 16, 2), ((1, 1), (1, 1), 16, 32, 3), ((1, 1), (4, 1), 16, 32, 3),
               ((1, 1), (4, 1), 16, 64, 8), ((2, 1), (1, 1), 16, 32, 3), ((2, 1), (2, 1), 16, 32, 3),
               ((2, 1), (2, 1), 16, 32, 5), ((2, 1), (4, 1), 16, 64, 8), ((4, 1), (4, 1), 16, 64, 8),
               ((4, 2), (4, 1), 16, 32, 5), ((2, 1), (2, 1), 32, 16, 2), ((4, 1), (2, 1), 32, 32, 5),
               ((2, 2), (4, 1), 16, 32, 5), ((4, 2), (4, 2), 16, 16, 1))


def _f32_clocks(view, tiles, m, n, mf, bk, depth, groups, call=False):
    """Predicted clocks (2.38 GHz) of an fp32 contraction on the busiest compute unit, see _default_f32; or of a whole
    ``call``, to be held against tiles without LDS, see _pick_f32."""
    (wm, rm), (wn, rn) = m, n
    bm, bn = wm * rm * mf, wn * rn * mf
    steps = ceil_div(view.K, bk * groups)
    nw = wm * wn * groups
    lds = groups * (1 if depth == 1 else 2) * 4 * (bm + bn) * bk
    if lds > LDS_BYTES:
        return None
    share = ceil_div(tiles, NUM_CUS)                                # output tiles of the busiest unit
    beside = max(1, min(LDS_BYTES // lds, 32 // nw))                # of which run side by side
    step = rm * rn * mf * mf * 2 * bk / 64.0                        # matrix clocks of one wavefront's k step
    matrix = ceil_div(share * nw, 4) * step * steps                 # four matrix cores
    latency = {1: 100, 2: 110, 3: 370, 5: 450, 8: 420}[depth] * (1 + 0.12 * bk / 32) + 30 * nw
    overlap = {1: 0.2, 2: 0.8, 3: 0.4, 5: 0.3, 8: 0.35}[depth]      # share of a step's own MFMAs the chain waits for
    turns = ceil_div(share, beside)
    chain = turns * (steps * (latency + step * ceil_div(nw, 4) * overlap) + 930)
    # the lower rate was fitted when only counts that 8 divides were renumbered by XCD; it still steers to those, which
    # end in whole rounds (one rate for all: 24 drawn batches 1 % faster in the mean, single pointwise layers up to 16 % slower)
    rate = 31 if call or view.groups == 1 or tiles % 8 == 0 else 14
    operands = tiles * (bm + bn) * steps * bk * groups * 4.0 / NUM_CUS / rate
    longest = max(matrix, chain, operands)
    clocks = (longest + 0.35 * (matrix + chain + operands - longest) + share * bm * bn * 4 * 4.8 / 64
              + (38 * rm * rn * mf * mf / 64 * (groups - 1)))
    if not call:
        return clocks
    # what the picks' times showed beside the launch: vectors of rows that are no whole ones lie across two lines each, and
    # several workgroups of wavefront groups on one unit are in each other's way (210 and 294 tiles of 80 and
    # 112x1500x667: 6.7 and 10.2 us)
    clocks *= 0.976
    vectors = share * steps * bk * groups * 4 / 64.0
    clocks += 0.6 * vectors * ((bm if view.K % 4 else 0) + (bn if view.N % 4 else 0))
    if groups > 1 and min(share, beside) > 1:
        clocks += 0.29 * chain
    return clocks + 4150


def _default_f32(view, padded=False, direct=True):
    """Tile, K tile, pipeline and K division of an fp32 GEMM (or a batch of them) nobody tuned: the smallest
    predicted time over F32_KERNELS, which between them are within 2 % of the best measured kernel everywhere.

    An fp32 MFMA is slow next to the loads that feed it (16x16x4: 32 clocks), so what decides is how evenly
    the tiles fill 256 compute units of four matrix cores, and for few tiles the chain of k steps (load, barrier,
    LDS round trip) that nothing hides. The prediction takes, for the busiest unit, the longest of its matrix
    clocks, that chain, and its share of the operand traffic (31 bytes per clock and unit), adds a third of the
    other two, the stores of C and the sum over wavefront groups. Constants fitted to 5 200 timings over 72
    sizes (M, N, K 8 .. 4096, batches of 26 .. 128; half of them no multiples of 4); the pick is within 5 % of the
    best measured in the geometric mean and 1.6 times as fast as the rule before it (square-ish power-of-two
    tiles until every unit has one, K tiles of 32): 1100x1301x900 47.1 -> 30.0 us, 863x1862x1280 (B^T) 69.7 ->
    44.4, 96 x 74x96x133 6.8 -> 5.4, 32x4096x3072 43.6 -> 16.5. Batches whose tiles are no multiple of 8 go at a lower
    rate (14 bytes per clock and unit, fitted when such grids were not renumbered; 86 batches measured: 3.8 % off the best kernel, with
    one rate for all 11.5 % off and up to 1.5 times as slow as the rule before): 121 x 35x80x124 6.33 -> 4.16 us,
    114 x 68x110x63 (B^T) 6.38 -> 4.88, 63 x 52x80x274 7.01 -> 5.21. K streaming is left to the search: a plan that owns a
    workspace cannot run on two streams at once, and a default plan can.
    """
    cfg, _, call = _pick_f32(view, F32_KERNELS, _f32_clocks, padded, direct)
    return _or_split(view, cfg, call) if direct and not padded else cfg


# kernels without LDS tiles that the defaults choose among: MFMA tiles per wavefront along M and N, k steps ahead
DIRECT_KERNELS = ((1, 1, 2), (1, 2, 2), (2, 2, 2), (1, 4, 2))


def _direct_clocks(view, m, n, pd, groups):
    """Predicted clocks (2.38 GHz) of a call on tiles without LDS, the launch included; see _pick_f32."""
    tiles = ceil_div(view.M, m * 16) * ceil_div(view.N, n * 16)
    steps = ceil_div(ceil_div(view.K, 32), groups)
    share = ceil_div(tiles, NUM_CUS)
    beside = max(1, min(share, min(8, 512 // (4 * m * n + 8 * (m + n) * pd + 40)) * 4 // groups))
    step = m * n * 256                                              # matrix clocks of a wavefront's k step
    # clocks a unit spends on a step's loads: two vectors per row block; per column one float and k (with a stride of 2
    # along the rows a load spreads over twice the lines), or a vector of n floats. Before the first step: the operands'
    # latency, or the gathered operand's table of offsets and its pixels' padding bits, both once; the table's entries
    # are read anew in every step.
    if view.conv:
        loads = (2 * m * 23 + 8 * n * 7.4 * (2 if view.conv["CSTRW"] > 1 else 1)) * (1 + 0.056 * (groups - 1))
        once = 186.0 * view.K / (64 * groups) + 144 * n * (view.conv["CR"] + view.conv["CS"])
        start, mix, store, sums, launch, entries = 0, 0.34, 9.7, 0, 4600, 62
    else:
        # rows of B that are no whole vectors: four neighbouring floats lie across two 16-byte pieces
        column = {1: 8.2, 2: 17, 4: 23} if view.N % 4 == 0 else {1: 12.8, 2: 18.4, 4: 25.5}
        loads = (2 * m * 44 + 8 * column[n]) * (1 + 0.025 * (groups - 1))
        once, start, mix, store, sums, launch, entries = 0, 844, 0.24, 8.9, 9.4, 4380, 0
    # wavefronts of one matrix core; two workgroups of two wavefronts go as if they shared two of the four (timed, not traced)
    wavefronts = 2 if share == groups == 2 else ceil_div(share * groups, 4)
    matrix = wavefronts * steps * step
    memory = share * groups * steps * loads
    chain = ceil_div(share, beside) * (steps * max(94.0 / pd + 0.19 * step, step) + start) + once
    # operands once at the rate of a large copy
    stream = 0 if view.conv else (view.M * view.K + view.K * view.N) * 4 / 1930.0
    longest = max(matrix, memory, chain)
    return (max(longest + mix * (matrix + memory + chain - longest), stream) + share * m * n * 1024 * store / 64
            + entries * share * groups * steps + sums * m * n * (groups - 1) + launch)


def _pick_f32(view, kernels, predict, padded, direct):
    """The config of the kernel and number of wavefront K groups with the smallest predicted time, that time (the
    LDS kernel's also where tiles without LDS are taken), and the predicted time of a call; where the LDS rows are to be padded, among the kernels whose tiles
    pass through registers, with K undivided (the groups' tiles lie beside each other in LDS).

    Against it stand the tiles without LDS, which for GEMMs have to be predicted 8 % faster, for windows faster at all. The
    two predictions of a call are off by 10 % each (one standard deviation), fitted to the LDS picks and to 1 368 timings of
    the tiles without LDS over 400 GEMMs (8 .. 4096 rows, half of them with K and N multiples of 16), for windows to 1 887
    and 1 233 timings over 230 layers. Over 357 GEMMs timed on both, the picks take 0.979 times the LDS kernels' time in the
    geometric mean, ten are more than 3 % slower than those, four more than 8 %. One rule whatever the rows and their
    alignment: 64x1500x667 6.9 us with LDS and 7.3 without, 32x4096x4096 18.7 and 19.2, 74x3120x1200 22.7 and 14.3,
    57x1610x1067 11.1 and 8.9, 112x4096x4096 36.6 and 50.4.
    Not for 1x1 windows, whose gathers the LDS kernels do without index arithmetic (7 x 259x90x90 -> 25 16.4 us, 18.4
    without LDS); not for strides of more than 2 along the rows, where the few layers timed took up to 1.5 times the predicted
    time (16x208x51x15 -> 164 1x3 stride 3 10.9 us, 16.4 without LDS); and not for B stored [N][K] nor for batches: with few
    k steps the operands' latency is all there is, and tiles that share it through LDS have it once (96 x 197x64x197 10.0 us,
    14.5 without LDS; 57x1249x714 with B^T 5.3 and 7.0)."""
    best = None
    window = view.conv["CR"] * view.conv["CS"] if view.conv else 1
    for m, n, mf, bk, depth in kernels:
        if padded and depth >= 5:
            continue
        bm, bn = m[0] * m[1] * mf, n[0] * n[1] * mf
        if bm >= 2 * max(view.M, 16) or bn >= 2 * max(view.N, 16):
            continue
        if depth >= 5 and view.trans_a:
            if bm % 64 or view.M % 4:
                continue
        elif depth >= 5 and view.K < 4:
            continue
        tm, tn = ceil_div(view.M, bm), ceil_div(view.N, bn)
        tiles = tm * tn * view.groups
        for groups in (1, 2, 4, 8, 16):
            if groups > 1 and (padded or tiles > 400 or groups * m[0] * n[0] > 16):
                break
            steps = ceil_div(view.K, bk * groups)
            kp = steps * bk * groups
            if kp not in view.KP_options and kp * 4 > view.K * 5:
                break
            # its matrix clocks alone are more than the best: not worth a prediction
            if best is not None and -(-tiles // NUM_CUS) * m[0] * n[0] * groups * m[1] * n[1] * mf * mf * bk * steps > best[0] * 128:
                continue
            clocks = predict(view, tiles, m, n, mf, bk, depth, groups)
            if clocks is not None and (best is None or clocks < best[0]):
                best = (clocks, [tm, m[0], m[1], mf], [tn, n[0], n[1], mf], [groups, steps, bk], depth)
                kernel = (tiles, m, n, mf, bk, depth, groups)
    call = predict(view, *kernel, call=True)
    if direct and view.groups == 1 and view.mode != 2 and not view.trans_a and view.K >= 32 \
            and (not view.conv or 1 < window <= 31 and view.K * 8 + 256 < LDS_BYTES and view.conv["CSTRW"] <= 2):
        limit = call / (1 if view.conv else 1.08)
        for m, n, pd in DIRECT_KERNELS:
            if m * 16 >= 2 * max(view.M, 16) or n * 16 >= 2 * max(view.N, 16):
                continue
            tm, tn = ceil_div(view.M, m * 16), ceil_div(view.N, n * 16)
            if tm * tn * m * n * view.K * 8.0 / (4 * NUM_CUS) > limit:          # matrix clocks alone
                continue
            for groups in (1, 2, 4, 8):
                kp = ceil_div(view.K, 32 * groups) * 32 * groups
                if groups > 1 and tm * tn > 3000 or tm * tn * groups < 128 \
                        or -(-tm * tn // NUM_CUS) * groups // 4 * (kp // (32 * groups)) * m * n * 256 > limit or kp * 4 > view.K * 5 and kp not in view.KP_options:
                    continue
                clocks = _direct_clocks(view, m, n, pd, groups)
                if clocks < limit:
                    limit = call = clocks
                    best = (best[0], [tm, 1, m, 16], [tn, 1, n, 16], [groups, kp // (32 * groups), 32], pd, 1)
    cfg = _empty_config()
    cfg["spatial"] = [best[1], best[2]]
    cfg["reduce"] = [best[3]]
    cfg["unroll"] = [[best[4], 1]]
    cfg["fuse"] = [[4]]
    cfg["reorder"] = [[1, 1 if best[3][0] > 1 else 0, 0] + list(best[5:])]
    return cfg, best[0], call


# kernels of products in bf16 parts that the defaults choose among: (wavefronts, MFMA tiles per wavefront) along M and N,
# MFMA edge, K groups, pipeline depth; and 32x32 MFMA tiles along M and N of a wavefront on its own, K groups
SPLIT_KERNELS = (((2, 2), (4, 1), 32, 1, 9), ((4, 1), (2, 1), 32, 1, 9), ((4, 1), (2, 1), 32, 2, 9), ((2, 2), (4, 1), 16, 1, 9),
                 ((2, 2), (4, 1), 16, 2, 10), ((2, 1), (4, 1), 16, 1, 9))
ALONE_KERNELS = ((2, 2, 8), (2, 2, 4), (2, 1, 8), (1, 1, 8), (1, 1, 4))


def _split_step(m, n, mf, groups):
    """What the step of such a kernel costs one unit whatever the operator: tile, wavefronts, instructions of a thread for
    its share of the tile's elements and of the gathered ones, of the MFMAs (one keeps the others out for 8 clocks, 10 the
    large one, another instruction for 4), LDS (six bytes an element in at 70 bytes a clock, out at 230), and the bytes of
    LDS."""
    (wm, rm), (wn, rn) = m, n
    bm, bn, waves = wm * rm * mf, wn * rn * mf, wm * wn
    return (bm, bn, waves * groups, (bm + bn) * 3.0 / waves, bn * 1.0 / waves, 6 * rm * rn * (20 if mf == 32 else 8),
            groups * ((bm + bn) * 192 / 70.0 + waves * (rm + rn) * mf * 192 / 230.0), groups * 384 * (bm + bn) + 16)


SPLIT_STEPS = {k[:4]: _split_step(*k[:4]) for k in SPLIT_KERNELS}


def _split_clocks(view, m, n, mf, groups):
    """Predicted clocks (2.38 GHz) of a call of the split kernel of igemm_f32.hip; see _or_split."""
    bm, bn, waves, share_ab, share_b, matrix, lds, lds_bytes = SPLIT_STEPS[m, n, mf, groups]
    share = -(-(-(-view.M // bm) * -(-view.N // bn) * view.groups) // NUM_CUS)
    steps = -(-view.K // (32 * groups))
    turns = -(-share // max(1, min(share, LDS_BYTES // lds_bytes, 32 // waves)))
    # rows of whole lines by the kilobyte, a vector less where rows are no whole ones; the gathered operand by 64 elements
    loads = groups * bm * (4.55 if view.K % 4 else 3.5)
    if view.conv:
        vector = share_ab + share_b
        loads += groups * bn * (9.27 if view.conv["CSTRW"] > 1 else 5.55)
        latency, start, mix, store, sums, launch, lds = 1007 + 17.2 * waves, 1310, 0.518, 6.45, 139, 4110, 0.97 * lds
    else:
        vector = share_ab
        loads += groups * bn * (0.84 if (view.K if view.mode == 2 else view.N) % 4 else 0.64)
        latency, start, mix, store, sums, launch, lds = 616 + 4.8 * waves, 412, 0.467, 6.93, 134, 3780, 0.86 * lds
    issue = waves * (matrix + 4 * (vector + 1)) / 4
    longest = max(issue, lds, loads)
    work = longest + mix * (issue + lds + loads - longest)
    return (max(share * steps * work, turns * steps * (latency + 0.6 * work)) + turns * start + share * bm * bn * store / 16
            + sums * bm * bn / 64.0 * (groups - 1) * groups / waves + launch)


def _alone_clocks(view, rm, rn, groups):
    """Predicted clocks (2.38 GHz) of a call of the split kernel of direct_f32.hip; see _or_split."""
    conv = view.conv is not None
    tiles = ceil_div(view.M, 32 * rm) * ceil_div(view.N, 32 * rn) * view.groups
    share, steps = ceil_div(tiles, NUM_CUS), ceil_div(ceil_div(view.K, 32), groups)
    lds = max(groups * (rm + (rn if view.mode == 2 else 0)) * 8192 + (view.K * 8 if conv else 0), groups * rm * rn * 4096)
    turns = ceil_div(share, max(1, min(share, LDS_BYTES // lds, max(1, (8 if rm * rn > 2 else 12) // groups))))
    issue = groups * (120 * rm * rn + 4 * ((rm + rn) * 96 + (48 * rn if conv else 0))) / 4.0
    if conv:
        loads = groups * (rm * 4 * 4.4 * (1.3 if view.K % 4 else 1) + 16 * rn * 3.5 * (4.43 if view.conv["CSTRW"] > 1 else 1))
        latency, mix, store, sums, launch = 1020 + 123, 0.394, 20, 263, 4530
        start = 25 + 38.6 * rn * (view.conv["CR"] + view.conv["CS"]) + 1480.0 * view.K / (groups * 64)
    else:
        rows = rm * 4 + (rn * 4 if view.mode == 2 else 0)
        loads = groups * (rows * 11.8 * (1.3 if view.K % 4 else 1)
                          + (0 if view.mode == 2 else 16 * 1.49 * (1 if rn == 2 else 0.75) * (1.3 if view.N % 4 else 1)))
        latency, start, mix, store, sums, launch = 1490, 1180, 1.34, 14.9, 274, 2170
    longest = max(issue, loads)
    work = longest + mix * (issue + loads - longest)
    return (max(share * steps * work, turns * steps * (latency + 0.5 * work)) + turns * start + share * rm * rn * 1024 * store / 16
            + sums * rm * rn * (groups - 1) + launch)


def _or_split(view, cfg, call):
    """``cfg``, whose call is predicted to take ``call`` clocks, or the best predicted kernel with products in bf16 parts
    where that is 8 % and 500 clocks faster.

    Both predictions were fitted to 2 427 timings over 150 operators (GEMMs of 8 .. 4096 an axis, batches of 8 .. 128, 3x3 and
    1x1 layers of 1 .. 16 images, 16 .. 512 channels, stride 1 and 2) and are off by 10 % (one standard deviation), like
    those of the fp32 kernels. Over these operators the picks take 0.954 times the time without them in the geometric mean
    (0.937 if every pick were the fastest), four are more than 2 % slower (10.3 us at 1.11), and all of them together 1 866
    us for 2 149: what is long gains most. These timings are of parts of x itself; parts of 2^23 x take the kernel of
    direct_f32.hip 3 % longer in the mean, 5 .. 9 % with one block a wavefront. 94 operators drawn since that it changes: 0.866,
    13 more than 2 % slower, one at 1.14 (0.852, ten and 1.10 with parts of x). With the factor in the prediction six of
    them go back, three of which were at 0.80 .. 0.89 and two above 1, so it is left out.
    Four blocks of a wavefront on its own have one set of accumulators, which rounds 1.3 times as much as the fp32 kernels
    do with K divided alike: they are for at least twice the groups."""
    if view.trans_a or view.K < 32 or view.conv and (
            view.groups > 1 or view.conv["CR"] * view.conv["CS"] > 31 or view.conv["CSTRW"] > 2 or view.K > 4096):
        return cfg
    limit, best = (call - 500) / 1.08, None
    before = cfg["reduce"][0][0]
    for m, n, mf, groups, depth in SPLIT_KERNELS:
        if m[0] * m[1] * mf >= 2 * max(view.M, 16) or n[0] * n[1] * mf >= 2 * max(view.N, 16) \
                or view.conv and _gathered_bytes(view.conv, 1) >= 2 ** 31:
            continue
        # launch, chain of steps, and matrix clocks alone: not worth a prediction
        steps = -(-view.K // (32 * groups))
        if view.K < 64 * groups or 3780 + steps * 616 > limit or steps * m[0] * n[0] * groups * m[1] * n[1] * mf * mf * 0.09 > limit:
            continue
        if groups > 1 and -(-view.M // (m[0] * m[1] * mf)) * -(-view.N // (n[0] * n[1] * mf)) * view.groups > 2 * NUM_CUS:
            continue                                # not among the timed: K divided where tiles are many
        clocks = _split_clocks(view, m, n, mf, groups)
        if clocks < limit:
            limit, best = clocks, ((m[0], m[1], mf), (n[0], n[1], mf), groups, depth)
    for rm, rn, groups in ALONE_KERNELS:
        if rm * 32 >= 2 * max(view.M, 32) or rn * 32 >= 2 * max(view.N, 32) or view.K < 32 * groups \
                or rm * rn == 4 and groups < 2 * before or 2170 + -(-view.K // (32 * groups)) * 1020 > limit:
            continue
        if groups > 4 and -(-view.M // (32 * rm)) * -(-view.N // (32 * rn)) * view.groups > 4 * NUM_CUS:
            continue
        lds = groups * 8192 * (rm + (rn if view.mode == 2 else 0)) + (ceil_div(view.K, 32) * 256 if view.conv else 0)
        clocks = _alone_clocks(view, rm, rn, groups) if lds <= LDS_BYTES else limit
        if clocks < limit:
            limit, best = clocks, ((1, rm, 32), (1, rn, 32), groups, 11)
    if best is None:
        return cfg
    (wm, rm, mf), (wn, rn, _), groups, depth = best
    cfg = _empty_config()
    cfg["spatial"] = [[ceil_div(view.M, wm * rm * mf), wm, rm, mf], [ceil_div(view.N, wn * rn * mf), wn, rn, mf]]
    cfg["reduce"] = [[groups, ceil_div(view.K, 32 * groups), 32]]
    cfg["unroll"] = [[depth, 1]]
    cfg["fuse"] = [[4]]
    cfg["reorder"] = [[1, 1 if groups > 1 else 0, 0]]
    return cfg


# kernels of the convolution's default, as F32_KERNELS: for windows of one pixel, and for larger ones
CONV_KERNELS = (((1, 1), (1, 1), 16, 16, 2), ((1, 1), (1, 1), 16, 32, 3), ((2, 1), (2, 1), 16, 32, 3),
                ((4, 1), (2, 1), 16, 32, 3), ((2, 2), (4, 1), 16, 16, 2), ((2, 1), (4, 1), 16, 16, 2),
                ((4, 2), (4, 1), 16, 32, 5), ((2, 1), (2, 1), 32, 16, 3))
WINDOW_KERNELS = (((1, 1), (1, 1), 16, 16, 2), ((2, 1), (4, 1), 16, 16, 2), ((2, 2), (4, 1), 16, 16, 2),
                  ((2, 1), (2, 1), 32, 16, 3),                                         # any K
                  ((1, 1), (1, 1), 16, 32, 3), ((2, 1), (2, 1), 16, 32, 3), ((4, 1), (2, 1), 16, 32, 3),
                  ((2, 1), (4, 1), 16, 32, 5), ((4, 2), (4, 1), 16, 32, 3), ((4, 1), (4, 1), 16, 32, 8),
                  ((4, 1), (4, 1), 16, 64, 8),
                  ((2, 1), (2, 1), 16, 144, 8), ((2, 1), (2, 1), 32, 72, 8), ((4, 1), (2, 1), 32, 72, 8))


def _conv_clocks(view, tiles, m, n, mf, bk, depth, groups, call=False):
    """Predicted clocks (2.38 GHz) of a convolution on the busiest compute unit, or of a whole ``call``; see
    _default_conv. The numbers are fitted, and those of the gather stand for all that a load costs there."""
    (wm, rm), (wn, rn) = m, n
    bm, bn = wm * rm * mf, wn * rn * mf
    steps = ceil_div(view.K, bk * groups)
    nw = wm * wn * groups
    lds = groups * 2 * 4 * (bm + bn) * bk
    window = view.conv["CR"] * view.conv["CS"]
    if lds > LDS_BYTES or bk in (72, 144) and bk % window:              # those K tiles are for the whole windows they hold
        return None
    share = ceil_div(tiles, NUM_CUS)
    turns = ceil_div(share, max(1, min(LDS_BYTES // lds, 32 // nw)))
    step = rm * rn * mf * mf * 2 * bk / 64.0                            # matrix clocks of one wavefront's k step
    gathered = groups * bn * bk / 64.0                                  # loads of a step's gather, all wavefronts
    if window == 1:
        latency = {2: 129, 3: 125, 5: 457, 8: 1499}[depth] * (1 + 0.12 * bk / 32) + 33 * nw
        overlap = {2: 0.8, 3: 0.4, 5: 0.3, 8: 0.35}[depth]
        gather, gather_chain, start, mix, store, sums = 3.7, 0, 3230, 0.47, 3.0, 82
        rate = 16 if tiles % 8 == 0 else 9                              # as in _f32_clocks
        operands = tiles * (bm + bn) * steps * bk * groups * 4.0 / NUM_CUS / rate
    else:
        latency = {2: 132, 3: 31, 5: 117, 8: 166 if bk > 64 else 3}[depth] * (1 + 0.12 * bk / 32) + 18 * nw
        overlap, mix, store, sums = 0.13, 1.0, 4.7, 45
        # channel and tap: hoisted out of the loop (what is left are the loads), scalars, or lane by lane; before the
        # loop, per element of a thread its offset, or per pixel of a thread its padding bits
        threads = wm * wn * 64
        elements = ceil_div(bn * bk, threads)
        pixels = 1 if threads % bn == 0 else elements
        if bk % window == 0:
            gather, gather_chain, start = 41, 0, 255 * elements
        else:
            gather, gather_chain = (30, 98) if bn % 64 == 0 else (52, 118)
            start = pixels * 54 * (view.conv["CR"] + view.conv["CS"])
            if window > 31:                                             # position and predicate for every element
                gather, gather_chain, start = gather * 1.4, gather_chain * 1.4, 255 * pixels
        if view.conv["CSTRW"] > 1:                                      # a load's lanes lie in more lines
            gather *= 1.3
        operands = 0                                                    # nothing that the gather's loads do not show
    compute = ceil_div(share * nw, 4) * step * steps + share * steps * gathered * gather / 4
    chain = turns * (steps * (latency + step * ceil_div(nw, 4) * overlap + gather_chain * gathered / nw) + start)
    longest = max(compute, chain, operands)
    return (longest + mix * (compute + chain + operands - longest) + share * bm * bn * 4 * store / 64
            + sums * rm * rn * mf * mf / 64 * (groups - 1) + (3550 if call else 0))


def _default_conv(view, padded=False, direct=True, by_image=False):
    """Tile, K tile, pipeline and K division of a convolution nobody tuned, by predicted time like _default_f32.

    What differs from the plain product is the gathered operand: one float per lane and load, with its own address.
    Where the K tile holds whole windows (or the window is one pixel) the address advances by a constant; else an
    element costs its channel and tap, which are scalars where a wavefront loads from one row of the tile. Windows of
    several pixels (2x2 .. 11x11 and single rows and columns, strides 1 .. 4, dilation 1 and 2, 1 .. 4 groups; 3 .. 512
    channels): fitted to 1 887 timings over 230 layers together with the tiles without LDS; the pick is 4 % off the best
    measured kernel in the geometric mean and 1.29 times for the worst layer.
    One pixel: 5 % off (1 .. 16 images, 16 .. 512 channels). Pointwise layers whose tiles are no multiple of 8 go at
    the lower rate of grids that were not renumbered by XCD: 4 x 464x49x49 -> 48 stride 2 11.96 -> 7.93 us, 8 x 144x30x30 -> 192
    stride 2 6.84 -> 5.09, 15 x 131x21x21 -> 45 5.42 -> 4.29 (with one rate up to 15 % slower than the rule before).

    A pointwise layer whose images are matrices as they lie in memory goes image by image: 16-byte loads instead of one
    float per lane and load, tiles that end with every image. Over 30 layers (1 .. 16 images of 117 .. 11 664 pixels) the
    pick is 5 % off the best kernel of both kinds, the gather's pick 20 % (2x240x35x35 -> 160 4.8 us for 5.9,
    10x459x92x92 -> 17 37.3 for 48.6, 10x336x17x111 -> 17 8.9 for 14.0); the two predicted times are both mended by what
    their picks took.
    """
    window = view.conv["CR"] * view.conv["CS"]
    cfg, clocks, call = _pick_f32(view, WINDOW_KERNELS if window > 1 else CONV_KERNELS, _conv_clocks, padded, direct)
    if window == 1:
        call = 0.78 * clocks + 3660
    # images of few pixels end in tiles that are partly empty, and several of them keep the gather's larger tiles
    if view.pixels is not None and by_image and (view.pixels[0] == 1 or view.pixels[1] >= 512):
        image, image_clocks, _ = _pick_f32(view.by_image(), F32_KERNELS, _f32_clocks, padded, False)
        if 0.98 * image_clocks + 4130 < call:
            if direct and not padded:
                image = _or_split(view.by_image(), image, 0.98 * image_clocks + 4130)
            image["reorder"] = [image["reorder"][0] + [2]]
            return image
    return _or_split(view, cfg, call) if direct and not padded else cfg


def default_config(op, padded=False, direct=False):
    """A reasonable untuned config: the point a search begins with, and with ``direct`` (tiles without LDS stand for
    choice too, which are not in the space) for all operators but the convolution what an untuned task runs on
    (untuned_config)."""
    cfg = _empty_config()
    if op.kind == "gemm_int8":
        return _default_i8(GemmView(op), padded)
    if op.kind in ("gemm", "batch_gemm"):
        return _default_f32(GemmView(op), padded, direct)
    if op.kind in GEMM_KINDS:
        view = GemmView(op)

        def tile(extent, want, mf):
            """[grid, waves, reps, mfma] with a tile close to ``want``."""
            w, r = 1, 1
            while w * r * mf * 2 <= want and w * r * mf * 2 <= max(extent, mf):
                if w < 2:
                    w *= 2
                else:
                    r *= 2
            return [ceil_div(extent, w * r * mf), w, r, mf]

        mf = 32 if min(view.M, view.N) >= 64 else 16
        # the largest square-ish tile that still yields one workgroup per CU
        want = 128
        while True:
            tm, tn = tile(view.M, want, mf), tile(view.N, want, mf)
            if tm[0] * tn[0] >= 256 or want <= mf:
                break
            want //= 2
        cfg["spatial"] = [tm, tn]
        kblk = 4 * (64 // mf)
        bk = None
        for cand in sorted(F32_BK, reverse=True):
            if view.KP % cand == 0 and cand % kblk == 0 and cand <= 32:
                bk = cand
                break
        if bk is None:
            for cand in sorted(F32_BK):
                if view.KP % cand == 0 and cand % kblk == 0:
                    bk = cand
                    break
        if bk is None:
            raise InvalidConfig("K=%d has no admissible LDS tile extent" % view.K)
        cfg["reduce"] = [[1, view.KP // bk, bk]]
        cfg["unroll"] = [[3, 1]]
        cfg["fuse"] = [[4]]
        cfg["reorder"] = [[1, 0, 0]]
    elif op.kind == "depthwise_conv2d_nchw":
        b, c, p, q = [x.extent for x in op.axis]
        # Rows per lane patch: 4 (3 at stride 2, where a row more is two more input rows to hold), fewer while
        # that leaves less than a wavefront per SIMD; small workgroups of two wavefronts, which retire and
        # start at a finer grain. Over 22 layers (1 .. 31 images, 24 .. 511 channels, 10 .. 104 rows; 3x3 and 5x5,
        # stride 1 and 2) this is 4 % off the best of 1 .. 8 rows and 1 .. 4 wavefronts in the geometric mean, 4 rows
        # and 4 wavefronts everywhere are 19 % off: 17x413x66x20 5x5 stride 2 33.9 -> 17.6 us.
        tw = 4 if q >= 4 else 1
        th = max(1, min(4 if op.attrs["stride"][0] == 1 else 3, p))        # no rows at all: refused in the lowering
        while th > 1 and b * c * ceil_div(p, th) * ceil_div(q, tw) < 64 * 4 * NUM_CUS:
            th //= 2
        cfg["spatial"] = [[b, 1, 1, 1], [c, 1, 1, 1], [ceil_div(p, th), 1, 1, th],
                          [ceil_div(q, tw), 1, 1, tw]]
        cfg["fuse"] = [[2]]
    return cfg


def untuned_config(op, special=None):
    """What schedule_with_config falls back to when a task has no tuned entry. The convolution's search keeps
    beginning at a square-ish tile with K undivided, beside which its other seed points lie. An LDS layout that
    the graph config names (``special``) is one that tiles straight into LDS may not be able to have, and that tiles
    without LDS do not have at all."""
    padded = _special(special, "lds_pad") != SPECIAL_DEFAULTS["lds_pad"]
    direct = not (special and "lds_pad" in special)
    if op.kind in ("conv2d_nchw", "col_gemm"):
        return _default_conv(GemmView(op), padded, direct, bool(int(_special(special, "image_as_matrix")[0])))
    return default_config(op, padded, direct)


def seed_configs(op, limit=24):
    """Points worth measuring before the random warm-up: the default config
    and variations of it along the knobs that decided the hand-tuned shapes
    (tile aspect and MFMA edge, LDS tile extent incl. whole 3x3 windows,
    pipeline depth incl. tiles straight into LDS, K streaming when the tiles
    are fewer than the compute units, and for layers with few tiles and a
    long K a grid-level K split sized to fill the compute units, or with
    small tiles wavefront groups that share K inside the workgroup; a third
    of the points is kept for those). The variations are entities of the op's
    space (the default config itself need not be: it may waste more of an
    edge tile than the space admits); points the templates refuse are
    dropped by the caller."""
    base = default_config(op)
    if op.kind not in GEMM_KINDS:
        return [base]
    view = GemmView(op)
    i8 = view.dtype == "int8"
    out = [base]

    def tile(extent, w, r, mf):
        return [ceil_div(extent, w * r * mf), w, r, mf]

    if i8:
        shapes = [((4, 4, 16), (2, 8, 16)), ((4, 4, 16), (4, 4, 16)), ((4, 2, 32), (4, 2, 32))]
        bks, depths, streams = [128, 64], [7, 6, 2], [0]
    else:
        shapes = [((4, 1, 16), (4, 1, 16)), ((4, 1, 32), (2, 1, 32)), ((2, 1, 32), (2, 1, 32)),
                  ((4, 1, 16), (1, 1, 16)), ((4, 1, 16), (2, 1, 16)), ((2, 2, 16), (4, 1, 16)),
                  ((2, 1, 16), (4, 1, 16))]
        bks = [b for b in (144, 72, 64, 48, 32) if b in F32_BK]
        depths, streams = [8, 5, 3, 2, 1], [0, 1]
    def in_space(extent, t):
        # the tile space's own rules: no tile a smaller one covers as well, bounded edge waste
        size = t[1] * t[2] * t[3]
        if t[0] == 1:
            return size - extent < t[3]
        return t[0] * size - extent <= 0.25 * extent or t[0] * size - extent < t[3]

    split_seeds = []
    for (m_w, m_r, mf), (n_w, n_r, _) in shapes:
        tm, tn = tile(view.M, m_w, m_r, mf), tile(view.N, n_w, n_r, mf)
        if not (in_space(view.M, tm) and in_space(view.N, tn)):
            continue
        tiles = tm[0] * tn[0] * view.groups
        for bk in bks:
            kps = [kp for kp in view.KP_options if kp % bk == 0]
            if not kps:
                continue
            # K streaming first where the tiles alone cannot fill the compute units
            order = [(d, st) for st in (streams[::-1] if tiles < NUM_CUS else streams) for d in depths]
            for depth, stream in order:
                if not (stream and (i8 or tiles >= 2 * NUM_CUS)):
                    cfg = _empty_config()
                    cfg["spatial"] = [tm, tn]
                    cfg["reduce"] = [[1, kps[0] // bk, bk]]
                    cfg["unroll"] = [[depth, 1]]
                    cfg["fuse"] = [[8]]
                    cfg["reorder"] = [[1, 0, stream]]
                    out.append(cfg)
                if depth == depths[0] and stream == 0 and tiles * 2 <= NUM_CUS:
                    # few tiles and a long K (weights streamed past a small image): K parts across
                    # workgroups, as many as fill the compute units
                    split = 1
                    while split * 2 * tiles <= NUM_CUS and split < 16 and (kps[0] // bk) % (split * 2) == 0:
                        split *= 2
                    if split > 1:
                        cfg = _empty_config()
                        cfg["spatial"] = [tm, tn]
                        cfg["reduce"] = [[split, kps[0] // (bk * split), bk]]
                        cfg["unroll"] = [[depth, 1]]
                        cfg["fuse"] = [[8]]
                        cfg["reorder"] = [[1, 0, 0]]
                        split_seeds.append(cfg)
    group_seeds = []
    if not i8:
        # a few small tiles and a long K (1x1 layers on a 7x7 image): one launch whose wavefront
        # groups share K inside the workgroup and add up in LDS, with single-wavefront tiles
        for (m_w, n_w) in ((1, 1), (2, 1), (1, 2)):
            tm, tn = tile(view.M, m_w, 1, 16), tile(view.N, n_w, 1, 16)
            if not (in_space(view.M, tm) and in_space(view.N, tn)) or tm[0] * tn[0] * view.groups * 2 > NUM_CUS:
                continue
            kps = [kp for kp in view.KP_options if kp % 16 == 0]
            for groups in range(16 // (m_w * n_w), 1, -1):
                if kps and (kps[0] // 16) % groups == 0:
                    cfg = _empty_config()
                    cfg["spatial"] = [tm, tn]
                    cfg["reduce"] = [[groups, kps[0] // (16 * groups), 16]]
                    cfg["unroll"] = [[3, 1]]
                    cfg["fuse"] = [[8]]
                    cfg["reorder"] = [[1, 1, 0]]
                    group_seeds.append(cfg)
                    break

    # spread over the variations instead of exhausting the first tile shape
    def spread(lst, n):
        if len(lst) <= n:
            return lst
        step = (len(lst) - 1) / float(max(n - 1, 1))
        return [lst[int(round(i * step))] for i in range(n)]

    def spread_groups(first, lst, n):
        """``first`` and n - 1 of ``lst``: the (tile, BK) groups are visited in turn, and each visit
        of a group takes its next (depth, streaming) variant, starting at a variant that moves
        with the group, so that every tile shape and every pipeline depth gets measured."""
        if len(lst) + 1 <= n:
            return [first] + lst
        groups, index = [], {}
        for c in lst:
            gkey = json.dumps([c["spatial"], c["reduce"]])
            if gkey not in index:
                index[gkey] = len(groups)
                groups.append([])
            groups[index[gkey]].append(c)
        picked, taken, k = [first], [0] * len(groups), 0
        while len(picked) < n:
            gi = k % len(groups)
            g = groups[gi]
            if taken[gi] < len(g):
                # the start moves through the depths with the group; the streaming choice listed
                # first for the group stays first
                picked.append(g[(taken[gi] + gi % len(depths)) % len(g)])
                taken[gi] += 1
            k += 1
        return picked

    group_seeds = group_seeds[:max(limit // 3, 0)]
    nsplit = max(0, min(len(split_seeds), limit // 3 - len(group_seeds)))
    return (spread_groups(out[0], out[1:], max(limit - nsplit - len(group_seeds), 1)) + group_seeds +
            spread(split_seeds, nsplit))[:max(limit, 1)]
