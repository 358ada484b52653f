"""GPU parity: every C-ABI kernel against the CPU oracle on the same seeded inputs (small shapes)."""
import ctypes as C_

import numpy as np
import pytest
import torch

import oracle as O
from rembrandt_amd import _lib, ops, synth
from conftest import assert_close, say
from test_gpu_step_graph import profile_records, profile_tags

pytestmark = pytest.mark.gpu


def T(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def N(t):
    return t.detach().cpu().numpy()


CONV_CASES = [
    # N, C, H, W, K, R, stride, pad
    (2, 3, 9, 7, 4, 3, 1, 1),        # tiny, ragged everything
    (3, 5, 13, 13, 20, 5, 1, 2),     # LeNet-like 5x5 pad 2, K=20
    (2, 3, 35, 35, 96, 11, 4, 0),    # AlexNet conv1-like: 11x11 stride 4, K=96
    (4, 16, 14, 14, 50, 5, 1, 2),    # K=50 -> 64-row tile
    (2, 96, 13, 13, 256, 5, 1, 2),   # AlexNet conv2-like channels, 128-row tile, K_gemm 2400
    (3, 40, 9, 9, 130, 3, 1, 1),     # K just above a tile boundary
    (2, 24, 12, 12, 24, 1, 1, 0),    # 1x1
    (2, 6, 15, 15, 10, 3, 2, 1),     # stride 2 with pad
    (1, 4, 10, 10, 8, 3, 3, 0),      # stride 3
    (70, 2, 6, 6, 5, 3, 1, 1),       # many images, pixel tiles straddle images
    # strided backward-data by residue classes: classes without filter taps (1x1), odd extents whose last rows no
    # window covers, 7x7 stride 2 pad 3, stride 4 with padding, a contraction deep enough to be cut into slices,
    # and a stride beyond the class form (zero-dilated copy)
    (2, 8, 12, 12, 16, 1, 2, 0),
    (2, 5, 14, 11, 6, 3, 2, 0),
    (2, 3, 30, 30, 16, 7, 2, 3),
    (2, 4, 21, 21, 6, 5, 4, 2),
    (2, 8, 14, 14, 256, 3, 2, 1),
    (1, 3, 16, 16, 4, 5, 5, 0),
    # 832 / 885 column tiles of 32 x 256 on 768 block slots: the tiles past the last multiple of the CU count are cut
    # into slices of the contraction although the grid takes more than one round (forward and backward-data)
    (52, 32, 66, 66, 32, 3, 1, 0),
    # stride 1 with output rows a multiple of four pixels long on a 128-row tile, padded and unpadded image
    (3, 8, 12, 16, 128, 3, 1, 1),
    (2, 16, 10, 12, 130, 1, 1, 0),
    # 1x1, stride 1, no padding, at most 128 channels on both sides: the register-resident streaming kernel (forward
    # and backward-data) and the pixel loaders for both operands of backward-filter.  Odd channel counts (a last
    # channel pair with one live half), column tiles that straddle images and end ragged, all four row-tile counts.
    (3, 5, 7, 9, 33, 1, 1, 0),
    (2, 96, 9, 11, 96, 1, 1, 0),
    (1, 128, 6, 5, 128, 1, 1, 0),
    (5, 17, 8, 8, 100, 1, 1, 0),
    (2, 64, 13, 13, 20, 1, 1, 0),
    # enough column tiles (313 / 1250) for the per-XCD ranges, with a ragged last range and tiles that straddle images
    (4, 64, 50, 50, 64, 1, 1, 0),
    (5, 32, 89, 90, 96, 1, 1, 0),
    # contractions of 96 and more with full row tiles and channel pairs and an even pixel count per image: the form
    # of the streaming kernel that moves two pixels per lane (forward, masked backward-data) or four (backward-data,
    # pixel count a multiple of four, up to three row tiles); groups of columns that straddle images and end ragged,
    # enough groups for the per-XCD ranges; a short contraction beside them (the one-pixel form)
    (3, 96, 12, 12, 96, 1, 1, 0),
    (2, 128, 10, 10, 64, 1, 1, 0),
    (6, 32, 20, 22, 32, 1, 1, 0),
    (3, 64, 9, 10, 96, 1, 1, 0),
    (4, 96, 64, 66, 96, 1, 1, 0),
    # filter gradients of at most 32 x 64 and 32 x 128 (first layers): the narrow tiles of the gather path
    (4, 1, 12, 12, 20, 5, 1, 2),
    (3, 3, 10, 11, 32, 5, 1, 2),
    (2, 2, 9, 9, 8, 3, 2, 1),
    (2, 4, 8, 8, 30, 5, 1, 0),
]


ALGOS = {"auto": 0, "gather": _lib.RH_ALGO_GATHER, "scalar_offset": _lib.RH_ALGO_SCALAR_OFFSET}


@pytest.mark.parametrize("algo", sorted(ALGOS))
@pytest.mark.parametrize("case", CONV_CASES, ids=[str(c) for c in CONV_CASES])
def test_conv2d_all_passes(dev, case, algo):
    Nn, C, H, W, K, R, st, pad = case
    say("conv case", case, algo)
    algo = ALGOS[algo]
    x = synth.normal(11, 1, (Nn, C, H, W))
    w = synth.normal(11, 2, (K, C, R, R))
    b = synth.normal(11, 3, (K,))
    y_ref = O.conv2d_fwd(x, w, st, pad)
    dy = synth.normal(11, 4, y_ref.shape)
    xd, wd, bd, dyd = T(x, dev), T(w, dev), T(b, dev), T(dy, dev)

    y = ops.conv2d_fwd(xd, wd, st, pad, algo=algo)
    assert_close(N(y), y_ref, "conv fwd")

    # fused bias + relu epilogue == K1 -> K2 -> K3
    yf = ops.conv2d_fwd(xd, wd, st, pad, bias=bd, relu=True, algo=algo)
    ref_f = O.rect_inplace(O.add_bias_nchw(b, y_ref.copy()))
    assert_close(N(yf), ref_f, "conv fwd fused bias+relu")

    # alpha / beta blend
    y0 = synth.normal(11, 5, y_ref.shape)
    yb = ops.conv2d_fwd(xd, wd, st, pad, alpha=0.5, beta=2.0, y=T(y0, dev), algo=algo)
    assert_close(N(yb), O.conv2d_fwd(x, w, st, pad, alpha=0.5, beta=2.0, y=y0.copy()), "conv fwd alpha/beta")

    dw_ref = O.conv2d_bwd_filter(x, dy, w.shape, st, pad)
    dw = ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, algo=algo)
    assert_close(N(dw), dw_ref, "conv bwd filter")
    dw0 = synth.normal(11, 6, w.shape)
    dwa = ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, alpha=1.0, beta=1.0, dw=T(dw0, dev), algo=algo)
    assert_close(N(dwa), O.conv2d_bwd_filter(x, dy, w.shape, st, pad, 1.0, 1.0, dw0.copy()), "conv bwd filter beta=1")
    # the scaled accumulation of the gen-2 layers: backward(batch, scale) passes `scale` as alpha (src/layer_new.rs:1093-1101)
    dws = ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, alpha=0.25, beta=1.0, dw=T(dw0, dev), algo=algo)
    assert_close(N(dws), O.conv2d_bwd_filter(x, dy, w.shape, st, pad, 0.25, 1.0, dw0.copy()), "conv bwd filter alpha=0.25 beta=1")
    dws = ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, alpha=-3.0, beta=0.5, dw=T(dw0, dev), algo=algo)
    assert_close(N(dws), O.conv2d_bwd_filter(x, dy, w.shape, st, pad, -3.0, 0.5, dw0.copy()), "conv bwd filter alpha=-3 beta=0.5")

    db = ops.conv2d_bwd_bias(dyd)
    assert_close(N(db), O.conv2d_bwd_bias(dy), "conv bwd bias")
    db0 = synth.normal(11, 7, (K,))
    db2 = ops.conv2d_bwd_bias(dyd, alpha=0.5, beta=1.0, db=T(db0, dev), two_stage=True)
    assert_close(N(db2), O.conv2d_bwd_bias(dy, 0.5, 1.0, db0.copy()), "conv bwd bias (two-stage)")

    # both gradients in one call: the filter gradient bit-identical to the call of its own, the bias gradient within
    # tolerance of the oracle (where the pass over dy carries the plane sums it is added up in another order)
    for alpha, beta in ((1.0, 0.0), (0.25, 1.0)):
        dwc, dbc = ops.conv2d_bwd_filter_bias(xd, dyd, w.shape, st, pad, alpha=alpha, beta=beta, dw=T(dw0, dev), db=T(db0, dev),
                                              algo=algo)
        dws = ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, alpha=alpha, beta=beta, dw=T(dw0, dev), algo=algo)
        assert torch.equal(dwc, dws), "filter gradient of the combined call"
        assert_close(N(dbc), O.conv2d_bwd_bias(dy, alpha, beta, db0.copy()), "bias gradient of the combined call")
        dbc2 = ops.conv2d_bwd_filter_bias(xd, dyd, w.shape, st, pad, alpha=alpha, beta=beta, dw=T(dw0, dev), db=T(db0, dev),
                                          algo=algo)[1]
        assert torch.equal(dbc, dbc2), "the combined call is not deterministic"

    dx_ref = O.conv2d_bwd_data(w, dy, x.shape, st, pad)
    dx = ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, algo=algo)
    assert_close(N(dx), dx_ref, "conv bwd data")
    # with the backward of the ReLU that produced x applied as dx is written: bit-identical to the data gradient
    # followed by the in-place mask (x here stands for that ReLU's output: its sign pattern is all that matters)
    if ops.conv2d_bwd_data_relu_supported(x.shape, w.shape, st, pad):
        dx0 = synth.normal(11, 8, x.shape)
        for alpha, beta in ((1.0, 0.0), (0.5, 2.0)):
            two = ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, alpha=alpha, beta=beta, dx=T(dx0, dev), algo=algo)
            ops.rect_backprop_inplace(xd, two)
            one = ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, alpha=alpha, beta=beta, dx=T(dx0, dev), algo=algo, relu_of=xd)
            assert torch.equal(one, two), "masked data gradient alpha=%g beta=%g" % (alpha, beta)
    else:
        assert st > 1
    torch.cuda.synchronize()


# Stride-1 layers with both operands staged in LDS: each tile shape (rows x pixels, "_q2": two channel quads a stage) that
# either filter extent is chosen with, whole and in slices of the channels where both are, sizes with remainders everywhere
# (rows, pixels, channels; tiles that span images), the smallest there is, a 5x5 layer without padding, and as many slices
# as there are.  With each case the shape and the slices of its forward pass and of its data gradient.
STAGED_CASES = [
    # N, C, H, W, K, R, pad
    ((1, 1, 1, 1, 1, 3, 1), ("32x32", 1), ("32x32", 1)),
    ((2, 5, 9, 7, 21, 5, 0), ("32x64", 1), ("32x128", 6)),
    ((3, 2, 4, 30, 33, 3, 2), ("32x128", 1), ("32x64", 5)),
    ((16, 3, 56, 56, 33, 3, 1), ("64x128", 1), ("32x128", 1)),
    ((11, 66, 31, 32, 33, 3, 1), ("64x128", 5), ("32x128", 1)),
    ((25, 3, 28, 28, 130, 5, 2), ("64x128", 1), ("32x128", 3)),
    ((22, 33, 27, 28, 33, 5, 2), ("64x128", 3), ("64x128", 3)),
    ((5, 3, 40, 41, 33, 5, 2), ("64x64", 1), ("32x64", 1)),
    ((19, 20, 13, 13, 33, 5, 2), ("64x64", 5), ("32x64", 5)),
    ((1, 132, 13, 13, 65, 3, 1), ("32x32", 5), ("32x32", 5)),
    ((1, 3, 5, 5, 20, 3, 1), ("32x128", 1), ("32x128", 5)),
    ((1, 20, 5, 6, 20, 5, 2), ("32x128", 5), ("32x128", 5)),
    ((20, 12, 27, 29, 96, 5, 2), ("32x128", 1), ("32x128", 4)),
    ((1, 8, 5, 6, 20, 3, 1), ("32x64", 1), ("32x128", 5)),
    ((1, 33, 5, 5, 33, 5, 2), ("32x64", 5), ("32x64", 5)),
    ((9, 40, 20, 20, 70, 3, 1), ("32x64", 1), ("32x128", 6)),
    ((1, 66, 5, 5, 20, 3, 1), ("32x32", 5), ("32x128", 5)),
    ((1, 13, 5, 5, 20, 5, 2), ("32x32", 1), ("32x128", 5)),
    ((32, 32, 16, 16, 32, 5, 2), ("32x32", 1), ("32x32", 1)),
    ((27, 8, 17, 18, 33, 5, 2), ("32x128_q2", 1), ("32x128", 3)),
    ((2, 33, 28, 29, 33, 5, 2), ("32x128_q2", 5), ("32x128_q2", 5)),
    ((1, 20, 5, 5, 20, 3, 1), ("32x128", 5), ("32x128", 5)),
    ((1, 256, 13, 13, 384, 3, 1), ("32x128", 16), ("32x128", 32)),
    ((1, 33, 5, 5, 20, 3, 1), ("32x64", 5), ("32x128", 5)),
    ((1, 512, 7, 7, 512, 3, 1), ("32x64", 32), ("32x64", 32)),
    ((24, 66, 15, 15, 33, 3, 1), ("64x64", 6), ("32x64", 1)),
    ((1, 384, 13, 13, 384, 3, 1), ("64x64", 24), ("64x64", 24)),
    ((24, 8, 37, 37, 130, 3, 1), ("32x128_q2", 1), ("32x128", 3)),
    ((24, 130, 37, 37, 32, 3, 1), ("32x128", 3), ("32x128_q2", 1)),
    ((1, 70, 5, 5, 20, 5, 2), ("32x32", 5), ("32x128", 5)),
    ((1, 9, 7, 9, 96, 5, 2), ("32x32", 1), ("32x128", 24)),
]


def staged_forms(records, pass_, elems):
    """Shapes and slices of the staged convolutions among launch records, one result of `elems` values each: the slices from
    the bytes that the reduction behind a sliced one moves, 4 (slices + 1) a value."""
    at = [i for i, (tag, _) in enumerate(records) if tag.startswith("conv_%s_lds_" % pass_)]
    return [(records[i][0][len("conv_%s_lds_" % pass_):],
             int(records[i + 1][1] / 4.0 / elems) - 1 if records[i + 1:] and records[i + 1][0] == "split_reduce" else 1) for i in at]


@pytest.mark.parametrize("case,fwd,bwd", STAGED_CASES, ids=lambda v: str(v) if len(v) > 2 else "%s/%d" % v)
def test_conv2d_staged_operands(dev, case, fwd, bwd):
    """Forward and backward-data against the oracle at the edges of the staged form's tiles, with its epilogues."""
    Nn, C, H, W, K, R, pad = case
    say("staged case", case)
    x, w, b = synth.normal(17, 1, (Nn, C, H, W)), synth.normal(17, 2, (K, C, R, R)), synth.normal(17, 3, (K,))
    y_ref = O.conv2d_fwd(x, w, 1, pad)
    dy = synth.normal(17, 4, y_ref.shape)
    y0, dx0 = synth.normal(17, 5, y_ref.shape), synth.normal(17, 6, x.shape)
    xd, wd, bd, dyd = T(x, dev), T(w, dev), T(b, dev), T(dy, dev)
    (y, dx), records = profile_records(lambda: (ops.conv2d_fwd(xd, wd, 1, pad), ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad)))
    assert staged_forms(records, "fwd", y.numel()) == [fwd] and staged_forms(records, "bwd_data", dx.numel()) == [bwd], records
    assert_close(N(y), y_ref, "staged fwd")
    assert_close(N(dx), O.conv2d_bwd_data(w, dy, x.shape, 1, pad), "staged bwd data")
    yf = ops.conv2d_fwd(xd, wd, 1, pad, bias=bd, relu=True)
    assert torch.equal(torch.clamp_min(y + bd.view(1, -1, 1, 1), 0.0), yf), "fused epilogue == conv, add_bias, rect"
    yb = ops.conv2d_fwd(xd, wd, 1, pad, alpha=0.5, beta=2.0, y=T(y0, dev))
    assert_close(N(yb), O.conv2d_fwd(x, w, 1, pad, alpha=0.5, beta=2.0, y=y0.copy()), "staged fwd alpha/beta")
    one = ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, alpha=0.5, beta=2.0, dx=T(dx0, dev), relu_of=xd)
    two = ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, alpha=0.5, beta=2.0, dx=T(dx0, dev))
    ops.rect_backprop_inplace(xd, two)
    assert torch.equal(one, two), "masked data gradient"


@pytest.mark.parametrize("case", [(64, 20, 14, 14, 50, 5, 2), (37, 32, 16, 16, 32, 5, 2), (5, 96, 27, 27, 256, 5, 2),
                                  (9, 128, 28, 28, 128, 3, 1), (9, 256, 14, 14, 256, 3, 1)], ids=str)
def test_conv2d_staged_operands_error(dev, case):
    """Error of the staged form against 64-bit sums.  A chain of n rounded additions of independent terms has a relative
    rms error of sqrt(0.09 n) 2^-24 (a rounding's variance is u^2 / 3 of the power of two below the partial sum, 0.54 of its
    square on average, and the partial sums grow as a random walk: n / 2 of the last one's); chains of F terms added up
    in a chain of n / F have that of a chain of F + n / F, and the products' and the result's own roundings stand for
    four more.  A quarter on top for the spread between tensors; a chain over the whole contraction is 2 to 4 times as far off."""
    Nn, C, H, W, K, R, pad = case
    say("staged error case", case)
    x, w = synth.normal(19, 1, (Nn, C, H, W)), synth.normal(19, 2, (K, C, R, R))
    dy = synth.normal(19, 3, (Nn, K, H, W))
    xd, wd, dyd = T(x, dev), T(w, dev), T(dy, dev)
    D = _lib.RH_ALGO_DIRECT
    (y, dx), tags = profile_tags(lambda: (ops.conv2d_fwd(xd, wd, 1, pad, algo=D), ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, algo=D)))
    assert any(t.startswith("conv_fwd_lds") for t in tags) and any(t.startswith("conv_bwd_data_lds") for t in tags), tags
    for got, ref, chans in ((y, O.conv2d_fwd(x, w, 1, pad), C), (dx, O.conv2d_bwd_data(w, dy, x.shape, 1, pad), K)):
        terms, chain = chans * R * R, 36 if R == 3 else 52
        bound = 1.25 * 2.0 ** -24 * (0.09 * (chain + terms / chain + 4)) ** 0.5
        err = np.linalg.norm(N(got).astype(np.float64) - ref) / np.linalg.norm(ref.astype(np.float64))
        assert err <= bound, (terms, err, bound)


@pytest.mark.parametrize("case", [(256, 1, 28, 28, 20, 5, 2), (60, 5, 29, 29, 477, 3, 1), (72, 2, 23, 28, 273, 5, 1)], ids=str)
def test_conv2d_few_channels_on_many_pixels_keep_the_engine(dev, case):
    """One, two or five input channels fill a quarter to two thirds of the staged form's quads; on grids that fill the GPU the
    engine is the faster one (16 us against 21, 40 against 52, 25 against 32)."""
    Nn, C, H, W, K, R, pad = case
    x, w = torch.zeros((Nn, C, H, W), device=dev), torch.zeros((K, C, R, R), device=dev)
    tags = profile_tags(lambda: ops.conv2d_fwd(x, w, 1, pad))[1]
    assert not any(t.startswith("conv_fwd_lds") for t in tags), tags


@pytest.mark.parametrize("case", [(16, 96, 27, 27, 256, 5, 2), (48, 48, 17, 17, 160, 3, 1), (21, 320, 33, 33, 100, 3, 1), (56, 130, 17, 17, 96, 3, 1)], ids=str)
def test_conv2d_one_tile_and_a_little_per_cu_is_staged(dev, case):
    """The engine slices only the tiles past a multiple of 256, and a whole tile's chain of K steps is the shortest that such a
    call can be: 1.0 to 1.8 tiles a CU take the staged form (123 us against 152, 30 against 39, 170 against 191)."""
    Nn, C, H, W, K, R, pad = case
    x, w = synth.normal(29, 1, (Nn, C, H, W)), synth.normal(29, 2, (K, C, R, R))
    y, tags = profile_tags(lambda: ops.conv2d_fwd(T(x, dev), T(w, dev), 1, pad, algo=_lib.RH_ALGO_DIRECT))
    assert any(t.startswith("conv_fwd_lds") for t in tags), tags
    assert_close(N(y), O.conv2d_fwd(x, w, 1, pad), "staged fwd")


# 3x3 stride-1 layers in the Winograd F(2x2, 3x3) form: odd and even extents (tiles that hang over the edge), every
# padding it takes, channel counts that do not fill a group of four, filter counts around the 128-row tile, tile counts
# that are no multiple of the 32-tile block, more blocks than CUs, and the sizes the library takes the form for by itself
WINO_CASES = [
    # N, C, H, W, K, pad
    (2, 8, 6, 6, 8, 1),
    (3, 5, 7, 9, 130, 1),
    (1, 12, 8, 8, 16, 0),
    (2, 16, 5, 6, 20, 2),
    (1, 1, 3, 3, 1, 0),           # one output pixel
    (1, 2, 2, 2, 3, 1),
    (4, 70, 13, 13, 140, 1),
    (2, 64, 13, 13, 96, 1),
    (33, 64, 14, 15, 128, 1),
    (70, 66, 13, 13, 384, 1),     # 3 x 108 blocks
    (70, 64, 13, 13, 384, 1),     # forward: 324 blocks, the 68 past 256 in three slices of the channel loop (6, 6, 4 stages)
    (70, 384, 13, 13, 64, 1),     # the same in the data gradient
    (16, 128, 28, 28, 64, 1),
    (90, 64, 13, 13, 128, 1),     # 4410 tiles: the filter gradient in the form too, its tiles in several slices
    (1, 260, 7, 9, 130, 1),       # three blocks of 64 rows in thirteen slices of five stages
    (5, 132, 12, 14, 64, 1),      # seven blocks of 64 rows in nine slices of four stages (the last one of one)
    (24, 252, 13, 13, 244, 1),    # 74 blocks in three slices (21, 21, 20 stages of 63) of two chains
]


@pytest.mark.parametrize("case", WINO_CASES, ids=str)
def test_conv2d_winograd(dev, case):
    """RH_ALGO_WINOGRAD against the oracle's direct convolution, forward and backward-data, with every epilogue the
    direct kernels have; the masked data gradient bit-identical to gradient + in-place mask; RH_ALGO_DIRECT and the
    loader bits keep the direct form; other geometries are refused."""
    Nn, C, H, W, K, pad = case
    say("winograd case", case)
    WG = _lib.RH_ALGO_WINOGRAD
    x = synth.normal(15, 1, (Nn, C, H, W))
    w = synth.normal(15, 2, (K, C, 3, 3))
    b = synth.normal(15, 3, (K,))
    y_ref = O.conv2d_fwd(x, w, 1, pad)
    dy = synth.normal(15, 4, y_ref.shape)
    xd, wd, bd, dyd = T(x, dev), T(w, dev), T(b, dev), T(dy, dev)
    y = ops.conv2d_fwd(xd, wd, 1, pad, algo=WG)
    assert_close(N(y), y_ref, "winograd fwd")
    yf = ops.conv2d_fwd(xd, wd, 1, pad, bias=bd, relu=True, algo=WG)
    assert_close(N(yf), O.rect_inplace(O.add_bias_nchw(b, y_ref.copy())), "winograd fwd fused bias+relu")
    # the fused epilogue is the separate passes' arithmetic
    two = ops.conv2d_fwd(xd, wd, 1, pad, algo=WG)
    assert torch.equal(torch.clamp_min(two + bd.view(1, -1, 1, 1), 0.0), yf), "winograd fused epilogue == conv, add_bias, rect"
    y0 = synth.normal(15, 5, y_ref.shape)
    yb = ops.conv2d_fwd(xd, wd, 1, pad, alpha=0.5, beta=2.0, y=T(y0, dev), algo=WG)
    assert_close(N(yb), O.conv2d_fwd(x, w, 1, pad, alpha=0.5, beta=2.0, y=y0.copy()), "winograd fwd alpha/beta")
    dx_ref = O.conv2d_bwd_data(w, dy, x.shape, 1, pad)
    dx = ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, algo=WG)
    assert_close(N(dx), dx_ref, "winograd bwd data")
    dx0 = synth.normal(15, 8, x.shape)
    dxb = ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, alpha=0.5, beta=2.0, dx=T(dx0, dev), algo=WG)
    assert_close(N(dxb), O.conv2d_bwd_data(w, dy, x.shape, 1, pad, 0.5, 2.0, dx0.copy()), "winograd bwd data alpha/beta")
    for alpha, beta in ((1.0, 0.0), (0.5, 2.0)):
        two = ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, alpha=alpha, beta=beta, dx=T(dx0, dev), algo=WG)
        ops.rect_backprop_inplace(xd, two)
        one = ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, alpha=alpha, beta=beta, dx=T(dx0, dev), algo=WG, relu_of=xd)
        assert torch.equal(one, two), "winograd masked data gradient alpha=%g beta=%g" % (alpha, beta)
    # the filter gradient in the same form (its sums run over the tiles, cut into slices added in a fixed order)
    dw_ref = O.conv2d_bwd_filter(x, dy, w.shape, 1, pad)
    dw = ops.conv2d_bwd_filter(xd, dyd, w.shape, 1, pad, algo=WG)
    assert_close(N(dw), dw_ref, "winograd bwd filter")
    dw0 = synth.normal(15, 6, w.shape)
    for alpha, beta in ((1.0, 1.0), (0.25, 1.0), (-3.0, 0.5)):
        dwa = ops.conv2d_bwd_filter(xd, dyd, w.shape, 1, pad, alpha=alpha, beta=beta, dw=T(dw0, dev), algo=WG)
        assert_close(N(dwa), O.conv2d_bwd_filter(x, dy, w.shape, 1, pad, alpha, beta, dw0.copy()),
                     "winograd bwd filter alpha=%g beta=%g" % (alpha, beta))
    db0 = synth.normal(15, 7, (K,))
    dwc, dbc = ops.conv2d_bwd_filter_bias(xd, dyd, w.shape, 1, pad, alpha=0.25, beta=1.0, dw=T(dw0, dev), db=T(db0, dev), algo=WG)
    assert torch.equal(dwc, ops.conv2d_bwd_filter(xd, dyd, w.shape, 1, pad, alpha=0.25, beta=1.0, dw=T(dw0, dev), algo=WG))
    assert_close(N(dbc), O.conv2d_bwd_bias(dy, 0.25, 1.0, db0.copy()), "bias gradient of the combined call (winograd)")
    # run to run the same bits
    assert torch.equal(ops.conv2d_fwd(xd, wd, 1, pad, algo=WG), y)
    assert torch.equal(ops.conv2d_bwd_filter(xd, dyd, w.shape, 1, pad, algo=WG), dw)
    # RH_ALGO_SHARED_GPU (other kernels run beside the call): no sliced tail behind a whole round of blocks; the same result
    # up to summation order where a tail was sliced, the same bits where none was or the grid is under one round
    SH = _lib.RH_ALGO_SHARED_GPU
    ys = ops.conv2d_fwd(xd, wd, 1, pad, algo=WG | SH)
    dxs = ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, algo=WG | SH)
    assert_close(N(ys), y_ref, "winograd fwd, shared-GPU hint")
    assert_close(N(dxs), dx_ref, "winograd bwd data, shared-GPU hint")
    blocks_b = -(-C // 128) * -(-(Nn * -(-H // 2) * -(-W // 2)) // 32)
    blocks_f = -(-K // 128) * -(-(Nn * -(-y_ref.shape[2] // 2) * -(-y_ref.shape[3] // 2)) // 32)
    if blocks_f <= 256 or C % 4: assert torch.equal(ys, y)
    if blocks_b <= 256 or K % 4: assert torch.equal(dxs, dx)
    # what the library picks by itself is what it says it picks
    auto = ops.conv2d_fwd(xd, wd, 1, pad)
    direct = ops.conv2d_fwd(xd, wd, 1, pad, algo=_lib.RH_ALGO_DIRECT)
    assert_close(N(direct), y_ref, "RH_ALGO_DIRECT fwd")
    takes = ops.conv2d_winograd_flops(x.shape, w.shape, 1, pad) > 0
    assert torch.equal(auto, y if takes else direct), "library's choice"
    torch.cuda.synchronize()


@pytest.mark.parametrize("case", [(24, 128, 28, 28, 128, 1), (19, 384, 13, 13, 384, 1), (27, 512, 7, 7, 512, 1),
                                  (40, 384, 6, 6, 1024, 1), (9, 128, 30, 30, 256, 0), (29, 256, 13, 13, 384, 1)], ids=str)
def test_conv2d_winograd_error_on_small_grids(dev, case):
    """Where the direct form's tiles are few it cuts its contraction into slices, whose short chains of sums lose few bits:
    the Winograd form has no larger an error against 64 bits on such grids (two correct results' errors differ by
    about the inverse root of their million elements; 3 % for that and for the fit that the chains are chosen by)."""
    Nn, C, H, W, K, pad = case
    say("winograd error case", case)
    x, w, dy = synth.normal(23, 1, (Nn, C, H, W)), synth.normal(23, 2, (K, C, 3, 3)), synth.normal(23, 3, (Nn, K, H, W))
    xd, wd, dyd = T(x, dev), T(w, dev), T(dy, dev)
    for ref, run in ((O.conv2d_fwd(x, w, 1, pad), lambda algo: ops.conv2d_fwd(xd, wd, 1, pad, algo=algo)),
                     (O.conv2d_bwd_data(w, dy, x.shape, 1, pad), lambda algo: ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, algo=algo))):
        err = [float(np.linalg.norm(N(run(algo)).astype(np.float64) - ref)) for algo in (_lib.RH_ALGO_WINOGRAD, _lib.RH_ALGO_SCALAR_OFFSET)]
        assert err[0] <= 1.03 * err[1], err


@pytest.mark.parametrize("case", [(3, 4, 9, 7, 64, 1), (2, 8, 13, 13, 64, 1), (2, 12, 8, 9, 33, 0), (3, 16, 7, 7, 50, 2), (2, 20, 11, 6, 64, 1),
                                  (1, 24, 10, 10, 7, 1), (2, 28, 5, 5, 64, 1), (3, 64, 14, 14, 192, 1), (1, 4, 1, 1, 64, 1),
                                  (9, 64, 56, 56, 64, 1), (24, 64, 56, 55, 64, 1)], ids=str)
def test_conv2d_winograd_64_rows(dev, case):
    """The 64-row tiles of up to 64, 192, ... filters: channel loops of one to seven stages (every way the pipeline starts
    and drains) and of sixteen, ragged rows and tiles, borders of 0, 1, 2, blocks under one round in slices (14 x 14) and
    whole (9 images), and a whole round with a sliced last one (24);
    forward with the fused epilogue, the data gradient masked and blended; the library's own choice."""
    Nn, C, H, W, K, pad = case
    say("winograd 64-row case", case)
    WG = _lib.RH_ALGO_WINOGRAD
    x, w, b = synth.normal(15, 1, (Nn, C, H, W)), synth.normal(15, 2, (K, C, 3, 3)), synth.normal(15, 3, (K,))
    y_ref = O.conv2d_fwd(x, w, 1, pad)
    dy, dx0 = synth.normal(15, 4, y_ref.shape), synth.normal(15, 8, x.shape)
    xd, wd, bd, dyd = T(x, dev), T(w, dev), T(b, dev), T(dy, dev)
    y = ops.conv2d_fwd(xd, wd, 1, pad, algo=WG)
    assert_close(N(y), y_ref, "winograd fwd")
    yf = ops.conv2d_fwd(xd, wd, 1, pad, bias=bd, relu=True, algo=WG)
    assert torch.equal(torch.clamp_min(y + bd.view(1, -1, 1, 1), 0.0), yf), "fused epilogue == conv, add_bias, rect"
    assert_close(N(ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, algo=WG)), O.conv2d_bwd_data(w, dy, x.shape, 1, pad), "winograd bwd data")
    for alpha, beta in ((1.0, 0.0), (0.5, 2.0)):
        two = ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, alpha=alpha, beta=beta, dx=T(dx0, dev), algo=WG)
        assert_close(N(two), O.conv2d_bwd_data(w, dy, x.shape, 1, pad, alpha, beta, dx0.copy()), "winograd bwd data alpha/beta")
        ops.rect_backprop_inplace(xd, two)
        one = ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, alpha=alpha, beta=beta, dx=T(dx0, dev), algo=WG, relu_of=xd)
        assert torch.equal(one, two), "masked data gradient alpha=%g beta=%g" % (alpha, beta)
    assert torch.equal(ops.conv2d_fwd(xd, wd, 1, pad, algo=WG), y), "run to run the same bits"
    if Nn >= 24:
        assert torch.equal(ops.conv2d_fwd(xd, wd, 1, pad), y), "library's choice"


WINO5_CASES = [
    # N, C, H, W, K, pad
    (2, 3, 9, 9, 8, 2),
    (1, 1, 5, 5, 1, 0),            # one output pixel
    (3, 5, 8, 11, 130, 1),
    (2, 8, 7, 6, 20, 4),
    (2, 16, 12, 13, 64, 3),
    (4, 32, 27, 27, 96, 2),
    (40, 32, 27, 27, 256, 2),      # 490 blocks: a whole round and an unsliced last one
    (70, 96, 13, 14, 128, 2),
    (44, 64, 27, 27, 128, 2),      # 270 blocks: a whole round and 14 blocks in sixteen slices
]


@pytest.mark.parametrize("case", WINO5_CASES, ids=str)
def test_conv2d_winograd_5x5_forward(dev, case):
    """RH_ALGO_WINOGRAD on a 5x5 stride-1 layer (forward only): the filter as four 3x3 blocks of its 6x6 zero extension,
    F(2x2, 3x3) on each over the shifted input, added in the transform domain; against the oracle's direct convolution,
    with every epilogue; the backward passes refuse the bit; the library's own choice and RH_ALGO_DIRECT."""
    Nn, C, H, W, K, pad = case
    say("winograd 5x5 case", case)
    WG = _lib.RH_ALGO_WINOGRAD
    x = synth.normal(17, 1, (Nn, C, H, W))
    w = synth.normal(17, 2, (K, C, 5, 5))
    b = synth.normal(17, 3, (K,))
    y_ref = O.conv2d_fwd(x, w, 1, pad)
    xd, wd, bd = T(x, dev), T(w, dev), T(b, dev)
    y = ops.conv2d_fwd(xd, wd, 1, pad, algo=WG)
    assert_close(N(y), y_ref, "winograd 5x5 fwd")
    yf = ops.conv2d_fwd(xd, wd, 1, pad, bias=bd, relu=True, algo=WG)
    assert_close(N(yf), O.rect_inplace(O.add_bias_nchw(b, y_ref.copy())), "winograd 5x5 fwd fused bias+relu")
    assert torch.equal(torch.clamp_min(y + bd.view(1, -1, 1, 1), 0.0), yf), "fused epilogue == conv, add_bias, rect"
    y0 = synth.normal(17, 5, y_ref.shape)
    yb = ops.conv2d_fwd(xd, wd, 1, pad, alpha=0.5, beta=2.0, y=T(y0, dev), algo=WG)
    assert_close(N(yb), O.conv2d_fwd(x, w, 1, pad, alpha=0.5, beta=2.0, y=y0.copy()), "winograd 5x5 fwd alpha/beta")
    assert torch.equal(ops.conv2d_fwd(xd, wd, 1, pad, algo=WG), y), "run to run the same bits"
    assert_close(N(ops.conv2d_fwd(xd, wd, 1, pad, algo=WG | _lib.RH_ALGO_SHARED_GPU)), y_ref, "winograd 5x5 fwd, shared-GPU hint")
    assert ops.conv2d_winograd_flops(x.shape, w.shape, 1, pad, "fwd", algo=WG) == \
        2.0 * 16 * K * 4 * C * Nn * (-(-y_ref.shape[2] // 2)) * (-(-y_ref.shape[3] // 2))
    # forward only
    dy = T(synth.normal(17, 4, y_ref.shape), dev)
    for fn in (lambda: ops.conv2d_bwd_data(wd, dy, x.shape, 1, pad, algo=WG), lambda: ops.conv2d_bwd_filter(xd, dy, w.shape, 1, pad, algo=WG)):
        with pytest.raises(_lib.RembrandtHipError):
            fn()
    # what the library picks by itself is what it says it picks (which that is: test_conv2d_winograd_by_itself)
    auto = ops.conv2d_fwd(xd, wd, 1, pad)
    direct = ops.conv2d_fwd(xd, wd, 1, pad, algo=_lib.RH_ALGO_DIRECT)
    assert_close(N(direct), y_ref, "RH_ALGO_DIRECT fwd (5x5)")
    takes = ops.conv2d_winograd_flops(x.shape, w.shape, 1, pad) > 0
    assert torch.equal(auto, y if takes else direct), "library's choice (5x5)"
    torch.cuda.synchronize()


@pytest.mark.parametrize("case,takes", [
    ((16, 256, 13, 13, 384, 3, 1), True),    # 75 blocks in three slices, data gradient 50 blocks in five of two chains
    ((5, 256, 13, 13, 384, 3, 1), False),    # too few images: the staged form
    ((18, 64, 56, 56, 64, 3, 1), True),      # 441 blocks on 64 rows, under one round of them
    ((13, 64, 56, 56, 64, 3, 1), False),     # 319 of them: two blocks on some CUs
    ((70, 128, 13, 13, 128, 3, 1), True),    # 108 blocks on 128 rows
    ((44, 256, 13, 13, 256, 3, 1), True),    # 136 blocks
    ((29, 96, 27, 27, 256, 5, 2), True),     # 5x5: 356 blocks of two row tiles, one round and a sliced one
    ((19, 96, 27, 27, 256, 5, 2), False),    # 234: under one round
], ids=str)
def test_conv2d_winograd_by_itself(dev, case, takes):
    """Where the library takes the Winograd form without being asked, by the estimates of the forms: the calls under one round
    of blocks and the 5x5 layers under two.  The same bits as with RH_ALGO_WINOGRAD, right against the oracle."""
    Nn, C, H, W, K, R, pad = case
    say("winograd by itself", case)
    x, w = synth.normal(25, 1, (Nn, C, H, W)), synth.normal(25, 2, (K, C, R, R))
    y_ref = O.conv2d_fwd(x, w, 1, pad)
    dy = synth.normal(25, 3, y_ref.shape)
    xd, wd, dyd = T(x, dev), T(w, dev), T(dy, dev)
    for pass_, ref, run in (("fwd", y_ref, lambda algo: ops.conv2d_fwd(xd, wd, 1, pad, algo=algo)),
                            ("bwd_data", None, lambda algo: ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, algo=algo))):
        if R == 5 and pass_ == "bwd_data":
            continue
        y, tags = profile_tags(lambda: run(0))
        assert ("conv_%s_wino" % pass_ in tags) == takes, tags
        if takes:
            assert torch.equal(y, run(_lib.RH_ALGO_WINOGRAD)), pass_
        assert_close(N(y), O.conv2d_bwd_data(w, dy, x.shape, 1, pad) if ref is None else ref, pass_)


def test_conv2d_winograd_refused_geometries(dev):
    import ctypes as C
    x = torch.zeros((2, 4, 8, 8), device=dev)
    ws = torch.zeros((1 << 22,), dtype=torch.uint8, device=dev)
    for R, st, pad, extra in ((5, 2, 2, 0), (7, 1, 3, 0), (3, 2, 1, 0), (1, 1, 0, 0), (3, 1, 3, 0), (3, 1, 1, _lib.RH_ALGO_GATHER),
                              (3, 1, 1, _lib.RH_ALGO_DIRECT), (3, 1, 1, _lib.RH_MATH_BF16_MFMA_FP32ACC)):
        g = _lib.ConvGeom(2, 4, 8, 8, 4, R, R, st, pad)
        w = torch.zeros((4, 4, R, R), device=dev)
        P = (8 + 2 * pad - R) // st + 1
        y = torch.zeros((2, 4, P, P), device=dev)
        rc = _lib.lib().rh_conv2d_fwd(C.byref(g), 1.0, x.data_ptr(), w.data_ptr(), 0.0, y.data_ptr(), None, ws.data_ptr(), ws.numel(),
                                      _lib.RH_ALGO_WINOGRAD | extra, None)
        assert rc == _lib.RH_E_UNSUPPORTED, (R, st, pad, extra, rc)
        if not (extra & _lib.RH_MATH_BF16_MFMA_FP32ACC):
            rc = _lib.lib().rh_conv2d_bwd_data(C.byref(g), 1.0, w.data_ptr(), y.data_ptr(), 0.0, x.data_ptr(), ws.data_ptr(), ws.numel(),
                                               _lib.RH_ALGO_WINOGRAD | extra, None)
            assert rc == _lib.RH_E_UNSUPPORTED, ("bwd", R, st, pad, extra, rc)
            rc = _lib.lib().rh_conv2d_bwd_filter(C.byref(g), 1.0, x.data_ptr(), y.data_ptr(), 0.0, w.data_ptr(), ws.data_ptr(), ws.numel(),
                                                 _lib.RH_ALGO_WINOGRAD | extra, None)
            assert rc == _lib.RH_E_UNSUPPORTED, ("bwd filter", R, st, pad, extra, rc)


# RH_ALGO_BF16X3: fp32 contractions on bf16 matrix instructions, each operand as the sum of three bf16 values.  Contracted
# channel counts of one group of eight, of an odd number of groups (a K step that two taps share) and of many; an odd number
# of groups in all (a last K step with a half of zeros); one to 128 K steps against a ring of three; row counts around the
# 64-, 96- and 128-row tiles; ragged pixels; batches around a group of eight images; strides; contractions in slices, and a
# sliced tail past a whole round of tiles; channels that no pass but the filter gradient takes.
X3_CASES = [
    # N, C, H, W, K, R, stride, pad
    (2, 8, 9, 7, 8, 3, 1, 1),
    (1, 8, 4, 4, 3, 1, 1, 0),
    (3, 24, 13, 13, 40, 3, 1, 1),
    (1, 16, 5, 5, 64, 3, 1, 0),
    (8, 40, 11, 12, 130, 3, 1, 2),
    (9, 64, 14, 15, 65, 5, 1, 2),
    (17, 96, 9, 9, 96, 1, 1, 0),
    (2, 96, 13, 13, 256, 5, 1, 2),
    (7, 128, 12, 12, 192, 3, 2, 1),
    (3, 16, 20, 20, 128, 5, 4, 2),
    (33, 32, 28, 28, 64, 3, 1, 1),
    (80, 128, 21, 21, 128, 3, 1, 1),
    (1, 512, 7, 7, 512, 3, 1, 1),
    (5, 3, 23, 22, 33, 7, 2, 3),
]


@pytest.mark.parametrize("case", X3_CASES, ids=str)
def test_conv2d_bf16x3(dev, case):
    """All passes in the split-operand form against the oracle, with every epilogue."""
    Nn, C, H, W, K, R, st, pad = case
    say("bf16x3 case", case)
    X3 = _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_DIRECT
    x, w, b = synth.normal(33, 1, (Nn, C, H, W)), synth.normal(33, 2, (K, C, R, R)), synth.normal(33, 3, (K,))
    y_ref = O.conv2d_fwd(x, w, st, pad)
    dy, y0, dx0, dw0, db0 = (synth.normal(33, 4 + i, s) for i, s in enumerate((y_ref.shape, y_ref.shape, x.shape, w.shape, (K,))))
    xd, wd, bd, dyd = T(x, dev), T(w, dev), T(b, dev), T(dy, dev)
    if C % 8 == 0:
        y, tags = profile_tags(lambda: ops.conv2d_fwd(xd, wd, st, pad, algo=X3))
        assert any(t.startswith("conv_fwd_tri_") for t in tags), tags
        assert_close(N(y), y_ref, "bf16x3 fwd")
        yf = ops.conv2d_fwd(xd, wd, st, pad, bias=bd, relu=True, algo=X3)
        assert torch.equal(torch.clamp_min(y + bd.view(1, -1, 1, 1), 0.0), yf), "fused epilogue == conv, add_bias, rect"
        yb = ops.conv2d_fwd(xd, wd, st, pad, alpha=0.5, beta=2.0, y=T(y0, dev), algo=X3)
        assert_close(N(yb), O.conv2d_fwd(x, w, st, pad, alpha=0.5, beta=2.0, y=y0.copy()), "bf16x3 fwd alpha/beta")
        assert torch.equal(ops.conv2d_fwd(xd, wd, st, pad, algo=X3), y), "run to run the same bits"
    else:
        with pytest.raises(_lib.RembrandtHipError):
            ops.conv2d_fwd(xd, wd, st, pad, algo=X3)
    if K % 8 == 0 and st == 1 and pad <= R - 1:
        assert_close(N(ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, algo=X3)), O.conv2d_bwd_data(w, dy, x.shape, st, pad), "bf16x3 bwd data")
        for alpha, beta in ((1.0, 0.0), (0.5, 2.0)):
            two = ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, alpha=alpha, beta=beta, dx=T(dx0, dev), algo=X3)
            assert_close(N(two), O.conv2d_bwd_data(w, dy, x.shape, st, pad, alpha, beta, dx0.copy()), "bf16x3 bwd data alpha/beta")
            ops.rect_backprop_inplace(xd, two)
            one = ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, alpha=alpha, beta=beta, dx=T(dx0, dev), algo=X3, relu_of=xd)
            assert torch.equal(one, two), "masked data gradient alpha=%g beta=%g" % (alpha, beta)
    else:
        with pytest.raises(_lib.RembrandtHipError):
            ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, algo=X3)
    dw, tags = profile_tags(lambda: ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, algo=X3))
    assert any(t.startswith("conv_bwd_filter_tri_") for t in tags), tags
    assert_close(N(dw), O.conv2d_bwd_filter(x, dy, w.shape, st, pad), "bf16x3 bwd filter")
    dwc, dbc = ops.conv2d_bwd_filter_bias(xd, dyd, w.shape, st, pad, alpha=0.25, beta=1.0, dw=T(dw0, dev), db=T(db0, dev), algo=X3)
    assert_close(N(dwc), O.conv2d_bwd_filter(x, dy, w.shape, st, pad, 0.25, 1.0, dw0.copy()), "bf16x3 bwd filter alpha/beta")
    assert_close(N(dbc), O.conv2d_bwd_bias(dy, 0.25, 1.0, db0.copy()), "bf16x3 bias gradient")
    assert torch.equal(ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, algo=X3), dw), "run to run the same bits"
    X3 |= _lib.RH_ALGO_BF16X3_WIDE
    wide, tags = profile_tags(lambda: ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, algo=X3))
    assert any(t.startswith("conv_bwd_filter_tri_wide_") for t in tags), tags
    assert_close(N(wide), O.conv2d_bwd_filter(x, dy, w.shape, st, pad), "bf16x3 wide bwd filter")
    dwc, dbc = ops.conv2d_bwd_filter_bias(xd, dyd, w.shape, st, pad, alpha=0.25, beta=1.0, dw=T(dw0, dev), db=T(db0, dev), algo=X3)
    assert_close(N(dwc), O.conv2d_bwd_filter(x, dy, w.shape, st, pad, 0.25, 1.0, dw0.copy()), "bf16x3 wide bwd filter alpha/beta")
    assert_close(N(dbc), O.conv2d_bwd_bias(dy, 0.25, 1.0, db0.copy()), "bf16x3 wide bias gradient")
    assert torch.equal(ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, algo=X3), wide), "run to run the same bits"


# The reduction of a filter gradient's slices: channels that end in a chunk of their own (4 of 20, 8 of 136, 2 of 18), no multiple of
# four, one channel; taps in chunks and a chunk of fewer; one tap; one slice and many; chunks of the widest result of a block.
@pytest.mark.parametrize("case", [(16, 20, 14, 14, 50, 5, 1, 0), (2, 136, 9, 9, 8, 3, 1, 1), (40, 18, 21, 20, 70, 3, 1, 1), (9, 3, 60, 59, 33, 11, 4, 2),
                                  (24, 5, 17, 17, 300, 3, 1, 1), (31, 1, 24, 24, 20, 5, 1, 0), (6, 72, 25, 25, 520, 1, 1, 0), (1, 8, 3, 3, 3, 3, 1, 0),
                                  (8, 516, 6, 6, 513, 3, 1, 1)], ids=str)
def test_conv2d_bwd_filter_slices(dev, case):
    Nn, C, H, W, K, R, st, pad = case
    say("filter slices case", case)
    x = synth.normal(71, 1, (Nn, C, H, W))
    w_shape = (K, C, R, R)
    dy = synth.normal(71, 2, (Nn, K, (H + 2 * pad - R) // st + 1, (W + 2 * pad - R) // st + 1))
    dw0, db0 = synth.normal(71, 3, w_shape), synth.normal(71, 4, (K,))
    xd, dyd = T(x, dev), T(dy, dev)
    for algo in (_lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_DIRECT, _lib.RH_ALGO_F16X2 | _lib.RH_ALGO_DIRECT):
        for alpha, beta in ((1.0, 0.0), (0.25, 1.0)):
            dw, db = ops.conv2d_bwd_filter_bias(xd, dyd, w_shape, st, pad, alpha=alpha, beta=beta, dw=T(dw0, dev), db=T(db0, dev), algo=algo)
            assert_close(N(dw), O.conv2d_bwd_filter(x, dy, w_shape, st, pad, alpha, beta, dw0.copy()), "filter gradient from slices")
            assert_close(N(db), O.conv2d_bwd_bias(dy, alpha, beta, db0.copy()), "bias gradient beside it")
        assert torch.equal(ops.conv2d_bwd_filter_bias(xd, dyd, w_shape, st, pad, alpha=0.25, beta=1.0, dw=T(dw0, dev), db=T(db0, dev), algo=algo)[0], dw)


# Backward-data of stride 2 to 4 by residue classes in the split-operand form: odd extents (classes of different sizes), classes
# without taps (a filter smaller than the stride) and without pixels, an odd number of groups (8, 24, 40 filters), rows past the
# 64-, 96- and 128-row tiles, one to many tiles a class, no padding and more than the filter needs.
X3_STRIDED_CASES = [
    # N, C, H, W, K, R, stride, pad
    (3, 64, 9, 7, 40, 3, 2, 1),
    (1, 65, 1, 5, 8, 3, 2, 1),
    (2, 96, 13, 12, 24, 5, 2, 2),
    (1, 128, 11, 11, 8, 7, 3, 3),
    (5, 70, 10, 9, 16, 3, 2, 0),
    (2, 64, 17, 16, 64, 2, 4, 0),
    (9, 250, 14, 15, 72, 5, 4, 1),
    (4, 64, 8, 8, 64, 3, 2, 3),
    (24, 64, 56, 56, 128, 3, 2, 1),
    (2, 256, 14, 13, 512, 3, 2, 1),      # the long classes in slices, of unequal numbers
    (1, 128, 9, 11, 200, 5, 3, 2),
    (8, 64, 28, 28, 264, 4, 2, 1),
]


@pytest.mark.parametrize("case", X3_STRIDED_CASES, ids=str)
def test_conv2d_bf16x3_strided_bwd_data(dev, case):
    """Against the oracle and no further from its sums than the form it replaces; the alpha / beta blend; infinities."""
    Nn, C, H, W, K, R, st, pad = case
    say("bf16x3 strided bwd data", case)
    X3 = _lib.RH_ALGO_BF16X3
    P, Q = (H + 2 * pad - R) // st + 1, (W + 2 * pad - R) // st + 1
    w, dy, dx0 = synth.normal(41, 1, (K, C, R, R)), synth.normal(41, 2, (Nn, K, P, Q)), synth.normal(41, 3, (Nn, C, H, W))
    wd, dyd = T(w, dev), T(dy, dev)
    got, tags = profile_tags(lambda: ops.conv2d_bwd_data(wd, dyd, dx0.shape, st, pad, algo=X3))
    assert any(t.startswith("conv_bwd_data_tri_") for t in tags), tags
    ref = O.conv2d_bwd_data(w, dy, dx0.shape, st, pad)
    assert_close(N(got), ref, "strided bf16x3")
    before = ops.conv2d_bwd_data(wd, dyd, dx0.shape, st, pad)
    # (of the oracle's sums, which are in 64 bits and then rounded; 1e-8: what that rounding moves, at most half an ulp)
    err, old = (float(np.linalg.norm(N(t).astype(np.float64) - ref) / np.linalg.norm(ref.astype(np.float64))) for t in (got, before))
    assert err <= old + 1e-8, (err, old)
    blend = ops.conv2d_bwd_data(wd, dyd, dx0.shape, st, pad, alpha=0.5, beta=2.0, dx=T(dx0, dev), algo=X3)
    assert_close(N(blend), O.conv2d_bwd_data(w, dy, dx0.shape, st, pad, 0.5, 2.0, dx0.copy()), "strided bf16x3 alpha/beta")
    # (products with the largest float stay in range, |dy| < 8 / 8: a finite overflow beside an infinity of the other sign is -inf, inf
    # or NaN by the order of the additions)
    dy *= np.float32(0.125)
    dy[0, 0, 0, 0], w[-1, -1, 0, 0] = np.inf, np.finfo(np.float32).max
    a, b = (ops.conv2d_bwd_data(T(w, dev), T(dy, dev), dx0.shape, st, pad, algo=f) for f in (X3, _lib.RH_ALGO_GATHER))
    assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b))


# Layers with the passes that the library takes in this form by itself: under a chain limit that asks for slices, against the staged,
# the engine's and the Winograd form, with stride, with one image and with nine (a group of eight and one more in the filter gradient)
X3_ERROR_CASES = [
    # N, C, H, K, R, stride, pad, passes
    (16, 256, 13, 384, 3, 1, 1, "fdw"),
    (9, 96, 27, 256, 5, 1, 2, "fdw"),
    (24, 256, 14, 256, 3, 1, 1, "fdw"),
    (64, 512, 7, 512, 3, 1, 1, "fdw"),
    (24, 128, 28, 128, 3, 1, 1, "fdw"),
    (64, 128, 28, 128, 3, 1, 1, "w"),
    (32, 64, 28, 64, 3, 1, 1, "w"),
    (50, 1024, 6, 1024, 1, 1, 0, "fdw"),
    (50, 128, 28, 256, 3, 2, 1, "fdw"),
    (50, 64, 56, 128, 3, 2, 1, "fdw"),
    (1, 384, 13, 384, 3, 1, 1, ""),
    (1, 512, 7, 512, 3, 1, 1, ""),     # filter gradient: faster by the estimates, but one chain of 25 steps where the engine's is of 49 terms
]


def _conv_sums64(x, w, dy, st, pad):
    """Forward, data gradient and filter gradient of device tensors as plain matrix products in 64 bits."""
    import torch.nn.functional as F
    (Nn, C, H, W), (K, _, R, S), (P, Q) = x.shape, w.shape, dy.shape[2:]
    w2, y, dx = w.double().reshape(K, -1), torch.empty(dy.shape, dtype=torch.float64, device=x.device), torch.empty(x.shape, dtype=torch.float64, device=x.device)
    wt, dw = w2.t().contiguous(), torch.zeros_like(w2)
    step = max(1, 10 ** 8 // (C * R * S * P * Q))
    for i in range(0, Nn, step):
        n = min(step, Nn - i)
        col = F.unfold(x[i:i + n].double(), (R, S), padding=pad, stride=st).permute(1, 0, 2).reshape(C * R * S, -1).contiguous()
        rows = dy[i:i + n].double().reshape(n, K, -1).permute(1, 0, 2).reshape(K, -1).contiguous()
        y[i:i + n] = (w2 @ col).reshape(K, n, P * Q).permute(1, 0, 2).reshape(n, K, P, Q)
        dx[i:i + n] = F.fold((wt @ rows).reshape(C * R * S, n, P * Q).permute(1, 0, 2).contiguous(), (H, W), (R, S), padding=pad, stride=st)
        dw += rows @ col.t().contiguous()
    return y, dx, dw.reshape(w.shape)


def _chain_bound(terms):
    """The large products add to a sum of 16 terms per MFMA; with two roundings each at the size of the sum (the instruction's own
    order is not documented) a chain of n steps has a relative rms error of sqrt(0.09 * 2 n + 4) 2^-24 (a rounding's variance as in
    test_conv2d_staged_operands_error; four more for the small products' own chain and the result).  A quarter on top."""
    return 1.25 * 2.0 ** -24 * (0.18 * terms / 16 + 4) ** 0.5


@pytest.mark.parametrize("data", ["normal", "half_zeros", "positive"])
@pytest.mark.parametrize("case", X3_ERROR_CASES, ids=str)
def test_conv2d_bf16x3_error(dev, case, data):
    """Error against 64-bit sums, all passes: within the bound of the form's own chain, and where the library takes it by itself (it
    does in the passes named) no larger than that of the form it replaces.  positive: all three tensors of one sign, whose sums grow
    with every term; such operands are held to the bound only (tri_max_chain is made for others)."""
    Nn, C, H, K, R, st, pad, takes = case
    say("bf16x3 error", case, data)
    P = (H + 2 * pad - R) // st + 1
    make = synth.uniform if data == "positive" else synth.normal
    x, w, dy = (T(make(35, 1 + i, s), dev) for i, s in enumerate(((Nn, C, H, H), (K, C, R, R), (Nn, K, P, P))))
    if data == "half_zeros":
        x = x.clamp_min(0.0)
    refs = _conv_sums64(x, w, dy, st, pad)
    for key, name, terms, ref, run in (("f", "fwd", C * R * R, refs[0], lambda algo: ops.conv2d_fwd(x, w, st, pad, algo=algo)),
                                       ("d", "bwd_data", K * R * R, refs[1], lambda algo: ops.conv2d_bwd_data(w, dy, x.shape, st, pad, algo=algo)),
                                       ("w", "bwd_filter", Nn * P * P, refs[2], lambda algo: ops.conv2d_bwd_filter(x, dy, w.shape, st, pad, algo=algo))):
        auto, tags = profile_tags(lambda: run(_lib.RH_ALGO_BF16X3))
        assert any(t.startswith("conv_%s_tri_" % name) for t in tags) == (key in takes), (name, tags)
        form = auto if key in takes else None if key == "d" and st > 1 else run(_lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_DIRECT)
        if form is None:
            continue
        err = float((form.double() - ref).norm() / ref.norm())
        assert err <= _chain_bound(terms), (name, terms, err)
        if key in takes and data != "positive":
            before = float((run(0).double() - ref).norm() / ref.norm())
            assert err <= before, (name, err, before)


@pytest.mark.parametrize("case", [(48, 64, 56, 64, 3, 1), (24, 64, 56, 128, 3, 2), (64, 96, 28, 96, 3, 1), (64, 128, 28, 256, 3, 2), (24, 256, 14, 256, 3, 1)], ids=str)
def test_conv2d_bf16x3_deltas_behind_a_batch_norm(dev, case):
    """Filter gradients of positive inputs and deltas with a small value of one sign almost everywhere: one value in ten is large and each
    channel's mean is taken off.  No larger an error against 64-bit sums than the fp32 instruction's, and infinities, NaNs and the
    values that have no sum of three stay where they are."""
    Nn, C, H, K, R, st = case
    say("bf16x3 wide", case)
    P = (H + 2 - R) // st + 1
    x = (1.5 + 0.6 * T(synth.normal(51, 1, (Nn, C, H, H)), dev)).clamp_min(0.01)
    dy = T(synth.normal(51, 2, (Nn, K, P, P)) * (synth.uniform(51, 3, (Nn, K, P, P)) < 0.1), dev)
    dy = dy - dy.mean((0, 2, 3), keepdim=True)
    shape = (K, C, R, R)
    X3 = _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_BF16X3_WIDE
    ref = _conv_sums64(x, torch.zeros(shape, device=dev), dy, st, 1)[2]
    got, before = (ops.conv2d_bwd_filter(x, dy, shape, st, 1, algo=algo).double() for algo in (X3 | _lib.RH_ALGO_DIRECT, _lib.RH_ALGO_SCALAR_OFFSET))
    err, err0 = (float((t - ref).norm() / ref.norm()) for t in (got, before))
    assert err <= err0, (err, err0)


def test_conv2d_bf16x3_wide_marks(dev):
    """The wide form's marks in the last bit of a part: powers of two over the whole range beside a large value, exact products, so that
    every result is known; with an infinity of dy, or a value whose parts need that bit, in the group of eight images."""
    X3 = _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_BF16X3_WIDE | _lib.RH_ALGO_DIRECT
    say("bf16x3 wide marks")
    Nn, C, K = 8, 8, 64
    exps = np.linspace(-149, 100, K).astype(int)
    odd = np.float64(1.0 + 2.0 ** -23)    # 24 significant bits where the exponent has them
    for image in range(Nn):
        for extra in (0.0, 2.0 ** 101, -(2.0 ** 127), np.inf):
            dy = np.zeros((Nn, K, 1, 1), np.float32)
            dy[image, :, 0, 0] = (odd * 2.0 ** exps).astype(np.float32)
            other = (image + 3) % Nn
            dy[other, :, 0, 0] = extra
            x = np.zeros((Nn, C, 1, 1), np.float32)
            x[image], x[other, 4:] = 1.0, 1.0
            got = N(ops.conv2d_bwd_filter(T(x, dev), T(dy, dev), (K, C, 1, 1), 1, 0, algo=X3))[:, :, 0, 0]
            alone = dy[image, :, 0, 0].astype(np.float64)
            if extra == np.inf:
                assert np.all(got[:, 4:] == np.inf) and np.all(np.isnan(got[:, :4]))   # (0 x inf)
                continue
            want = np.stack([alone] * 4 + [alone + extra] * 4, 1).astype(np.float32)
            assert np.all(np.abs(got - want) <= np.spacing(np.abs(want))), (image, extra)
            assert np.array_equal(got[:, :4], want[:, :4]), (image, extra)


# RH_ALGO_F16X2: every operand value as the sum of two scaled fp16 values.  X3_CASES are at its edges too (64 rows to a block of a tile;
# 64 x 256, 96 x 128 and 128 x 128 tiles); then K steps around a chain's end and the ring's (8 K steps and 4 or 5 buffers).
F16X2_CASES = X3_CASES + [(1, 16 * n, 3, 3, 70, 1, 1, 0) for n in (4, 5, 11, 12, 13, 20, 21)] + [(1, 16 * n, 2, 2, 128, 1, 1, 0) for n in (11, 12, 29)] + \
    [(8, 8, 1, 2 * n, 128, 1, 1, 0) for n in (3, 13, 27)]


@pytest.mark.parametrize("case", F16X2_CASES, ids=str)
def test_conv2d_f16x2(dev, case):
    """All passes with operands of two parts against the oracle, with every epilogue; images, filters and channels far apart in size."""
    Nn, C, H, W, K, R, st, pad = case
    say("f16x2 case", case)
    F2 = _lib.RH_ALGO_F16X2 | _lib.RH_ALGO_DIRECT
    x, w, b = synth.normal(37, 1, (Nn, C, H, W)), synth.normal(37, 2, (K, C, R, R)), synth.normal(37, 3, (K,))
    y_ref = O.conv2d_fwd(x, w, st, pad)
    dy, y0, dx0, dw0, db0 = (synth.normal(37, 4 + i, s) for i, s in enumerate((y_ref.shape, y_ref.shape, x.shape, w.shape, (K,))))
    xd, wd, bd, dyd = T(x, dev), T(w, dev), T(b, dev), T(dy, dev)
    image, row = ((2.0 ** (10 * synth.normal(38, i, (n,))).astype(int)[:, None, None, None]).astype(np.float32) for i, n in ((0, Nn), (1, K)))
    if C % 8 == 0:
        y, tags = profile_tags(lambda: ops.conv2d_fwd(xd, wd, st, pad, algo=F2))
        assert any(t.startswith("conv_fwd_duo_") for t in tags), tags
        assert_close(N(y), y_ref, "f16x2 fwd")
        yf = ops.conv2d_fwd(xd, wd, st, pad, bias=bd, relu=True, algo=F2)
        assert torch.equal(torch.clamp_min(y + bd.view(1, -1, 1, 1), 0.0), yf), "fused epilogue == conv, add_bias, rect"
        yb = ops.conv2d_fwd(xd, wd, st, pad, alpha=0.5, beta=2.0, y=T(y0, dev), algo=F2)
        assert_close(N(yb), O.conv2d_fwd(x, w, st, pad, alpha=0.5, beta=2.0, y=y0.copy()), "f16x2 fwd alpha/beta")
        assert torch.equal(ops.conv2d_fwd(xd, wd, st, pad, algo=F2), y), "run to run the same bits"
        scaled = ops.conv2d_fwd(T(x * image, dev), T(w * row, dev), st, pad, algo=F2)
        assert np.array_equal(N(scaled), N(y) * image * row.reshape(1, -1, 1, 1)), "powers of two of an image and a filter"
    else:
        with pytest.raises(_lib.RembrandtHipError):
            ops.conv2d_fwd(xd, wd, st, pad, algo=F2)
    if K % 8 == 0 and st == 1 and pad <= R - 1:
        dx, tags = profile_tags(lambda: ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, algo=F2))
        assert any(t.startswith("conv_bwd_data_duo_") for t in tags), tags
        assert_close(N(dx), O.conv2d_bwd_data(w, dy, x.shape, st, pad), "f16x2 bwd data")
        two = ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, alpha=0.5, beta=2.0, dx=T(dx0, dev), algo=F2)
        assert_close(N(two), O.conv2d_bwd_data(w, dy, x.shape, st, pad, 0.5, 2.0, dx0.copy()), "f16x2 bwd data alpha/beta")
        ops.rect_backprop_inplace(xd, two)
        one = ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, alpha=0.5, beta=2.0, dx=T(dx0, dev), algo=F2, relu_of=xd)
        assert torch.equal(one, two), "masked data gradient"
        assert np.array_equal(N(ops.conv2d_bwd_data(wd, T(dy * image, dev), x.shape, st, pad, algo=F2)), N(dx) * image), "powers of two of an image"
    else:
        with pytest.raises(_lib.RembrandtHipError):
            ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad, algo=F2)
    dw, tags = profile_tags(lambda: ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, algo=F2))
    assert any(t.startswith("conv_bwd_filter_duo_") for t in tags), tags
    assert_close(N(dw), O.conv2d_bwd_filter(x, dy, w.shape, st, pad), "f16x2 bwd filter")
    dwc, dbc = ops.conv2d_bwd_filter_bias(xd, dyd, w.shape, st, pad, alpha=0.25, beta=1.0, dw=T(dw0, dev), db=T(db0, dev), algo=F2)
    assert_close(N(dwc), O.conv2d_bwd_filter(x, dy, w.shape, st, pad, 0.25, 1.0, dw0.copy()), "f16x2 bwd filter alpha/beta")
    assert_close(N(dbc), O.conv2d_bwd_bias(dy, 0.25, 1.0, db0.copy()), "f16x2 bias gradient")
    assert torch.equal(ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, algo=F2), dw), "run to run the same bits"
    scaled = ops.conv2d_bwd_filter(xd, T(dy * row.reshape(1, -1, 1, 1), dev), w.shape, st, pad, algo=F2)
    assert np.array_equal(N(scaled), N(dw) * row), "powers of two of a channel"


def test_conv2d_f16x2_values_out_of_range(dev):
    """What two parts cannot hold is formed again from the operands: values far below the largest of their image or channel, infinities,
    NaNs, the largest and the smallest floats."""
    say("f16x2 values")
    F2, big = _lib.RH_ALGO_F16X2 | _lib.RH_ALGO_DIRECT, np.finfo(np.float32).max
    Nn, C, H, K, R = 9, 24, 12, 72, 3
    x, w = synth.normal(39, 1, (Nn, C, H, H)), 0.01 * synth.normal(39, 2, (K, C, R, R))
    dy = synth.normal(39, 3, (Nn, K, H, H))
    x[0, :, 2, 2], x[1] = 1e25, x[1] * 1e-30             # one pixel beside which the others of its image have no bits; a small image
    x[2, 3, 5, 5], x[3, 4, 1, 1], x[4, 0, 0, 0] = np.inf, np.nan, -np.inf
    x[5] *= np.float32(1e-42)                            # denormal
    w[7] *= np.float32(1e-38)
    dy[:, 5, 0, 0] = 0.0
    dy[8, 5, 3, 3] = 1e28
    magnitudes = [np.abs(np.where(np.isfinite(t), t, 0.0)) for t in (x, w, dy)]
    passes = (lambda x, w, dy: O.conv2d_fwd(x, w, 1, 1), lambda x, w, dy: O.conv2d_bwd_filter(x, dy, w.shape, 1, 1),
              lambda x, w, dy: O.conv2d_bwd_data(w, dy, x.shape, 1, 1))
    for name, run, oracle in (("fwd", lambda a: ops.conv2d_fwd(T(x, dev), T(w, dev), 1, 1, algo=a), passes[0]),
                              ("bwd filter", lambda a: ops.conv2d_bwd_filter(T(x, dev), T(dy, dev), w.shape, 1, 1, algo=a), passes[1]),
                              ("bwd data", lambda a: ops.conv2d_bwd_data(T(w, dev), T(dy, dev), x.shape, 1, 1, algo=a), passes[2])):
        got, other, ref = N(run(F2)), N(run(_lib.RH_ALGO_GATHER)), oracle(x, w, dy)
        assert np.array_equal(np.isnan(got), np.isnan(other)) and np.array_equal(np.isinf(got), np.isinf(other)), name
        ok = np.isfinite(ref) & np.isfinite(got) & (np.abs(ref) >= 2.0 ** -126)
        # 2^-21 for what the parts lose and some hundred roundings of 2^-24 (1296 products at most), of the sum of the products' magnitudes
        size = oracle(*magnitudes)
        assert ok.any() and np.all(np.abs(got[ok].astype(np.float64) - ref[ok]) <= 2.0 ** -18 * size[ok]), name
        # of each result plane, whose sums are of one size; 24 x 9 terms of relative error 2^-22 at most each, in quadrature below 2^-21
        for g, r, m in zip(got.reshape(-1, got.shape[-1] ** 2).astype(np.float64), ref.reshape(-1, got.shape[-1] ** 2).astype(np.float64), ok.reshape(-1, got.shape[-1] ** 2)):
            if not m.any() or np.abs(r[m]).max() > 1e3 * np.median(np.abs(r[m])):   # (a plane with the large pixel: its far results below)
                continue
            assert np.linalg.norm(g[m] - r[m]) <= 2.0 ** -21 * np.linalg.norm(r[m]), name
        if name == "fwd":   # away from the large pixel of image 0
            far = np.s_[0, :, 5:, 5:]
            assert np.linalg.norm((got[far] - ref[far]).astype(np.float64)) <= 2.0 ** -21 * np.linalg.norm(ref[far].astype(np.float64))
    x = np.zeros((1, 8, 1, 8), np.float32)
    x[0, 3] = [big, -big, 1.0, 2.0 ** -149, 2.0 ** -126, 0.0, -0.0, 3.0]
    w = np.zeros((64, 8, 1, 1), np.float32)
    w[:, 3, 0, 0] = 1.0
    got = N(ops.conv2d_fwd(T(x, dev), T(w, dev), 1, 0, algo=F2))
    assert np.array_equal(got[0], np.broadcast_to(x[0, 3], (64, 1, 8)))


def _f16x2_range_passes(dev, algo):
    """name, run(filter, input), the same by the oracle, for the two passes whose operands share groups of eight channels: stride 1, extents kept."""
    pad = lambda w: w.shape[2] // 2
    yield "fwd", lambda w, x: N(ops.conv2d_fwd(T(x, dev), T(w, dev), 1, pad(w), algo=algo)), lambda w, x: O.conv2d_fwd(x, w, 1, pad(w))
    flip = lambda w: np.ascontiguousarray(w.transpose(1, 0, 2, 3))   # contracted: the filters
    shape = lambda w, x: (len(x), len(w)) + x.shape[2:]
    yield ("bwd data", lambda w, x: N(ops.conv2d_bwd_data(T(flip(w), dev), T(x, dev), shape(w, x), 1, pad(w), algo=algo)),
           lambda w, x: O.conv2d_bwd_data(flip(w), x, shape(w, x), 1, pad(w)))


@pytest.mark.parametrize("k", [20, 29, 31, 36, 45, 52, 80, 120])
def test_conv2d_f16x2_small_values_beside_large_ones(dev, k):
    """Every channel but the eighth of each group 2^-k as large, in the input where the eighth's weight is 0 and in the filter where the
    eighth's input is: the result is of the small values alone, and has the bits of any other.  16 x 9 products of relative error 2^-21 at
    most each, and sums of a hundred roundings of 2^-24 at most: 2^-18 of the sum of magnitudes."""
    say("f16x2 small beside large", k)
    x0, w0 = synth.normal(40, 1, (3, 16, 7, 6)), 0.1 * synth.normal(40, 2, (70, 16, 3, 3))
    eighth = np.arange(16) % 8 == 7
    for small, other in ((0, 1), (1, 0)):
        pair = [x0.copy(), w0.copy()]
        pair[small][:, ~eighth] *= np.float32(2.0) ** -k
        pair[other][:, eighth] = 0.0
        x, w = pair
        for name, run, ref in _f16x2_range_passes(dev, _lib.RH_ALGO_F16X2 | _lib.RH_ALGO_DIRECT):
            got, want, size = run(w, x), ref(w, x), ref(np.abs(w), np.abs(x))
            assert np.all(np.abs(got.astype(np.float64) - want) <= 2.0 ** -18 * size), (name, small)


def test_conv2d_f16x2_values_of_all_sizes(dev):
    """Values of every size beside one another, zeros among them: each result as exact against the sum of its products' magnitudes."""
    say("f16x2 all sizes")
    x, w = synth.normal(41, 1, (5, 8, 17, 16)), synth.normal(41, 2, (136, 8, 1, 1))
    x *= np.float32(2.0) ** -np.floor(50 * synth.uniform(41, 3, x.shape)) * (synth.uniform(41, 4, x.shape) < 0.7)
    for spread, zeros in ((0, 0.0), (12, 0.0), (12, 0.6), (50, 0.6)):
        ww = w * np.float32(2.0) ** -np.floor(spread * synth.uniform(41, 5, w.shape)) * (synth.uniform(41, 6, w.shape) >= zeros)
        for name, run, ref in _f16x2_range_passes(dev, _lib.RH_ALGO_F16X2 | _lib.RH_ALGO_DIRECT):
            got, want, size = run(ww, x), ref(ww, x), ref(np.abs(ww), np.abs(x))
            assert np.all(np.abs(got.astype(np.float64) - want) <= 2.0 ** -20 * size), (name, spread, zeros)


@pytest.mark.parametrize("k", [20, 29, 31, 36, 45, 52, 80, 120])
def test_conv2d_f16x2_filter_gradient_of_small_values(dev, k):
    """The same for the filter gradient: one sample's values large where the other operand's are 0, the others' 2^-k as large, a few of
    them or all.  18 x 56 products at most: 2^-18 of the sum of magnitudes."""
    say("f16x2 small in a batch", k)
    x0, dy0, shape = synth.normal(42, 1, (18, 10, 8, 7)), synth.normal(42, 2, (18, 70, 8, 7)), (70, 10, 3, 3)
    few = synth.uniform(42, 3, (18, 1, 8, 7)) < 0.01
    for small, other in ((0, 1), (1, 0)):
        for some in (few, np.ones_like(few)):
            pair = [x0.copy(), dy0.copy()]
            pair[small][1:] *= np.float32(2.0) ** -k * some[1:]
            pair[other][0] = 0.0
            x, dy = pair
            got = N(ops.conv2d_bwd_filter(T(x, dev), T(dy, dev), shape, 1, 1, algo=_lib.RH_ALGO_F16X2 | _lib.RH_ALGO_DIRECT))
            want, size = O.conv2d_bwd_filter(x, dy, shape, 1, 1), O.conv2d_bwd_filter(np.abs(x), np.abs(dy), shape, 1, 1)
            assert np.all(np.abs(got.astype(np.float64) - want) <= 2.0 ** -18 * size), (small, some.all())


@pytest.mark.parametrize("kind", ["none", "one", "many", "x", "nan"])
def test_conv2d_f16x2_filter_gradient_in_three_parts(dev, kind):
    """Where the library takes two parts by itself, beside RH_ALGO_BF16X3: a value that two parts cannot hold, or that is no finite number,
    makes it the call with RH_ALGO_BF16X3 alone."""
    say("f16x2 or three parts", kind)
    Nn, C, H, K, R, pad = 128, 96, 27, 96, 5, 2
    x, dy = T(synth.normal(43, 1, (Nn, C, H, H)), dev).clamp_min(0.0), T(synth.normal(43, 2, (Nn, K, H, H)), dev)
    x, dy = (torch.where(t.abs() < 1e-4, torch.zeros_like(t), t) for t in (x, dy))   # (none by chance)
    X3, F2, shape = _lib.RH_ALGO_BF16X3, _lib.RH_ALGO_F16X2, (K, C, R, R)
    x[0], x[:, 5] = 0.0, 0.0
    if kind == "one":
        dy[77, 11, 26, 26] = 2.0 ** -41
    elif kind == "many":
        dy[1:] *= 2.0 ** -40
    elif kind == "x":
        x[127, 95, 0, 0] = 2.0 ** -45
    elif kind == "nan":
        dy[3, 2], x[40, 3, 3, 3], x[41, 17, 0, 0] = float("nan"), float("inf"), float("nan")
    call = lambda algo: ops.conv2d_bwd_filter_bias(x, dy, shape, 1, pad, alpha=0.5, algo=algo)
    (got, db), tags = profile_tags(lambda: call(X3 | F2))
    assert any(t.startswith("conv_bwd_filter_duo_") for t in tags) and "tri_rest" in tags, tags
    (three, db3), tags = profile_tags(lambda: call(X3))
    assert any(t.startswith("conv_bwd_filter_tri_") for t in tags), tags
    same = torch.equal(torch.isnan(got), torch.isnan(three)) and torch.equal(got.nan_to_num(), three.nan_to_num())
    assert same == (kind != "none")
    assert torch.allclose(got, three, rtol=1e-5, atol=1e-5 * float(three.nan_to_num().abs().max()), equal_nan=True)
    assert torch.allclose(db, db3, rtol=1e-5, atol=1e-5 * float(db3.nan_to_num().abs().max()), equal_nan=True)
    again = call(X3 | F2)
    assert torch.equal(again[0].nan_to_num(), got.nan_to_num()) and torch.equal(again[1].nan_to_num(), db.nan_to_num()), "run to run the same bits"


@pytest.mark.parametrize("case", [(90, 256, 14, 256, 3, 1), (24, 512, 7, 512, 3, 1)], ids=str)
def test_conv2d_f16x2_deltas_behind_a_batch_norm(dev, case):
    """A filter gradient whose caller sets RH_ALGO_BF16X3_WIDE stays with three parts."""
    Nn, C, H, K, R, st = case
    say("f16x2 wide", case)
    P = (H + 2 - R) // st + 1
    x = (1.5 + 0.6 * T(synth.normal(51, 1, (Nn, C, H, H)), dev)).clamp_min(0.01)
    dy = T(synth.normal(51, 2, (Nn, K, P, P)) * (synth.uniform(51, 3, (Nn, K, P, P)) < 0.1), dev)
    dy = dy - dy.mean((0, 2, 3), keepdim=True)
    shape, X3 = (K, C, R, R), _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_BF16X3_WIDE
    got, tags = profile_tags(lambda: ops.conv2d_bwd_filter(x, dy, shape, st, 1, algo=X3 | _lib.RH_ALGO_F16X2))
    assert any(t.startswith("conv_bwd_filter_tri_wide_") for t in tags), tags
    assert torch.equal(got, ops.conv2d_bwd_filter(x, dy, shape, st, 1, algo=X3))


# Layers with the passes that the library takes in this form by itself beside RH_ALGO_BF16X3: whole contractions, slices, a sliced
# tail, 64- and 96-row tiles
F16X2_ERROR_CASES = [
    # N, C, H, K, R, stride, pad, passes
    (50, 384, 13, 384, 3, 1, 1, "fd"),
    (24, 96, 27, 256, 5, 1, 2, "f"),
    (128, 96, 27, 256, 5, 1, 2, "fw"),
    (64, 128, 28, 128, 3, 1, 1, "fd"),
    (200, 64, 56, 64, 3, 1, 1, "fd"),
    (128, 512, 7, 512, 3, 1, 1, "fd"),
    (16, 96, 27, 256, 1, 1, 0, ""),
]


@pytest.mark.parametrize("data", ["normal", "half_zeros", "positive"])
@pytest.mark.parametrize("case", F16X2_ERROR_CASES, ids=str)
def test_conv2d_f16x2_error(dev, case, data):
    """Error against 64-bit sums where the library takes the form by itself: no larger than that of the form it replaces.  positive: all three
    tensors of one sign, where the instruction's cuts add up; each of the eight products that it adds at once loses up to 2^-24 of the
    largest of them, which is no larger than their sum (2^-21 of it at most), whatever the sum's length."""
    Nn, C, H, K, R, st, pad, takes = case
    say("f16x2 error", case, data)
    P = (H + 2 * pad - R) // st + 1
    x, w, dy = (T(synth.normal(36, 1 + i, s), dev) for i, s in enumerate(((Nn, C, H, H), (K, C, R, R), (Nn, K, P, P))))
    if data == "half_zeros":
        x, dy = x.clamp_min(0.0), dy * (T(synth.uniform(36, 4, dy.shape), dev) < 0.5)
    elif data == "positive":
        x, w, dy = x.abs(), w.abs(), dy.abs()
    X3 = _lib.RH_ALGO_BF16X3
    refs = _conv_sums64(x, w, dy, st, pad)
    for key, name, ref, run in (("f", "fwd", refs[0], lambda algo: ops.conv2d_fwd(x, w, st, pad, algo=algo)),
                                ("d", "bwd_data", refs[1], lambda algo: ops.conv2d_bwd_data(w, dy, x.shape, st, pad, algo=algo)),
                                ("w", "bwd_filter", refs[2], lambda algo: ops.conv2d_bwd_filter(x, dy, w.shape, st, pad, algo=algo))):
        got, tags = profile_tags(lambda: run(X3 | _lib.RH_ALGO_F16X2))
        assert any(t.startswith("conv_%s_duo_" % name) for t in tags) == (key in takes), (name, tags)
        before = run(X3)
        if key in takes:
            err, err0 = (float((t.double() - ref).norm() / ref.norm()) for t in (got, before))
            assert err <= err0, (name, err, err0)
        else:
            assert torch.equal(got, before), name
        if data == "positive":
            form = run(_lib.RH_ALGO_F16X2 | _lib.RH_ALGO_DIRECT)
            assert float((form.double() - ref).norm() / ref.norm()) <= 2.0 ** -21 + 2.0 ** -23, name


# Data gradients of deltas that are zeros for nine in ten, as behind a max-pool, where what three parts round is less; whether two are taken:
# tiles that three parts sum in shorter chains (a tail in slices), whole contractions in slices, one long chain.
@pytest.mark.parametrize("case", [(105, 384, 13, 256, 3, False), (97, 384, 13, 256, 3, False), (105, 256, 14, 256, 3, False), (64, 512, 7, 512, 3, False),
                                  (24, 1024, 6, 1024, 3, False), (200, 384, 13, 384, 3, True), (105, 96, 27, 256, 5, True)], ids=str)
def test_conv2d_f16x2_error_of_sparse_deltas(dev, case):
    """As test_conv2d_f16x2_error; with RH_ALGO_BF16X3_WIDE (few deltas are zeros) the choice is another, on such operands."""
    Nn, C, H, K, R, takes = case
    say("f16x2 sparse deltas", case)
    X3, F2, WIDE = _lib.RH_ALGO_BF16X3, _lib.RH_ALGO_F16X2, _lib.RH_ALGO_BF16X3_WIDE
    x, w = torch.zeros((Nn, C, H, H), device=dev), T(synth.normal(45, 1, (K, C, R, R)), dev)
    dense = T(synth.normal(45, 2, (Nn, K, H, H)), dev)
    sparse = dense * (T(synth.uniform(45, 3, (Nn, K, H, H)), dev) < 0.1)
    for dy, flags, taken in ((sparse, X3, takes), (dense, X3 | WIDE, None)):
        run = lambda algo: ops.conv2d_bwd_data(w, dy, x.shape, 1, R // 2, algo=algo)
        got, tags = profile_tags(lambda: run(flags | F2))
        assert taken is None or any(t.startswith("conv_bwd_data_duo_") for t in tags) == taken, tags
        ref = _conv_sums64(x, w, dy, 1, R // 2)[1]
        err, err0 = (float((t.double() - ref).norm() / ref.norm()) for t in (got, run(flags)))
        assert err <= err0, (flags, err, err0)


@pytest.mark.parametrize("case", [(9, 16, 14, 11, 40, 3, 5, 1, 2), (3, 24, 9, 12, 72, 1, 4, 1, 0), (8, 40, 12, 9, 64, 5, 1, 1, 1),
                                  (5, 16, 13, 10, 33, 2, 3, 2, 1), (24, 64, 30, 28, 128, 2, 3, 2, 1)], ids=str)
def test_conv2d_bf16x3_filters_that_are_not_square(dev, case):
    """R != S through the C interface: forward and filter gradient have the form; the data gradient has it by residue classes, with a
    stride, and with RH_ALGO_DIRECT is RH_E_UNSUPPORTED."""
    import ctypes as C
    Nn, Cc, H, W, K, R, S, st, pad = case
    say("bf16x3 not square", case)
    lib, X3 = _lib.lib(), _lib.RH_ALGO_BF16X3
    forced = X3 | _lib.RH_ALGO_DIRECT
    g = _lib.ConvGeom(Nn, Cc, H, W, K, R, S, st, pad)
    P, Q = (H + 2 * pad - R) // st + 1, (W + 2 * pad - S) // st + 1
    x, w, dy = (T(synth.normal(51, 1 + i, s), dev) for i, s in enumerate(((Nn, Cc, H, W), (K, Cc, R, S), (Nn, K, P, Q))))
    y_ref, dx_ref, dw_ref = _conv_sums64(x, w, dy, st, pad)
    size = max(lib.rh_conv2d_workspace_bytes_for(C.byref(g), p, f) for p in range(3) for f in (X3, forced))
    ws = torch.empty(size + 256, dtype=torch.uint8, device=dev)
    at = (ws.data_ptr() + 255) // 256 * 256
    y, dw, dx, dx0 = torch.empty_like(dy), torch.empty_like(w), torch.zeros_like(x), torch.zeros_like(x)
    assert lib.rh_conv2d_fwd(C.byref(g), 1.0, x.data_ptr(), w.data_ptr(), 0.0, y.data_ptr(), None, at, size, forced, None) == 0
    assert lib.rh_conv2d_bwd_filter(C.byref(g), 1.0, x.data_ptr(), dy.data_ptr(), 0.0, dw.data_ptr(), at, size, forced, None) == 0
    bwd_data = lambda out, flags: lib.rh_conv2d_bwd_data(C.byref(g), 1.0, w.data_ptr(), dy.data_ptr(), 0.0, out.data_ptr(), at, size, flags, None)
    assert bwd_data(dx, forced) == _lib.RH_E_UNSUPPORTED
    rc, tags = profile_tags(lambda: bwd_data(dx, X3))
    classes = any(t.startswith("conv_bwd_data_tri_") for t in tags)
    assert rc == 0 and classes == (case[0] == 24), tags
    assert bwd_data(dx0, 0) == 0
    torch.cuda.synchronize()
    for got, ref, terms in ((y, y_ref, Cc * R * S), (dw, dw_ref, Nn * P * Q)) + (((dx, dx_ref, K * R * S),) if classes else ()):
        err = float((got.double() - ref).norm() / ref.norm())
        assert err <= _chain_bound(terms), (err, terms)
    assert classes or torch.equal(dx, dx0)


def test_conv2d_bf16x3_infinities_and_largest_floats(dev):
    """What is not finite comes out as fp32 multiplication makes it: infinities where no NaN is, NaNs where there are (the
    products of an infinity's zero parts are NaNs inside); values that round to an infinity in bf16 stay finite."""
    X3 = _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_DIRECT
    Nn, C, H, W, K, R, pad = 19, 40, 13, 13, 72, 3, 1
    x, w = synth.normal(37, 1, (Nn, C, H, W)), synth.normal(37, 2, (K, C, R, R))
    dy = synth.normal(37, 3, (Nn, K, H, W))
    x[3, 5, 4, 4], x[4, 7, 0, 12], x[6, 1, 1, 1] = np.inf, -np.inf, np.nan
    x[7, 2, 3, 3], x[8, 2, 3, 3] = 3.4e38, -np.finfo(np.float32).max
    w[5, :, 1, 1], w[6] = 0.5, 0.125
    dy[2, 3, 1, 1] = np.inf
    w[:, 2] *= 0.125   # (the largest floats' products stay in range)
    xd, wd, dyd = T(x, dev), T(w, dev), T(dy * 0.125, dev)
    G = _lib.RH_ALGO_SCALAR_OFFSET
    wide = X3 | _lib.RH_ALGO_BF16X3_WIDE
    for form, run in ((X3, lambda algo: ops.conv2d_fwd(xd, wd, 1, pad, algo=algo)), (X3, lambda algo: ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, algo=algo)),
                      (X3, lambda algo: ops.conv2d_bwd_filter(xd, dyd, w.shape, 1, pad, algo=algo)),
                      (wide, lambda algo: ops.conv2d_bwd_filter(xd, dyd, w.shape, 1, pad, algo=algo))):
        got, ref = run(form), run(G)
        assert bool(torch.isinf(ref).any())
        assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
        keep = torch.isfinite(ref)
        assert torch.equal(got[torch.isinf(ref)], ref[torch.isinf(ref)])
        assert bool(((got - ref).abs()[keep] <= 1e-4 * (1.0 + ref.abs()[keep])).all())


def test_conv2d_bf16x3_largest_floats_beside_an_infinity(dev):
    """A result that is formed again in fp32 because of an infinity takes the largest floats as they are: their first two parts add
    up to 2^128, and an infinity of the other sign would make a NaN of the result."""
    X3 = _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_DIRECT
    x, w = torch.full((1, 8, 4, 4), -0.125, device=dev), torch.full((16, 8, 1, 1), 0.5, device=dev)
    x[0, 0], w[:, 1] = float("inf"), torch.finfo(torch.float32).max
    assert bool((ops.conv2d_fwd(x, w, 1, 0, algo=X3) == float("inf")).all())


def _redo_bound(terms):
    """Relative error of sums on the fp32 instruction in two levels, chains of 128 terms and the sum of them: a rounding's variance
    as in test_conv2d_staged_operands_error, a quarter on top."""
    return 1.25 * 2.0 ** -24 * (0.09 * (128 + terms / 128) + 4) ** 0.5


@pytest.mark.parametrize("exponent", [-112, -120, -126, -140])
def test_conv2d_bf16x3_small_operands(dev, exponent):
    """Operands whose last bits lie under bf16's smallest value, 2^-133, beside large ones: no bit of them is lost.  Both of a
    pass's operands in turn, all of a tensor or one value in a hundred (of which the others' results must not suffer)."""
    X3 = _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_DIRECT
    Nn, C, H, W, K, R, pad = 9, 40, 12, 11, 72, 3, 1
    shapes = (Nn, C, H, W), (K, C, R, R), (Nn, K, H, W)
    big = np.float32(2.0 ** 100)
    for tiny in range(3):
        for share in (1.0, 0.01):
            say("bf16x3 small operands", exponent, tiny, share)
            t = [synth.normal(43, 1 + i, s) for i, s in enumerate(shapes)]
            small = (t[tiny].astype(np.float64) * 2.0 ** exponent).astype(np.float32)
            assert np.any(small != 0)
            t = [a * big for a in t]
            t[tiny] = small if share == 1.0 else np.where(synth.uniform(43, 9, t[tiny].shape) < share, small, t[tiny] / big)
            x, w, dy = t
            xd, wd, dyd = T(x, dev), T(w, dev), T(dy, dev)
            for name, operands, terms, ref, run in (
                    ("fwd", (0, 1), C * R * R, lambda: O.conv2d_fwd(x, w, 1, pad), lambda: ops.conv2d_fwd(xd, wd, 1, pad, algo=X3)),
                    ("bwd_data", (1, 2), K * R * R, lambda: O.conv2d_bwd_data(w, dy, x.shape, 1, pad), lambda: ops.conv2d_bwd_data(wd, dyd, x.shape, 1, pad, algo=X3)),
                    ("bwd_filter", (0, 2), Nn * H * W, lambda: O.conv2d_bwd_filter(x, dy, w.shape, 1, pad), lambda: ops.conv2d_bwd_filter(xd, dyd, w.shape, 1, pad, algo=X3)),
                    ("bwd_filter wide", (0, 2), Nn * H * W, lambda: O.conv2d_bwd_filter(x, dy, w.shape, 1, pad),
                     lambda: ops.conv2d_bwd_filter(xd, dyd, w.shape, 1, pad, algo=X3 | _lib.RH_ALGO_BF16X3_WIDE))):
                if tiny not in operands:
                    continue
                want = ref().astype(np.float64)
                err = np.linalg.norm(N(run()).astype(np.float64) - want) / np.linalg.norm(want)
                assert err <= _redo_bound(terms), (name, err)


@pytest.mark.parametrize("exponent", [-112, -126, -140])
def test_conv2d_bf16x3_strided_small_operands(dev, exponent):
    """As above, the data gradient by residue classes."""
    Nn, C, H, W, K, R, st, pad = X3_STRIDED_CASES[0]
    P, Q = (H + 2 * pad - R) // st + 1, (W + 2 * pad - R) // st + 1
    w, dy = synth.normal(45, 1, (K, C, R, R)), synth.normal(45, 2, (Nn, K, P, Q))
    for a, b in ((exponent, 100), (100, exponent)):
        ws, dys = ((t.astype(np.float64) * 2.0 ** e).astype(np.float32) for t, e in ((w, a), (dy, b)))
        got, tags = profile_tags(lambda: ops.conv2d_bwd_data(T(ws, dev), T(dys, dev), (Nn, C, H, W), st, pad, algo=_lib.RH_ALGO_BF16X3))
        assert any(t.startswith("conv_bwd_data_tri_") for t in tags), tags
        want = O.conv2d_bwd_data(ws, dys, (Nn, C, H, W), st, pad).astype(np.float64)
        err = np.linalg.norm(N(got).astype(np.float64) - want) / np.linalg.norm(want)
        assert err <= _redo_bound(K * R * R), err


def test_conv2d_bf16x3_what_the_parts_leave_cancels(dev):
    """Two values of a group of eight of which nothing fits the parts, of opposite signs: each counts by itself."""
    X3 = _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_DIRECT
    x, w = torch.zeros((1, 8, 4, 4), device=dev), torch.zeros((16, 8, 1, 1), device=dev)
    x[0, 0], x[0, 1] = 2.0 ** -149, -2.0 ** -149
    w[:, 0], w[:8, 1] = 2.0 ** 100, -2.0 ** 101
    y = ops.conv2d_fwd(x, w, 1, 0, algo=X3)
    assert bool((y[:, :8] == 3 * 2.0 ** -49).all()) and bool((y[:, 8:] == 2.0 ** -49).all())


def test_conv2d_bf16x3_where_it_pays(dev):
    """RH_ALGO_BF16X3 alone: the form where it is expected to be the fastest, and the others' bits elsewhere."""
    for (Nn, C, H, K, R, st, pad), takes in (((37, 256, 13, 384, 3, 1, 1), True), ((24, 128, 28, 256, 3, 2, 1), True), ((8, 96, 27, 256, 5, 1, 2), True),
                                             ((16, 96, 54, 96, 1, 1, 0), False), ((1, 256, 13, 384, 3, 1, 1), False), ((4, 12, 20, 24, 3, 1, 1), False)):
        x, w = T(synth.normal(39, 1, (Nn, C, H, H)), dev), T(synth.normal(39, 2, (K, C, R, R)), dev)
        y, tags = profile_tags(lambda: ops.conv2d_fwd(x, w, st, pad, algo=_lib.RH_ALGO_BF16X3))
        assert any(t.startswith("conv_fwd_tri_") for t in tags) == takes, (Nn, C, H, K, R, tags)
        other = ops.conv2d_fwd(x, w, st, pad)
        if not takes:
            assert torch.equal(y, other)
        assert bool(((y - other).norm() <= 2e-6 * other.norm()).item())


def test_conv2d_bf16x3_without_room_for_it(dev):
    """RH_ALGO_BF16X3 alone with the scratch of a caller that does not know the bit, in all passes and with a stride: taken, in the
    form that runs without it; with room for the form, that form.  With RH_ALGO_DIRECT, which leaves no other, refused."""
    import ctypes as C
    lib, X3 = _lib.lib(), _lib.RH_ALGO_BF16X3
    for Nn, Cc, H, K, R, st, pad in ((37, 256, 13, 384, 3, 1, 1), (24, 64, 56, 128, 3, 2, 1)):
        say("bf16x3 without room", (Nn, Cc, H, K, R, st))
        g = _lib.ConvGeom(Nn, Cc, H, H, K, R, R, st, pad)
        P = (H + 2 * pad - R) // st + 1
        x, w, dy = (T(synth.normal(49, 1 + i, s), dev) for i, s in enumerate(((Nn, Cc, H, H), (K, Cc, R, R), (Nn, K, P, P))))
        for pass_, name in ((_lib.RH_CONV_FWD, "fwd"), (_lib.RH_CONV_BWD_DATA, "bwd_data"), (_lib.RH_CONV_BWD_FILTER, "bwd_filter")):
            plain, need = lib.rh_conv2d_workspace_bytes(C.byref(g), pass_), lib.rh_conv2d_workspace_bytes_for(C.byref(g), pass_, X3)
            ws = torch.empty(max(plain, need) + 256, dtype=torch.uint8, device=dev)
            at = (ws.data_ptr() + 255) // 256 * 256

            def call(flags, room):
                out = torch.zeros_like({"fwd": dy, "bwd_data": x, "bwd_filter": w}[name])
                o = out.data_ptr()
                if name == "fwd":
                    rc = lib.rh_conv2d_fwd(C.byref(g), 1.0, x.data_ptr(), w.data_ptr(), 0.0, o, None, at, room, flags, None)
                elif name == "bwd_data":
                    rc = lib.rh_conv2d_bwd_data(C.byref(g), 1.0, w.data_ptr(), dy.data_ptr(), 0.0, o, at, room, flags, None)
                else:
                    rc = lib.rh_conv2d_bwd_filter(C.byref(g), 1.0, x.data_ptr(), dy.data_ptr(), 0.0, o, at, room, flags, None)
                torch.cuda.synchronize()
                return rc, out
            (rc0, without), (rc1, small) = call(0, plain), call(X3, plain)
            assert rc0 == 0 and rc1 == 0, (name, rc0, rc1)
            (rc2, _), tags = profile_tags(lambda: call(X3, need))
            took = any(t.startswith("conv_%s_tri_" % name) for t in tags)
            assert rc2 == 0 and (took or name == "bwd_filter" and st == 2), (name, tags)
            if need > plain or not took:
                assert torch.equal(without, small), name
            if st == 1:
                forced = lib.rh_conv2d_bf16x3_workspace_bytes(C.byref(g), pass_)
                if forced > plain:
                    assert call(X3 | _lib.RH_ALGO_DIRECT, plain)[0] == _lib.RH_E_WORKSPACE, name


def test_conv2d_bf16x3_on_one_row_tile_of_filters(dev):
    """Layers of up to 128 filters take the form where it is the faster one as others do: the filter gradient (98 -> 64, 139 -> 92
    us) and the 5x5 forward pass (198 -> 141 us), no further from 64-bit sums than the Winograd form."""
    for (Nn, C, H, K, R, pad), pass_ in (((37, 128, 28, 128, 3, 1), "bwd_filter"), ((64, 128, 28, 128, 3, 1), "bwd_filter"), ((128, 64, 24, 128, 5, 2), "fwd")):
        say("bf16x3 one row tile", (Nn, C, H, K, R, pass_))
        x, w, dy = synth.normal(47, 1, (Nn, C, H, H)), synth.normal(47, 2, (K, C, R, R)), synth.normal(47, 3, (Nn, K, H, H))
        xd, wd, dyd = T(x, dev), T(w, dev), T(dy, dev)
        run = ((lambda algo: ops.conv2d_fwd(xd, wd, 1, pad, algo=algo)) if pass_ == "fwd" else
               (lambda algo: ops.conv2d_bwd_filter(xd, dyd, w.shape, 1, pad, algo=algo)))
        got, tags = profile_tags(lambda: run(_lib.RH_ALGO_BF16X3))
        assert any(t.startswith("conv_%s_tri_" % pass_) for t in tags), tags
        before, tags = profile_tags(lambda: run(0))
        assert "conv_%s_wino" % pass_ in tags, tags
        ref = (O.conv2d_fwd(x, w, 1, pad) if pass_ == "fwd" else O.conv2d_bwd_filter(x, dy, w.shape, 1, pad)).astype(np.float64)
        err, old = (np.linalg.norm(N(t).astype(np.float64) - ref) for t in (got, before))
        assert err <= old, (err, old)


# input channels a multiple of 8 take the packed-operand form (bf16 copies of image and filter in 16-byte groups of
# eight channels): channel groups that do not fill a 64-wide tile, rectangular images, stride with padding, no padding,
# more filters than one row tile, a contraction shorter than one K step
BF16_PACKED_CASES = [
    (3, 72, 11, 9, 40, 3, 2, 1),
    (2, 8, 17, 17, 200, 5, 1, 2),
    (5, 16, 9, 12, 24, 3, 1, 0),
    (2, 8, 6, 6, 3, 1, 1, 0),
    (130, 8, 5, 5, 16, 3, 1, 1),
    # long contractions on grids of 256 and more 256-row tiles take the direct-to-LDS kernel: ragged rows and columns,
    # two row tiles, a strided layer, a 1x1 layer whose contraction is exactly four ring buffers long plus twelve steps;
    # the last two are grids as large on short contractions (the 128x128 kernel)
    (80, 24, 30, 30, 130, 5, 1, 2),
    (40, 64, 31, 29, 500, 3, 1, 1),
    (120, 64, 47, 45, 200, 3, 2, 1),
    (70, 512, 34, 33, 256, 1, 1, 0),
    (70, 8, 34, 33, 384, 1, 1, 0),
    (80, 8, 30, 30, 130, 5, 1, 2),
]


@pytest.mark.parametrize("case", CONV_CASES + BF16_PACKED_CASES, ids=[str(c) for c in CONV_CASES + BF16_PACKED_CASES])
def test_conv2d_fwd_bf16_operands(dev, case):
    """RH_MATH_BF16_MFMA_FP32ACC: operands rounded to bf16 (nearest even), products accumulated in fp32.
    Reference = the fp64-accumulating oracle on operands rounded the same way."""
    Nn, C, H, W, K, R, st, pad = case
    say("bf16 conv case", case)
    x = synth.normal(12, 1, (Nn, C, H, W))
    w = synth.normal(12, 2, (K, C, R, R))
    b = synth.normal(12, 3, (K,))
    y_ref = O.conv2d_fwd(O.round_bf16(x), O.round_bf16(w), st, pad)
    y = ops.conv2d_fwd(T(x, dev), T(w, dev), st, pad, algo=_lib.RH_MATH_BF16_MFMA_FP32ACC)
    assert_close(N(y), y_ref, "bf16 conv fwd")
    yf = ops.conv2d_fwd(T(x, dev), T(w, dev), st, pad, bias=T(b, dev), relu=True, algo=_lib.RH_MATH_BF16_MFMA_FP32ACC)
    assert_close(N(yf), O.rect_inplace(O.add_bias_nchw(b, y_ref.copy())), "bf16 conv fwd fused bias+relu")
    # operands that are already bf16 values give the fp32 path's result up to summation order
    xr, wr = O.round_bf16(x), O.round_bf16(w)
    y32 = ops.conv2d_fwd(T(xr, dev), T(wr, dev), st, pad)
    y16 = ops.conv2d_fwd(T(xr, dev), T(wr, dev), st, pad, algo=_lib.RH_MATH_BF16_MFMA_FP32ACC)
    assert_close(N(y16), N(y32), "bf16 path on bf16-exact operands == fp32 path")
    torch.cuda.synchronize()


BF16_CHAIN_CASES = [
    # N, C, H, W, K, R, stride, pad, halo of the packed result
    (3, 72, 11, 9, 40, 3, 2, 1, 0),
    (2, 8, 17, 17, 200, 5, 1, 2, 2),
    (5, 16, 9, 12, 24, 3, 1, 0, 1),
    (130, 8, 5, 5, 16, 3, 1, 1, 0),
    (80, 24, 30, 30, 136, 5, 1, 2, 1),     # the direct-to-LDS kernel
    (70, 512, 34, 33, 256, 1, 1, 0, 0),
    (4, 3, 35, 35, 16, 7, 2, 0, 0),        # grouped by filter columns: fp32 image in, packed result out
    # 1x1 layers of up to 128 channels with a packed result: the streaming kernel (pixel counts that are not a
    # multiple of the 32-pixel tile, every tile height, rows shorter than a tile, a bordered result)
    (3, 96, 54, 54, 96, 1, 1, 0, 0),
    (5, 32, 7, 5, 128, 1, 1, 0, 2),
    (2, 128, 13, 11, 32, 1, 1, 0, 1),
    (7, 64, 3, 3, 64, 1, 1, 0, 0),
    (3, 256, 9, 10, 256, 1, 1, 0, 1),     # two chunks of 128 output channels, the deep contraction
    (2, 256, 5, 5, 192, 1, 1, 0, 0),      # two chunks of 96
]


@pytest.mark.parametrize("case", BF16_CHAIN_CASES, ids=[str(c) for c in BF16_CHAIN_CASES])
def test_conv2d_fwd_bf16_packed_chain_forms(dev, case):
    """The forms of the bf16 forward that a forward-only chain uses are bit-identical to rh_conv2d_fwd with
    RH_MATH_BF16_MFMA_FP32ACC: a converted filter kept between calls, a packed bf16 input, and a packed bf16 result,
    which holds the fp32 result rounded to nearest even inside a border that stays zero."""
    Nn, C, H, W, K, R, st, pad, halo = case
    say("bf16 chain case", case)
    x = synth.normal(14, 1, (Nn, C, H, W))
    w = synth.normal(14, 2, (K, C, R, R))
    b = synth.normal(14, 3, (K,))
    xd, wd, bd = T(x, dev), T(w, dev), T(b, dev)
    for relu in (False, True):
        legacy = ops.conv2d_fwd(xd, wd, st, pad, bias=bd, relu=relu, algo=_lib.RH_MATH_BF16_MFMA_FP32ACC)
        y = ops.conv2d_fwd_bf16_packed(xd, wd, st, pad, bias=bd, relu=relu)
        assert torch.equal(y, legacy), "fp32 image in, fp32 result"
        yp = ops.conv2d_fwd_bf16_packed(xd, wd, st, pad, bias=bd, relu=relu, out_halo=halo)
        want = O.round_bf16(N(legacy))
        assert np.array_equal(N(ops.bf16_unpack(yp, legacy.shape, halo)), want), "packed result == rounded fp32 result"
        # the border of the packed result is untouched (zero): re-packing the unpacked interior reproduces every byte
        assert torch.equal(ops.bf16_pack(T(want, dev), halo), yp), "border"
        if C % 8 == 0:
            xp = ops.bf16_pack(xd, pad)
            assert np.array_equal(N(ops.bf16_unpack(xp, x.shape, pad)), O.round_bf16(x)), "pack / unpack"
            y2 = ops.conv2d_fwd_bf16_packed(xd, wd, st, pad, bias=bd, relu=relu, x_packed=xp)
            assert torch.equal(y2, legacy), "packed image in, fp32 result"
            yp2 = ops.conv2d_fwd_bf16_packed(xd, wd, st, pad, bias=bd, relu=relu, x_packed=xp, out_halo=halo)
            assert torch.equal(yp2, yp), "packed image in, packed result"
            # (the streaming 1x1 kernel wherever it can run, also where the tiled kernel is the one chosen)
            yp3 = ops.conv2d_fwd_bf16_packed(xd, wd, st, pad, bias=bd, relu=relu, x_packed=xp, out_halo=halo,
                                             algo=_lib.RH_ALGO_SCALAR_OFFSET)
            assert torch.equal(yp3, yp), "packed image in, packed result, streaming kernel where it runs"
    torch.cuda.synchronize()


@pytest.mark.parametrize("case,form", [
    ((1, 48, 13, 13, 72, 5, 1, 2, 1), "64x64_k4"), ((1, 136, 13, 13, 72, 3, 1, 1, 0), "64x64_k4"),
    ((16, 72, 13, 13, 136, 3, 1, 1, 1), "64x64_k2"), ((37, 72, 13, 13, 384, 3, 1, 1, 1), "128x128_k2"),
    ((40, 40, 13, 13, 264, 3, 1, 1, 0), "128x128"), ((1, 1024, 6, 6, 1000, 1, 1, 0, 0), "64x64_k4"),
    ((16, 384, 13, 13, 384, 1, 1, 0, 0), "64x64_k2"), ((28, 128, 13, 13, 384, 3, 1, 1, 1), "128x128_k2"),
    ((16, 16, 13, 13, 48, 3, 1, 1, 1), "64x128")], ids=str)
def test_conv2d_fwd_bf16_small_grids(dev, case, form):
    """The forms for grids of few tiles: 64 x 64 with four groups of waves over the K steps (38 steps: 9, 10, 9, 10; 40),
    64 x 64 with two, 128 x 128 with two and with one, 64 x 128; ragged rows and columns; fp32 and packed results."""
    _, tags = profile_tags(lambda: (test_conv2d_fwd_bf16_packed_chain_forms(dev, case), test_conv2d_fwd_bf16_operands(dev, case[:8])))
    assert {t for t in tags if t.startswith("conv_fwd_bf16p_")} == {"conv_fwd_bf16p_" + form}, tags


BF16_POOL_CASES = [
    # N, C, H, W, size, stride, pad, rounding, halo of the result
    (3, 16, 13, 13, 3, 2, 0, 0, 1),
    (2, 96, 54, 54, 3, 2, 0, 1, 2),     # ceil extent: clipped windows at the bottom / right edge
    (4, 8, 9, 7, 2, 2, 0, 0, 0),
    (2, 24, 10, 11, 3, 2, 1, 0, 1),     # padded windows: padding never wins
    (1, 8, 5, 5, 3, 1, 1, 1, 0),
]


@pytest.mark.parametrize("case", BF16_POOL_CASES, ids=[str(c) for c in BF16_POOL_CASES])
def test_pool2d_fwd_bf16_packed(dev, case):
    """Max pooling of packed bf16 activations == the fp32 pooling's result rounded to bf16 (rounding is monotone),
    bit for bit, on inputs with ties, negative values and all-negative windows."""
    Nn, C, H, W, k, st, pad, rnd, halo = case
    say("bf16 pool case", case)
    x = synth.normal(15, 1, (Nn, C, H, W))
    x[:, :, ::3, ::2] = np.float32(-0.75)     # ties
    xd = T(x, dev)
    want = O.round_bf16(N(ops.pool2d_fwd(xd, k, st, pad, _lib.RH_POOL_MAX, rnd)))
    want_oracle = O.round_bf16(O.pool2d_fwd(x, k, st, pad, O.POOL_MAX, rnd))
    assert np.array_equal(want, want_oracle)
    yp, shape = ops.pool2d_fwd_bf16_packed(ops.bf16_pack(xd, 0), x.shape, k, st, pad, rnd, out_halo=halo)
    assert np.array_equal(N(ops.bf16_unpack(yp, shape, halo)), want)
    assert torch.equal(ops.bf16_pack(T(want, dev), halo), yp), "border"
    torch.cuda.synchronize()


SGEMM_CASES = [
    # transA, transB, m, n, k
    (1, 0, 500, 64, 2450),   # affine forward  Y = W^T X
    (0, 1, 300, 500, 64),    # affine bwd-W    dW += X dY^T
    (0, 0, 300, 64, 500),    # affine bwd-X    dX = W dY
    (1, 1, 37, 29, 53),
    (0, 0, 1, 10, 64),
    (0, 1, 1, 130, 70),      # the bias-gradient GEMV shape
    (1, 0, 4096, 32, 1024),  # few tiles, deep contraction -> split path
    # a side of at most sixteen: the plain kernels (a wave per element for long contractions, a thread per element
    # otherwise): a ten-class classifier's forward, data-gradient and weight-gradient products, every transposition
    (1, 0, 10, 64, 500),
    (0, 0, 500, 64, 10),
    (0, 1, 500, 10, 64),
    (0, 1, 64, 10, 128),
    (1, 1, 10, 33, 200),
    (1, 0, 16, 256, 129),
    (0, 0, 3, 5, 1),
]


@pytest.mark.parametrize("case", SGEMM_CASES, ids=[str(c) for c in SGEMM_CASES])
@pytest.mark.parametrize("use_ws", [True, False])
def test_sgemm(dev, case, use_ws):
    tA, tB, m, n, k = case
    say("sgemm case", case, "ws", use_ws)
    a_shape = (m, k) if tA else (k, m)   # memory shape (row-major view of a column-major array)
    b_shape = (k, n) if tB else (n, k)
    lda, ldb, ldc = a_shape[1] + 3, b_shape[1] + 1, m + 2
    A = synth.normal(12, 1, (a_shape[0], lda))
    B = synth.normal(12, 2, (b_shape[0], ldb))
    C0 = synth.normal(12, 3, (n, ldc))
    for alpha, beta in ((1.0, 0.0), (0.5, 1.0)):
        ref = O.sgemm(tA, tB, m, n, k, alpha, A, lda, B, ldb, beta, C0.copy(), ldc)
        Cd = T(C0, dev)
        ops.sgemm(tA, tB, m, n, k, alpha, T(A, dev), lda, T(B, dev), ldb, beta, Cd, ldc, use_workspace=use_ws)
        got = N(Cd)
        assert_close(got[:, :m], ref[:, :m], "sgemm alpha=%g beta=%g" % (alpha, beta))
        assert np.array_equal(got[:, m:], C0[:, m:]), "sgemm wrote outside ldc padding"


@pytest.mark.parametrize("case", [
    # (m = out channels, n = batch, k = in channels): one block, several tiles, a split contraction with the dense
    # 16-byte reduction, one with the many-slice reduction, odd extents with a padded result (scalar reduction)
    (10, 4, 50), (10, 64, 500), (500, 64, 800), (4096, 32, 1024), (96, 16, 9216), (1001, 33, 2450), (1000, 256, 4096),
])
def test_sgemm_bias_act(dev, case):
    """rh_sgemm_bias_act = matrix product, bias row, activation of the affine forward pass in one call: bit-identical
    to the library's own three calls, and within tolerance of the oracle's."""
    m, n, k = case
    W = synth.normal(14, 1, (m, k))
    X = synth.normal(14, 2, (n, k))
    b = synth.normal(14, 3, (m,))
    for ldc, use_ws, relu, beta in ((m, True, True, 0.0), (m + (4 if m % 4 == 0 else 3), True, True, 0.0),
                                    (m, False, False, 0.0), (m, True, True, 0.5)):
        say("sgemm_bias_act", case, "ldc", ldc, "ws", use_ws, "relu", relu, "beta", beta)
        C0 = synth.normal(14, 4, (n, ldc))
        ref = O.sgemm(1, 0, m, n, k, 1.0, W, k, X, k, beta, C0.copy(), ldc)
        ref[:, :m] += b[None, :]
        if relu:
            ref[:, :m] = np.maximum(ref[:, :m], 0)
        Cd = T(C0, dev)
        ops.sgemm(1, 0, m, n, k, 1.0, T(W, dev), k, T(X, dev), k, beta, Cd, ldc, use_workspace=use_ws, bias=T(b, dev), relu=relu)
        got = N(Cd)
        assert_close(got[:, :m], ref[:, :m], "sgemm_bias_act")
        assert np.array_equal(got[:, m:], C0[:, m:]), "wrote into the ldc padding"
        if ldc == m:
            Cs = T(C0, dev)
            ops.sgemm(1, 0, m, n, k, 1.0, T(W, dev), k, T(X, dev), k, beta, Cs, ldc, use_workspace=use_ws)
            ops.add_bias_nchw(T(b, dev), Cs.view(n, m, 1, 1))
            if relu:
                ops.rect_inplace(Cs)
            assert np.array_equal(N(Cs), got), "fused and separate calls differ"


# The products of affine layers with RH_ALGO_BF16X3.  Rows (n) around the 32-, 64- and 128-row blocks and two of them; columns
# (m) that do not fill a block of 128, a wave's 32 or a group of 8; contractions of one K step, of fewer than a block's ring of
# steps (4, 5 and 7), of an odd number, in slices whose last one is shorter, and with a last step that is not full (where k is no
# contiguous extent of A).  Padded lda, ldb, ldc.
SGEMM_X3_CASES = [
    # tA, tB, m, n, k
    (1, 0, 4, 1, 16), (1, 0, 132, 31, 48), (1, 0, 260, 33, 80), (1, 0, 96, 64, 112), (1, 0, 100, 65, 64), (1, 0, 516, 129, 496),
    (1, 0, 1000, 37, 4096), (1, 0, 2052, 256, 2064),
    (0, 0, 4, 1, 3), (0, 0, 132, 32, 50), (0, 0, 260, 40, 77), (0, 0, 36, 63, 129), (0, 0, 100, 100, 16), (0, 0, 516, 130, 1000),
    (0, 0, 4096, 50, 1000),
    (0, 1, 4, 1, 1), (0, 1, 132, 129, 9), (0, 1, 500, 1000, 50), (0, 1, 1028, 260, 256),
]


@pytest.mark.parametrize("case", SGEMM_X3_CASES, ids=str)
def test_sgemm_bf16x3(dev, case):
    """The split-operand form against the oracle, its error against 64-bit sums, and what is not finite.  Bound of the error: as
    in test_conv2d_bf16x3_error, a chain of n steps of 16 terms has sqrt(0.18 n + 4) 2^-24, a quarter on top."""
    tA, tB, m, n, k = case
    say("sgemm bf16x3", case)
    X3 = _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_DIRECT
    a_shape, b_shape = ((m, k) if tA else (k, m)), ((k, n) if tB else (n, k))
    lda, ldb, ldc = (a_shape[1] + 7) // 4 * 4, b_shape[1] + 1, m + 2
    A, B, C0 = synth.normal(16, 1, (a_shape[0], lda)), synth.normal(16, 2, (b_shape[0], ldb)), synth.normal(16, 3, (n, ldc))
    bias = synth.normal(16, 4, (m,))
    Ad, Bd = T(A, dev), T(B, dev)
    opA = (A[:, :k].T if tA else A[:, :m]).astype(np.float64)     # [k][m]
    opB = (B[:, :n].T if tB else B[:, :k]).astype(np.float64)     # [n][k]
    exact = opB @ opA
    for alpha, beta, relu in ((1.0, 0.0, False), (0.5, 1.0, False), (1.0, 0.0, True)):
        Cd = T(C0, dev)
        ops.sgemm(tA, tB, m, n, k, alpha, Ad, lda, Bd, ldb, beta, Cd, ldc, bias=T(bias, dev) if relu else None, relu=relu, algo=X3)
        got, ref = N(Cd), alpha * exact + beta * C0[:, :m]
        if relu:
            ref = np.maximum(ref + bias, 0.0)
        assert_close(got[:, :m], ref.astype(np.float32), "sgemm bf16x3 alpha=%g beta=%g" % (alpha, beta))
        assert np.array_equal(got[:, m:], C0[:, m:]), "wrote outside ldc padding"
        if alpha == 1.0 and not relu:
            err = np.linalg.norm(got[:, :m] - exact) / np.linalg.norm(exact)
            assert err <= 1.25 * 2.0 ** -24 * (0.18 * k / 16 + 4) ** 0.5, err
    # an infinity, a NaN and values that round to an infinity in bf16, in either operand
    A[0, 0], B[n // 2 if not tB else 0, 0] = np.inf, -3.4e38
    A[-1, (k if tA else m) - 1] = -np.inf
    B[-1, (n if tB else k) - 1] = np.nan if n > 2 and not tB else 2.0
    A[:, :] *= np.float32(0.125)
    out = []
    for algo in (X3, _lib.RH_ALGO_GATHER):
        Cd = T(C0, dev)
        ops.sgemm(tA, tB, m, n, k, 1.0, T(A, dev), lda, T(B, dev), ldb, 0.0, Cd, ldc, algo=algo)
        out.append(N(Cd)[:, :m])
    assert np.array_equal(np.isnan(out[0]), np.isnan(out[1])) and np.array_equal(np.isinf(out[0]), np.isinf(out[1]))
    keep = np.isfinite(out[1])
    assert np.array_equal(out[0][np.isinf(out[1])], out[1][np.isinf(out[1])])
    assert np.all(np.abs(out[0][keep].astype(np.float64) - out[1][keep]) <= 1e-4 * (1.0 + np.abs(out[1][keep].astype(np.float64))))


@pytest.mark.parametrize("exponent", [-112, -126, -140])
@pytest.mark.parametrize("case", [(1, 0, 132, 31, 48), (1, 0, 516, 129, 496), (0, 0, 260, 40, 77), (0, 0, 516, 130, 1000), (0, 1, 500, 1000, 50)], ids=str)
def test_sgemm_bf16x3_small_operands(dev, case, exponent):
    """As test_conv2d_bf16x3_small_operands: either operand all below bf16's parts, or one value in a hundred."""
    tA, tB, m, n, k = case
    X3 = _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_DIRECT
    base = synth.normal(18, 1, (m, k) if tA else (k, m)), synth.normal(18, 2, (k, n) if tB else (n, k))
    for tiny in (0, 1):
        for share in (1.0, 0.01):
            say("sgemm bf16x3 small operands", case, exponent, tiny, share)
            t = [a * np.float32(2.0 ** 100) for a in base]
            small = (base[tiny].astype(np.float64) * 2.0 ** exponent).astype(np.float32)
            t[tiny] = small if share == 1.0 else np.where(synth.uniform(18, 9, small.shape) < share, small, base[tiny])
            A, B = t
            C = torch.empty(n, m, device=dev)
            ops.sgemm(tA, tB, m, n, k, 1.0, T(A, dev), A.shape[1], T(B, dev), B.shape[1], 0.0, C, m, algo=X3)
            exact = (B.T if tB else B).astype(np.float64) @ (A.T if tA else A).astype(np.float64)
            err = np.linalg.norm(N(C).astype(np.float64) - exact) / np.linalg.norm(exact)
            assert err <= _redo_bound(k), err


def test_sgemm_bf16x3_where_it_pays(dev):
    """RH_ALGO_BF16X3 alone: the form on large affine products, with no larger error against 64-bit sums than the form that it
    replaces, half of the activations zeros; the other forms' bits elsewhere and where the scratch does not hold it."""
    for tA, tB, m, n, k, takes in ((1, 0, 4096, 32, 4096, True), (1, 0, 2048, 16, 8192, False), (0, 0, 4096, 24, 4096, True), (0, 0, 6144, 8, 4096, False),
                                   (0, 0, 9216, 32, 4096, True), (0, 0, 9216, 33, 4096, True), (1, 0, 4096, 31, 4080, False), (1, 0, 1000, 33, 4096, True), (1, 0, 512, 64, 1024, False),
                                   (1, 0, 1000, 129, 4096, True), (1, 0, 1024, 200, 2048, False), (0, 0, 4096, 37, 1000, True), (0, 0, 4096, 256, 4096, True),
                                   (0, 1, 4096, 4096, 50, True), (0, 1, 4096, 1000, 96, False), (0, 1, 4096, 1000, 97, True), (0, 1, 4096, 4096, 256, True),
                                   (0, 1, 800, 500, 128, False)):
        say("sgemm bf16x3 pays", (tA, tB, m, n, k))
        A, B = synth.normal(17, 1, (m, k) if tA else (k, m)), synth.normal(17, 2, (k, n) if tB else (n, k))
        B = np.maximum(B, 0.0)
        Ad, Bd, C = T(A, dev), T(B, dev), torch.empty(n, m, device=dev)
        run = lambda algo, ws=True: N(ops.sgemm(tA, tB, m, n, k, 1.0, Ad, A.shape[1], Bd, B.shape[1], 0.0, C, m, use_workspace=ws, algo=algo)).copy()
        got, tags = profile_tags(lambda: run(_lib.RH_ALGO_BF16X3))
        assert any(t.startswith("sgemm_tri_") for t in tags) == takes, ((tA, tB, m, n, k), tags)
        before = run(0)
        exact = (B.T if tB else B).astype(np.float64) @ (A.T if tA else A).astype(np.float64)
        assert np.linalg.norm(got - exact) <= np.linalg.norm(before - exact), (tA, tB, m, n, k)
        if not takes:
            assert np.array_equal(got, before)
        assert np.array_equal(run(_lib.RH_ALGO_BF16X3, False), run(0, False))


def test_sgemm_bf16x3_refused(dev):
    """No such form: both operands transposed, m no multiple of 4, k no multiple of 16 with A transposed, A or lda not aligned."""
    X3 = _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_DIRECT
    buf = torch.zeros(1 << 16, device=dev)
    ws = torch.empty(1 << 20, dtype=torch.uint8, device=dev)
    for tA, tB, m, n, k, lda, shift in ((1, 1, 64, 64, 64, 64, 0), (0, 0, 66, 8, 16, 68, 0), (1, 0, 64, 8, 24, 24, 0), (1, 0, 64, 8, 32, 33, 0), (0, 0, 64, 8, 16, 64, 1)):
        C = torch.full((n, m), 7.0, device=dev)
        rc = _lib.lib().rh_sgemm(tA, tB, m, n, k, 1.0, buf.data_ptr() + 4 * shift, lda, buf.data_ptr(), max(n, k), 0.0, C.data_ptr(), m,
                                 ws.data_ptr(), ws.numel(), X3, None)
        assert rc == _lib.RH_E_UNSUPPORTED, (tA, tB, m, n, k, rc)
        torch.cuda.synchronize()
        assert bool((C == 7.0).all())


def test_bias_relu(dev):
    for shape in [(3, 7, 5, 9), (2, 96, 27, 27), (64, 500), (5, 3, 16, 20)]:
        say("bias/relu", shape)
        y = synth.normal(13, 1, shape)
        b = synth.normal(13, 2, (shape[1],))
        yd = T(y, dev)
        ops.add_bias_nchw(T(b, dev), yd)
        ref = O.add_bias_nchw(b, y.copy())
        assert_close(N(yd), ref, "add_bias")
        ops.rect_inplace(yd)
        ref = O.rect_inplace(ref)
        assert np.array_equal(N(yd) > 0, ref > 0)
        assert_close(N(yd), ref, "rect")
        dy = synth.normal(13, 3, shape)
        dyd = T(dy, dev)
        ops.rect_backprop_inplace(yd, dyd)
        assert np.array_equal(N(dyd), O.rect_backprop_inplace(ref, dy.copy())), "rect backprop is a pure mask"


POOL_CASES = [
    # N, C, H, size, stride, pad
    (2, 3, 9, 3, 2, 0), (2, 3, 9, 3, 2, 1), (3, 4, 8, 2, 2, 0), (2, 2, 10, 3, 2, 0), (2, 5, 27, 3, 2, 0),
    (1, 2, 6, 6, 1, 0), (2, 3, 7, 3, 1, 1), (2, 2, 13, 3, 3, 1),
    (1, 3, 112, 3, 2, 1),   # planes above a block's LDS share: forward in bands of output rows, backward with
    (1, 2, 130, 3, 2, 0),   # several windows per thread and colour / (130: above 60 KB) by the gather kernel
    (1, 1, 20, 7, 3, 2),    # three colours per axis: gather backward
]


@pytest.mark.parametrize("case", POOL_CASES, ids=[str(c) for c in POOL_CASES])
@pytest.mark.parametrize("mode", [_lib.RH_POOL_MAX, _lib.RH_POOL_AVG_INCL_PAD])
@pytest.mark.parametrize("rounding", [_lib.RH_ROUND_FLOOR, _lib.RH_ROUND_CEIL])
def test_pool2d(dev, case, mode, rounding):
    Nn, C, H, k, st, pad = case
    say("pool case", case, mode, rounding)
    x = synth.normal(14, 1, (Nn, C, H, H + 1))
    # repeated values so that the first-maximum tie rule is exercised
    x = np.round(x * 2) / 2
    y_ref, am_ref = O.pool2d_fwd(x, k, st, pad, mode, rounding, want_argmax=True)
    if y_ref.size == 0:
        pytest.skip("empty output")
    xd = T(x, dev)
    y, am = ops.pool2d_fwd(xd, k, st, pad, mode, rounding, want_argmax=True)
    assert_close(N(y), y_ref, "pool fwd")
    if mode == _lib.RH_POOL_MAX:
        assert np.array_equal(N(am), am_ref), "arg-max mask is bit-exact"
    dy = synth.normal(14, 2, y_ref.shape)
    dx_ref = O.pool2d_bwd(x, y_ref, dy, k, st, pad, mode, rounding)
    dx = ops.pool2d_bwd(xd, y, T(dy, dev), k, st, pad, mode, rounding)
    assert_close(N(dx), dx_ref, "pool bwd (recomputed arg-max)")
    if mode == _lib.RH_POOL_MAX:
        dx2 = ops.pool2d_bwd(xd, y, T(dy, dev), k, st, pad, mode, rounding, argmax=am)
        # same elements, same values up to the order in which an element's (at most four) contributions are added
        assert np.array_equal(N(dx2) == 0, N(dx) == 0), "mask-driven backward routes to the same elements"
        assert_close(N(dx2), dx_ref, "pool bwd (arg-max mask)")
        assert np.allclose(N(dx2), N(dx), rtol=1e-6, atol=2e-6), "mask-driven backward equals recomputed"
        again = ops.pool2d_bwd(xd, y, T(dy, dev), k, st, pad, mode, rounding, argmax=am)
        assert np.array_equal(N(dx2), N(again)), "the mask-driven backward is deterministic"


@pytest.mark.parametrize("case", POOL_CASES + [(2, 3, 55, 3, 2, 0), (3, 2, 31, 5, 4, 2)], ids=str)
@pytest.mark.parametrize("rounding", [_lib.RH_ROUND_FLOOR, _lib.RH_ROUND_CEIL])
def test_pool2d_one_byte_mask(dev, case, rounding):
    """The one-byte mask (the winner's slot r*size + s inside its window, 255 for none) names the same elements as the
    int32 plane index, bit for bit; the pooled values are identical; the backward pass from it, without and with the ReLU
    mask of the operator below folded in, is bit-identical to the one from the int32 mask."""
    Nn, C, H, k, st, pad = case
    shape = (Nn, C, H, H + 1)
    say("pool one-byte mask case", case, rounding)
    if not ops.pool2d_slot_supported(shape, k, st, pad, rounding):
        g = ops.pool_geom(shape, k, st, pad, _lib.RH_POOL_MAX, rounding)
        dummy = torch.zeros(16, device=dev)
        assert _lib.lib().rh_pool2d_fwd_slot(C_.byref(g), dummy.data_ptr(), dummy.data_ptr(), dummy.data_ptr(), None) == _lib.RH_E_UNSUPPORTED
        pytest.skip("no one-byte form for this geometry (three colours per axis or planes beyond the LDS kernels)")
    x = np.round(synth.normal(17, 1, shape) * 2) / 2 - np.float32(0.5)     # ties, and windows that are all negative
    xd = T(x, dev)
    y, am = ops.pool2d_fwd(xd, k, st, pad, _lib.RH_POOL_MAX, rounding, want_argmax=True)
    y2, slot = ops.pool2d_fwd_slot(xd, k, st, pad, rounding)
    assert torch.equal(y, y2)
    am_h, slot_h = N(am), N(slot).astype(np.int64)
    P, Q = am_h.shape[2], am_h.shape[3]
    hs = (np.arange(P) * st - pad)[:, None]
    ws = (np.arange(Q) * st - pad)[None, :]
    plane = (hs + slot_h // k) * shape[3] + ws + slot_h % k
    assert np.array_equal(np.where(slot_h == 255, -1, plane), am_h), "slot names the element the plane index names"
    assert (slot_h[slot_h != 255] < k * k).all()
    dy = T(synth.normal(17, 2, tuple(y.shape)), dev)
    assert torch.equal(ops.pool2d_bwd_slot(shape, dy, slot, k, st, pad, rounding),
                       ops.pool2d_bwd(xd, y, dy, k, st, pad, _lib.RH_POOL_MAX, rounding, argmax=am))
    assert torch.equal(ops.pool2d_bwd_slot(shape, dy, slot, k, st, pad, rounding, relu_y=y),
                       ops.pool2d_bwd_relu(shape, y, dy, k, st, pad, am, rounding))
    torch.cuda.synchronize()


@pytest.mark.parametrize("shape", [(64, 10), (256, 1000), (7, 1), (3, 5000)])
def test_softmax_loss_argmax(dev, shape):
    Nn, C = shape
    say("softmax case", shape)
    x = synth.normal(15, 1, shape, 0.0, 3.0)
    labels = synth.integers(15, 2, (Nn,), C)
    weights = synth.uniform(15, 3, (Nn,), 0.1, 1.0)
    xd, ld, wd = T(x, dev), T(labels, dev), T(weights, dev)
    p_ref = O.softmax_fwd(x)
    p = ops.softmax_fwd(xd)
    assert_close(N(p), p_ref, "softmax", atol=1e-7)
    d = ops.softmax_kl_backward(p, ld, wd)
    assert_close(N(d), O.softmax_kl_backward(N(p), labels, weights), "kl backward", atol=1e-7)
    l1 = ops.softmax_kl_loss1(p, ld, wd)
    l1_ref = O.softmax_kl_loss1(N(p), labels, weights)
    assert_close(N(l1), l1_ref, "kl loss1")
    l1b = ops.softmax_kl_loss1(p, ld, wd, beta=1.0, loss1=l1.clone())
    assert_close(N(l1b), 2 * l1_ref, "kl loss1 accumulate")
    tot = ops.blockreduce_sum(l1.reshape(1, Nn))
    assert_close(N(tot), O.blockreduce_sum(N(l1).reshape(1, Nn)), "loss sum")
    mx, idx = ops.blockreduce_argmax(p)
    mx_ref, idx_ref = O.blockreduce_argmax(N(p))
    assert np.array_equal(N(idx), idx_ref), "arg-max is bit-exact"
    assert np.array_equal(N(mx), mx_ref)


@pytest.mark.parametrize("shape", [(1, 1), (3, 10), (64, 10), (128, 1000), (256, 1000), (700, 37), (5, 3000)])
def test_softmax_kl_step_equals_separate_calls(dev, shape):
    """The one-launch form of the loss operator's train step is bit-identical to the five separate kernels, three
    calls in a row on one counter word (the kernel leaves it at zero)."""
    Nn, C = shape
    counter = None
    for rep in range(3):
        say("softmax_kl_step", shape, "call", rep)
        x = synth.normal(17, rep + 1, shape, 0.0, 3.0)
        if rep == 2 and C > 2:
            x[:, 1] = x[:, 0] = x.max(axis=1) + 1.0      # ties for the maximum: the lowest index wins
        labels = synth.integers(17, 10 + rep, (Nn,), C)
        weights = synth.uniform(17, 20 + rep, (Nn,), 0.1, 1.0)
        xd, ld, wd = T(x, dev), T(labels, dev), T(weights, dev)
        p, mx, idx, l1, tot, dx, counter = ops.softmax_kl_step(xd, ld, wd, counter)
        p_s = ops.softmax_fwd(xd)
        mx_s, idx_s = ops.blockreduce_argmax(p_s)
        l1_s = ops.softmax_kl_loss1(p_s, ld, wd)
        tot_s = ops.blockreduce_sum(l1_s.reshape(1, Nn))
        dx_s = ops.softmax_kl_backward(p_s, ld, wd)
        for name, a, b in (("p", p, p_s), ("max", mx, mx_s), ("argmax", idx, idx_s), ("loss1", l1, l1_s), ("loss", tot, tot_s),
                           ("dx", dx, dx_s)):
            assert np.array_equal(N(a), N(b)), name
        assert int(N(counter)[0]) == 0
        assert_close(N(p), O.softmax_fwd(x), "softmax", atol=1e-7)
        assert np.array_equal(N(idx), O.blockreduce_argmax(N(p))[1])


AFFINE2_CASES = [
    # B, I, H, C, relu
    (64, 800, 160, 10, True),     # a LeNet-like classifier of 2^17 weights
    (128, 1024, 64, 10, True),    # the CIFAR-10 network's
    (1, 7, 5, 3, False),
    (5, 33, 130, 64, True),       # ragged wave groups, the widest class count
    (37, 1022, 1, 2, False),      # odd input count: the element-wise weight-gradient form
    (256, 4096, 32, 17, True),    # the widest input the form takes
]


@pytest.mark.parametrize("case", AFFINE2_CASES)
def test_affine2_softmax_kl_step(dev, case):
    """The classifier tail in two launches against the oracle's separate operators: two affine layers, softmax,
    arg-max, loss, KL delta, the data gradients of both layers, then all four parameter gradients (beta 0 and 1);
    two calls in a row on one counter word."""
    B, I, H, Cc, relu = case
    assert ops.affine2_softmax_kl_step_supported(B, I, H, Cc)
    counter = None
    for rep in range(2):
        say("affine2_softmax_kl_step", case, "call", rep)
        x = synth.normal(41, 10 * rep + 1, (B, I))
        w1 = synth.normal(41, 10 * rep + 2, (H, I), 0.0, 1.0 / np.sqrt(I))
        b1 = synth.normal(41, 10 * rep + 3, (H,), 0.0, 0.5)
        w2 = synth.normal(41, 10 * rep + 4, (Cc, H), 0.0, 1.0 / np.sqrt(H))
        b2 = synth.normal(41, 10 * rep + 5, (Cc,), 0.0, 0.5)
        labels = synth.integers(41, 10 * rep + 6, (B,), Cc)
        weights = synth.uniform(41, 10 * rep + 7, (B,), 0.1, 1.0)
        # the oracle's operators, one after the other (column-major products as AffineOperator issues them)
        h = O.sgemm(1, 0, H, B, I, 1.0, w1, I, x, I, 0.0, np.zeros((B, H), np.float32), H) + b1
        if relu:
            h = np.maximum(h, 0.0).astype(np.float32)
        logits = O.sgemm(1, 0, Cc, B, H, 1.0, w2, H, h, H, 0.0, np.zeros((B, Cc), np.float32), Cc) + b2
        p = O.softmax_fwd(logits)
        dl = O.softmax_kl_backward(p, labels, weights)
        l1 = O.softmax_kl_loss1(p, labels, weights)
        dh = O.sgemm(0, 0, H, B, Cc, 1.0, w2, H, dl, Cc, 0.0, np.zeros((B, H), np.float32), H)
        if relu:
            dh = dh * (h > 0)
        dx = O.sgemm(0, 0, I, B, H, 1.0, w1, I, dh, H, 0.0, np.zeros((B, I), np.float32), I)
        out = ops.affine2_softmax_kl_step(T(x, dev), T(w1, dev), T(b1, dev), T(w2, dev), T(b2, dev), T(labels, dev), T(weights, dev),
                                          relu1=relu, want_dx=(rep == 0), counter=counter)
        counter = out["counter"]
        assert int(N(counter)[0]) == 0
        assert_close(N(out["h"]), h, "affine2 h")
        assert_close(N(out["logits"]), logits, "affine2 logits")
        assert_close(N(out["p"]), p, "affine2 softmax", atol=1e-6)
        assert np.array_equal(N(out["idx"]), O.blockreduce_argmax(N(out["p"]))[1]), "affine2 arg-max of its own probabilities"
        assert np.array_equal(N(out["max"]), N(out["p"]).max(axis=1))
        assert_close(N(out["loss1"]), l1, "affine2 loss1")
        assert_close(N(out["loss"]), np.array([l1.astype(np.float64).sum()], np.float32), "affine2 loss sum")
        assert_close(N(out["dlogits"]), dl, "affine2 dlogits")
        # the hidden delta is masked by the GPU's own h (an h within rounding of 0 may differ in sign from the oracle's)
        dh_gpu_mask = O.sgemm(0, 0, H, B, Cc, 1.0, w2, H, N(out["dlogits"]), Cc, 0.0, np.zeros((B, H), np.float32), H)
        if relu:
            dh_gpu_mask = dh_gpu_mask * (N(out["h"]) > 0)
        assert_close(N(out["dh"]), dh_gpu_mask, "affine2 dh")
        if rep == 0:
            dx_ref = O.sgemm(0, 0, I, B, H, 1.0, w1, I, N(out["dh"]), H, 0.0, np.zeros((B, I), np.float32), I)
            assert_close(N(out["dx"]), dx_ref, "affine2 dx")
            if not relu:
                assert_close(N(out["dx"]), dx, "affine2 dx (oracle chain)")
        # parameter gradients from the GPU's own activations and deltas
        hh, dhh, dll = N(out["h"]), N(out["dh"]), N(out["dlogits"])
        for beta1, beta2 in ((0.0, 0.0), (1.0, 1.0), (0.5, 0.0)):
            dw1_0, db1_0 = synth.normal(41, 10 * rep + 8, (H, I)), synth.normal(41, 10 * rep + 9, (H,))
            dw2_0, db2_0 = synth.normal(41, 10 * rep + 10, (Cc, H)), synth.normal(41, 10 * rep + 11, (Cc,))
            dw1, db1, dw2, db2 = T(dw1_0, dev), T(db1_0, dev), T(dw2_0, dev), T(db2_0, dev)
            ops.affine2_bwd_params(T(x, dev), out["h"], out["dh"], out["dlogits"], dw1, db1, dw2, db2, beta1, beta2)
            r1 = O.sgemm(0, 1, I, H, B, 1.0, x, I, dhh, H, beta1, dw1_0.copy(), I)
            r2 = O.sgemm(0, 1, H, Cc, B, 1.0, hh, H, dll, Cc, beta2, dw2_0.copy(), H)
            assert_close(N(dw1), r1, "affine2 dW1 beta %g" % beta1)
            assert_close(N(dw2), r2, "affine2 dW2 beta %g" % beta2)
            assert_close(N(db1), (dhh.astype(np.float64).sum(axis=0) + beta1 * db1_0).astype(np.float32), "affine2 db1 beta %g" % beta1)
            assert_close(N(db2), (dll.astype(np.float64).sum(axis=0) + beta2 * db2_0).astype(np.float32), "affine2 db2 beta %g" % beta2)


@pytest.mark.parametrize("case", [(64, 500, 10, True), (3, 2048, 64, False), (130, 1, 2, True), (256, 384, 17, True)])
def test_affine_softmax_kl_step_from_h(dev, case):
    """The form that starts from the first layer's output (I = 0, x = NULL): second layer, loss step and the hidden
    delta in one launch, dW2 and db2 in another; h and the first layer's gradients are left untouched."""
    B, H, Cc, relu = case
    assert ops.affine2_softmax_kl_step_supported(B, 0, H, Cc)
    counter = None
    for rep in range(2):
        say("affine_softmax_kl_step_from_h", case, "call", rep)
        h = synth.normal(43, 10 * rep + 1, (B, H))
        if relu:
            h = np.maximum(h, 0.0).astype(np.float32)
        w2 = synth.normal(43, 10 * rep + 4, (Cc, H), 0.0, 1.0 / np.sqrt(H))
        b2 = synth.normal(43, 10 * rep + 5, (Cc,), 0.0, 0.5)
        labels = synth.integers(43, 10 * rep + 6, (B,), Cc)
        weights = synth.uniform(43, 10 * rep + 7, (B,), 0.1, 1.0)
        logits = O.sgemm(1, 0, Cc, B, H, 1.0, w2, H, h, H, 0.0, np.zeros((B, Cc), np.float32), Cc) + b2
        p = O.softmax_fwd(logits)
        dl = O.softmax_kl_backward(p, labels, weights)
        l1 = O.softmax_kl_loss1(p, labels, weights)
        h_dev = T(h, dev)
        out = ops.affine_softmax_kl_step_from_h(h_dev, T(w2, dev), T(b2, dev), T(labels, dev), T(weights, dev), relu1=relu,
                                                counter=counter)
        counter = out["counter"]
        assert int(N(counter)[0]) == 0
        assert np.array_equal(N(h_dev), h), "h is an input here"
        assert_close(N(out["logits"]), logits, "from_h logits")
        assert_close(N(out["p"]), p, "from_h softmax", atol=1e-6)
        assert np.array_equal(N(out["idx"]), O.blockreduce_argmax(N(out["p"]))[1])
        assert np.array_equal(N(out["max"]), N(out["p"]).max(axis=1))
        assert_close(N(out["loss1"]), l1, "from_h loss1")
        assert_close(N(out["loss"]), np.array([l1.astype(np.float64).sum()], np.float32), "from_h loss sum")
        assert_close(N(out["dlogits"]), dl, "from_h dlogits")
        dh = O.sgemm(0, 0, H, B, Cc, 1.0, w2, H, N(out["dlogits"]), Cc, 0.0, np.zeros((B, H), np.float32), H)
        if relu:
            dh = dh * (h > 0)
        assert_close(N(out["dh"]), dh, "from_h dh")
        dll = N(out["dlogits"])
        for beta2 in (0.0, 1.0):
            dw2_0, db2_0 = synth.normal(43, 10 * rep + 10, (Cc, H)), synth.normal(43, 10 * rep + 11, (Cc,))
            dw2, db2 = T(dw2_0, dev), T(db2_0, dev)
            ops.affine_bwd_params_from_h(h_dev, out["dlogits"], dw2, db2, beta2)
            r2 = O.sgemm(0, 1, H, Cc, B, 1.0, h, H, dll, Cc, beta2, dw2_0.copy(), H)
            assert_close(N(dw2), r2, "from_h dW2 beta %g" % beta2)
            assert_close(N(db2), (dll.astype(np.float64).sum(axis=0) + beta2 * db2_0).astype(np.float32), "from_h db2 beta %g" % beta2)
            # with dh and db1: the first layer's bias gradient too, the second layer's unchanged bit for bit
            db1_0 = synth.normal(43, 10 * rep + 12, (H,))
            dw2b, db2b, db1 = T(dw2_0, dev), T(db2_0, dev), T(db1_0, dev)
            ops.affine_bwd_params_from_h(h_dev, out["dlogits"], dw2b, db2b, beta2, dh=out["dh"], db1=db1, beta1=beta2)
            assert torch.equal(dw2b, dw2) and torch.equal(db2b, db2)
            assert_close(N(db1), (N(out["dh"]).astype(np.float64).sum(axis=0) + beta2 * db1_0).astype(np.float32),
                         "from_h db1 beta %g" % beta2)
        # db1 without dh is refused
        assert _lib.lib().rh_affine2_bwd_params(B, 0, H, Cc, None, h_dev.data_ptr(), None, out["dlogits"].data_ptr(), 0.0, None,
                                                db1.data_ptr(), 0.0, dw2.data_ptr(), db2.data_ptr(), None) == _lib.RH_E_INVALID


def test_affine2_softmax_kl_step_limits(dev):
    x8 = torch.zeros((2, 8), device=dev)
    # I = 0 goes with x = NULL and the other way round
    assert _lib.lib().rh_affine2_softmax_kl_step(2, 0, 4, 2, 1, *([x8.data_ptr()] * 19), None) == _lib.RH_E_INVALID
    assert _lib.lib().rh_affine2_softmax_kl_step(2, 8, 4, 2, 1, None, *([x8.data_ptr()] * 18), None) == _lib.RH_E_INVALID
    assert ops.affine2_softmax_kl_step_supported(64, 0, 500, 10)
    assert not ops.affine2_softmax_kl_step_supported(64, 0, 2049, 10)
    assert not ops.affine2_softmax_kl_step_supported(64, 4097, 10, 10)
    assert not ops.affine2_softmax_kl_step_supported(64, 2450, 500, 10)     # more than 2^17 weights in the first layer
    assert not ops.affine2_softmax_kl_step_supported(1024, 4096, 32, 10)    # more than 2^26 multiply-adds over the batch
    assert not ops.affine2_softmax_kl_step_supported(64, 100, 100, 65)
    x = torch.zeros((2, 8), device=dev)
    z = lambda *s: torch.zeros(s, device=dev)
    rc = _lib.lib().rh_affine2_softmax_kl_step(2, 8, 4, 65, 1, *([x.data_ptr()] * 19), None)
    assert rc == _lib.RH_E_UNSUPPORTED


def test_argmax_ties(dev):
    x = np.zeros((4, 700), np.float32)
    x[0, [5, 300, 699]] = 2.0
    x[1, :] = 1.0
    x[2, 699] = 3.0
    x[3, [64, 65]] = 7.0
    mx, idx = ops.blockreduce_argmax(T(x, dev))
    assert N(idx).tolist() == [5, 0, 699, 64]
    assert N(mx).tolist() == [2.0, 1.0, 3.0, 7.0]


@pytest.mark.parametrize("n", [1, 5, 1000, 1 << 20 | 3])
def test_blas1_sgd(dev, n):
    say("blas1/sgd n", n)
    x = synth.normal(16, 1, (n,))
    y = synth.normal(16, 2, (n,))
    yd = T(y, dev)
    ops.saxpy(0.25, T(x, dev), yd)
    assert_close(N(yd), O.saxpy(0.25, x, y.copy()), "saxpy")
    ops.sscal(-1.5, yd)
    assert_close(N(yd), O.sscal(-1.5, O.saxpy(0.25, x, y.copy())), "sscal")
    # unaligned views
    if n > 8:
        yd2 = T(y, dev)
        ops.saxpy(2.0, T(x, dev)[1:], yd2[1:])
        assert_close(N(yd2)[1:], O.saxpy(2.0, x[1:].copy(), y[1:].copy()), "saxpy unaligned")
        assert N(yd2)[0] == y[0]
    W, g, v = synth.normal(16, 3, (n,)), synth.normal(16, 4, (n,)), synth.normal(16, 5, (n,))
    for (l2, scale, mu, apply, zg) in [(5e-4, -0.01, 0.9, 1.0, True), (0.0, 1.0, 0.9, -0.01, False)]:
        Wd, gd, vd = T(W, dev), T(g, dev), T(v, dev)
        ops.sgd_momentum_step(Wd, gd, vd, l2, scale, mu, apply, zg)
        Wr, gr, vr = W.copy(), g.copy(), v.copy()
        O.sgd_momentum_step(Wr, gr, vr, l2, scale, mu, apply, zg)
        assert_close(N(Wd), Wr, "sgd W", atol=1e-7)
        assert_close(N(vd), vr, "sgd v", atol=1e-7)
        assert_close(N(gd), gr, "sgd g", atol=1e-7)
    Wd, gd = T(W, dev), T(g, dev)
    ops.descend(Wd, gd, 0.05, 1e-3)
    Wr, gr = W.copy(), g.copy()
    O.descend(Wr, gr, 0.05, 1e-3)
    assert_close(N(Wd), Wr, "descend W", atol=1e-7)
    assert_close(N(gd), gr, "descend g", atol=1e-7)


def test_sgd_multi_tensor_step(dev):
    """One launch over many parameter blocks == one rh_sgd_momentum_step per block, bit for bit, and the oracle:
    lengths around the 1024-element block and the 4-element vector boundaries, an empty block, unaligned views,
    per-block l2 (zero for some), more blocks than one launch's table holds (48), both zero_grad settings."""
    lens = [1, 3, 4, 5, 96, 1023, 1024, 1025, 4096, 0, 2049, 34848, 1 << 18 | 1] + [7 * i + 1 for i in range(60)]
    say("multi-tensor sgd over", len(lens), "blocks")
    for zg in (True, False):
        host, multi, single = [], [], []
        for k, n in enumerate(lens):
            off = k % 3 if n > 16 else 0        # some blocks start 4 or 8 bytes off a 16-byte boundary
            W, g, v = (synth.normal(17, 10 * k + j, (n + off,)) for j in range(3))
            l2 = 0.0 if k % 4 == 0 else 1e-3 * (1 + k % 5)
            host.append((W[off:].copy(), g[off:].copy(), v[off:].copy(), l2))
            multi.append(tuple(T(a, dev)[off:] for a in (W, g, v)) + (l2,))
            single.append(tuple(T(a, dev)[off:] for a in (W, g, v)) + (l2,))
        ops.sgd_momentum_step_multi(multi, -0.01, 0.9, 1.0, zg)
        for (W, g, v, l2) in single:
            if W.numel():
                ops.sgd_momentum_step(W, g, v, l2, -0.01, 0.9, 1.0, zg)
        for k, ((Wm, gm, vm, _), (Ws, gs, vs, _), (Wh, gh, vh, l2)) in enumerate(zip(multi, single, host)):
            assert torch.equal(Wm, Ws) and torch.equal(gm, gs) and torch.equal(vm, vs), "block %d" % k
            if Wh.size:
                O.sgd_momentum_step(Wh, gh, vh, l2, -0.01, 0.9, 1.0, zg)
                assert_close(N(Wm), Wh, "multi sgd W[%d]" % k, atol=1e-7)
                assert_close(N(vm), vh, "multi sgd v[%d]" % k, atol=1e-7)
                assert_close(N(gm), gh, "multi sgd g[%d]" % k, atol=1e-7)
    assert _lib.lib().rh_sgd_momentum_step_multi(1, None, 1.0, 0.9, 1.0, 1, None) == _lib.RH_E_INVALID
    # keep_grad: those tensors' gradients are read for the update and left untouched (not zeroed, not regularised in
    # place); W and v as in the plain step, the other tensors as without the flag
    lens = (5, 4099, 1 << 16)
    host = [(synth.normal(19, 3 * k + 1, (n,)), synth.normal(19, 3 * k + 2, (n,)), synth.normal(19, 3 * k + 3, (n,))) for k, n in enumerate(lens)]
    for zg in (True, False):
        a = [tuple(T(x, dev) for x in h) + (0.01,) for h in host]
        b = [tuple(T(x, dev) for x in h) + (0.01,) for h in host]
        ops.sgd_momentum_step_multi(a, -0.01, 0.9, 1.0, zg, keep_grad=(0, 2))
        ops.sgd_momentum_step_multi(b, -0.01, 0.9, 1.0, zg)
        for k in range(3):
            assert torch.equal(a[k][0], b[k][0]) and torch.equal(a[k][2], b[k][2]), "keep_grad changed W or v of block %d" % k
            if k in (0, 2):
                assert np.array_equal(N(a[k][1]), host[k][1]), "a kept gradient was written"
            else:
                assert torch.equal(a[k][1], b[k][1])
    torch.cuda.synchronize()


def test_cast_and_fill(dev):
    x = (synth.integers(17, 1, (1000003,), 256)).astype(np.uint8)
    y = ops.cast_u8_f32(T(x, dev), 1.0 / 255.0)
    assert np.array_equal(N(y), O.cast_u8_f32(x, 1.0 / 255.0))
    t = torch.empty(1027, device=dev)
    ops.memset_f32(t[1:], 1.0)
    assert (N(t)[1:] == 1.0).all()


def test_preproc_kernels(dev):
    say("preproc kernels")
    x = synth.normal(13, 1, (5, 3, 37, 41))
    xd = T(x, dev)
    for (cw, ch, ow, oh) in ((41, 37, 0, 0), (32, 32, 9, 5), (1, 1, 40, 36), (17, 3, 0, 34)):
        assert np.array_equal(N(ops.crop_nchw(xd, cw, ch, ow, oh)), O.crop_nchw(x, cw, ch, ow, oh))
    assert np.array_equal(N(ops.flip_x(xd)), O.flip_x(x))
    wide = synth.normal(13, 2, (2, 1, 3, 300))     # wider than the 256 the reference asserts
    assert np.array_equal(N(ops.flip_x(T(wide, dev))), O.flip_x(wide))
    alphas, svals, svecs = synth.normal(13, 3, (15,)), synth.uniform(13, 4, (3,)), synth.normal(13, 5, (9,))
    assert_close(N(ops.pca3_noise(xd, T(alphas, dev), T(svals, dev), T(svecs, dev))), O.pca3_noise(x, alphas, svals, svecs),
                 "pca3 noise")
    # mean subtraction is the bias-add kernel with one "channel" per frame element
    mean = synth.normal(13, 6, (3, 37, 41))
    for normalize in (False, True):
        y = T(x, dev).clone()
        ops.add_bias_nchw(T(mean.ravel(), dev), y.view(5, -1, 1), alpha=(-1.0 / 255.0 if normalize else -1.0), beta=1.0)
        assert_close(N(y), O.subtract_mean(x, mean, normalize), "subtract mean")
    torch.cuda.synchronize()


def test_dropout_and_device_rng(dev):
    say("dropout / device rng")
    n = (1 << 18) + 77
    host = synth.uniform(31, 9, (n + 1000,))
    got = ops.rng_uniform01_device(31, 9, 1000, n, dev)
    assert np.array_equal(N(got), host[1000:]), "device generator == host generator, element by element"
    x, dy = synth.normal(14, 1, (n,)), synth.normal(14, 2, (n,))
    for ratio in (0.5, 0.1, 0.0, 1.0):
        y, mask = ops.dropout(T(x, dev), ratio, 1.0, got)
        y_ref, m_ref = O.dropout(x, ratio, 1.0, host[1000:])
        assert np.array_equal(N(mask), m_ref) and np.array_equal(N(y), y_ref)
        assert np.array_equal(N(ops.dropout_backprop(T(dy, dev), ratio, 1.0, mask)), O.dropout_backprop(dy, 1.0, m_ref))
    torch.cuda.synchronize()


@pytest.mark.parametrize("case", [((2, 7, 5, 6), 5), ((3, 96, 27, 27), 5), ((1, 3, 4, 4), 5), ((2, 10, 3, 3), 4), ((2, 4, 3, 3), 1)])
def test_lrn(dev, case):
    shape, size = case
    say("lrn", case)
    scale, power, min_div = 1e-4, 0.75, 2.0
    x = synth.normal(15, 1, shape) * np.float32(20.0)
    dy = synth.normal(15, 2, shape)
    y, d = ops.lrn_fwd(T(x, dev), size, scale, power, min_div)
    y_ref, d_ref = O.lrn_fwd(x, size, scale, power, min_div)
    assert_close(N(d), d_ref, "lrn denominators")
    assert_close(N(y), y_ref, "lrn fwd")
    dx = ops.lrn_bwd(T(x, dev), y, d, T(dy, dev), size, scale, power, min_div)
    assert_close(N(dx), O.lrn_bwd(x, dy, size, scale, power, min_div), "lrn bwd")
    torch.cuda.synchronize()


@pytest.mark.parametrize("shape", [(4, 3, 5, 6), (6, 5, 1, 1), (3, 2, 7, 7), (1, 4, 3, 3), (8, 64, 56, 56), (16, 512, 7, 7),
                                   (2, 3, 112, 112), (5, 7, 13, 9), (3, 8, 2, 2), (2, 4, 14, 14)])
def test_bnorm(dev, shape):
    """Spatial batch normalisation: training forward (batch statistics, moving averages, blend, fused ReLU),
    inference forward and backward against the fp64 restatement; one channel carries a mean 25x its deviation.
    (Two values per channel are left out: there dx cancels to ~epsilon analytically and has no stable digits.)"""
    say("bnorm", shape)
    C = shape[1]
    x = synth.normal(17, 1, shape) * np.float32(2.0) + np.linspace(-1, 50, C, dtype=np.float32)[None, :, None, None]
    dy = synth.normal(17, 2, shape)
    y0 = synth.normal(17, 3, shape)
    scale, bias = synth.normal(17, 4, (C,)) + np.float32(1.0), synth.normal(17, 5, (C,))
    rm, ri = synth.normal(17, 6, (C,)), np.abs(synth.normal(17, 7, (C,))) + np.float32(0.5)
    eps, ema = 1e-5, 0.1
    y_ref, cm_ref, ci_ref, rm_ref, ri_ref = O.bnorm_fwd_train(x, scale, bias, rm, ri, ema, eps)
    xd, sd, bd = T(x, dev), T(scale, dev), T(bias, dev)
    rmd, rid = T(rm, dev), T(ri, dev)
    y, cm, ci = ops.bnorm_fwd_train(xd, sd, bd, rmd, rid, ema, eps)
    assert_close(N(cm), cm_ref, "batch mean")
    assert_close(N(ci), ci_ref, "batch inverse deviation")
    assert_close(N(rmd), rm_ref, "running mean")
    assert_close(N(rid), ri_ref, "running inverse deviation")
    # normalised values of a channel with |mean| >> deviation lose |mean|/deviation ulps of x itself (fp32 inputs)
    assert_close(N(y), y_ref, "bnorm fwd", atol=2e-5)
    # blend into an existing tensor with the ReLU fused (the residual add of the stacked operators)
    yb = T(y0, dev)
    rm2, ri2 = T(rm, dev), T(ri, dev)
    ops.bnorm_fwd_train(xd, sd, bd, rm2, ri2, ema, eps, alpha=1.0, beta=1.0, y=yb, relu=True)
    want = O.bnorm_fwd_train(x, scale, bias, rm, ri, ema, eps, alpha=1.0, beta=1.0, y=y0)[0]
    got = N(yb)
    unsure = np.abs(want) < 1e-4 * max(1.0, float(np.sqrt((want ** 2).mean())))
    assert np.array_equal((got > 0)[~unsure], (want > 0)[~unsure])
    assert_close(got, np.maximum(want, 0), "bnorm fwd blend + relu", atol=2e-5)
    assert np.array_equal(N(rm2), N(rmd)) and np.array_equal(N(ri2), N(rid)), "statistics do not depend on the blend"
    yi = ops.bnorm_fwd_infer(xd, sd, bd, T(rm, dev), T(ri, dev), eps)
    assert_close(N(yi), O.bnorm_fwd_infer(x, scale, bias, rm, ri), "bnorm inference", atol=2e-5)
    # backward on the statistics the device cached; parameter gradients accumulate with beta_param = 1
    dx_ref, ds_ref, db_ref = O.bnorm_bwd(x, dy, scale, N(cm), N(ci))
    ds0, db0 = synth.normal(17, 8, (C,)), synth.normal(17, 9, (C,))
    dsd, dbd = T(ds0, dev), T(db0, dev)
    dx, _, _ = ops.bnorm_bwd(xd, T(dy, dev), sd, cm, ci, eps, dscale=dsd, dbias=dbd, beta_param=1.0)
    assert_close(N(dx), dx_ref, "bnorm bwd dx", atol=2e-5)
    assert_close(N(dsd), ds_ref.astype(np.float64) + ds0, "bnorm dscale", atol=2e-5)
    assert_close(N(dbd), db_ref.astype(np.float64) + db0, "bnorm dbias", atol=2e-5)
    dx2 = T(y0, dev)
    ops.bnorm_bwd(xd, T(dy, dev), sd, cm, ci, eps, alpha_data=1.0, beta_data=1.0, dx=dx2)
    assert_close(N(dx2), dx_ref.astype(np.float64) + y0, "bnorm bwd dx blended", atol=2e-5)
    # backward through the ReLU the forward pass fused: the mask is the device's own forward output, and must be that
    # exactly (an element the two passes disagree on would be off by a whole dy)
    yr, _, _ = ops.bnorm_fwd_train(xd, sd, bd, T(rm, dev), T(ri, dev), ema, eps, relu=True)
    dym = np.where(N(yr) > 0, dy, np.float32(0.0)).astype(np.float32)
    dxm_ref, dsm_ref, dbm_ref = O.bnorm_bwd(x, dym, scale, N(cm), N(ci))
    dxm, dsm, dbm = ops.bnorm_bwd(xd, T(dy, dev), sd, cm, ci, eps, relu_bias=bd)
    assert_close(N(dxm), dxm_ref, "bnorm bwd through fused relu: dx", atol=2e-5)
    assert_close(N(dsm), dsm_ref, "bnorm bwd through fused relu: dscale", atol=2e-5)
    assert_close(N(dbm), dbm_ref, "bnorm bwd through fused relu: dbias", atol=2e-5)
    same = ops.bnorm_bwd(xd, T(dym, dev), sd, cm, ci, eps)
    assert np.array_equal(N(dxm), N(same[0])) and np.array_equal(N(dsm), N(same[1])), "identical to masking dy beforehand"
    torch.cuda.synchronize()


@pytest.mark.parametrize("shape", [(1, 3, 16, 128), (9, 3, 4, 57), (4, 2, 32, 64), (3, 2, 4, 683), (5, 2, 64, 64), (1, 2, 4, 5121),
                                   (512, 3, 1, 3), (29, 3, 1, 53), (2048, 3, 1, 3), (5, 2, 1, 1229), (4096, 2, 1, 5), (2, 2, 1, 10241)])
def test_bnorm_at_the_bounds_of_its_forms(dev, shape):
    """Values per channel at and just past what each block size of the one-launch form holds (2048 / 8192 / 20480 in
    16-byte units, 1536 / 6144 / 20480 single), where the last is the bound to the form of three launches; results written over
    their own input are those written elsewhere."""
    test_bnorm(dev, shape)
    C = shape[1]
    x = synth.normal(18, 1, shape) * np.float32(2.0) + np.float32(3.0)
    scale, bias = T(synth.normal(18, 4, (C,)), dev), T(synth.normal(18, 5, (C,)), dev)
    stats = [T(np.zeros(C, np.float32), dev) for _ in range(4)]
    apart, cm, ci = ops.bnorm_fwd_train(T(x, dev), scale, bias, stats[0], stats[1], 0.1, 1e-5)
    over = T(x, dev)
    ops.bnorm_fwd_train(over, scale, bias, stats[2], stats[3], 0.1, 1e-5, y=over)
    assert np.array_equal(N(over), N(apart))
    dy = T(synth.normal(18, 2, shape), dev)
    dx = N(ops.bnorm_bwd(T(x, dev), dy, scale, cm, ci, 1e-5)[0])
    ops.bnorm_bwd(T(x, dev), dy, scale, cm, ci, 1e-5, dx=dy)
    assert np.array_equal(N(dy), dx)


@pytest.mark.parametrize("shape", [(3, 2, 4, 5), (2, 3, 3, 3), (4, 2, 32, 65), (3, 2, 83, 83), (5, 2, 64, 66), (1, 1, 1, 1)])
def test_residual_sum_and_its_gradient(dev, shape):
    """The batch norm that adds another tensor gives what the blend with a copy of it gives (one launch, three, single values
    and 16-byte units, a tensor at a 4-byte offset), and the ReLU backward with a second result what the pass and a copy do."""
    C = shape[1]
    x, r, dy = synth.normal(19, 1, shape), synth.normal(19, 2, shape), synth.normal(19, 3, shape)
    scale, bias = T(synth.normal(19, 4, (C,)), dev), T(synth.normal(19, 5, (C,)), dev)
    off = torch.empty(r.size + 1, device=dev)[1:].view(shape)
    off.copy_(T(r, dev))
    for relu in (False, True):
        for y0, same_units in ((T(r, dev), True), (off, shape[2] * shape[3] % 4 != 0)):
            stats = [torch.full((C,), 0.5, device=dev) for _ in range(4)]
            want = ops.bnorm_fwd_train(T(x, dev), scale, bias, stats[0], stats[1], 0.1, 1e-5, alpha=0.5, beta=1.5, y=T(r, dev), relu=relu)
            got = ops.bnorm_fwd_train(T(x, dev), scale, bias, stats[2], stats[3], 0.1, 1e-5, alpha=0.5, beta=1.5, y0=y0, relu=relu)
            for a, b in zip(got + (stats[2], stats[3]), want + (stats[0], stats[1])):
                # (another unit, another order of the sums)
                assert torch.equal(a, b) if same_units else torch.allclose(a, b, rtol=1e-5, atol=1e-5)
            assert np.array_equal(N(y0), r), "the added tensor is read only"
            want = ops.bnorm_fwd_infer(T(x, dev), scale, bias, stats[0], stats[1], 1e-5, beta=1.0, y=T(r, dev), relu=relu)
            got = ops.bnorm_fwd_infer(T(x, dev), scale, bias, stats[0], stats[1], 1e-5, beta=1.0, y0=y0, relu=relu)
            assert torch.equal(got, want)
    for y in (T(r, dev), off):
        one, two, copy = T(dy, dev), T(dy, dev), torch.full(shape, 7.0, device=dev)
        ops.rect_backprop_copy(y, one, copy)
        ops.rect_backprop_inplace(y, two)
        assert torch.equal(one, two) and torch.equal(copy, two)


# A batch norm behind a forward pass at inference: whole results and a sliced tail (the batch norm in a launch of its own), contractions in
# slices of each form (split operands, the engine, staged), planes and channels that are no multiple of four; which of the four calls
# below have slices throughout and form the batch norm in their reduction.
@pytest.mark.parametrize("case, fused", [((9, 64, 56, 56, 64, 3, 1, 1), ""), ((9, 128, 28, 28, 128, 3, 1, 1), "xds"), ((9, 512, 7, 7, 512, 3, 1, 1), "0xds"),
                                         ((9, 256, 14, 14, 512, 1, 2, 0), "0xds"), ((5, 256, 13, 11, 70, 3, 2, 1), "0xds"), ((1, 24, 5, 7, 40, 3, 1, 1), "0xds"),
                                         ((33, 96, 27, 27, 250, 5, 1, 2), ""), ((2, 3, 30, 30, 33, 7, 2, 3), "0xds"), ((60, 256, 14, 14, 256, 3, 1, 1), "")],
                         ids=str)
def test_conv2d_fwd_bnorm_infer(dev, case, fused):
    """rh_conv2d_fwd_bnorm_infer against the two calls that it stands for: the same bits in both results."""
    Nn, C, H, W, K, R, st, pad = case
    say("conv bnorm infer case", case)
    x, w = T(synth.normal(73, 1, (Nn, C, H, W)), dev), T(synth.normal(73, 2, (K, C, R, R)), dev)
    scale, bias, mean = (T(synth.normal(73, 3 + i, (K,)), dev) for i in range(3))
    ivar = T(np.abs(synth.normal(73, 6, (K,))) + 0.1, dev)
    for key, algo in (("0", 0), ("x", _lib.RH_ALGO_BF16X3 | _lib.RH_ALGO_F16X2), ("d", _lib.RH_ALGO_DIRECT), ("s", _lib.RH_ALGO_SCALAR_OFFSET)):
        pre = ops.conv2d_fwd(x, w, st, pad, algo=algo)
        y0 = T(synth.normal(73, 7, tuple(pre.shape)), dev)
        for beta, old, relu in ((0.0, None, True), (1.0, y0, True), (0.5, y0, False)):
            want = ops.bnorm_fwd_infer(pre, scale, bias, mean, ivar, 1e-5, beta=beta, y0=old, relu=relu)
            (got_pre, got), tags = profile_tags(lambda: ops.conv2d_fwd_bnorm_infer(x, w, st, pad, scale, bias, mean, ivar, 1e-5, beta=beta,
                                                                                  y0=old, relu=relu, algo=algo))
            assert torch.equal(got_pre, pre) and torch.equal(got, want), (algo, beta, relu)
            assert ("bnorm_fwd_apply" not in tags) == (key in fused), (key, tags)



@pytest.mark.parametrize("case", [(2, 3, 9, 3, 2, 0), (2, 3, 9, 3, 2, 1), (3, 4, 8, 2, 2, 0), (2, 5, 27, 3, 2, 0), (2, 2, 13, 3, 3, 1)])
@pytest.mark.parametrize("rounding", [_lib.RH_ROUND_FLOOR, _lib.RH_ROUND_CEIL])
def test_pool2d_bwd_with_folded_relu_mask(dev, case, rounding):
    """rh_pool2d_bwd_relu == max-pool backward followed by the ReLU backward mask of the pool's input
    (Pool2dOperator::backward then the producer's rect_backprop), on inputs with whole windows of zeros."""
    Nn, C, H, k, st, pad = case
    say("pool bwd + relu case", case, rounding)
    x = O.rect_inplace(synth.normal(16, 1, (Nn, C, H, H)) - np.float32(0.8))     # ~80 % zeros: some windows are all zero
    xd = T(x, dev)
    y, am = ops.pool2d_fwd(xd, k, st, pad, _lib.RH_POOL_MAX, rounding, want_argmax=True)
    assert (N(y) == 0).any() and (N(y) > 0).any()
    dy = synth.normal(16, 2, tuple(y.shape))
    want = O.pool2d_bwd(x, N(y), dy, k, st, pad, O.POOL_MAX, rounding)
    O.rect_backprop_inplace(x, want)
    got = N(ops.pool2d_bwd_relu(x.shape, y, T(dy, dev), k, st, pad, am, rounding))
    assert np.array_equal(got == 0, want == 0), "same elements are masked"
    assert_close(got, want, "pool bwd with folded relu mask")    # elements fed by several windows add in another order
    # and it is bit-identical to the two GPU kernels it replaces
    two = ops.pool2d_bwd(xd, y, T(dy, dev), k, st, pad, _lib.RH_POOL_MAX, rounding, argmax=am)
    ops.rect_backprop_inplace(xd, two)
    assert np.array_equal(got, N(two))
    torch.cuda.synchronize()


@pytest.mark.parametrize("case", [(2, 3, 9, 3, 2, 0), (2, 3, 9, 3, 2, 1), (3, 4, 8, 2, 2, 0), (2, 5, 27, 3, 2, 0), (2, 2, 13, 3, 3, 1)])
@pytest.mark.parametrize("rounding", [_lib.RH_ROUND_FLOOR, _lib.RH_ROUND_CEIL])
def test_avg_pool2d_bwd_with_folded_relu_mask(dev, case, rounding):
    """rh_pool2d_bwd_avg_relu == average-pool backward followed by the ReLU backward mask of the pool's input: against the
    oracle's two passes, and bit-identical to the two GPU kernels it replaces; max pooling is refused."""
    Nn, C, H, k, st, pad = case
    say("avg pool bwd + relu case", case, rounding)
    x = O.rect_inplace(synth.normal(18, 1, (Nn, C, H, H)) - np.float32(0.3))
    xd = T(x, dev)
    y = ops.pool2d_fwd(xd, k, st, pad, _lib.RH_POOL_AVG_INCL_PAD, rounding)
    dy = synth.normal(18, 2, tuple(y.shape))
    want = O.pool2d_bwd(x, N(y), dy, k, st, pad, O.POOL_AVG, rounding)
    O.rect_backprop_inplace(x, want)
    got = ops.pool2d_bwd_avg_relu(xd, T(dy, dev), k, st, pad, rounding)
    assert_close(N(got), want, "avg pool bwd with folded relu mask")
    two = ops.pool2d_bwd(xd, y, T(dy, dev), k, st, pad, _lib.RH_POOL_AVG_INCL_PAD, rounding)
    ops.rect_backprop_inplace(xd, two)
    assert torch.equal(got, two)
    import ctypes as C
    g = ops.pool_geom(x.shape, k, st, pad, _lib.RH_POOL_MAX, rounding)
    assert _lib.lib().rh_pool2d_bwd_avg_relu(C.byref(g), xd.data_ptr(), T(dy, dev).data_ptr(), got.data_ptr(), None) == _lib.RH_E_UNSUPPORTED
    torch.cuda.synchronize()


def test_context_memory_calls(dev):
    """rh_malloc (zero-filled), rh_host_malloc (page-locked, zero-filled), rh_load_sync / rh_store_sync round trip,
    rh_store_begin / rh_store_wait."""
    import ctypes as C
    lib = _lib.lib()
    ctx = C.c_void_p()
    _lib.check(lib.rh_ctx_create(0, C.byref(ctx)), "rh_ctx_create")
    n = 3 * 1000 + 1   # not a multiple of four bytes
    d, h, back = C.c_void_p(), C.c_void_p(), C.c_void_p()
    _lib.check(lib.rh_malloc(ctx, n, C.byref(d)), "rh_malloc")
    _lib.check(lib.rh_host_malloc(ctx, n, C.byref(h)), "rh_host_malloc")
    _lib.check(lib.rh_host_malloc(ctx, n, C.byref(back)), "rh_host_malloc")
    host = (C.c_uint8 * n).from_address(h.value)
    out = (C.c_uint8 * n).from_address(back.value)
    assert not any(host) and not any(out), "page-locked memory starts zeroed"
    _lib.check(lib.rh_store_sync(ctx, back, d, n), "rh_store_sync")
    assert not any(out), "device memory starts zeroed, odd tail included"
    pattern = synth.integers(21, 1, (n,), 256).astype(np.uint8)
    C.memmove(h, pattern.ctypes.data, n)
    _lib.check(lib.rh_load_sync(ctx, d, h, n), "rh_load_sync")
    _lib.check(lib.rh_store_sync(ctx, back, d, n), "rh_store_sync")
    assert np.array_equal(np.frombuffer(out, np.uint8), pattern)
    assert lib.rh_host_malloc(ctx, 16, None) == _lib.RH_E_INVALID and lib.rh_host_free(None, h) == _lib.RH_E_INVALID
    # the store in two halves: the copy is ordered behind what the context's stream holds when it is begun (a fill
    # kernel here), not behind what is enqueued afterwards (a second fill, which the copy must not see)
    nf = 1 << 20
    big, hb = C.c_void_p(), C.c_void_p()
    _lib.check(lib.rh_malloc(ctx, 4 * nf, C.byref(big)), "rh_malloc")
    _lib.check(lib.rh_host_malloc(ctx, 8, C.byref(hb)), "rh_host_malloc")
    stream = C.c_void_p(lib.rh_ctx_stream(ctx))
    assert lib.rh_store_wait(ctx) == 0, "nothing begun: returns at once"
    _lib.check(lib.rh_memset_f32(big, 3.5, nf, stream), "rh_memset_f32")
    _lib.check(lib.rh_store_begin(ctx, hb, C.c_void_p(big.value + 4 * (nf - 2)), 8), "rh_store_begin")
    _lib.check(lib.rh_store_wait(ctx), "rh_store_wait")
    assert list((C.c_float * 2).from_address(hb.value)) == [3.5, 3.5]
    _lib.check(lib.rh_ctx_sync(ctx), "rh_ctx_sync")
    assert lib.rh_store_begin(ctx, None, big, 8) == _lib.RH_E_INVALID and lib.rh_store_begin(None, hb, big, 8) == _lib.RH_E_INVALID
    assert lib.rh_store_begin(ctx, hb, big, 0) == 0 and lib.rh_store_wait(None) == _lib.RH_E_INVALID
    _lib.check(lib.rh_host_free(ctx, hb), "rh_host_free")
    _lib.check(lib.rh_free(ctx, big), "rh_free")
    for p_ in (h, back):
        _lib.check(lib.rh_host_free(ctx, p_), "rh_host_free")
    _lib.check(lib.rh_free(ctx, d), "rh_free")
    _lib.check(lib.rh_ctx_destroy(ctx), "rh_ctx_destroy")


def _check_conv_case_all_passes(dev, case, seed, idx):
    """All three passes, the forced scalar-offset backward-filter and the bf16-operand forward of one geometry."""
    Nn, C, H, W, K, R, st, pad = case
    x = synth.normal(seed, idx * 4 + 1, (Nn, C, H, W))
    w = synth.normal(seed, idx * 4 + 2, (K, C, R, R))
    b = synth.normal(seed, idx * 4 + 3, (K,))
    y_ref = O.conv2d_fwd(x, w, st, pad)
    dy = synth.normal(seed, idx * 4 + 4, y_ref.shape)
    xd, wd, bd, dyd = T(x, dev), T(w, dev), T(b, dev), T(dy, dev)
    tag = " %s" % (case,)
    y = ops.conv2d_fwd(xd, wd, st, pad, bias=bd, relu=True)
    assert_close(N(y), O.rect_inplace(O.add_bias_nchw(b, y_ref.copy())), "fwd" + tag)
    y16 = ops.conv2d_fwd(xd, wd, st, pad, algo=_lib.RH_MATH_BF16_MFMA_FP32ACC)
    assert_close(N(y16), O.conv2d_fwd(O.round_bf16(x), O.round_bf16(w), st, pad), "fwd bf16" + tag)
    dw_ref = O.conv2d_bwd_filter(x, dy, w.shape, st, pad)
    assert_close(N(ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad)), dw_ref, "bwd_filter" + tag)
    assert_close(N(ops.conv2d_bwd_filter(xd, dyd, w.shape, st, pad, algo=_lib.RH_ALGO_SCALAR_OFFSET)), dw_ref,
                 "bwd_filter scalar-offset" + tag)
    assert_close(N(ops.conv2d_bwd_data(wd, dyd, x.shape, st, pad)), O.conv2d_bwd_data(w, dy, x.shape, st, pad),
                 "bwd_data" + tag)


def test_conv2d_random_geometries(dev):
    """A seeded sweep over convolution geometries (filter 1-7, stride 1-4, any padding below the filter size, channel
    counts on both sides of every tile and group size): all three passes, the forced scalar-offset backward-filter and
    the bf16-operand forward against the oracle.  The hand-picked cases above name the paths; this guards the seams."""
    import random
    rnd = random.Random(20160417)
    done = 0
    while done < 60:
        R = rnd.choice([1, 1, 2, 3, 3, 3, 4, 5, 7])
        st = rnd.choice([1, 1, 1, 2, 2, 3, 4])
        pad = rnd.randint(0, max(0, R - 1))
        C = rnd.choice([1, 2, 3, 4, 7, 8, 12, 16, 24, 33, 40, 64, 72, 96])
        K = rnd.choice([1, 3, 5, 8, 16, 20, 32, 50, 64, 96, 100, 128, 130, 200, 256])
        H, W = rnd.randint(max(R - 2 * pad, 1), 24), rnd.randint(max(R - 2 * pad, 1), 24)
        Nn = rnd.choice([1, 2, 3, 5, 9, 17, 40])
        if Nn * C * H * W * K * R * R > 6e8:
            Nn = 2
        if (H + 2 * pad - R) // st + 1 < 1 or (W + 2 * pad - R) // st + 1 < 1:
            continue
        case = (Nn, C, H, W, K, R, st, pad)
        say("random conv case", done, case)
        _check_conv_case_all_passes(dev, case, 31, done)
        done += 1
    torch.cuda.synchronize()


def test_conv2d_random_midsize_geometries(dev):
    """A seeded sweep over layer-sized geometries (16-256 input and 32-512 output channels, planes of 7-56, batches up
    to 128, capped at 30 GFLOP a pass): grids of tens to over a thousand tiles, so contraction splits, sliced tails in
    one and in several rounds of tiles, the per-layer loader choice of backward-filter and the stride-2 class
    decomposition of backward-data are all met at sizes the hand-picked cases do not name."""
    import random
    rnd = random.Random(20160418)
    done = 0
    while done < 24:
        R = rnd.choice([1, 3, 3, 3, 5])
        st = rnd.choice([1, 1, 1, 2])
        pad = rnd.choice([0, R // 2, R // 2])
        C = rnd.choice([16, 24, 32, 48, 64, 96, 128, 160, 256])
        K = rnd.choice([32, 64, 96, 128, 192, 256, 384, 512])
        H = rnd.randint(7, 56)
        W = rnd.choice([H, H, rnd.randint(7, 56)])
        Nn = rnd.choice([8, 16, 24, 32, 52, 64, 100, 128])
        P, Q = (H + 2 * pad - R) // st + 1, (W + 2 * pad - R) // st + 1
        if P < 1 or Q < 1:
            continue
        while 2.0 * Nn * C * K * R * R * P * Q > 3e10 and Nn > 1:
            Nn //= 2
        case = (Nn, C, H, W, K, R, st, pad)
        say("random mid-size conv case", done, case, "forward tiles", -(-K // 128) * -(-(Nn * P * Q) // 128))
        _check_conv_case_all_passes(dev, case, 51, done)
        done += 1
    torch.cuda.synchronize()


def test_sgemm_and_pool_random_shapes(dev):
    """Seeded sweeps: SGEMM over transposes, odd extents, padded leading dimensions, alpha / beta pairs, with and
    without scratch; pooling over window, stride, padding, both modes and both roundings on rectangular planes."""
    import random
    rnd = random.Random(20160418)
    for it in range(40):
        tA, tB = rnd.randint(0, 1), rnd.randint(0, 1)
        m = rnd.choice([1, 2, 7, 10, 31, 64, 100, 128, 129, 300, 500, 1000, 4096])
        n = rnd.choice([1, 3, 16, 32, 64, 100, 128, 200, 256])
        k = rnd.choice([1, 2, 15, 16, 17, 64, 100, 256, 1000, 2450, 4096])
        if m * n * k > 3e8:
            k = 64
        use_ws = rnd.random() < 0.7
        a_shape = (m, k) if tA else (k, m)
        b_shape = (k, n) if tB else (n, k)
        lda, ldb, ldc = a_shape[1] + rnd.randint(0, 3), b_shape[1] + rnd.randint(0, 2), m + rnd.randint(0, 2)
        alpha, beta = rnd.choice([(1.0, 0.0), (0.5, 1.0), (1.0, 1.0), (-2.0, 0.25)])
        say("random sgemm", it, (tA, tB, m, n, k, lda, ldb, ldc, alpha, beta, use_ws))
        A = synth.normal(41, it * 3 + 1, (a_shape[0], lda))
        B = synth.normal(41, it * 3 + 2, (b_shape[0], ldb))
        C0 = synth.normal(41, it * 3 + 3, (n, ldc))
        ref = O.sgemm(tA, tB, m, n, k, alpha, A, lda, B, ldb, beta, C0.copy(), ldc)
        Cd = T(C0, dev)
        ops.sgemm(tA, tB, m, n, k, alpha, T(A, dev), lda, T(B, dev), ldb, beta, Cd, ldc, use_workspace=use_ws)
        assert_close(N(Cd), ref, "sgemm %d" % it)
    for it in range(40):
        k = rnd.choice([2, 2, 3, 3, 4, 5])
        st = rnd.choice([1, 2, 2, 3])
        pad = rnd.randint(0, k // 2)
        H, W = rnd.randint(k, 40), rnd.randint(k, 40)
        Nn, C = rnd.choice([1, 2, 5]), rnd.choice([1, 3, 8, 17])
        mode = rnd.choice([_lib.RH_POOL_MAX, _lib.RH_POOL_AVG_INCL_PAD])
        rounding = rnd.choice([_lib.RH_ROUND_FLOOR, _lib.RH_ROUND_CEIL])
        say("random pool", it, (Nn, C, H, W, k, st, pad, mode, rounding))
        x = np.round(synth.normal(42, it * 2 + 1, (Nn, C, H, W)) * 2) / 2
        y_ref, am_ref = O.pool2d_fwd(x, k, st, pad, mode, rounding, want_argmax=True)
        if y_ref.size == 0:
            continue
        xd = T(x, dev)
        y, am = ops.pool2d_fwd(xd, k, st, pad, mode, rounding, want_argmax=True)
        assert_close(N(y), y_ref, "pool fwd %d" % it)
        if mode == _lib.RH_POOL_MAX:
            assert np.array_equal(N(am), am_ref), "arg-max mask %d" % it
        dy = synth.normal(42, it * 2 + 2, y_ref.shape)
        dx_ref = O.pool2d_bwd(x, y_ref, dy, k, st, pad, mode, rounding)
        assert_close(N(ops.pool2d_bwd(xd, y, T(dy, dev), k, st, pad, mode, rounding)), dx_ref, "pool bwd %d" % it)
        if mode == _lib.RH_POOL_MAX:
            assert_close(N(ops.pool2d_bwd(xd, y, T(dy, dev), k, st, pad, mode, rounding, argmax=am)), dx_ref,
                         "pool bwd from the mask %d" % it)
    torch.cuda.synchronize()

