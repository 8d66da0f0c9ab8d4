"""Conv2d and MaxPool through the C ABI and the session: exact on integer-valued
data against the oracle and the definition, bounded on random data; padding forms, strides, dilation,
groups, SAME_UPPER, and the ViT patch embedding feeding the token layout."""
import numpy as np
import pytest

import oracle as O
from altius_amd.graph import Model, Op
from altius_amd.session import HipSessionBuilder
from conftest import assert_bits_equal
from test_oracle import CONV_CASES, direct_conv

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(41)


@pytest.mark.parametrize("case_", CONV_CASES)
def test_conv2d(ctx, case, case_):
    case(f"conv2d {case_}")
    args = dict(strides=(1, 1), pads=(0, 0, 0, 0), dilations=(1, 1), group=1)
    args.update({k: v for k, v in case_.items() if k not in ("x", "w")})
    x = RNG.integers(-3, 4, size=case_["x"]).astype(np.float32)
    w = RNG.integers(-3, 4, size=case_["w"]).astype(np.float32)
    bias = RNG.integers(-3, 4, size=case_["w"][0]).astype(np.float32)
    for b in (bias, None):
        got = ctx.conv2d(x, w, b, **args)
        assert_bits_equal(got, O.conv2d(x, w, b, **args), "vs oracle")
        assert_bits_equal(got, direct_conv(x, w, b, **args).astype(np.float32), "vs the definition")
    xr, wr = RNG.standard_normal(case_["x"]).astype(np.float32), RNG.standard_normal(case_["w"]).astype(np.float32)
    k = int(np.prod(case_["w"][1:]))
    exact = direct_conv(xr, wr, bias, **args)
    bound = (k + 3) * 2.0 ** -24 * direct_conv(np.abs(xr), np.abs(wr), np.abs(bias), **args)
    got = ctx.conv2d(xr, wr, bias, **args)
    assert np.all(np.abs(got - exact) <= bound)
    assert np.allclose(got, O.conv2d(xr, wr, bias, **args), rtol=1e-5, atol=1e-5 * np.sqrt(k))


@pytest.mark.parametrize("x, w, args", [
    # depthwise: planes of one, several planes per block, rows and columns cut into tiles, one and four rows per thread
    ((1, 5, 1, 1), (5, 1, 3, 3), dict(pads=(1, 1, 1, 1), group=5)),
    ((3, 37, 7, 7), (37, 1, 5, 5), dict(pads=(2, 2, 2, 2), group=37)),
    ((2, 3, 67, 131), (3, 1, 5, 5), dict(pads=(2, 2, 2, 2), group=3)),
    ((40, 96, 29, 30), (96, 1, 3, 3), dict(pads=(1, 1, 1, 1), group=96)),
    ((40, 96, 29, 31), (96, 1, 5, 5), dict(pads=(2, 2, 2, 2), strides=(2, 2), group=96)),
    ((40, 96, 29, 31), (96, 1, 5, 5), dict(pads=(2, 2, 2, 2), group=96)),
    ((40, 96, 28, 31), (96, 1, 3, 3), dict(pads=(1, 1, 1, 1), strides=(2, 2), group=96)),
    ((2, 6, 20, 23), (12, 1, 3, 5), dict(pads=(1, 2, 3, 0), strides=(1, 3), dilations=(2, 1), group=6)),
    ((1, 2, 9, 300), (2, 1, 9, 150), dict(group=2)),
    # products: edges of the 16, 32 and 64 x 128 tiles, k below, at and past a step, images that end inside a tile
    ((1, 1, 1, 1), (1, 1, 1, 1), dict()),
    ((1, 16, 4, 4), (16, 16, 1, 1), dict()),
    ((2, 17, 5, 5), (33, 17, 1, 1), dict()),
    ((1, 576, 7, 7), (96, 576, 1, 1), dict()),
    ((9, 40, 64, 64), (65, 40, 1, 1), dict()),
    ((33, 15, 47, 43), (63, 15, 1, 1), dict()),
    ((70, 3, 57, 53), (16, 3, 3, 3), dict(pads=(1, 1, 1, 1), strides=(2, 2))),
    ((1, 24, 19, 21), (36, 12, 3, 3), dict(pads=(1, 1, 1, 1), group=2)),
    ((1, 64, 30, 30), (40, 64, 1, 1), dict(strides=(2, 2))),
    ((33, 8, 33, 33), (130, 8, 3, 3), dict(pads=(0, 1, 0, 1), dilations=(2, 1))),
])
def test_conv2d_kernel_edges(ctx, case, x, w, args):
    """Small integers: every product and partial sum is exact in fp32 whatever the order, so the result is the oracle's."""
    case(f"conv2d edges {x} {w} {args}")
    args = {**dict(strides=(1, 1), pads=(0, 0, 0, 0), dilations=(1, 1), group=1), **args}
    xi, wi = RNG.integers(-3, 4, size=x).astype(np.float32), RNG.integers(-3, 4, size=w).astype(np.float32)
    bias = RNG.integers(-3, 4, size=w[0]).astype(np.float32)
    for b in (bias, None):
        assert_bits_equal(ctx.conv2d(xi, wi, b, **args), O.conv2d(xi, wi, b, **args), "vs oracle")


@pytest.mark.parametrize("x, w, args", [
    # many channels and values of k: products of the input as it lies (1 x 1) or of an unfolded copy
    ((1, 700, 12, 12), (128, 700, 3, 3), dict(pads=(1, 1, 1, 1))),                              # k in slices
    ((3, 257, 19, 23), (301, 257, 3, 3), dict(pads=(1, 0, 1, 2))),
    ((2, 40, 40, 40), (300, 40, 3, 3), dict(pads=(1, 1, 1, 1), dilations=(2, 2))),
    ((2, 129, 30, 31), (260, 129, 5, 3), dict(pads=(2, 1, 2, 1), strides=(1, 2))),
    ((1, 3, 224, 224), (768, 3, 16, 16), dict(strides=(16, 16))),
    ((3, 250, 33, 31), (270, 125, 3, 3), dict(pads=(1, 1, 1, 1), group=2)),
    ((8, 256, 28, 28), (130, 256, 1, 1), dict()),
    ((4, 601, 16, 16), (515, 601, 1, 1), dict()),
])
def test_conv2d_unfolded(ctx, case, x, w, args):
    case(f"conv2d unfolded {x} {w} {args}")
    args = {**dict(strides=(1, 1), pads=(0, 0, 0, 0), dilations=(1, 1), group=1), **args}
    xi, wi = RNG.integers(-3, 4, size=x).astype(np.float32), RNG.integers(-3, 4, size=w).astype(np.float32)
    bias = RNG.integers(-3, 4, size=w[0]).astype(np.float32)
    for b in (bias, None):
        assert_bits_equal(ctx.conv2d(xi, wi, b, **args), O.conv2d(xi, wi, b, **args), "vs oracle")


@pytest.mark.parametrize("x", [(1, 512, 243, 244), (3, 256, 208, 209)])
def test_conv2d_unfolded_in_passes(ctx, case, x):
    """An image whose unfolded copy is more than the workspace's 1 GiB is taken in bands of rows, a batch in groups of images; the
    last one of either is smaller.  Whole numbers, at the corners of every image, around the bands' seam and at random places."""
    b, c, h, wd = x
    oc = 256
    case(f"conv2d in passes {x}")
    xi = RNG.integers(-3, 4, size=x).astype(np.float32)
    wi = RNG.integers(-3, 4, size=(oc, c, 3, 3)).astype(np.float32)
    bias = RNG.integers(-3, 4, size=oc).astype(np.float32)
    got = ctx.conv2d(xi, wi, bias, pads=(1, 1, 1, 1))
    assert got.shape == (b, oc, h, wd)
    padded = np.pad(xi, ((0, 0), (0, 0), (1, 1), (1, 1)))
    rows, cols = [0, h // 2 - 1, h // 2, h // 2 + 1, h - 1], [0, 1, wd - 1]
    at = [(i, y, z) for i in range(b) for y in rows for z in cols]
    at += list(zip(RNG.integers(0, b, 200), RNG.integers(0, h, 200), RNG.integers(0, wd, 200)))
    patches = np.stack([padded[i, :, y:y + 3, z:z + 3].reshape(-1) for i, y, z in at]).astype(np.float64)
    want = patches @ wi.reshape(oc, -1).T.astype(np.float64) + bias
    assert np.array_equal(np.stack([got[i, :, y, z] for i, y, z in at]), want)


def test_unfolded_convolutions_of_a_session_replayed(case):
    """Two of them share the workspace; the recorded run gives the eager run's bits."""
    case("session conv2d unfolded, recorded")
    m = Model(opset_version=13)
    v = m.new_val_named_and_shaped("x", [2, 96, 20, 22])
    m.add_input(v)
    w = [RNG.integers(-2, 3, size=s).astype(np.float32) for s in ((256, 96, 3, 3), (300, 256, 3, 3))]
    y = v
    for a in w:
        out = m.new_val()
        m.add_node(Op.Conv2d, [y, m.new_initializer(a)], [out], kernel_shape=[3, 3], strides=[1, 1], pads=[1, 1, 1, 1])
        y = out
    m.add_output(y)
    session = HipSessionBuilder(m).with_graph_replay().build()
    for _ in range(4):
        x = RNG.integers(-2, 3, size=(2, 96, 20, 22)).astype(np.float32)
        want = x
        for a in w:
            want = O.conv2d(want, a, None, pads=(1, 1, 1, 1))
        assert_bits_equal(session.run([x])[0], want, "vs oracle")
    assert session.graph_replays() > 0


@pytest.mark.parametrize("x, w, args", [
    ((1, 1, 520, 7), (1, 1, 2, 1), dict(dilations=(500, 1))),                       # few outputs to a tile of 8192 values
    ((2, 3, 33, 33), (3, 1, 3, 3), dict(dilations=(36, 36), pads=(36,) * 4, group=3)),
    ((2, 3, 40, 41), (3, 1, 3, 3), dict(dilations=(24, 24), pads=(24,) * 4, group=3)),
    ((1, 2, 70, 70), (2, 1, 64, 64), dict(group=2)),                                # thousands of taps
    ((1, 2, 1, 5000), (4, 1, 1, 3), dict(dilations=(1, 2048), group=2)),
    ((3, 2, 64, 64), (2, 1, 16, 16), dict(strides=(16, 16), group=2)),
])
def test_depthwise_that_reads_far_apart(ctx, case, x, w, args):
    case(f"depthwise far apart {x} {w} {args}")
    args = {**dict(strides=(1, 1), pads=(0, 0, 0, 0), dilations=(1, 1), group=1), **args}
    xi, wi = RNG.integers(-3, 4, size=x).astype(np.float32), RNG.integers(-3, 4, size=w).astype(np.float32)
    bias = RNG.integers(-3, 4, size=w[0]).astype(np.float32)
    for b in (bias, None):
        assert_bits_equal(ctx.conv2d(xi, wi, b, **args), O.conv2d(xi, wi, b, **args), "vs oracle")


def test_depthwise_of_more_tiles_than_a_grid_holds(ctx, case):
    """A tile of this geometry holds four outputs: 2^24 of them are 2^32 threads."""
    rows, cols, apart = 2000, 33600, 2000
    case(f"depthwise [1,1,{rows + apart},{cols}], 2 x 1, dilation {apart}")
    x = RNG.integers(-3, 4, size=(1, 1, rows + apart, cols)).astype(np.float32)
    got = ctx.conv2d(x, np.array([2.0, -3.0], np.float32).reshape(1, 1, 2, 1), None, dilations=(apart, 1))
    assert np.array_equal(got, 2.0 * x[:, :, :rows] - 3.0 * x[:, :, apart:])


def test_max_pool(ctx, case):
    case("maxpool")
    x = RNG.standard_normal((2, 5, 33, 31)).astype(np.float32)
    x[0, 0, 0, 0] = np.nan
    for kernel, strides, pads in [((2, 2), (2, 2), (0, 0, 0, 0)), ((3, 3), (2, 2), (1, 1, 1, 1)), ((3, 2), (1, 3), (0, 1, 2, 0)), ((33, 31), (1, 1), (0, 0, 0, 0))]:
        assert_bits_equal(ctx.max_pool(x, kernel, strides, pads), O.max_pool(x, kernel, strides, pads), f"maxpool {kernel} {strides} {pads}")
    lowest = np.full((1, 1, 2, 2), np.finfo(np.float32).min, np.float32)
    assert_bits_equal(ctx.max_pool(lowest, (2, 2), (2, 2)), np.zeros((1, 1, 1, 1), np.float32), "f32::MIN window")


def test_vit_patch_embedding_and_cnn_stem_through_the_session(case):
    case("session: Conv -> Reshape -> Transpose (ViT tokens); Conv SAME_UPPER -> Relu -> MaxPool")
    x = RNG.integers(-2, 3, size=(2, 3, 32, 32)).astype(np.float32)
    w = RNG.integers(-2, 3, size=(24, 3, 8, 8)).astype(np.float32)
    b = RNG.integers(-2, 3, size=24).astype(np.float32)
    m = Model(opset_version=13)
    v = m.new_val_named_and_shaped("x", x.shape)
    c, r, t = m.new_val(), m.new_val(), m.new_val()
    m.add_node(Op.Conv2d, [v, m.new_initializer(w), m.new_initializer(b)], [c], kernel_shape=[8, 8], strides=[8, 8])
    m.add_node(Op.Reshape, [c, m.new_initializer(np.array([2, 24, 16], np.int64))], [r])
    m.add_node(Op.Transpose, [r], [t], perm=[0, 2, 1])
    m.add_input(v)
    m.add_output(t)
    (tokens,) = HipSessionBuilder(m).build().run([x])
    want = direct_conv(x, w, b, (8, 8), (0, 0, 0, 0), (1, 1), 1).astype(np.float32).reshape(2, 24, 16).transpose(0, 2, 1)
    assert_bits_equal(tokens, want, "patch tokens")

    x2 = RNG.integers(-2, 3, size=(1, 3, 15, 17)).astype(np.float32)
    w2 = RNG.integers(-2, 3, size=(8, 3, 3, 3)).astype(np.float32)
    m = Model(opset_version=13)
    v = m.new_val_named_and_shaped("x", x2.shape)
    c, a, p = m.new_val(), m.new_val(), m.new_val()
    m.add_node(Op.Conv2d, [v, m.new_initializer(w2)], [c], kernel_shape=[3, 3], strides=[2, 2], auto_pad="SAME_UPPER")
    m.add_node(Op.ReLU, [c], [a])
    m.add_node(Op.MaxPool, [a], [p], kernel_shape=[2, 2], strides=[2, 2])
    m.add_input(v)
    m.add_output(p)
    (got,) = HipSessionBuilder(m).build().run([x2])
    # SAME_UPPER for 15x17, k 3, s 2: out 8x9, total pad 2 -> (1,1) and 2 -> (1,1)  (shape.rs:48-61)
    conv = direct_conv(x2, w2, None, (2, 2), (1, 1, 1, 1), (1, 1), 1).astype(np.float32)
    assert conv.shape == (1, 8, 8, 9)
    assert_bits_equal(got, O.max_pool(np.maximum(conv, 0), (2, 2), (2, 2)), "cnn stem")


def test_resize(ctx, case):
    case("resize")
    x = RNG.standard_normal((2, 3, 13, 17)).astype(np.float32)
    for out_hw in [(26, 34), (13, 17), (39, 51), (20, 25), (6, 8), (1, 1)]:
        for nearest in (True, False):
            assert_bits_equal(ctx.resize(x, out_hw, nearest), O.resize(x, out_hw, nearest), f"resize {out_hw} nearest={nearest}")
    # through the session, with `scales` (3 inputs) and with `sizes` (4 inputs)
    for extra, mode in (([np.zeros(0, np.float32), np.array([1, 1, 2, 2], np.float32)], "nearest"),
                        ([np.zeros(0, np.float32), np.zeros(0, np.float32), np.array([2, 3, 30, 40], np.int64)], "linear")):
        m = Model(opset_version=13)
        v = m.new_val_named_and_shaped("x", x.shape)
        y = m.new_val()
        m.add_node(Op.Resize, [v] + [m.new_initializer(e) for e in extra], [y], mode=mode, coordinate_transformation_mode="asymmetric",
                   nearest_mode="floor")
        m.add_input(v)
        m.add_output(y)
        (got,) = HipSessionBuilder(m).build().run([x])
        want = O.resize(x, (26, 34), True) if mode == "nearest" else O.resize(x, (30, 40), False)
        assert_bits_equal(got, want, f"session resize {mode}")


def test_more_groups_than_a_grid_has_rows(ctx, case):
    groups = 65535 + 7
    case(f"conv2d of {groups} groups of two channels")
    x = RNG.integers(-3, 4, size=(2, 2 * groups, 1, 3)).astype(np.float32)
    w = RNG.integers(-3, 4, size=(groups, 2, 1, 1)).astype(np.float32)
    bias = RNG.integers(-3, 4, size=groups).astype(np.float32)
    want = (x.reshape(2, groups, 2, 1, 3) * w[None, :, :, :, :]).sum(axis=2) + bias[None, :, None, None]
    assert_bits_equal(ctx.conv2d(x, w, bias, group=groups), want, "against the definition")
