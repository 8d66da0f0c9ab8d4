"""What stands behind a convolution and is done while its result is written (BatchNormalization, an activation, a residual Add),
an average pool in one kernel, and a hard swish behind an element-wise chain: the bits of the nodes run apart."""
import numpy as np
import pytest

from altius_amd import device as D
from altius_amd import graphs
from altius_amd.graph import Model, Op
from altius_amd.session import HipSessionBuilder
from conftest import assert_bits_equal

pytestmark = pytest.mark.gpu

# batch, channels, image, output channels, kernel, stride, group: every kernel a convolution may take, ragged
GEOMETRIES = [
    (1, 6, 9, 6, 3, 1, 6),       # depthwise, one output per thread
    (8, 240, 23, 240, 5, 1, 240),  # depthwise, four outputs per thread
    (2, 5, 11, 10, 2, 1, 5),     # depthwise, general kernel, two outputs per channel
    (1, 19, 7, 21, 1, 1, 1),     # tiles of 16 x 16
    (1, 3, 21, 17, 3, 2, 1),
    (4, 8, 13, 12, 3, 1, 2),     # groups
    (32, 16, 57, 70, 1, 1, 1),   # tiles of 32 x 32 or larger
    (16, 3, 113, 67, 3, 2, 1),
    (32, 96, 14, 576, 1, 1, 1),
    (32, 512, 14, 511, 1, 1, 1),  # products of the images as they lie
    (2, 256, 33, 192, 3, 1, 1),  # unfolded
]
AFTER = ["relu", "hard_sigmoid", "hard_swish", "add", "norm", "norm relu", "norm hard_swish", "norm add", "relu seen"]


def hard_swish(m, v):
    s, out = m.new_val(), m.new_val()
    m.add_node(Op.HardSigmoid, [v], [s], alpha=1.0 / 6.0, beta=0.5)
    m.add_node(Op.Mul, [v, s], [out])
    return out


def graph(b, c, size, oc, k, stride, group, after, bias):
    rng = np.random.default_rng(oc + k)
    const = lambda *s: m.new_initializer(rng.standard_normal(s).astype(np.float32))  # noqa: E731
    m = Model(opset_version=13)
    side = (size + 2 * (k // 2) - k) // stride + 1
    x, r = m.new_val_named_and_shaped("x", [b, c, size, size]), m.new_val_named_and_shaped("r", [b, oc, side, side])
    m.add_input(x)
    m.add_input(r)

    def op(kind, inputs, **attrs):
        out = m.new_val()
        m.add_node(kind, inputs, [out], **attrs)
        return out

    conv = v = op(Op.Conv2d, [x, const(oc, c // group, k, k)] + ([const(oc)] if bias else []), kernel_shape=[k, k], strides=[stride, stride], pads=[k // 2] * 4,
                  group=group)
    for kind in after.split():
        if kind == "norm":
            var = m.new_initializer((0.5 + rng.random(oc)).astype(np.float32))
            v = op(Op.BatchNormalization, [v, const(oc), const(oc), const(oc), var], epsilon=1e-5)
        elif kind == "relu":
            v = op(Op.ReLU, [v])
        elif kind == "hard_sigmoid":
            v = op(Op.HardSigmoid, [v], alpha=0.2, beta=0.5)
        elif kind == "hard_swish":
            v = hard_swish(m, v)
        elif kind == "add":
            v = op(Op.Add, [v, r])
        else:  # "seen": the convolution's own result is asked for
            m.add_output(conv)
    m.add_output(v)
    m.fuse_elemwise_ops(extended=True)
    return m, (b, c, size, size), (b, oc, side, side)


@pytest.mark.parametrize("after", AFTER)
@pytest.mark.parametrize("geometry", GEOMETRIES)
def test_behind_a_convolution(case, geometry, after):
    case(f"conv {geometry}, {after}")
    m, x_dims, r_dims = graph(*geometry, after, bias=geometry[3] % 2 == 0)
    rng = np.random.default_rng(5)
    x, r = (3 * rng.standard_normal(d).astype(np.float32) for d in (x_dims, r_dims))
    together, apart = HipSessionBuilder(m).build(), HipSessionBuilder(m).with_strided_views(False).build()
    for _ in range(2):
        for a, w in zip(together.run([x, r]), apart.run([x, r])):
            assert_bits_equal(a, w, "the nodes together and apart")
    assert apart.copies_avoided() == 0
    if after != "relu seen":  # the last two geometries are products, which have no normalisation
        assert together.copies_avoided() == (0 if "norm" in after and geometry in GEOMETRIES[-2:] else len(after.split()))


# Pointwise convolutions whose products would take longer than the kernels that read x in place (those do a normalisation along), and
# some whose products are faster.
@pytest.mark.parametrize("geometry,in_place", [((30, 48, 14, 144, 1, 1, 1), True), ((31, 40, 15, 240, 1, 1, 1), True), ((44, 96, 7, 576, 1, 1, 1), True),
                                               ((8, 40, 16, 240, 1, 1, 1), True), ((29, 144, 14, 48, 1, 1, 1), True), ((44, 138, 11, 89, 1, 1, 1), True),
                                               ((41, 576, 6, 96, 1, 1, 1), False), ((7, 383, 42, 421, 1, 1, 1), False)])
def test_small_images_are_read_in_place(case, geometry, in_place):
    case(f"conv {geometry}, norm")
    m, x_dims, r_dims = graph(*geometry, "norm", bias=True)
    rng = np.random.default_rng(8)
    x, r = (3 * rng.standard_normal(d).astype(np.float32) for d in (x_dims, r_dims))
    together, apart = HipSessionBuilder(m).build(), HipSessionBuilder(m).with_strided_views(False).build()
    assert_bits_equal(together.run([x, r])[0], apart.run([x, r])[0], "the nodes together and apart")
    assert together.copies_avoided() == (1 if in_place else 0)


# From 128 images on a product of small ones without a bias is the kernel of many small matrices, in one chunk of k and in several.
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("after", ["relu", "hard_swish", "add"])
@pytest.mark.parametrize("geometry", [(128, 64, 14, 192, 1, 1, 1), (128, 1024, 7, 192, 1, 1, 1), (144, 64, 14, 200, 1, 1, 1), (127, 64, 14, 192, 1, 1, 1)])
def test_behind_products_of_many_images(case, geometry, after, bias):
    case(f"conv {geometry}, {after}, bias {bias}")
    m, x_dims, r_dims = graph(*geometry, after, bias=bias)
    rng = np.random.default_rng(6)
    x, r = (3 * rng.standard_normal(d).astype(np.float32) for d in (x_dims, r_dims))
    together, apart = HipSessionBuilder(m).build(), HipSessionBuilder(m).with_strided_views(False).build()
    assert_bits_equal(together.run([x, r])[0], apart.run([x, r])[0], "the nodes together and apart")
    assert together.copies_avoided() == (1 if bias or geometry[0] < 128 else 0)


def test_norm_whose_scale_an_input_replaces(case):
    """An initializer that is an input of the graph too: the run's value counts."""
    case("conv, BatchNormalization with a scale that is an input")
    m = Model(opset_version=13)
    x = m.new_val_named_and_shaped("x", [1, 3, 9, 9])
    m.add_input(x)
    rng = np.random.default_rng(2)
    const = lambda *s: m.new_initializer(rng.random(s).astype(np.float32) + np.float32(0.5))  # noqa: E731
    c, y, scale = m.new_val(), m.new_val(), const(5)
    m.add_input(scale)
    m.add_node(Op.Conv2d, [x, const(5, 3, 3, 3)], [c], kernel_shape=[3, 3], pads=[1] * 4)
    m.add_node(Op.BatchNormalization, [c, scale, const(5), const(5), const(5)], [y], epsilon=1e-5)
    m.add_output(y)
    feed = [rng.standard_normal((1, 3, 9, 9)).astype(np.float32), np.arange(5, dtype=np.float32)]
    together, apart = HipSessionBuilder(m).build(), HipSessionBuilder(m).with_strided_views(False).build()
    got = together.run(feed)[0]
    assert_bits_equal(got, apart.run(feed)[0], "the nodes together and apart")
    assert np.ptp(got[0, 0]) == 0.0  # scaled by the input's zero


# planes below and above every kernel that row sums take, rows that start anywhere, few planes that are cut into parts
@pytest.mark.parametrize("planes,side", [(3, 1), (5, 2), (70, 4), (40, 7), (3, 14), (9, 16), (12, 28), (6, 33), (4, 56), (3, 64), (2, 113), (1, 301)])
def test_average_pool(case, ctx, planes, side):
    case(f"average pool of {planes} planes of {side} x {side}")
    x = np.random.default_rng(side).standard_normal((1, planes, side, side)).astype(np.float32)
    m = graphs.single_input_model([1, planes, side, side], lambda m, v: pooled(m, v))
    sums = ctx.reduce(D.REDUCE_SUM, x, planes, side * side, 1)
    got = HipSessionBuilder(m).build().run([x])[0]
    assert_bits_equal(got.reshape(planes), sums.reshape(planes) / np.float32(side * side), "one kernel, and a sum that is then divided")


def pooled(m, v):
    out = m.new_val()
    m.add_node(Op.GlobalAveragePool, [v], [out])
    return out


@pytest.mark.parametrize("side", [1, 7, 12, 14])
@pytest.mark.parametrize("steps", [1, 2, 15, 16])
def test_hard_swish_behind_a_chain(case, side, steps):
    """x * HardSigmoid(s), more steps behind it up to as many as a kernel takes, then a hard swish."""
    case(f"chain of {steps + 1} steps on planes of {side} x {side}, then a hard swish")
    m = Model(opset_version=13)
    b, c = 3, 10
    x, s = m.new_val_named_and_shaped("x", [b, c, side, side]), m.new_val_named_and_shaped("s", [b, c, 1, 1])
    m.add_input(x)
    m.add_input(s)
    v = m.new_val()
    m.add_node(Op.HardSigmoid, [s], [v], alpha=1.0 / 6.0, beta=0.5)
    half = m.new_initializer(np.array(0.75, np.float32))
    for k in range(steps):
        u = m.new_val()
        m.add_node(Op.Mul if k == 0 else Op.Add, [v, x if k == 0 else half], [u])
        v = u
    m.add_output(hard_swish(m, v))
    m.fuse_elemwise_ops(extended=True)
    rng = np.random.default_rng(side)
    inputs = [3 * rng.standard_normal(d).astype(np.float32) for d in ((b, c, side, side), (b, c, 1, 1))]
    inputs[0].flat[:3] = [np.inf, -np.inf, np.nan]
    together, apart = HipSessionBuilder(m).build(), HipSessionBuilder(m).with_strided_views(False).build()
    assert_bits_equal(together.run(inputs)[0], apart.run(inputs)[0], "the swish in the chain's kernel and behind it")
