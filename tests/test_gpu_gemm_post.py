"""A Relu, Gelu or residual Add behind a Gemm, with and without a Reshape between them: the session that has the product's kernel do
it returns the bits of the session that runs the nodes apart, and leaves apart what it cannot take along."""
import numpy as np
import pytest

from altius_amd import device as D
from altius_amd.graph import Model, Op
from altius_amd.session import HipSessionBuilder
from conftest import assert_bits_equal

pytestmark = pytest.mark.gpu

# b, t, k, n: one tile, ragged tiles, k cut into slices, larger tiles
SIZES = [(1, 1, 4, 4), (2, 33, 20, 35), (1, 77, 3072, 768), (4, 256, 64, 3072)]


def graph(b, t, k, n, after, reshape, form, trans):
    rng = np.random.default_rng(k)
    const = lambda *s: m.new_initializer(rng.standard_normal(s).astype(np.float32))  # noqa: E731
    m = Model(opset_version=13)
    x = m.new_val_named_and_shaped("x", [b * t, k])
    shape = [b, t, n] if reshape else [b * t, n]
    r = m.new_val_named_and_shaped("r", {"row": [n], "wide": [2] + shape}.get(form, shape))
    y, z = m.new_val(), m.new_val()
    m.add_input(x)
    m.add_input(r)
    w = const(n, k) if trans else const(k, n)
    m.add_node(Op.Gemm, [x, w, const(n)], [y], trans_b=trans, alpha=0.5, beta=2.0)
    v = y
    if reshape:
        v = m.new_val()
        m.add_node(Op.Reshape, [y, m.new_initializer(np.array(shape, np.int64))], [v])
    if after == Op.Add:
        m.add_node(Op.Add, [r, v] if form == "second" else [v, r], [z])
    else:
        u = m.new_val()
        m.add_node(after, [v], [u])
        m.add_node(Op.Add, [u, r], [z])
    if form == "twice":  # another reader of the product
        q = m.new_val()
        m.add_node(Op.Mul, [v, z], [q])
        m.add_output(q)
    if form == "seen":
        m.add_output(v)
    m.add_output(z)
    return m


@pytest.mark.parametrize("after", [Op.Add, Op.ReLU, Op.Gelu])
@pytest.mark.parametrize("reshape", [False, True])
@pytest.mark.parametrize("form", ["first", "second", "row", "wide", "twice", "seen"])
def test_behind_a_gemm(case, after, reshape, form):
    for b, t, k, n in SIZES:
        for trans in (0, 1):
            case(f"gemm {b, t, k, n} trans_b {trans}, {after}, reshape {reshape}, {form}")
            m = graph(b, t, k, n, after, reshape, form, trans)
            rng = np.random.default_rng(9)
            x = rng.standard_normal((b * t, k)).astype(np.float32)
            shape = [b, t, n] if reshape else [b * t, n]
            r = rng.standard_normal({"row": [n], "wide": [2] + shape}.get(form, shape)).astype(np.float32)
            together, apart = HipSessionBuilder(m).build(), HipSessionBuilder(m).with_strided_views(False).build()
            for _ in range(2):
                got = together.run([x, r])
                for a, w in zip(got, apart.run([x, r])):
                    assert_bits_equal(a, w, "the nodes together and apart")
            if form in ("first", "second") or (form in ("row", "wide") and after != Op.Add):
                assert together.copies_avoided() > apart.copies_avoided()


@pytest.mark.parametrize("after", [Op.Add, Op.Gelu])
# slices of 64 x 64 and of 128 x 128 blocks, ragged; 128 x 128 blocks behind which an activation follows, 128 x 64 where none does
@pytest.mark.parametrize("t,k,n", [(551, 1481, 2305), (1411, 6162, 2516), (4301, 100, 4304)])
def test_behind_a_gemm_of_other_tiles(case, after, t, k, n):
    case(f"gemm {t, k, n}, {after}")
    m = graph(1, t, k, n, after, False, "first", 0)
    rng = np.random.default_rng(13)
    x, r = (rng.standard_normal(d).astype(np.float32) for d in ((t, k), (t, n)))
    together, apart = HipSessionBuilder(m).build(), HipSessionBuilder(m).with_strided_views(False).build()
    assert_bits_equal(together.run([x, r])[0], apart.run([x, r])[0], "the nodes together and apart")
    assert together.copies_avoided() > apart.copies_avoided()


@pytest.mark.parametrize("product", ["MatMul", "Gemm", "Gemm and Reshape"])
def test_behind_a_residual_that_is_still_owed(case, product):
    """s = a + b stands in front of a LayerNormalization that leaves the sum to its own kernel, which runs behind the product
    (its scale is computed by a later node): the product's kernel must not read s before anybody has written it."""
    case(f"{product} + a sum that waits for a LayerNormalization")
    b, t, k, n, wide = 2, 512, 64, 768, 3072
    rows, rng = b * t, np.random.default_rng(11)
    normal = lambda *shape: rng.standard_normal(shape).astype(np.float32)  # noqa: E731
    m = Model(opset_version=17)
    const = lambda *shape: m.new_initializer(normal(*shape))  # noqa: E731

    def op(kind, inputs, **attrs):
        out = m.new_val()
        m.add_node(kind, inputs, [out], **attrs)
        return out

    shape = [rows, n] if product == "Gemm" else [b, t, n]
    u_shape = [b, t, k] if product == "MatMul" else [rows, k]
    shapes = {"a": shape, "b": shape, "u": u_shape, "p": [n], "q": [n]}
    v = {name: m.new_val_named_and_shaped(name, dims) for name, dims in shapes.items()}
    for x in v.values():
        m.add_input(x)
    s = op(Op.Add, [v["a"], v["b"]])
    if product == "MatMul":
        g = op(Op.MatMul, [v["u"], const(k, n)])
    else:
        g = op(Op.Gemm, [v["u"], const(k, n), const(n)])
        if product != "Gemm":
            g = op(Op.Reshape, [g, m.new_initializer(np.array(shape, np.int64))])
    y = op(Op.Add, [g, s])
    gamma = op(Op.Add, [v["p"], v["q"]])
    h = op(Op.LayerNormalization, [s, gamma, const(n)], axis=-1)
    z = op(Op.MatMul, [h, const(n, wide)])
    m.add_output(y)
    m.add_output(z)
    sessions = [HipSessionBuilder(m).with_gemm_algorithm(D.GEMM_AUTO).with_strided_views(views).build() for views in (True, False)]
    for _ in range(3):
        inputs = [normal(*dims) for dims in shapes.values()]
        (y0, z0), (y1, z1) = (x.run(inputs) for x in sessions)
        assert_bits_equal(y0, y1, "the product and the sum")
        assert_bits_equal(z0, z1, "the product behind the LayerNormalization")
