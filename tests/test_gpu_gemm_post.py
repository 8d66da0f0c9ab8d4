"""A Relu, Gelu or residual Add behind a Gemm, with and without a Reshape between them: the session that has the product's kernel do
it returns the bits of the session that runs the nodes apart, and leaves apart what it cannot take along."""
import numpy as np
import pytest

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
