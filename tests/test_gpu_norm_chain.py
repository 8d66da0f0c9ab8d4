"""A written-out LayerNormalization in a session that runs the graph as it stands: one kernel where nobody sees the steps between,
the nine operators elsewhere.  Rows of small whole numbers over a power of two have exact sums, so there every rounding of the nine
steps is checked to the bit; other rows against the oracle's nine steps."""
import numpy as np
import pytest

import oracle as O
from altius_amd.graph import Model, Op
from altius_amd.graphs import layer_norm_chain
from altius_amd.session import HipSessionBuilder
from conftest import assert_bits_equal, assert_close

pytestmark = pytest.mark.gpu


def nine_steps(x, gamma, beta, eps):
    mean = O.reduce(O.REDUCE_MEAN, x, [x.ndim - 1], True)
    d = O.binary(O.SUB, x, mean)
    var = O.reduce(O.REDUCE_MEAN, O.binary(O.POW, d, np.array(2.0, np.float32)), [x.ndim - 1], True)
    s = O.unary(O.SQRT, O.binary(O.ADD, var, np.array(eps, np.float32)))
    return O.binary(O.ADD, O.binary(O.MUL, O.binary(O.DIV, d, s), gamma), beta)


def chain(shape, gamma, beta, eps, see=None):
    """see: a step's output that is an output of the graph as well (0: the mean ... 7: the product with gamma)."""
    m = Model()
    x = m.new_val_named_and_shaped("x", list(shape))
    m.add_input(x)
    out, _, _ = layer_norm_chain(m, x, gamma, beta, eps=eps)
    m.add_output(out)
    if see is not None:
        m.add_output(m.nodes()[see]["outputs"][0])
    return m


@pytest.mark.parametrize("length", [1, 4, 5, 64, 252, 256, 260, 768, 1028, 2052, 3072, 4096, 4100])
def test_lengths(case, length):
    case(f"norm chain length {length}")
    rng = np.random.default_rng(length)
    for rows in (1, 7):
        x = rng.standard_normal((rows, length)).astype(np.float32) * 3 + 1
        g, b = rng.standard_normal(length).astype(np.float32), rng.standard_normal(length).astype(np.float32)
        session = HipSessionBuilder(chain(x.shape, g, b, 1e-5)).build()
        (got,) = session.run([x])
        assert_close(got, nine_steps(x, g, b, 1e-5), what=f"{rows} rows")
        assert session.copies_avoided() == (8 if length % 4 == 0 and 32 < length < 4096 else 0), "one kernel for the nine steps"


@pytest.mark.parametrize("length", [4, 64, 256, 1024, 4096])
def test_every_rounding_where_the_sums_are_exact(case, length):
    case(f"norm chain bits, length {length}")
    rng = np.random.default_rng(length + 1)
    x = rng.integers(0, 4, size=(2, 3, length)).astype(np.float32)
    x[..., : length // 2] = 3 - x[..., length // 2:]  # mean 1.5, squares of halves
    x[1, 2] = 2.0                                     # variance 0
    g, b = rng.standard_normal(length).astype(np.float32), rng.standard_normal(length).astype(np.float32)
    session = HipSessionBuilder(chain(x.shape, g, b, 1e-5)).build()
    (got,) = session.run([x])
    assert_bits_equal(got, nine_steps(x, g, b, 1e-5), "result")
    assert session.copies_avoided() == (8 if 32 < length < 4096 else 0)


def test_infinities_and_zero_over_zero(case):
    case("norm chain: infinities, NaN, 0 / 0")
    x = np.ones((4, 256), np.float32)
    x[0, 3], x[1, 5], x[2, 7] = np.inf, -np.inf, np.nan
    g, b = np.full(256, 2.0, np.float32), np.full(256, 1.0, np.float32)
    (got,) = HipSessionBuilder(chain(x.shape, g, b, 0.0)).build().run([x])
    np.testing.assert_array_equal(np.isnan(got), np.isnan(nine_steps(x, g, b, 0.0)))


@pytest.mark.parametrize("see", [0, 1, 2, 5, 7])
def test_a_step_that_is_seen_keeps_the_operators(case, see):
    case(f"norm chain, step {see} is an output")
    rng = np.random.default_rng(3)
    x = rng.integers(0, 4, size=(5, 256)).astype(np.float32)
    g, b = rng.standard_normal(256).astype(np.float32), rng.standard_normal(256).astype(np.float32)
    plain = HipSessionBuilder(chain(x.shape, g, b, 1e-5)).build().run([x])[0]
    session = HipSessionBuilder(chain(x.shape, g, b, 1e-5, see)).build()
    got, step = session.run([x])
    assert session.copies_avoided() == 0
    assert_close(got, plain, what="result")
    assert step.size in (5, 5 * 256)


def test_scale_that_the_caller_may_replace_and_other_forms(case):
    case("norm chain: gamma as an input with a default, middle axis, exponent 3, squeezed mean")
    rng = np.random.default_rng(4)
    x = rng.standard_normal((4, 8, 8)).astype(np.float32)
    g, b = rng.standard_normal(8).astype(np.float32), rng.standard_normal(8).astype(np.float32)
    for axis, exponent in ((-1, 2.0), (2, 2.0), (1, 2.0), (-1, 3.0)):
        m = Model()
        v = m.new_val_named_and_shaped("x", list(x.shape))
        m.add_input(v)

        def op(kind, inputs, **attrs):
            out = m.new_val()
            m.add_node(kind, inputs, [out], **attrs)
            return out

        const = lambda a: m.new_initializer(np.asarray(a, np.float32))  # noqa: E731
        d = op(Op.Sub, [v, op(Op.ReduceMean, [v], axes=[axis], keep_dims=True)])
        var = op(Op.ReduceMean, [op(Op.Pow, [d, const(exponent)])], axes=[axis], keep_dims=True)
        s = op(Op.Sqrt, [op(Op.Add, [const([10.0]), var])])
        m.add_output(op(Op.Add, [const(b), op(Op.Mul, [const(g), op(Op.Div, [d, s])])]))
        session = HipSessionBuilder(m).build()
        (got,) = session.run([x])
        assert session.copies_avoided() == 0  # rows of 8 are too short, and the others are no such chain
        y = x.astype(np.float64)
        y = y - y.mean(axis, keepdims=True)
        want = y / np.sqrt((y ** exponent).mean(axis, keepdims=True) + 10.0) * g + b
        np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("shape", [(3, 16), (70, 32), (70, 36), (65, 252), (9, 256), (70, 288), (5, 300), (70, 300), (64, 1024), (66, 1028), (2, 3, 3072), (5, 4092)])
def test_bits_of_the_operators_run_one_by_one(case, shape):
    """The sums run in the order of the reduction kernels: the same bits as a profiled session, which runs every node."""
    case(f"norm chain against node by node {shape}")
    rng = np.random.default_rng(sum(shape))
    x = (rng.standard_normal(shape) * 2 - 1).astype(np.float32)
    g, b = rng.standard_normal(shape[-1]).astype(np.float32), rng.standard_normal(shape[-1]).astype(np.float32)
    together, apart = HipSessionBuilder(chain(shape, g, b, 1e-5)).build(), HipSessionBuilder(chain(shape, g, b, 1e-5)).with_profiling_enabled(True).build()
    assert_bits_equal(together.run([x])[0], apart.run([x])[0], "one kernel against nine")
    rows, length = int(np.prod(shape[:-1])), shape[-1]
    grouped = rows >= 64 and 256 < length <= 1024 and length % 32 != 0  # rows that the reduction adds up through LDS
    assert together.copies_avoided() == (8 if length > 32 and not grouped else 0) and apart.copies_avoided() == 0
