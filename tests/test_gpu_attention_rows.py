"""Attention as one kernel: the bits of its nodes run apart, in every form of scale, condition and mask, at the edges of its tiles and
for every order of sums that the products alone would have; and apart after all where an operand is not one that the kernel takes."""
import ctypes

import numpy as np
import pytest

from altius_amd import device as D
from altius_amd._lib import AltiusHipError
from altius_amd.graph import Model, Op
from altius_amd.session import HipSessionBuilder
from conftest import assert_bits_equal
from test_gpu_graph_replay import hip_runtime

pytestmark = pytest.mark.gpu


def attention(b, h, tq, tk, d=64, scale="div", cond=None, mask=(1, 1, 1, "k"), value_late=False, k_form="transposed", seen=False, rewritten=True):
    """Inputs q [b, tq, h d], kv [b, tk, 2 h d], and cond / mask where asked for; the result [b, tq, h d]."""
    m = Model(opset_version=13)
    shapes = {"q": [b, tq, h * d], "kv": [b, tk, 2 * h * d]}
    ext = {"b": b, "h": h, "q": tq, "k": tk}
    for name, dims in (("cond", cond), ("mask", mask)):
        if dims:
            shapes[name] = [ext.get(x, x) for x in dims]
    v = {name: m.new_val_named_and_shaped(name, dims) for name, dims in shapes.items()}
    for x in v.values():
        m.add_input(x)

    def op(kind, inputs, n=1, **attrs):
        outs = [m.new_val() for _ in range(n)]
        m.add_node(kind, inputs, outs, **attrs)
        return outs[0] if n == 1 else outs

    i64 = lambda *a: m.new_initializer(np.array(a, np.int64))  # noqa: E731
    f32 = lambda a: m.new_initializer(np.array(a, np.float32))  # noqa: E731
    heads = lambda x, t, perm: op(Op.Transpose, [op(Op.Reshape, [x, i64(b, t, h, d)])], perm=perm)  # noqa: E731
    k, val = op(Op.Split, [v["kv"], i64(h * d, h * d)], 2, axis=2)
    q = heads(v["q"], tq, [0, 2, 1, 3])
    k = heads(k, tk, [0, 2, 3, 1]) if k_form == "transposed" else op(Op.Transpose, [heads(k, tk, [0, 2, 1, 3])], perm=[0, 1, 3, 2])
    if not value_late:
        val = heads(val, tk, [0, 2, 1, 3])
    s = op(Op.MatMul, [q, k])
    by = {"div": lambda: op(Op.Div, [s, f32(np.sqrt(d) + 0.1)]), "mul": lambda: op(Op.Mul, [f32(0.11), s]), "power": lambda: op(Op.Div, [s, f32(8.0)])}
    if scale:
        s = by[scale]()
    if cond:
        s = op(Op.Where, [op(Op.Greater, [v["cond"], f32(0.0)]), s, f32(-1e4)])
    if mask:
        s = op(Op.Add, [s, v["mask"]])
    p = op(Op.Softmax, [s], axis=-1)
    if value_late:  # not there yet when the first product is due
        val = heads(op(Op.Mul, [val, f32(1.0)]), tk, [0, 2, 1, 3])
    o = op(Op.MatMul, [p, val])
    if seen:
        m.add_output(p)
    m.add_output(op(Op.Reshape, [op(Op.Transpose, [o], perm=[0, 2, 1, 3]), i64(b, tq, h * d)]))
    if rewritten:
        m.fuse_softmax_prologue()
        m.fuse_transpose_matmul()
    return m, shapes


def has_kernel(heads, tq, tk):
    """More than one head, two to 448 keys (a single key's matrix reads as a column), and the operators' sums in an order that the kernel
    has: not the Softmax of rows that whole wavefronts take (whole 128-byte lines that fill three quarters of their loads), not the
    products of many small matrices."""
    whole_wavefronts = tk % 32 == 0 and 4 * tk >= 3 * (-(-tk // 256) * 256)
    small_matrices = heads >= 128 and tq <= 208
    return heads > 1 and 1 < tk <= 448 and not whole_wavefronts and not small_matrices


def check(case, b, h, tq, tk, taken=True, **form):
    case(f"attention b {b} h {h} tq {tq} tk {tk} {form}")
    m, shapes = attention(b, h, tq, tk, **form)
    rng = np.random.default_rng(tq + tk)
    x = {name: rng.standard_normal(dims).astype(np.float32) for name, dims in shapes.items()}
    if "mask" in x:
        x["mask"] = np.where(rng.random(x["mask"].shape) < 0.2, -1e4, 0.1 * x["mask"]).astype(np.float32)
    together, apart = HipSessionBuilder(m).build(), HipSessionBuilder(m).with_strided_views(False).build()
    for _ in range(2):
        got, ops = together.run(list(x.values())), apart.run(list(x.values()))
        for g, o in zip(got, ops):
            assert_bits_equal(g, o, "one kernel and the nodes apart")
        assert apart.fused_attentions() == 0
        assert together.fused_attentions() == (1 if taken and has_kernel(b * h, tq, tk) else 0)


# edges of tiles of 32 queries and keys, of turns of 16, 32 and 64 keys and of the lanes of a row; one key, as many as LDS holds and more
@pytest.mark.parametrize("tq,tk", [(1, 1), (1, 65), (5, 16), (16, 17), (17, 63), (33, 64), (77, 77), (31, 128), (48, 129), (64, 192), (15, 193), (197, 197),
                                   (20, 256), (257, 257), (16, 321), (40, 447), (40, 449), (7, 600)])
def test_sizes(case, tq, tk):
    assert D.attention_rows_fits(6, tq, tk) == has_kernel(6, tq, tk)
    check(case, 2, 3, tq, tk)


# many heads and few: products of 32 x 32, 64 x 64 and 128 x 64 tiles, and small matrices of one block each (from 128 heads on)
@pytest.mark.parametrize("b,h", [(1, 2), (1, 12), (3, 16), (8, 12), (127, 1), (16, 12), (60, 12)])
@pytest.mark.parametrize("tq,tk", [(50, 50), (77, 77), (128, 128), (197, 197), (300, 211), (64, 400)])
def test_orders_of_sums(case, b, h, tq, tk):
    check(case, b, h, tq, tk, scale="power")


@pytest.mark.parametrize("scale", [None, "div", "mul", "power"])
@pytest.mark.parametrize("cond", [None, (1, 1, "q", "k"), ("b", 1, 1, "k"), ("b", "h", "q", 1)])
@pytest.mark.parametrize("mask", [(1, 1, 1, "k"), ("b", 1, 1, "k"), (1, "h", "q", "k"), ("k",), ("b", 1, "q", 1)])
def test_forms(case, scale, cond, mask):
    check(case, 2, 3, 37, 45, scale=scale, cond=cond, mask=mask)


@pytest.mark.parametrize("form", [dict(mask=None), dict(mask=None, scale="power"), dict(value_late=True), dict(k_form="twice"), dict(seen=True), dict(rewritten=False), dict(d=32), dict(d=128)])
@pytest.mark.parametrize("b,h", [(1, 1), (1, 4), (3, 1), (5, 2)])
def test_operands_and_readers(case, b, h, form):
    check(case, b, h, 50, 70, taken=not form.get("seen") and form.get("d", 64) == 64, **form)


def test_rows_without_a_finite_score(case):
    """Minus infinity for every key of some rows, infinite values and NaN: what the nodes run apart give."""
    case("attention with infinities")
    m, shapes = attention(2, 2, 20, 40, mask=("b", 1, "q", "k"))
    rng = np.random.default_rng(3)
    x = {name: rng.standard_normal(dims).astype(np.float32) for name, dims in shapes.items()}
    x["mask"][:] = 0
    x["mask"][0, 0, 3] = -np.inf
    x["mask"][1, 0, 5, 7:] = -np.inf
    x["mask"][1, 0, 6, 2] = np.nan
    x["mask"][1, 0, 8] = np.finfo(np.float32).min
    x["kv"][1, 39, 70 * 2 - 1] = np.inf
    together, apart = HipSessionBuilder(m).build(), HipSessionBuilder(m).with_strided_views(False).build()
    got, want = together.run(list(x.values()))[0], apart.run(list(x.values()))[0]
    assert_bits_equal(got, want, "one kernel and the nodes apart")
    assert together.fused_attentions() == 1


@pytest.mark.parametrize("shared", ["keys", "values", "both"])
@pytest.mark.parametrize("heads,t", [(12, 77), (40, 200), (3, 50)])
def test_heads_that_share_keys_or_values(case, shared, heads, t):
    """One [t, 64] matrix for all heads: its product is one of all heads' rows, and the nodes run apart after they were held."""
    case(f"{heads} heads of {t} share {shared}")
    m = Model(opset_version=13)
    one, own = [64, t], [1, heads, 64, t]
    shapes = [[1, heads, t, 64], own if shared == "values" else one, [1, heads, t, 64] if shared == "keys" else [t, 64]]
    q, k, v = (m.new_val_named_and_shaped(n, s) for n, s in zip("qkv", shapes))
    for x in (q, k, v):
        m.add_input(x)
    s, s2, p, v2, o = (m.new_val() for _ in range(5))
    m.add_node(Op.MatMul, [q, k], [s])
    m.add_node(Op.Div, [s, m.new_initializer(np.array(8.0, np.float32))], [s2])
    m.add_node(Op.Softmax, [s2], [p], axis=-1)
    m.add_node(Op.Mul, [v, m.new_initializer(np.array(1.0, np.float32))], [v2])
    m.add_node(Op.MatMul, [p, v2], [o])
    m.add_output(o)
    rng = np.random.default_rng(t)
    x = [rng.standard_normal(d).astype(np.float32) for d in shapes]
    together, apart = HipSessionBuilder(m).build(), HipSessionBuilder(m).with_strided_views(False).build()
    for _ in range(2):
        assert_bits_equal(together.run(x)[0], apart.run(x)[0], "held and run apart, and apart")
        assert together.fused_attentions() == 0


@pytest.mark.parametrize("tq,tk", [(77, 77), (197, 197), (40, 447)])
def test_no_scores_in_memory(case, tq, tk):
    """Where the probabilities are asked for the nodes run apart, which takes blocks for the scores and for them."""
    allocations = []
    for seen in (False, True):
        case(f"blocks of an attention, tq {tq} tk {tk}, probabilities an output: {seen}")
        m, shapes = attention(1, 12, tq, tk, seen=seen)
        session = HipSessionBuilder(m).build()
        session.run([np.zeros(dims, np.float32) for dims in shapes.values()])
        allocations.append(session.device_allocations())
    assert allocations[0] < allocations[1]


@pytest.mark.parametrize("fused", [False, True])
def test_a_run_that_fails_between_the_products(case, fused):
    """The values' product, due when the first product's nodes already hold their operands, broadcasts in a way that is refused: the run
    raises, and the session gives all its memory back when it goes."""
    case(f"attention whose values cannot be computed, one-kernel attention allowed: {fused}")
    tq, tk = 1 << 16, 50
    m = Model(opset_version=13)
    shapes = [[2, 3, tq, 64], [2, 3, 64, tk], [2, 1, tk, 8], [1, 3, 8, 64]]
    q, k, a, b = (m.new_val_named_and_shaped(n, s) for n, s in zip("qkab", shapes))
    for x in (q, k, a, b):
        m.add_input(x)
    s, p, v, o = (m.new_val() for _ in range(4))
    m.add_node(Op.MatMul, [q, k], [s])
    m.add_node(Op.Softmax, [s], [p], axis=-1)
    m.add_node(Op.MatMul, [a, b], [v])
    m.add_node(Op.MatMul, [p, v], [o])
    m.add_output(o)
    hip = hip_runtime()

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    x = [np.zeros(d, np.float32) for d in shapes]
    before = []
    for _ in range(3):
        session = HipSessionBuilder(m).with_fused_attention(fused).build()
        before.append(free_bytes())
        with pytest.raises(AltiusHipError, match="broadcast against each other partially"):
            session.run(x)
        session.close()
    assert before[0] - before[2] < x[0].nbytes // 2, "device memory that a failed run kept"


def test_replayed(case):
    case("attention in a recorded graph")
    m, shapes = attention(2, 3, 33, 50, cond=(1, 1, "q", "k"))
    session = HipSessionBuilder(m).with_graph_replay(True).build()
    eager = HipSessionBuilder(m).build()
    for seed in range(5):
        rng = np.random.default_rng(seed)
        x = [rng.standard_normal(dims).astype(np.float32) for dims in shapes.values()]
        assert_bits_equal(session.run(x)[0], eager.run(x)[0], "recorded and not")
        assert session.fused_attentions() == eager.fused_attentions() == 1
    assert session.graph_replays() > 0
