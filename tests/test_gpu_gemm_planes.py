"""Products of a session with weights kept as bf16 planes (csrc/device/gemm_planes.h) at the edges of their tiles, against float64: no
further off than the fp32 kernel, and fp32 arithmetic's result for infinite, NaN, huge and denormal operand values."""
import contextlib
import ctypes
import threading

import numpy as np
import pytest

from altius_amd import device as D
from altius_amd.graph import Model, Op, Tensor
from altius_amd.session import HipSessionBuilder
from test_gpu_graph_replay import hip_runtime

pytestmark = pytest.mark.gpu


def product(rows, k, n, w, gemm=None, views=True):
    """x [rows, k] times the weights; gemm: (trans_b, bias) of a Gemm instead of a MatMul."""
    m = Model(opset_version=13)
    x, y = m.new_val_named_and_shaped("x", [rows, k]), m.new_val()
    m.add_input(x)
    if gemm is None:
        m.add_node(Op.MatMul, [x, m.new_initializer(w)], [y])
    else:
        m.add_node(Op.Gemm, [x, m.new_initializer(np.ascontiguousarray(w.T) if gemm[0] else w), m.new_initializer(gemm[1])], [y], trans_b=gemm[0])
    m.add_output(y)
    return HipSessionBuilder(m).with_strided_views(views).build()


def fp32_kernel(a, w):
    with D.Context(0) as ctx:
        return ctx.matmul(a, w)


# Rows at the edges of 64- and 128-row tiles and one past them; values of k that are no whole groups of 64, no whole float4s, and long enough
# to be cut; columns that are no whole 32, 64 or 128.
SIZES = [(1024, 768, 768), (1025, 768, 3072), (1089, 3072, 772), (4095, 772, 770), (3153, 770, 1537), (6304, 768, 768), (2049, 3076, 801), (8200, 381, 1000)]


@pytest.mark.parametrize("rows,k,n", SIZES)
def test_as_close_as_the_fp32_kernel(case, rows, k, n):
    case(f"[{rows},{k}] x [{k},{n}]")
    rng = np.random.default_rng(rows + k)
    a = rng.standard_normal((rows, k)).astype(np.float32)
    w = (rng.standard_normal((k, n)) * 0.05).astype(np.float32)
    session = product(rows, k, n, w)
    (got,) = session.run([a])
    (again,) = session.run([a])
    assert np.array_equal(got, again)
    some = np.unique(np.concatenate([np.arange(0, rows, 37), [rows - 1]]))
    want = a[some].astype(np.float64) @ w.astype(np.float64)
    plain = fp32_kernel(a, w)
    assert not np.array_equal(got, plain), "these sizes are meant to take the planes"
    off, off32 = np.linalg.norm(got[some] - want), np.linalg.norm(plain[some] - want)
    assert off <= off32
    # Three dropped terms below 2^-25 of a product each; at most a chain of k / 16 + 1 additions to the larger sums and five times as many to
    # the ones 2^-8 of them, each off by 2^-23 of what they add to; eight sums that meet behind them.
    bound = (3 * 2.0**-25 + (k / 16 + 1 + 8) * (1 + 5 * 2.0**-8) * 2.0**-23) * (np.abs(a[some]).astype(np.float64) @ np.abs(w).astype(np.float64))
    assert (np.abs(got[some] - want) <= bound).all()


# Sums of one sign, where roundings toward zero would add up: all four tiles (64 x 64, 64 x 128, 128 x 128 in two chains of k and in one).
@pytest.mark.parametrize("rows,k,n", [(1024, 3072, 768), (6304, 768, 768), (6304, 3072, 768), (6304, 768, 3072)])
@pytest.mark.parametrize("operands", ["unit", "relu", "equal"])
def test_sums_of_one_sign(case, rows, k, n, operands):
    case(f"{operands} operands, [{rows},{k}] x [{k},{n}]")
    rng = np.random.default_rng(4)
    if operands == "unit":
        a, w = rng.random((rows, k), dtype=np.float32), rng.random((k, n), dtype=np.float32)
    elif operands == "relu":
        a, w = np.maximum(rng.standard_normal((rows, k), dtype=np.float32), 0), np.abs(rng.standard_normal((k, n), dtype=np.float32))
    else:
        a, w = np.full((rows, k), 1.1, np.float32), np.full((k, n), 1.3, np.float32)
    some = np.unique(np.concatenate([np.arange(0, rows, 101), [rows - 1]]))
    want = a[some].astype(np.float64) @ w.astype(np.float64)
    got, plain = product(rows, k, n, w).run([a])[0][some], fp32_kernel(a, w)[some]
    assert np.linalg.norm(got - want) <= np.linalg.norm(plain - want)


@pytest.mark.parametrize("rows,k,n", [(77, 768, 16384), (129, 771, 16390)])
def test_few_rows_and_many_columns(case, rows, k, n):
    test_as_close_as_the_fp32_kernel(case, rows, k, n)


@pytest.mark.parametrize("rows,k,n", [(256, 768, 3072), (512, 3072, 768), (788, 1536, 384)])
def test_sizes_that_weights_from_memory_hold_up_stay_on_the_fp32_kernel(case, rows, k, n):
    case(f"[{rows},{k}] x [{k},{n}]")
    rng = np.random.default_rng(rows)
    a, w = (rng.standard_normal(s).astype(np.float32) for s in ((rows, k), (k, n)))
    assert np.array_equal(product(rows, k, n, w).run([a])[0], fp32_kernel(a, w))


@pytest.mark.parametrize("trans_b", [False, True])
def test_gemm_with_bias(case, trans_b):
    case(f"Gemm, trans_b {trans_b}")
    rng = np.random.default_rng(3)
    a, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((1100, 768), (768, 1500), (1500,)))
    (got,) = product(1100, 768, 1500, w, gemm=(trans_b, b)).run([a])
    (plain,) = product(1100, 768, 1500, w).run([a])
    assert np.array_equal(got, plain + b)


@pytest.mark.parametrize("rows,k,n", [(1100, 768, 1500), (1025, 771, 3070), (1089, 3072, 772)])
def test_every_operand_value(case, rows, k, n):
    case(f"infinite, NaN, huge and denormal operands, [{rows},{k}] x [{k},{n}]")
    rng = np.random.default_rng(5)
    a = rng.standard_normal((rows, k)).astype(np.float32)
    w = (rng.standard_normal((k, n)) * 0.05).astype(np.float32)
    a[3, 17], a[700, k - 1], a[rows - 1, 0], a[65, 40] = np.inf, -np.inf, np.inf, np.nan
    a[129, :] = 0
    a[129, 5], a[200, 9] = 3e38, -2e36
    a[300] *= np.float32(1e-38)
    a[301] *= np.float32(2.0**-100)
    w[:, 7] *= np.float32(2.0**-20)
    (got,) = product(rows, k, n, w).run([a])
    with np.errstate(over="ignore", invalid="ignore"):
        want = a.astype(np.float64) @ w.astype(np.float64)
        magnitude = np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64)
        want32 = want.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want32))
    infinite = np.isinf(want32)
    assert infinite[[3, 700, rows - 1]].all() and np.array_equal(got[infinite], want32[infinite])
    finite = np.isfinite(want32)
    # fp32 arithmetic: k roundings, each of 2^-24 or, below the smallest normal number, of a whole denormal.
    assert (np.abs(got[finite] - want[finite]) <= k * (2.0**-24 * magnitude + 2.0**-149)[finite]).all()
    assert not np.array_equal(got[finite], fp32_kernel(a, w)[finite]), "these sizes are meant to take the planes"
    assert not np.isfinite(product(rows, k, n, np.full_like(w, np.inf)).run([np.ones_like(a)])[0]).any()


def test_a_view_has_the_bits_of_its_copy(case):
    """Half of a Split's columns, read in place or copied first."""
    case("a strided view of the first operand")
    rng = np.random.default_rng(6)
    x, w = rng.standard_normal((4, 300, 1536)).astype(np.float32), (rng.standard_normal((768, 768)) * 0.05).astype(np.float32)

    def build(views):
        m = Model(opset_version=13)
        v = m.new_val_named_and_shaped("x", list(x.shape))
        m.add_input(v)
        left, right, y, z = (m.new_val() for _ in range(4))
        m.add_node(Op.Split, [v, m.new_initializer(np.array([768, 768], np.int64))], [left, right], axis=2)
        m.add_node(Op.MatMul, [right, m.new_initializer(w)], [y])
        m.add_node(Op.MatMul, [left, m.new_initializer(w)], [z])  # an output of the graph would have the Split copy
        m.add_output(y)
        m.add_output(z)
        return HipSessionBuilder(m).with_strided_views(views).build()

    views, copies = build(True), build(False)
    (in_place, left), (copied, left_copied) = views.run([x]), copies.run([x])
    assert views.copies_avoided() > copies.copies_avoided() == 0
    assert np.array_equal(in_place, copied) and np.array_equal(left, left_copied)
    assert not np.array_equal(left.reshape(1200, 768), fp32_kernel(np.ascontiguousarray(x[..., :768]).reshape(1200, 768), w)), "these sizes are meant to take the planes"
    assert np.array_equal(in_place.reshape(1200, 768), product(1200, 768, 768, w).run([np.ascontiguousarray(x[..., 768:]).reshape(1200, 768)])[0])


@pytest.mark.parametrize("shape,axis", [((4, 1, 600, 768), 2), ((4, 1, 1, 600, 768), 3), ((1, 4, 600, 768), 2), ((4, 600, 768), 1), ((2, 600, 1, 768), 1), ((4, 1, 300, 1536), 3),
                                        ((1, 1, 1200, 1536), 3)])
def test_parts_of_a_split_read_in_place(case, shape, axis):
    """Parts along the rows, behind axes of extent 1 too, start further apart than their rows go; parts along the columns do not."""
    case(f"both halves of a Split of {shape} along axis {axis}")
    rng = np.random.default_rng(7)
    x, w = rng.standard_normal(shape).astype(np.float32), (rng.standard_normal((768, 768)) * 0.05).astype(np.float32)
    half = shape[axis] // 2

    def build(views):
        m = Model(opset_version=13)
        v = m.new_val_named_and_shaped("x", list(shape))
        m.add_input(v)
        parts, products = [m.new_val(), m.new_val()], [m.new_val(), m.new_val()]
        m.add_node(Op.Split, [v, m.new_initializer(np.array([half, half], np.int64))], parts, axis=axis)
        for part, y in zip(parts, products):
            m.add_node(Op.MatMul, [part, m.new_initializer(w)], [y])
            m.add_output(y)
        return HipSessionBuilder(m).with_strided_views(views).build()

    in_place, copied = build(True), build(False)
    got, plain = in_place.run([x]), copied.run([x])
    assert in_place.copies_avoided() > copied.copies_avoided() == 0
    for y, z, part in zip(got, plain, np.split(x, 2, axis)):
        want, magnitude = part.astype(np.float64) @ w.astype(np.float64), np.abs(part).astype(np.float64) @ np.abs(w).astype(np.float64)
        # fp32 arithmetic: k roundings of 2^-24 each
        assert (np.abs(y - want) <= 768 * 2.0**-24 * magnitude).all() and (np.abs(z - want) <= 768 * 2.0**-24 * magnitude).all()


@pytest.mark.parametrize("b,t,c,n,planes", [(64, 196, 512, 256, False), (16, 1024, 768, 512, False), (32, 300, 1088, 770, False), (16, 1024, 768, 2048, True)])
def test_a_transposed_first_operand_counts_its_copy(case, b, t, c, n, planes):
    """Tokens mixed by a product over the middle axis: the fp32 kernel reads the Transpose's input where it lies, as it does with weights that
    are an input of the graph; by planes the tall operand is copied first, which few products are worth."""
    case(f"Transpose(0,2,1) of [{b},{t},{c}], then [{t},{n}]")
    rng = np.random.default_rng(8)
    x, w = rng.standard_normal((b, t, c)).astype(np.float32), (rng.standard_normal((t, n)) * 0.05).astype(np.float32)

    def build(constant, views=True):
        m = Model(opset_version=13)
        v = m.new_val_named_and_shaped("x", [b, t, c])
        m.add_input(v)
        weights = m.new_initializer(w) if constant else m.new_val_named_and_shaped("w", [t, n])
        if not constant:
            m.add_input(weights)
        turned, y = m.new_val(), m.new_val()
        m.add_node(Op.Transpose, [v], [turned], perm=[0, 2, 1])
        m.add_node(Op.MatMul, [turned, weights], [y])
        m.add_output(y)
        return HipSessionBuilder(m).with_strided_views(views).build()

    (got,) = build(True).run([x])
    assert np.array_equal(got, build(False).run([x, w])[0]) != planes
    if planes:
        assert np.array_equal(got, build(True, views=False).run([x])[0])
    some = np.arange(0, c, 37)
    assert np.abs(got[::7, some] - np.swapaxes(x[::7], 1, 2)[:, some].astype(np.float64) @ w).max() < 1e-4


@pytest.mark.parametrize("b,t,k,n,planes", [(8, 128, 768, 768, False), (12, 256, 384, 768, False), (32, 197, 768, 768, True), (8, 128, 768, 3072, True)])
def test_a_transpose_behind_counts_its_copy(case, b, t, k, n, planes):
    """A product whose result a Transpose reads is written in that layout by the fp32 kernel; planes are taken where they save more than the copy costs."""
    case(f"[{b},{t},{k}] x [{k},{n}], then Transpose(1,0,2)")
    rng = np.random.default_rng(9)
    x, w = rng.standard_normal((b, t, k)).astype(np.float32), (rng.standard_normal((k, n)) * 0.05).astype(np.float32)

    def build(constant, views=True):
        m = Model(opset_version=13)
        v = m.new_val_named_and_shaped("x", [b, t, k])
        m.add_input(v)
        weights = m.new_initializer(w) if constant else m.new_val_named_and_shaped("w", [k, n])
        if not constant:
            m.add_input(weights)
        y, turned = m.new_val(), m.new_val()
        m.add_node(Op.MatMul, [v, weights], [y])
        m.add_node(Op.Transpose, [y], [turned], perm=[1, 0, 2])
        m.add_output(turned)
        return HipSessionBuilder(m).with_strided_views(views).build()

    session = build(True)
    (got,), (plain,) = session.run([x]), build(False).run([x, w])
    assert np.array_equal(got, plain) != planes and session.copies_avoided() == (0 if planes else 1)
    if planes:
        assert np.array_equal(got, build(True, views=False).run([x])[0])
    assert np.abs(got[::5] - np.swapaxes(x, 0, 1)[::5].astype(np.float64) @ w).max() < 1e-4


def weights_and_room(rows, k, n, w):
    """rows of x times w, and the largest of `room` ones: a run that needs as much memory as its second input says."""
    m = Model(opset_version=13)
    x, shape = m.new_val_named_and_shaped("x", [rows, k]), m.new_val_named("shape")
    y, ones, z = m.new_val(), m.new_val(), m.new_val()
    m.add_input(x)
    m.add_input(shape)
    m.add_node(Op.MatMul, [x, m.new_initializer(w)], [y])
    m.add_node(Op.Expand, [m.new_initializer(np.ones(1, np.float32)), shape], [ones])
    m.add_node(Op.ReduceMax, [ones], [z], axes=[0, 1], keep_dims=1)
    m.add_output(y)
    m.add_output(z)
    return HipSessionBuilder(m)


def free_memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip_runtime().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@contextlib.contextmanager
def memory_left(nbytes):
    """All of the GPU's memory but that much is taken."""
    with D.Context(0) as holder:
        for least in (0, 64 << 20):  # the first one leaves more than what it was asked for
            if free_memory() > nbytes + least:
                holder.alloc(free_memory() - nbytes)
        yield


def test_planes_give_way_to_what_a_run_needs(case):
    """1 GiB of weights have 1.5 GiB of planes; a run that needs more than is left otherwise does without them, and so do later ones."""
    case("planes go when a run finds no memory")
    rng = np.random.default_rng(10)
    rows, k, n = 128, 8192, 32768
    x, w = rng.standard_normal((rows, k)).astype(np.float32), rng.standard_normal((k, n), dtype=np.float32)
    plain = fp32_kernel(x, w)
    session = weights_and_room(rows, k, n, w).build()
    small = np.array([4, 256], np.int64)
    assert not np.array_equal(session.run([x, small])[0], plain), "this size is meant to take the planes"
    with memory_left(1 << 30):
        for shape in (np.array([2048, 1 << 18], np.int64), small):  # 2 GiB
            y, z = session.run([x, shape])
            assert np.array_equal(y, plain) and np.array(z).ravel() == [1.0]


def test_planes_leave_room_for_what_comes_behind(case):
    """Planes take a third of what is free when a session is built, or are not made."""
    case("planes are not made where memory is short")
    rng = np.random.default_rng(11)
    rows, k, n = 128, 8192, 32768
    x, w = rng.standard_normal((rows, k)).astype(np.float32), rng.standard_normal((k, n), dtype=np.float32)
    plain = fp32_kernel(x, w)
    with memory_left(9 << 29):  # 4.5 GiB
        y, _ = weights_and_room(rows, k, n, w).build().run([x, np.array([4, 256], np.int64)])
    assert np.array_equal(y, plain)


def test_lanes_share_the_planes(case):
    """A further lane has its own copy of the weights and reads the first one's planes; when one lane needs their memory, all go on without."""
    case("planes of a session with lanes")
    rng = np.random.default_rng(12)
    rows, k, n = 128, 8192, 32768
    x, w = rng.standard_normal((rows, k)).astype(np.float32), rng.standard_normal((k, n), dtype=np.float32)
    small = np.array([4, 256], np.int64)
    plain = fp32_kernel(x, w)
    session = weights_and_room(rows, k, n, w).build()
    (by_planes, _), wrong = session.run([x, small]), []
    before = free_memory()

    def several(callers, runs, wanted):
        together = threading.Barrier(callers)

        def work():
            together.wait()
            try:
                for _ in range(runs):
                    y, _ = session.run([x, small])
                    if not any(np.array_equal(y, z) for z in wanted):
                        wrong.append(y)
            except Exception as e:  # noqa: BLE001 - reported below, in the main thread
                wrong.append(repr(e))

        threads = [threading.Thread(target=work) for _ in range(callers)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()

    several(2, 10, [by_planes])
    assert session.lanes() == 2 and not wrong, wrong
    assert before - free_memory() < 1.5 * w.nbytes
    with memory_left(1 << 30):  # (a third caller's lane would take the memory for its weights)
        other = threading.Thread(target=several, args=(1, 4, [by_planes, plain]))
        other.start()
        y, z = session.run([x, np.array([2048, 1 << 18], np.int64)])  # 2 GiB
        other.join()
        assert np.array_equal(y, plain) and not wrong, wrong
        several(2, 2, [plain])
        assert session.lanes() == 2
    assert not wrong, wrong


def test_recorded_launches_go_with_the_planes(case):
    """Lane 0 replays what it has recorded; a second lane finds no memory for its values and the planes go: lane 0 records anew."""
    case("planes of a session that replays, given back by another lane")
    rng = np.random.default_rng(13)
    rows, k, n = 16384, 4096, 16384
    x, w = rng.random((rows, k), dtype=np.float32) - np.float32(0.5), rng.random((k, n), dtype=np.float32) - np.float32(0.5)
    plain = fp32_kernel(x, w)
    m = Model(opset_version=13)
    v, y = m.new_val_named_and_shaped("x", [rows, k]), m.new_val()
    m.add_input(v)
    m.add_node(Op.MatMul, [v, m.new_initializer(w)], [y])
    m.add_output(y)
    session = HipSessionBuilder(m).with_graph_replay(True).build()
    for _ in range(3):
        (by_planes,) = session.run([x])
    assert session.graph_replays() and not np.array_equal(by_planes, plain)
    # The lane's weights and x take 0.5 GiB of 1.3, the product 1 GiB more, the planes have 0.4.
    together, wrong, right, held = threading.Barrier(2), [], [], Tensor.from_numpy(x)

    def work():
        together.wait()
        try:
            for _ in range(100):  # until two of them have overlapped, and a few more
                if session.lanes() == 2 and len(right) >= 4:
                    break
                some = session.run([held], copy=False)[0][::61]
                (right if np.array_equal(some, by_planes[::61]) or np.array_equal(some, plain[::61]) else wrong).append(1)
        except Exception as e:  # noqa: BLE001 - reported below, in the main thread
            wrong.append(repr(e))

    with memory_left(1331 << 20):
        threads = [threading.Thread(target=work) for _ in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert right and not wrong, wrong
        assert session.lanes() == 2
        for _ in range(4):
            assert np.array_equal(session.run([x])[0][::7], plain[::7])
