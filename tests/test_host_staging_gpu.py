"""The host-pointer calls on either side of what they stage through pinned memory (4 MiB each way) and of the parts a
routing call's tokens go in, against the oracle and against the same call in pieces; calls of several threads at once."""

import threading

import numpy as np
import pytest

from artlite_amd.moe import CHUNK, COLS
from artlite_amd.moe import plan as MP
from artlite_amd.moe import route as MR
from oracle import host_ref, layers

from .helpers import gpu_input, gpu_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(("T", "E", "k"), [(1, 32, 2), (1023, 128, 8), (1025, 128, 8), (8191, 128, 4), (8193, 128, 4),
                                           (40, 1000, 6),
                                           # (several parts, whose first and last rows share cache lines)
                                           (2100, 129, 8), (6001, 77, 5)])
def test_route_sizes(T: int, E: int, k: int) -> None:
    lg = np.random.default_rng(T).standard_normal((T, E)).astype(np.float32)
    ids, w = MP.route(lg, k)
    rids, rw = host_ref.moe_route(lg.reshape(-1), T, E, E, 0, E, k)
    assert np.array_equal(ids, rids)
    np.testing.assert_allclose(w, rw, rtol=1e-6)
    tids, tw = MR.top_k(lg, k)
    assert np.array_equal(tids, rids)
    np.testing.assert_allclose(tw, rw, rtol=1e-6)


def test_route_overlapping_rows() -> None:
    """Rows closer together than a token's logits reach: the reference's layout arguments allow it."""
    T, E, per_col, pitch, row = 700, 64, 16, 300, 20
    flat = np.random.default_rng(1).standard_normal((T - 1) * row + 3 * pitch + per_col).astype(np.float32)
    want = host_ref.moe_route(flat, T, row, per_col, pitch, E, 4)
    from artlite_amd import _hip

    c = _hip.ctypes
    ids, w = np.empty((T, 4), np.int32), np.empty((T, 4), np.float32)
    _hip.check(_hip.lib().artlite_moe_route(_hip.ptr(flat, c.c_float), flat.size, T, row, per_col, pitch, E, 4, 0,
                                            _hip.ptr(ids, c.c_int32), _hip.ptr(w, c.c_float)))
    assert np.array_equal(ids, want[0])
    np.testing.assert_allclose(w, want[1], rtol=1e-6)


@pytest.mark.parametrize(("T", "k", "E"), [(3, 2, 8), (20000, 8, 64), (60000, 8, 64)])
def test_plan_sizes(T: int, k: int, E: int) -> None:
    ids = np.argsort(np.random.default_rng(T).random((T, E)), axis=1)[:, :k].astype(np.int32)
    cap = -(-(E + -(-T * k // CHUNK)) // COLS)
    plan = MP.Plan.of(ids, cap=cap, E=E)
    ref = host_ref.moe_plan(ids, E, COLS, cap, CHUNK)
    assert plan.counts == ref["counts"].tolist() and np.array_equal(plan.pos, ref["pos"])
    for c in range(COLS):
        n = ref["counts"][c]
        assert np.array_equal(plan.experts[c], ref["experts"][c, :n])
        assert np.array_equal(plan.rows[c], ref["rows"][c, :n])


@pytest.mark.parametrize("x_dtype", ["bf16", "f32"])
def test_layer_call_sizes(x_dtype: str) -> None:
    """layer(x) at 1023 and 1025 tokens of 1024 values (an fp32 output on either side of 4 MiB) equals the same tokens
    staged, run and read, and what another thread's layer computes at the same time does not reach it."""
    spec = layers.Spec("call", H=1024, E=8, k=2, F=320, gate_type="Q8_0", down_type="Q8_0", scale=0.01, x_dtype=x_dtype)
    layer = layers.make_layer(spec, 0)
    with gpu_layer(layer, 1025) as g, gpu_layer(layer, 1025) as other:
        x2 = gpu_input(spec, layers.make_x(spec, 600, 5))
        want2 = other(x2)
        same = []

        def work() -> None:
            same.extend(np.array_equal(other(x2), want2) for _ in range(20))

        t = threading.Thread(target=work)
        t.start()
        for T in (1, 1023, 1025, 1022):
            x = gpu_input(spec, layers.make_x(spec, T, T))
            y = g(x)
            g.stage(x)
            g.run()
            assert np.array_equal(g.output().view(np.uint32), y.view(np.uint32)), T
        t.join()
        assert len(same) == 20 and all(same)
