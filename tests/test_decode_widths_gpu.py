"""Decode on the GEMV where a width is not a multiple of 256: the last unit of a row is partly past its end, in each
format of 32-value blocks, for the gate / up (hidden), the down (expert width) and the shared expert's down, at the
widths around a unit's edges (one 64 past it, one short of it) and the benchmark's own (1408, 2880). Widths that the prefill
tiles do not take (below 320) stay on the MFMA decode tiles."""

import numpy as np
import pytest

from oracle import layers, moe_ref

from .helpers import check_pairs_f64, gpu_input, gpu_layer, rel_l2

pytestmark = pytest.mark.gpu

Spec = layers.Spec
CASES = [
    (Spec("ds", H=2048, E=64, k=6, F=1408, gate_type="Q4_K", down_type="Q8_0", scale=2e-4, dmin_scale=1.5e-3,
          shared_F=2816, shared_type="Q4_K"), (1, 8, 42)),
    (Spec("wide", H=2880, E=8, k=2, F=2880, gate_type="Q8_0", down_type="Q8_0", scale=0.01, router="uniform"), (1, 5, 16)),
    (Spec("q4_0", H=320, E=16, k=4, F=448, gate_type="Q4_0", down_type="Q4_0", scale=0.02, x_dtype="f32"), (1, 16)),
    (Spec("q4_1", H=576, E=16, k=4, F=320, gate_type="Q4_1", down_type="IQ4_NL", scale=4e-3, x_dtype="f32",
          shared_F=448, shared_type="IQ4_NL", shared_down_type="Q4_1", shared_gated=True), (2, 16)),
]


@pytest.mark.parametrize(("spec", "tokens"), CASES, ids=[s.name for s, _ in CASES])
def test_partial_units(spec: Spec, tokens: tuple) -> None:
    layer = layers.make_layer(spec, 3)
    with gpu_layer(layer, max_tokens=max(tokens)) as g:
        for T in tokens[::-1] + tokens[:1]:  # (down and up in size: what a pass leaves behind does not reach the next)
            x = layers.make_x(spec, T, T)
            y = g(gpu_input(spec, x))
            assert "router_quant" in g.kernel_names(), g.kernel_names()
            ids, w = g.tap("ids"), g.tap("weights")
            rids, rw = moe_ref.moe_route(layers.logits(layer, x), spec.k)
            assert np.array_equal(ids, rids) and np.allclose(w, rw, rtol=1e-6)
            # int8 hi / lo planes hold a group's values to max |x| / 65024: a few 1e-5 of relative error
            assert rel_l2(y, layers.forward_f64(layer, x, ids, w)) < 1e-4, (spec.name, T)
            h = g.tap("h")
            order = g.tap("order")
            e = int(ids.reshape(-1)[order[0]])
            gw, uw, _ = (m.astype(np.float64) for m in layers.expert(layer)(e))
            xt = x.astype(np.float64)[order[0] // spec.k]
            a = xt @ gw.T
            assert rel_l2(h[0], a / (1 + np.exp(-a)) * (xt @ uw.T)) < 1e-4, (spec.name, T)


NARROW = [
    (Spec("w192", H=2048, E=16, k=4, F=192, gate_type="Q4_0", down_type="Q4_0", scale=0.02), (1, 16)),
    (Spec("h64", H=64, E=4, k=1, F=192, gate_type="Q8_0", down_type="Q4_0", scale=0.02), (3, 16)),
    (Spec("h192", H=192, E=16, k=4, F=1408, gate_type="Q4_1", down_type="IQ4_NL", scale=4e-3, x_dtype="f32"), (2, 16)),
    (Spec("f128", H=320, E=16, k=4, F=128, gate_type="IQ4_NL", down_type="Q8_0", scale=4e-3, shared_F=448,
          shared_type="Q8_0"), (2, 16)),
]


@pytest.mark.parametrize(("spec", "tokens"), NARROW, ids=[s.name for s, _ in NARROW])
def test_narrow_widths(spec: Spec, tokens: tuple) -> None:
    """Below the prefill tiles' widths decode holds x and h in bf16 hi + lo planes (2^-17 a value; bf16 x exactly): a pair's
    output is off by at most three such roundings (x in the gate and the up product, h), 2.3e-5, and the layer's, over many
    pairs, by less than 1e-5, where XQ (2^-16 of a group's largest) gives about 4.5e-5."""
    layer = layers.make_layer(spec, 3)
    with gpu_layer(layer, max_tokens=max(tokens)) as g:
        for T in tokens:
            x = layers.make_x(spec, T, T)
            y = g(gpu_input(spec, x))
            ids, w = g.tap("ids"), g.tap("weights")
            assert rel_l2(y, layers.forward_f64(layer, x, ids, w)) < 1e-5, (spec.name, T)
            check_pairs_f64(g, layer, x, g.tap("offsets"), g.tap("order"), list(range(spec.E)), 3 * 2.0**-17)
