"""The streamed small tiles (past the GEMV's sizes, up to a few dozen pairs per expert) against float64 math, in every
block format: token counts around the lines between tiles of 16, 32 and 64 rows and the first and last that take them,
widths of partial K-units and of partial 64-row blocks, tiles of one row and of a full one (uneven routing); a shared expert
beside them on either side of its own line; workgroups of several items each."""

from dataclasses import replace

import numpy as np
import pytest

from oracle import gguf_ref, layers

from .helpers import check_against_oracle, check_pairs_f64, gpu_input, gpu_layer, rel_l2

pytestmark = pytest.mark.gpu

Spec = layers.Spec
# (hidden and expert width; token counts: more than 4 pairs per expert, up to 14 (tiles of 16 rows), up to 38 (of 32))
CASES = [
    Spec("q4_0", H=448, E=8, k=2, F=336 + 48, gate_type="Q4_0", down_type="Q8_0", scale=0.02),
    Spec("q8_0", H=576, E=8, k=2, F=320, gate_type="Q8_0", down_type="Q4_0", scale=0.01, x_dtype="f32"),
    Spec("q4_1", H=320, E=8, k=2, F=448, gate_type="Q4_1", down_type="IQ4_NL", scale=4e-3, x_dtype="f32"),
    Spec("iq4_nl", H=704, E=8, k=2, F=512, gate_type="IQ4_NL", down_type="Q4_1", scale=4e-3),
    Spec("q4_k", H=512, E=8, k=2, F=768, gate_type="Q4_K", down_type="Q6_K", scale=2e-4, dmin_scale=1.5e-3),
    Spec("q5_k", H=768, E=8, k=2, F=512, gate_type="Q5_K", down_type="Q3_K", scale=1e-4, dmin_scale=1e-3),
    Spec("q6_k", H=512, E=8, k=2, F=512, gate_type="Q6_K", down_type="IQ4_XS", scale=5e-5),
    Spec("q3_k", H=512, E=8, k=2, F=512, gate_type="Q3_K", down_type="Q5_K", scale=1e-4, dmin_scale=1e-3),
    Spec("iq4_xs", H=512, E=8, k=2, F=512, gate_type="IQ4_XS", down_type="Q4_K", scale=5e-5, dmin_scale=1.5e-3),
]
# (pairs per expert that layers of this size stream up to in tiles of 32 rows, and the formats with tiles of 64 past 32 pairs)
LAST_32, LAST_64 = 38, {"Q4_0": 41, "Q4_K": 45, "Q8_0": 54}
CASES_64 = [
    CASES[0], CASES[1],
    Spec("q4_k", H=512, E=8, k=2, F=512, gate_type="Q4_K", down_type="Q8_0", scale=2e-4, dmin_scale=1.5e-3),
    Spec("q8_0_only", H=448, E=8, k=2, F=576, gate_type="Q8_0", down_type="Q8_0", scale=0.01),
]
# (a shared expert beside streamed routed ones: on the streamed dense rows up to 256 tokens, then on the prefill tiles; 16
# experts, whose few logits leave no near tie among 63 to 65 tokens, where one is more than the oracle's check allows)
SHARED = Spec("shared", H=512, E=16, k=2, F=384, gate_type="Q4_0", down_type="Q8_0", scale=0.02, shared_F=448,
              shared_type="Q8_0", shared_down_type="Q4_0", shared_gated=True)


def tiles(spec: Spec, T: int) -> str:
    """The variant of the products' names that these cases are made for, by formats and pairs per expert."""
    pairs, by64 = T * spec.k / spec.E, {spec.gate_type, spec.down_type} <= set(LAST_64)
    if by64 and pairs > 32:
        return "@stream64" if pairs <= min(LAST_64[spec.gate_type], LAST_64[spec.down_type]) else ""
    return "" if pairs > LAST_32 else "@stream16" if pairs <= 14 else "@stream32"


@pytest.mark.parametrize(("spec", "tokens"),
                         [(s, (17, 56, 57, 4 * LAST_32)) for s in CASES]
                         + [(s, (128, 129, n := 4 * min(LAST_64[s.gate_type], LAST_64[s.down_type]), n + 1)) for s in CASES_64]
                         + [(replace(SHARED, x_dtype=x), (63, 64, 65, 256, 257)) for x in ("bf16", "f32")])
def test_stream_tiles(spec: Spec, tokens: tuple) -> None:
    layer = layers.make_layer(spec, 7)
    # (uneven: expert 0 far ahead, expert 1 behind, so that tiles of every size come up)
    layer.router[0] += 0.08
    layer.router[1] -= 0.08
    with gpu_layer(layer, max_tokens=max(tokens)) as g:
        for T in tokens + tokens[:1]:
            x = np.abs(layers.make_x(spec, T, T))
            y = g(gpu_input(spec, x))
            names = g.kernel_names()
            assert "prefill_x" in names and ("gate_up" + tiles(spec, T)) in names and ("down" + tiles(spec, T)) in names, names
            if spec.shared_F:
                assert ("shared_down@stream" in names) == (T <= 256), names
                sg, su, sd = (gguf_ref.dequantize(q, m, c).astype(np.float64) for q, m, c in
                              zip((spec.shared_type, spec.shared_type, spec.sdown_type), layer.shared,
                                  (spec.H, spec.H, spec.shared_F)))
                a = x.astype(np.float64) @ sg.T
                ys = (a / (1 + np.exp(-a)) * (x.astype(np.float64) @ su.T)) @ sd.T
                # (streamed: x, in the gate and the up product, and h to 2^-17; prefill: h and the weights to 2^-11)
                assert rel_l2(g.tap("y_shared"), ys) < (3 * 2.0**-17 if T <= 256 else 1e-3), T
            taps = check_against_oracle(g, layer, x, y)
            counts = g.tap("counts")
            # h and the pair outputs: fp16 x (fp32 x rounded once), h rounded once (2^-11 each at most)
            check_pairs_f64(g, layer, x, taps["offsets"], taps["order"], list(np.flatnonzero(counts)), 1e-3)
            assert rel_l2(y, layers.forward_f64(layer, x, taps["ids"], taps["weights"])) < 1e-3, (spec.name, T)
            assert np.array_equal(g(gpu_input(spec, x)).view(np.uint32), y.view(np.uint32)), (spec.name, T)


MANY = [(Spec("q4_0", H=1024, E=64, k=8, F=1024, gate_type="Q4_0", down_type="Q4_0", scale=0.02), 288, "@stream64"),
        (Spec("q4_k", H=1024, E=64, k=8, F=1024, gate_type="Q4_K", down_type="Q4_K", scale=2e-4, dmin_scale=1.5e-3), 288,
         "@stream64"),
        (Spec("q8_0", H=1024, E=64, k=8, F=1024, gate_type="Q8_0", down_type="Q8_0", scale=0.01, x_dtype="f32"), 288,
         "@stream64"),
        # (8 waves a workgroup: 128 rows of gate and up, 256 of the down)
        (Spec("q6_k", H=1024, E=64, k=8, F=1024, gate_type="Q6_K", down_type="Q6_K", scale=5e-5), 150, "@stream32")]


@pytest.mark.parametrize(("spec", "T", "variant"), MANY, ids=[s.name for s, _, _ in MANY])
def test_stream_many_items(spec: Spec, T: int, variant: str) -> None:
    """More items than resident workgroups (one or two a CU, 256 CUs; 512 items of gate and up and more): each takes several in
    turn, an item's loads issued under the one before it."""
    layer = layers.make_layer(spec, 9)
    with gpu_layer(layer, max_tokens=T) as g:
        x = layers.make_x(spec, T, 4)
        y = g(gpu_input(spec, x))
        names = g.kernel_names()
        assert "gate_up" + variant in names and "down" + variant in names, names
        check_pairs_f64(g, layer, x, g.tap("offsets"), g.tap("order"), list(range(0, spec.E, 4)) + [spec.E - 1], 1e-3)
        # (the layer's output: every token's pairs by slot, as the taps hold them)
        w, slot = g.tap("weights"), g.tap("slot").reshape(T, spec.k)
        yp = g.tap("y_pairs")
        assert rel_l2(y, np.einsum("ti,tih->th", w, yp[slot])) < 1e-6
        for _ in range(3):
            assert np.array_equal(g(gpu_input(spec, x)).view(np.uint32), y.view(np.uint32))
