"""The streamed small tiles (past the GEMV's sizes, up to a few dozen pairs per expert) against float64 math, in every
block format: token counts around the line between tiles of 16 and of 32 rows and the first and last that take them,
widths of partial K-units and of partial 64-row blocks, tiles of one row and of a full one (uneven routing)."""

import numpy as np
import pytest

from oracle import layers

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
TOKENS = (17, 56, 57, 152)


@pytest.mark.parametrize("spec", CASES, ids=[s.name for s in CASES])
def test_stream_tiles(spec: Spec) -> None:
    layer = layers.make_layer(spec, 7)
    # (uneven: expert 0 far ahead, expert 1 behind, so that tiles of every size come up)
    layer.router[0] += 0.08
    layer.router[1] -= 0.08
    with gpu_layer(layer, max_tokens=max(TOKENS)) as g:
        for T in TOKENS + TOKENS[:1]:
            x = np.abs(layers.make_x(spec, T, T))
            y = g(gpu_input(spec, x))
            names = g.kernel_names()
            assert "prefill_x" in names and "router_quant" not in names, names
            taps = check_against_oracle(g, layer, x, y)
            counts = g.tap("counts")
            # h and the pair outputs: fp16 x (fp32 x rounded once), h rounded once (2^-11 each at most)
            check_pairs_f64(g, layer, x, taps["offsets"], taps["order"], list(np.flatnonzero(counts)), 1e-3)
            assert rel_l2(y, layers.forward_f64(layer, x, taps["ids"], taps["weights"])) < 1e-3, (spec.name, T)
            assert np.array_equal(g(gpu_input(spec, x)).view(np.uint32), y.view(np.uint32)), (spec.name, T)
