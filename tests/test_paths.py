"""Which kernels a pass takes, on the CPU: the names of a layer's kernels by format, widths and token count."""

from pathlib import Path

import pytest

from .fake_runtime import run_fake


@pytest.mark.parametrize(("H", "F", "fmt", "gemv"), [(2048, 192, "Q4_0", False), (64, 1408, "Q8_0", False),
                                                     (128, 128, "Q4_1", False), (192, 512, "IQ4_NL", False),
                                                     (2048, 320, "Q4_0", True), (2880, 2880, "Q8_0", True),
                                                     (256, 256, "Q4_0", True), (512, 256, "Q4_K", True)])
def test_decode_widths(tmp_path: Path, H: int, F: int, fmt: str, gemv: bool) -> None:
    """Decode of widths of partial units is the GEMV's where the prefill tiles take them, and stays on the MFMA decode
    tiles' bf16 planes below that; whole units of 256 are the GEMV's at any width."""
    run_fake(tmp_path, f"""
n = names(8, hidden={H}, n_experts=16, top_k=4, expert_ffn={F}, gate_type="{fmt}", down_type="{fmt}")
assert ("router_quant" in n) == {gemv} and "prefill_x" not in n, n
""")


@pytest.mark.parametrize(("H", "F"), [(1280, 2944), (320, 4032)])
def test_decode_of_many_wide_experts(tmp_path: Path, H: int, F: int) -> None:
    """1024 experts at 4 pairs each, more items than the GEMV's workgroups (one a CU at least) have table entries for: the
    pass takes the prefill tiles, as widths of partial units always did, and runs. One pair each stays on the GEMV."""
    run_fake(tmp_path, f"""
a = dict(hidden={H}, n_experts=1024, top_k=4, expert_ffn={F}, gate_type="Q8_0", down_type="Q8_0", max_tokens=1024)
with layer(**a) as L:
    for T, gemv in ((1024, False), (64, True)):
        L.stage(np.zeros((T, {H}), np.uint16))
        L.run()
        assert ("router_quant" in L.kernel_names()) == gemv, (T, L.kernel_names())
""")


def test_shared_expert_of_a_million_tokens(tmp_path: Path) -> None:
    """A shared expert narrower than the prefill tiles take, past the rows of one launch of the streamed dense rows."""
    run_fake(tmp_path, """
T = 65535 * 16 + 1
with layer(hidden=64, n_experts=4, top_k=1, expert_ffn=64, gate_type="Q8_0", down_type="Q8_0", shared_ffn=64,
           shared_type="Q8_0", max_tokens=T) as L:
    for n in (T - 1, T):
        L.stage(np.zeros((n, 64), np.uint16))
        L.run()
""")


@pytest.mark.parametrize(("gate", "down", "pairs"), [
    ("Q6_K", "Q6_K", 19), ("Q3_K", "Q3_K", 22), ("Q5_K", "Q5_K", 33), ("IQ4_XS", "IQ4_XS", 33), ("Q4_1", "Q4_1", 33),
    ("IQ4_NL", "IQ4_NL", 34), ("Q4_K", "Q6_K", 36), ("Q5_K", "Q6_K", 22), ("Q4_0", "Q6_K", 22), ("Q3_K", "Q4_K", 29),
    ("Q6_K", "Q4_0", 23), ("Q4_K", "Q5_K", 38), ("Q4_0", "Q4_0", 41), ("Q4_K", "Q4_K", 45), ("Q8_0", "Q8_0", 54),
    ("Q4_0", "Q8_0", 41)])
def test_streamed_lines(tmp_path: Path, gate: str, down: str, pairs: int) -> None:
    """The last pairs an expert that stream, by the formats: past them the prefill tiles are faster. Layers of few rows
    stream to 38 at least in every format; a shared expert of another format, while it streams along, adds six."""
    run_fake(tmp_path, f"""
def streams(T, **a): return any("gate_up@stream" in k for k in names(T, hidden=2048, gate_type="{gate}", down_type="{down}", **a))
for p, want in ((5, True), ({pairs}, True), ({pairs} + 1, False), (64, False)):
    assert streams(16 * p, n_experts=128, top_k=8, expert_ffn=768) == want, p
few = max({pairs}, 38)
for p, want in ((20, True), (few, True), (few + 1, False)):
    assert streams(8 * p, n_experts=16, top_k=2, expert_ffn=1024) == want, p
other = "Q4_1" if "{gate}" != "Q4_1" != "{down}" else "Q4_0"
own = dict(n_experts=128, top_k=32, expert_ffn=768, shared_ffn=512, shared_type=other)
for p, want in (({pairs} + 1, True), ({pairs} + 5 if {pairs} < 33 else 38, True), (max({pairs}, 38) + 1, False)):
    assert {pairs} >= 38 or streams(4 * p, **own) == want, p
""")


@pytest.mark.parametrize(("fmt", "down", "x", "last"), [
    ("Q6_K", "Q6_K", "bf16", 112), ("Q6_K", "Q6_K", "f32", 64), ("Q3_K", "Q3_K", "f32", 64), ("Q4_K", "Q6_K", "f32", 112),
    ("Q5_K", "Q6_K", "f32", 96), ("Q5_K", "Q5_K", "f32", 160), ("Q4_0", "Q4_0", "bf16", 224), ("Q4_K", "Q4_K", "f32", 200)])
def test_streamed_shared_expert(tmp_path: Path, fmt: str, down: str, x: str, last: int) -> None:
    """The last tokens (of these) at which 16 experts 1024 wide stream beside a shared one of 2048 of their formats: past
    them it is faster to join the prefill tiles' launches. Below 64 tokens it streams in any case."""
    run_fake(tmp_path, f"""
a = dict(hidden=2048, n_experts=16, top_k=2, expert_ffn=1024, gate_type="{fmt}", down_type="{down}", shared_ffn=2048,
         shared_type="{fmt}", shared_down_type="{down}")
for T in (33, 63, 64, 80, 96, 112, 128, 160, 200, 224, 225):
    n = names(T, "{x}", **a)
    assert any("@stream" in k for k in n) == (T <= {last}) == ("shared_down@stream" in n), (T, n)
""")
