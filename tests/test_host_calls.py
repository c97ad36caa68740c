"""The host-pointer calls' own errors and fall-backs, on the CPU (no kernel runs)."""

from pathlib import Path

from .fake_runtime import run_fake

CALLS = """
L = layer(hidden=1024, n_experts=8, top_k=2, expert_ffn=512, gate_type="Q8_0", down_type="Q8_0", max_tokens=64)
logits, x = np.zeros((5000, 128), np.float32), np.zeros((40, 1024), np.float32)
CALLS = dict(route=lambda: route(logits, 8), top_k=lambda: MR.top_k(logits, 8),
             plan=lambda: Plan.of(np.zeros((500, 8), np.int32), cap=200, E=128), layer=lambda: L(x))
"""


def test_without_pinned_memory(tmp_path: Path) -> None:
    """Where no pinned memory is to be had the calls take pageable copies, as they do beyond the pinned buffers' size."""
    run_fake(tmp_path, CALLS + """
hip.fail_host_malloc = 1
for name, call in CALLS.items():
    before = hip.copies
    call()
    assert hip.copies >= before + 2, name  # (to the device and back)
hip.fail_host_malloc = 0
for name, call in CALLS.items():
    before = hip.copies
    call()
    assert hip.copies == before, name
""")


def test_failed_launch_leaves_nothing_queued(tmp_path: Path) -> None:
    """Whichever launch of a call fails, what was queued on the thread's pinned buffers before it has run when the call
    returns: the next call writes them, and may free them for larger ones."""
    run_fake(tmp_path, CALLS + """
for name, call in CALLS.items():
    before = hip.launches
    call()
    n = hip.launches - before
    assert n >= 2 and hip.pending == 0, (name, n)
    for i in range(n):
        hip.fail_launch = hip.launches + i
        try:
            call()
        except _hip.Error as e:
            assert "invalid" in str(e), e
        else:
            raise AssertionError((name, i))
        assert hip.pending == 0, (name, i, n)
    hip.fail_launch = -1
    call()
L.close()
L = layer(hidden=1024, n_experts=8, top_k=2, expert_ffn=512, gate_type="Q8_0", down_type="Q8_0", max_tokens=512)
hip.fail_launch = hip.launches + 3
try: L(x)
except _hip.Error: pass
hip.fail_launch = -1
L(np.zeros((512, 1024), np.float32))  # (larger buffers: the others are freed)
assert hip.freed_busy == 0
""")


def test_layer_call_makes_no_stream(tmp_path: Path) -> None:
    """A layer's call runs on the layer's own stream: the thread's is made by the first call that needs it."""
    run_fake(tmp_path, CALLS + """
assert hip.streams == 1
L(x)
assert hip.streams == 1
CALLS["route"]()
CALLS["plan"]()
assert hip.streams == 2
""")


def test_call_before_the_upload_stages_its_input(tmp_path: Path) -> None:
    """layer(x) without its tensors is refused, and has staged x: once they are there, it runs."""
    run_fake(tmp_path, """
a = dict(hidden=1024, n_experts=8, top_k=2, expert_ffn=512, gate_type="Q8_0", down_type="Q8_0", max_tokens=64)
L = layer(ready=False, **a)
try: L(np.zeros((40, 1024), np.float32))
except _hip.Error as e: assert "not uploaded" in str(e), e
else: raise AssertionError
upload(L, a)
_hip.check(_hip.lib().artlite_moe_layer_run(L.handle, 40))
""")


def test_last_error_outlives_a_pass(tmp_path: Path) -> None:
    """Asking whether a launch takes a pass's items, and finding that it does not, leaves the thread's message alone."""
    run_fake(tmp_path, """
a = dict(hidden=1024, n_experts=1024, top_k=8, expert_ffn=4096, gate_type="Q4_0", down_type="Q4_0")
with layer(ready=False, max_tokens=128 * 36, **a) as L:
    try: L.upload("ffn_gate_inp", np.zeros(10, np.uint8))
    except _hip.Error as e: said = str(e)
    for pairs in (4, 33, 36):
        L.stage(np.zeros((128 * pairs, 1024), np.uint16))
        n = L.kernel_names()
        assert not any("@stream64" in k for k in n), n
        assert _hip.last_error() == said, (pairs, _hip.last_error())
""")
