"""Host code of the library on the CPU: a snippet run in a process of its own, where the library's HIP calls land in
``fake_hip.c``. It sees ``hip`` (the stand-in's counters and switches: ``hip.launches`` ..), ``_hip``, ``np``, ``MR``
(routing), ``route``, ``Plan``, ``MoELayer`` and ``layer(ready=True, **args)`` (a layer, by default with every tensor uploaded:
untouched zeros)."""

import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
PRELUDE = """
import ctypes, sys
sys.path.insert(0, {root!r})
_so = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
class _Fake:
    def __getattr__(self, name): return ctypes.c_int.in_dll(_so, "fake_" + name).value
    def __setattr__(self, name, v): ctypes.c_int.in_dll(_so, "fake_" + name).value = v
hip = _Fake()
import numpy as np
from artlite_amd import _hip
from artlite_amd.gguf_model import TYPE_ID
from artlite_amd.moe import route as MR
from artlite_amd.moe.layer import TENSORS, MoELayer
from artlite_amd.moe.plan import Plan, route
BLOCK = dict(Q4_0=(32, 18), Q4_1=(32, 20), Q8_0=(32, 34), Q3_K=(256, 110), Q4_K=(256, 144), Q5_K=(256, 176),
             Q6_K=(256, 210), IQ4_NL=(32, 18), IQ4_XS=(256, 136))
def upload(L, a):
    H, E, F, S = a["hidden"], a["n_experts"], a["expert_ffn"], a.get("shared_ffn", 0)
    def rows(n, cols, q): return n * (cols // BLOCK[q][0]) * BLOCK[q][1]
    sizes = dict(ffn_gate_inp=E * H * 4, ffn_gate_exps=rows(E * F, H, a["gate_type"]),
                 ffn_up_exps=rows(E * F, H, a["gate_type"]), ffn_down_exps=rows(E * H, F, a["down_type"]))
    if S:
        q = a["shared_type"]
        sizes.update(ffn_gate_shexp=rows(S, H, q), ffn_up_shexp=rows(S, H, q),
                     ffn_down_shexp=rows(H, S, a.get("shared_down_type") or q))
    for name, n in sizes.items(): L.upload(name, np.zeros(n, np.uint8))
def layer(ready=True, **a):
    L = MoELayer(**a)
    if ready: upload(L, a)
    return L
def names(T, x="bf16", **a):
    with layer(ready=False, max_tokens=T, **a) as L:
        L.stage(np.zeros((T, a["hidden"]), np.uint16 if x == "bf16" else np.float32))
        return L.kernel_names()
"""


def run_fake(tmp: Path, body: str) -> str:
    """What the snippet printed; an exception in it fails."""
    so = tmp / "fake_hip.so"
    if not so.exists():
        subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-Wall", "-Werror", "-o", str(so), str(HERE / "fake_hip.c")],
                       check=True)
    code = PRELUDE.format(root=str(HERE.parent), so=str(so)) + body
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
