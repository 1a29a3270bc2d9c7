"""Runs library calls in a child process over tests/fake_hip.cpp: a HIP runtime
without a device, which refuses allocations past a limit and writes launches down."""
import json
import os
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_built = None

_PRELUDE = """
import ctypes, json, sys
F = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)  # before libjev: its HIP calls bind here
F.fake_log.restype = ctypes.c_char_p
F.fake_live.restype = ctypes.c_size_t
F.fake_limit.argtypes = [ctypes.c_size_t]
sys.path[:0] = [{root!r} + "/llm-shield_amd", {root!r} + "/tests"]
import numpy as np
import jev
MIB = 1 << 20

def room(n=None):  # n bytes of device memory left; None: no limit
    F.fake_limit((1 << 63) if n is None else F.fake_live() + n)

def launches():  # since the last call: (kernel with its template arguments, grid, start event, stop event)
    out = []
    for line in F.fake_log().decode().splitlines():
        name, x, y, z, a, b = line.split("|")
        out.append((name, (int(x), int(y), int(z)), int(a), int(b)))
    F.fake_clear()
    return out

def model(heads=32, kv=8, cap=16384, **kw):
    cfg = jev.ModelConfig(n_layers=1, hidden=256, n_heads=heads, n_kv_heads=kv, head_dim=128, ffn=512, vocab=512,
                          initial_kv_capacity=cap, **kw)
    return jev.SynthModel(cfg, jev.TYPE_Q8_0).open(0)

def tokens(n):
    return jev.random_tokens(n, 512, 3)

def attention(log):  # the tree attention's form: (ds, "one" | "merged" | "split", grid z), and whether a merge kernel follows
    name, grid = [(n, g) for n, g, _, _ in log if "attn_tree_kernel" in n][0]
    ds, parts = name.split("attn_tree_kernelILi")[1].split("E")[:2]
    return int(ds), ["one", "merged", "split"][int(parts[2:])], grid[2], any("attn_merge_kernel" in n for n, _, _, _ in log)
"""


def run(code):
    """The value that `code` leaves in `result` (JSON)."""
    global _built
    if _built is None:
        _built = os.path.join(tempfile.mkdtemp(prefix="fake_hip"), "fake_hip.so")
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", "-o", _built, os.path.join(ROOT, "tests", "fake_hip.cpp")], check=True)
    p = subprocess.run([sys.executable, "-c", _PRELUDE.format(so=_built, root=ROOT) + code + "\nprint(json.dumps(result))"],
                       capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stderr[-2000:]
    return json.loads(p.stdout.splitlines()[-1])
