"""Runs the library's host code without a GPU and records which kernels it would
launch (tests/cpp/launch_recorder.cpp stands in for the HIP runtime).

run(snippet) executes `snippet` in a process of its own, where `L` is the
library, `R` the recorder, `P` a fake device address aligned to 1 MiB, `events()`
the recorded events so far, `Event` their type, and returns what the snippet
prints.  The process does not load torch: torch's own HIP runtime would come
first.
"""
import os
import subprocess
import sys
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "tests", "cpp", "launch_recorder.cpp")

_PRELUDE = """
import collections, ctypes, threading, time
R = ctypes.CDLL({recorder!r}, mode=ctypes.RTLD_GLOBAL)
R.recorder_log.restype = ctypes.c_size_t
for f in (R.recorder_close, R.recorder_set_capturing):
    f.argtypes = [ctypes.c_void_p] + [ctypes.c_int] * (f is R.recorder_set_capturing)
L = ctypes.CDLL({library!r})
I, V = ctypes.c_int, ctypes.c_void_p
P = 1 << 20
Event = collections.namedtuple("Event", "what thread stream grid block lds kernel")
def events():
    n = R.recorder_log(None, ctypes.c_size_t(0))
    b = ctypes.create_string_buffer(n + 1)
    R.recorder_log(b, ctypes.c_size_t(n + 1))
    out = []
    for line in b.value.decode().splitlines():
        w = line.split()
        if w[0] == "free":
            out.append(Event("free", int(w[1]), None, None, None, None, w[2]))
        else:
            s = 0 if w[2] == "(nil)" else int(w[2], 16)
            out.append(Event("launch", int(w[1]), s, tuple(map(int, w[3:6])), int(w[6]), int(w[7]), w[8]))
    return out
def ok(rc):
    L.qe_last_error.restype = ctypes.c_char_p
    assert rc == 0, L.qe_last_error()
def tune(key, value):
    ok(L.qe_set_tuning(key.encode(), value))
def attention(stream=0, rows=512, nq=12, nkv=2, max_seq=4096):
    ok(L.qe_launch_attention_gqa_prefill(V(P), V(P), V(P), V(P), V(0), I(rows), V(stream), I(nq), I(nkv), I(128),
                                         I(max_seq), I(nq * 128)))
def gemm(M, N, K, stream=0, tiled=False, scales=P):
    if tiled:
        ok(L.qe_launch_gemm_prefill_w4a16_tiled(V(P), V(scales), V(P), V(0), V(P), I(M), I(N), I(K), V(stream)))
    else:
        ok(L.qe_launch_gemm_prefill_w4a16(V(P), V(scales), V(P), V(0), V(P), I(M), I(N), I(K), V(stream), I(0)))
def gemm_noalloc(M, N, K, stream=0):
    ok(L.qe_launch_gemm_prefill_w4a16_noalloc(V(P), V(P), V(P), V(0), V(P), I(M), I(N), I(K), V(stream), I(0)))
def gemm_w4a8(M, N, K, stream=0):
    ok(L.qe_launch_gemm_prefill_w4a8(V(P), V(P), V(P), V(P), V(P), V(0), V(P), I(M), I(N), I(K), V(stream)))
def reserve(stream=0):
    ok(L.qe_gemm_reserve_workspace(V(stream)))
def release(stream=0):
    ok(L.qe_gemm_release_workspace(V(stream)))
"""


def build(folder) -> str:
    out = os.path.join(str(folder), "liblaunch_recorder.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", SOURCE, "-o", out, "-lpthread"], check=True)
    return out


def run(recorder: str, snippet: str) -> str:
    library = os.path.join(ROOT, "qwen-engine_amd", "libqe_amd.so")
    code = _PRELUDE.format(recorder=recorder, library=library) + textwrap.dedent(snippet)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
