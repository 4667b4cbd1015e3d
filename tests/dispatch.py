"""Runs calls of libqlin's C ABI on the CPU over the recording HIP runtime of fake_hip.cpp
and returns what each would have launched.  The library is loaded in a child process, which
no real HIP runtime reaches; device pointers are invented addresses."""
from __future__ import annotations

import ctypes
import json
import os
import pathlib
import subprocess
import sys

TESTS = pathlib.Path(__file__).resolve().parent
LIB = TESTS.parent / "qwen_3.5_comfy_prompt_enhancer_amd" / "kernels" / "libqlin.so"
WS = 256 << 20
F32, BF16, F16 = 3, 2, 1

X, XS, W, S, Z, OUT, Q, QS, SCRATCH = ((i + 1) << 36 for i in range(9))


def gemm_i8(M, K, N, ws=WS):
    return ["qlin_gemm_i8", X, XS, M, K, W, S, F32, N, OUT, N, None, 0, SCRATCH if ws else None, ws, None]


def gemm_w4(M, K, N, group=128, zeros=False, ws=WS):
    return ["qlin_gemm_w4", X, XS, M, K, W, S, BF16, Z if zeros else None, group, N, OUT, N, None, 0,
            SCRATCH if ws else None, ws, None]


def proj3_i8(M, K, n1, n2, n3, ws=WS):
    return ["qlin_proj3_i8", X, XS, M, K, W, S, n1, W, S, n2, W, S, n3, F32, OUT, n1 + n2 + n3, SCRATCH, ws, None]


def gate_up_i8(M, K, N, ws=WS):
    return ["qlin_mlp_gate_up_quant_i8", X, XS, M, K, W, S, W, S, F32, N, Q, QS, SCRATCH if ws else None, ws, None]


def gate_up_w4(M, K, N, group=128, zeros=False, ws=WS):
    z = Z if zeros else None
    return ["qlin_mlp_gate_up_quant_w4", X, XS, M, K, W, S, z, W, S, z, BF16, group, N, Q, QS,
            SCRATCH if ws else None, ws, None]


def linear_w8(M, K, N, ws=WS):
    return ["qlin_linear_w8", X, F16, M, K, K, W, S, F32, N, OUT, F16, N, None, 0, SCRATCH, ws, None]


def linear_w4(M, K, N, group=128, ws=WS):
    return ["qlin_linear_w4", X, F16, M, K, K, W, S, F16, None, group, N, OUT, F16, N, None, 0, SCRATCH, ws, None]


def requant_w8(K, N):
    return ["qlin_requant_w8_row", W, K, N, OUT, S, None]


def run(tmp, calls, env=None):
    """[(status, [(what, kernel, grid x, grid y)], message)] of each call; `env` is the
    library's environment (its tuning variables)."""
    fake = pathlib.Path(tmp) / "libfake_hip.so"
    if not fake.exists():
        subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", str(fake), str(TESTS / "fake_hip.cpp")], check=True)
    e = {k: v for k, v in os.environ.items() if not k.startswith("QLIN_")}
    r = subprocess.run([sys.executable, __file__, str(fake), str(LIB)], input=json.dumps(calls), text=True,
                       capture_output=True, env={**e, **(env or {})})
    assert r.returncode == 0, r.stderr
    return [(st, [tuple(e) for e in ev], msg) for st, ev, msg in json.loads(r.stdout)]


def _child(fake, lib):
    f = ctypes.CDLL(fake, mode=ctypes.RTLD_GLOBAL)
    f.fake_log.restype = ctypes.c_char_p
    q = ctypes.CDLL(lib)
    q.qlin_last_error.restype = ctypes.c_char_p
    out = []
    for name, *args in json.load(sys.stdin):
        f.fake_clear()
        # (every integer as 64 bits: the ABI's registers and stack slots hold either width)
        st = getattr(q, name)(*(None if a is None else ctypes.c_int64(a) for a in args))
        events = []
        for line in f.fake_log().decode().splitlines():
            what, kernel, *dims = line.split()
            events.append((what, kernel, *map(int, dims[:2])))
        out.append((st, events, q.qlin_last_error().decode()))
    json.dump(out, sys.stdout)


if __name__ == "__main__":
    _child(*sys.argv[1:])
