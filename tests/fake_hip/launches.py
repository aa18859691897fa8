"""Calls of the library's step functions on the fake HIP runtime.  Run as
`launches.py libfake_hip.so` with a script on standard input, which sees the
names below and leaves its result in `out`, printed as JSON."""
import ctypes
import json
import os
import sys
import threading
import time

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_take_log.restype = ctypes.c_void_p
fake.hipStreamBeginCapture.argtypes = [ctypes.c_void_p, ctypes.c_int]
fake.hipStreamEndCapture.argtypes = [ctypes.c_void_p, ctypes.c_void_p]

from multigpu_advectiondiffusion_amd import _capi  # noqa: E402

L = _capi.lib()
S = _capi.Scheme(_capi.WENO_Z, 2, 1e-40)


def log() -> str:
    return ctypes.string_at(fake.fake_take_log()).decode()


def problems(n=2):
    return (_capi.Problem * n)(*[_capi.Problem(0x1000, 0x2000, 0x3000, 0x4000, 32, 32, 32, .1, .1, .1)] * n)


def batch():
    b = _capi.Batch()
    rc = L.mgad_batch_init(None, _capi.F64, S, 2, problems(), 0x9000, 1 << 24, 8, 0.0, 1.0, 0.4, b)
    assert rc == 0
    log()
    return b


def call(kind, n, graph=1, stream=0x77, u=0x1000, nx=32, ny=16, nz=12):
    """n steps of one solver on buffers that exist by name only; the returned status."""
    s, w1, w2, w3, c = ctypes.c_void_p(stream), u + 0x100, u + 0x200, u + 0x300, u + 0x400
    if kind == "periodic":
        return L.mgad_burgers_steps(s, S, nx, ny, nz, .1, .1, .1, u, w1, w2, c, n, graph)
    if kind == "slab":
        return L.mgad_burgers_slab_steps(s, S, nx, ny, nz // 3, 3, .1, .1, .1, u, w1, w2, c, n, graph)
    if kind == "reference":
        return L.mgad_burgers_ref_steps(s, S, 1, nx, ny, nz, .1, .1, .1, .01, u, w1, w2, n, graph)
    if kind == "weno7":
        return L.mgad_weno7_steps(s, nx, ny, nz, .1, .1, .1, u, w1, w2, w3, c, n, graph)
    if kind == "heat13":
        return L.mgad_heat13_rk3_steps(s, nx, ny, nz, .01, u, w1, w2, n, graph)
    if kind == "heat7":
        return L.mgad_heat7_fe_steps(s, nx, ny, nz, .1, .1, .1, .01, u, w1, n, graph)
    if kind == "batch":
        return L.mgad_batch_steps(s, batch_, n, graph)
    return L.mgad_batch_steps_serial(s, batch_, problems(), n, graph)


batch_ = batch()
out = None
exec(sys.stdin.read())
print(json.dumps(out))
