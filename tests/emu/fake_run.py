"""libspeckle_hip.so's host code on fake_hip.cpp: `python fake_run.py FAKE_SO`
runs the program on its standard input with the names below.  In a process of
its own without torch, whose HIP runtime would come first."""
import ctypes
import importlib.util
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
fake = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_char_p
fake.fake_live.restype = ctypes.c_ulonglong
fake.fake_get.restype = ctypes.c_longlong
spec = importlib.util.spec_from_file_location(
    "_capi", os.path.join(ROOT, "als_speckle_amd", "_capi.py"))
capi = importlib.util.module_from_spec(spec)
sys.modules["_capi"] = capi
spec.loader.exec_module(capi)
lib = capi.load(os.path.join(ROOT, "als_speckle_amd", "libspeckle_hip.so"))

HIO, ER, DM = ((capi.HIO, 0, 0.9, 0.0, 0.0), (capi.ER, 0, 0.0, 0.0, 0.0),
               (capi.DM, 0, 0.7, 0.0, 0.0))


def knob(name, value):
    fake.fake_set(name.encode(), value)


def launches():
    """The launches since the last call, as lists of words."""
    out = [line.split() for line in fake.fake_log().decode().splitlines()]
    fake.fake_clear()
    return out


def kernels(which="k_"):
    return [w[1].split("<")[0] for w in launches() if which in w[1]]


def ok(rc):
    assert rc == 0, (rc, lib.spk_last_error())


ctx = ctypes.c_void_p()
ok(lib.spk_ctx_create(0, None, ctypes.byref(ctx)))


class Plan:
    def __init__(self, n, batch=1, shared=1, ipsf=False, **tune):
        self.n, self.batch = n, batch
        t = capi.SpkTune(**tune)
        self.h = ctypes.c_void_p()
        ok(lib.spk_plan_create(ctx, n, batch, shared, ctypes.byref(t), ctypes.byref(self.h)))
        x = ctypes.c_void_p(64)          # a device address; no kernel reads it
        ok(lib.spk_set_modulus(self.h, -1, x))
        ok(lib.spk_set_support(self.h, -1, x))
        ok(lib.spk_set_psi(self.h, -1, x, 0))
        if ipsf:
            ok(lib.spk_set_ipsf(self.h, x))
        launches()

    def iterate(self, steps, per_frame=0):
        """The call's status."""
        count = len(steps) // (self.batch if per_frame else 1)
        return lib.spk_iterate(self.h, capi.make_steps(steps), count, per_frame, None)

    def coherence(self, iterations=2):
        x = ctypes.c_void_p(64)
        return lib.spk_coherence_rl(self.h, x, self.n, self.n, x, iterations, 0, 0, x)

    def close(self):
        ok(lib.spk_plan_destroy(self.h))


if __name__ == "__main__":
    exec(compile(sys.stdin.read(), "program", "exec"))
