"""The step engine's host code on the CPU: the library's sources compiled for the host only and linked with
host_runtime.cpp, whose kernels keep the bookkeeping of a scripted solve."""
import ctypes
import os
import subprocess
import tempfile

from hobakv1_amd import build, lib

RUNS, MISFIT, LATE, LOST = 0, 1, 2, 3
_fake = None


def load():
    """The host-only library (built once per process)."""
    global _fake
    if _fake is None:
        hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
        here = os.path.dirname(os.path.abspath(__file__))
        with tempfile.TemporaryDirectory() as tmp:
            flags = ["--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-w", "-c"]
            sources = [os.path.join(build.CSRC, s) for s in build.HIP_SOURCES]
            sources.append(os.path.join(here, "host_runtime.cpp"))
            objs = [os.path.join(tmp, os.path.basename(s) + ".o") for s in sources]
            jobs = [subprocess.Popen([hipcc, *flags, "-x", "hip", s, "-o", o]) for s, o in zip(sources, objs)]
            assert all([j.wait() == 0 for j in jobs])
            undefined = subprocess.run(["nm", "-u", *objs], check=True, capture_output=True, text=True).stdout.split()
            fatbins = {f"-Wl,--defsym={u}=0" for u in undefined if u.startswith("__hip_fatbin_")}
            so = os.path.join(tmp, "libhobak_host.so")
            subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", *sorted(fatbins), *objs, "-o", so], check=True)
            _fake = ctypes.CDLL(so)
        for name, (res, args) in lib.SIGNATURES.items():
            getattr(_fake, name).restype, getattr(_fake, name).argtypes = res, args
        _fake.fake_log.restype = ctypes.c_char_p
    return _fake


class Engine:
    """A context of the host-only library, with what its launches did."""

    def __init__(self, **tuning):
        self.fake = load()
        self.fake.fake_reset()
        self.ctx = lib.Context(0, apply_table=False)
        self.ctx.set_tuning(**tuning)

    def script(self, inst, iters=10, sweeps=1, device=RUNS, die=RUNS, big=RUNS):
        self.fake.fake_script(inst.nv, sweeps, iters, device, die, big)

    def log(self):
        """The launches and waits since the last call, one word list each."""
        out = [line.split() for line in self.fake.fake_log().decode().splitlines()]
        self.fake.fake_clear()
        return out

    def forms(self):
        """Which PCG forms were launched since the last call, in order, repeats left out."""
        names = [line[0] for line in self.log() if line[0] in ("spmv", "device", "die", "big")]
        return [n for i, n in enumerate(names) if i == 0 or names[i - 1] != n]
