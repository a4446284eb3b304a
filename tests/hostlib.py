"""The library's host code on the CPU: its sources compiled for the host
alone and linked against hostrt/host_runtime.cpp in place of the HIP runtime."""
import concurrent.futures as cf
import ctypes
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
sys.path.insert(0, ROOT)
from __graft_entry__ import _load_build_module  # noqa: E402

LAUNCH_CB = ctypes.CFUNCTYPE(None, ctypes.c_char_p, ctypes.POINTER(ctypes.c_void_p))


def build(folder):
    """Path of the host library, compiled into folder."""
    b = _load_build_module()

    def run(cmd):
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(" ".join(cmd) + "\n" + r.stderr[-4000:])
        return r.stdout

    def compile_one(src):
        obj = os.path.join(folder, os.path.basename(src) + ".o")
        run([b.hipcc(), "--offload-arch=" + b.ARCH, "--offload-host-only", "-O1", "-std=c++17",
             "-fPIC", "-w", "-I" + os.path.join(ROOT, "include"), "-x", "hip", "-c", src, "-o",
             obj])
        return obj

    with cf.ThreadPoolExecutor(8) as ex:
        objs = list(ex.map(compile_one, b.sources()))
    # the device code that these objects do without
    fat = {line.split()[-1] for line in run(["nm", "--undefined-only"] + objs).splitlines()
           if "__hip_fatbin_" in line}
    out = os.path.join(folder, "libphyflow_host.so")
    run(["g++", "-shared", "-fPIC", "-O1", "-w", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
         "-I/opt/rocm/include", "-o", out, os.path.join(HERE, "hostrt", "host_runtime.cpp")] +
        objs + ["-lpthread", "-Wl,-z,defs", "-Wl,-Bsymbolic"] + ["-Wl,--defsym=%s=0" % f for f in sorted(fat)])
    return out


def load(path):
    """The library at path (its C ABI and the runtime's hr_* calls)."""
    h = ctypes.CDLL(path, mode=os.RTLD_LOCAL | os.RTLD_NOW)
    h.phf_last_error.restype = ctypes.c_char_p
    h.hr_calls.restype = h.hr_launches.restype = ctypes.c_long
    h.hr_fail_new.argtypes = [ctypes.c_long]
    h.hr_fail.argtypes = [ctypes.c_char_p, ctypes.c_long]
    return h
