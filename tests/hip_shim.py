"""A test process of its own in which hip_shim.c stands before the HIP runtime.

`run(function, ...)` starts it and calls `function` of hip_shim_checks with the
shim loaded; the function's assertions decide."""
import ctypes as C
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def run(function, *args):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), function, *map(str, args)], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=100)
    print(r.stdout)
    assert r.returncode == 0, r.stdout[-3000:]


class Shim:
    def __init__(self, path):
        self.lib = C.CDLL(path, mode=C.RTLD_GLOBAL)  # before libgzm.so, whose calls it then takes

    def __getattr__(self, name):
        return C.c_size_t.in_dll(self.lib, "shim_" + name).value if name in ("budget", "used", "peak") else \
            C.c_int.in_dll(self.lib, "shim_" + name).value

    def set(self, name, value):
        t = C.c_size_t if name in ("budget", "used", "peak") else C.c_int
        t.in_dll(self.lib, "shim_" + name).value = value

    def connect(self):
        """the runtime that libgzm.so brought with it"""
        with open("/proc/self/maps") as f:
            path = next(line.split()[-1] for line in f if "libamdhip64" in line)
        hip = C.CDLL(path)
        for name, symbol in (("malloc", "hipMalloc"), ("free", "hipFree"), ("set_device", "hipSetDevice")):
            C.c_void_p.in_dll(self.lib, "shim_" + name).value = C.cast(getattr(hip, symbol), C.c_void_p).value


def main():
    import tempfile
    for sub in ("oracle", "gizmo-public_amd", "tests"):
        sys.path.insert(0, os.path.join(ROOT, sub))
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "hip_shim.so")
        subprocess.run(["gcc", "-O1", "-fPIC", "-shared", "-o", path, os.path.join(HERE, "hip_shim.c"), "-lpthread"],
                       check=True)
        shim = Shim(path)
        import gzm
        gzm.load_library()
        shim.connect()
        import hip_shim_checks
        getattr(hip_shim_checks, sys.argv[1])(shim, *sys.argv[2:])


if __name__ == "__main__":
    main()
