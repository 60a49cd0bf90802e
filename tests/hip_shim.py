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
        return self._var(name).value

    def set(self, name, value):
        self._var(name).value = value

    def _var(self, name):
        t = C.c_size_t if name in ("budget", "unwanted", "used", "peak") else C.c_int
        return t.in_dll(self.lib, "shim_" + name)

    def recent(self):
        """(address, bytes) of the last allocations, in order"""
        ring = (C.c_size_t * 512).in_dll(self.lib, "shim_recent")
        return [(ring[2 * (k % 256)], ring[2 * (k % 256) + 1]) for k in
                range(max(0, self.n_recent - 256), self.n_recent)]

    def before_graph(self, function):
        self.hook = C.CFUNCTYPE(None)(function)
        C.c_void_p.in_dll(self.lib, "shim_before_graph").value = C.cast(self.hook, C.c_void_p).value

    def connect(self):
        """the runtime that libgzm.so brought with it"""
        with open("/proc/self/maps") as f:
            path = next(line.split()[-1] for line in f if "libamdhip64" in line)
        self.hip = C.CDLL(path)
        for name, symbol in (("malloc", "hipMalloc"), ("free", "hipFree"), ("set_device", "hipSetDevice"),
                             ("graph_launch", "hipGraphLaunch"), ("mem_info", "hipMemGetInfo")):
            C.c_void_p.in_dll(self.lib, "shim_" + name).value = C.cast(getattr(self.hip, symbol), C.c_void_p).value


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
