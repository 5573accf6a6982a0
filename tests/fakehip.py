"""Runs the library's host code on fake_hip.cpp's runtime, in a process of its
own: run(fake, steps) gives a dict a step.  A step is a list: an operation and
its arguments (the methods of _Child).  Each answer holds the call's status, the
kernels that it launched (name, template arguments, grid, block) and the
allocations so far (bytes, freed), in order."""
import ctypes
import json
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def build(folder):
    so = os.path.join(str(folder), "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-w",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", so], check=True)
    return so


def run(fake, steps, **env):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fake], input=json.dumps(steps), text=True,
                       capture_output=True, env=dict(os.environ, **env), timeout=120)
    assert r.returncode == 0, r.stderr
    return json.loads(r.stdout.splitlines()[-1])


class _Child:
    P = 0x10000  # a device address: nothing is ever read or written

    def __init__(self, fake):
        self.fake = ctypes.CDLL(fake, mode=ctypes.RTLD_GLOBAL)
        self.fake.fake_launch.restype = ctypes.c_char_p
        self.fake.fake_alloc_bytes.restype = ctypes.c_ulonglong
        sys.path.insert(0, ROOT)
        import chatokf_amd
        self.ok = chatokf_amd
        self.enc = chatokf_amd.Enc(0)

    def _w(self, fmt, M, K):
        return self.ok.QuantTensor(self.P, K, M, self.ok.BY_NAME[fmt])

    def gemm(self, fmt, M, K, N):
        self.enc.raw_gemm(self._w(fmt, M, K).c(), self.P, N, self.P)

    def tile(self, fmt, M, K, N):
        self.enc.gemm_tile(self._w(fmt, M, K), self.P, self.P, N)

    def gemv(self, fmt, M, K):
        self.enc.raw_gemv(self._w(fmt, M, K).c(), self.P, self.P)

    def gate_up(self, fmt, M, K):
        self.enc.gemv_gate_up(self._w(fmt, M, K), self._w(fmt, M, K), self.P, self.P, self.P)

    def argmax(self, n, rows):
        self.enc.argmax_rows(self.P, n, rows, self.P)

    def norm(self, n, rows, add):
        self.enc.add_rmsnorm(self.P, self.P if add else None, self.P, self.P, n, rows, 1e-6)

    def reserve(self, nk, n, rows):
        self.enc.reserve(nk, n, rows)

    def capture(self, on):
        self.fake.fake_capture(on)

    def fail_above(self, kib):
        self.fake.fake_fail_above(kib)

    def close(self):
        self.enc.close()

    def step(self, op, *args):
        first, status = self.fake.fake_launches(), 0
        try:
            getattr(self, op)(*args)
        except self.ok.OkfError as e:
            status = e.status
        launches = []
        for i in range(first, self.fake.fake_launches()):
            name, *dims = self.fake.fake_launch(i).decode().split()
            dims = [int(v) for v in dims]
            m = re.match(r"_ZN3okfL?(\d+)", name)
            n = int(m.group(1)) if m else 0
            base = name[m.end():m.end() + n] if m else name
            targs = [int(v) for v in re.findall(r"L[ijb](\d+)E", name[m.end() + n:])] if m else []
            launches.append({"name": base, "args": targs, "grid": dims[:3], "block": dims[3], "lds": dims[6]})
        allocs = [[self.fake.fake_alloc_bytes(i), self.fake.fake_alloc_freed(i)]
                  for i in range(self.fake.fake_allocs())]
        return {"status": status, "launches": launches, "allocs": allocs}


if __name__ == "__main__":
    steps = json.load(sys.stdin)
    child = _Child(sys.argv[1])
    print(json.dumps([child.step(*s) for s in steps]))
