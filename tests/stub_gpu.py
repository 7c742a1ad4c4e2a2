"""Tests of the engine's host side without a GPU: the real engine and kernel library over a HIP runtime whose device memory is
host memory and whose launches do nothing (native/hip_stub.cpp).  The stub stands in for the runtime of a whole process, so each
test runs in a child."""
import atexit
import ctypes as C
import functools
import importlib
import json
import os
import re
import shutil
import subprocess
import sys
import tempfile

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = os.path.join(ROOT, "tests", "native")


@functools.lru_cache(maxsize=1)
def _built():
    out = tempfile.mkdtemp(prefix="saga_stub_")
    atexit.register(shutil.rmtree, out, ignore_errors=True)
    for name in ("hip_stub", "plan_probe"):
        subprocess.check_call(["g++", "-O1", "-std=c++17", "-march=x86-64-v3", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                               "-I", os.path.join(ROOT, "saga_amd", "src"), "-I", os.path.join(ROOT, "include"),
                               "-I", "/opt/rocm/include", os.path.join(NATIVE, name + ".cpp"), "-o", os.path.join(out, name + ".so")])
    return out


def on_stub(fn):
    """Runs the test function in a child process on the stub."""

    @functools.wraps(fn)
    def run(**kwargs):
        code = "import sys; from tests import stub_gpu; stub_gpu._child(*sys.argv[1:])"
        r = subprocess.run([sys.executable, "-c", code, _built(), fn.__module__.split(".")[-1], fn.__name__, json.dumps(kwargs)], cwd=ROOT,
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr

    run.body = fn
    return run


def _child(libs, module, name, kwargs):
    global stub, probe
    from saga_amd import api

    stub = C.CDLL(os.path.join(libs, "hip_stub.so"), mode=C.RTLD_GLOBAL)  # before anything that needs the runtime
    stub.hipstub_set_memory.argtypes = [C.c_size_t]
    stub.hipstub_uploads.restype = stub.hipstub_replays.restype = C.c_long
    stub.hipstub_used.restype = stub.hipstub_peak.restype = C.c_size_t
    stub.hipstub_log.restype = C.c_char_p
    stub.hipstub_launches.argtypes, stub.hipstub_launches.restype = [C.c_char_p], C.c_long
    api.lib()
    probe = C.CDLL(os.path.join(libs, "plan_probe.so"))
    probe.probe_plan.argtypes = [C.c_void_p, C.c_char_p, C.c_size_t]
    for f in (probe.probe_access, probe.probe_access_data, probe.probe_last_batch):
        f.argtypes, f.restype = [C.c_void_p], C.c_void_p
    probe.probe_access_close.argtypes = [C.c_void_p]
    getattr(importlib.import_module("tests." + module), name).body(**json.loads(kwargs))


def launches(kernel):
    return stub.hipstub_launches(kernel.encode())


def launched():
    """The launches since the last call: (kernel, its whole-number template arguments, blocks, threads)."""
    out = []
    for line in stub.hipstub_log().decode().splitlines():
        name, grid, block = line.rsplit(" ", 2)
        m = re.match(r"_ZN12_GLOBAL__N_1(\d+)", name) or re.match(r"_Z(\d+)", name)
        base, rest = name[m.end():m.end() + int(m.group(1))], name[m.end() + int(m.group(1)):]
        # (the arguments of the function behind the template's hold no such numbers)
        out.append((base, tuple(int(v) for v in re.findall(r"L[ib](\d+)E", rest)), int(grid), int(block)))
    return out


def uploads():
    return stub.hipstub_uploads()


def replays():
    return stub.hipstub_replays()


def plan(program):
    """The operations of a finalized program as dicts (native/plan_probe.cpp)."""
    n = probe.probe_plan(program._h, None, 0)
    buf = C.create_string_buffer(n + 1)
    probe.probe_plan(program._h, buf, n + 1)
    return [json.loads(line) for line in buf.value.decode().splitlines()]


def overlapping(ops):
    """Pairs of storages at the same addresses of which one is written while the other still holds something that is read later
    (operations in the order of the list)."""
    life, place = {}, {}
    for i, op in enumerate(ops):
        for s, a, size, _ in op["reads"] + op["writes"]:
            if a:
                first, _ = life.get(s, (i, i))
                life[s], place[s] = (first, i), (a, a + size)
    return [(s, q) for s in life for q in life if s < q and place[s][0] < place[q][1] and place[q][0] < place[s][1]
            and life[s][0] <= life[q][1] and life[q][0] <= life[s][1]]


def unordered(ops):
    """Pairs of operations that touch the same addresses, one of them writing, and that neither the order of a stream nor an
    event puts one behind the other."""
    n = len(ops)
    behind = [set() for _ in range(n)]  # what operation i is known to run behind
    last = {0: None, 1: None}
    for i, op in enumerate(ops):
        before = last[op["side"]]
        if before is not None:
            behind[i] |= behind[before] | {before}
        if op["side"] and op["fork"] >= 0:
            behind[i] |= behind[op["fork"]] | {op["fork"]}
        if not op["side"] and op["needs"] >= 0:
            behind[i] |= behind[op["needs"]] | {op["needs"]}
        last[op["side"]] = i

    def spans(op, which):
        return [(a, a + size) for _, a, size, _ in op[which] if a]

    def meet(a, b):
        return any(x[0] < y[1] and y[0] < x[1] for x in a for y in b)

    bad = []
    for i in range(n):
        w, rw = spans(ops[i], "writes"), spans(ops[i], "writes") + spans(ops[i], "reads")
        for j in range(i):
            if j in behind[i]:
                continue
            w2, rw2 = spans(ops[j], "writes"), spans(ops[j], "writes") + spans(ops[j], "reads")
            if meet(w, rw2) or meet(rw, w2):
                bad.append((j, ops[j]["kind"], i, ops[i]["kind"]))
    return bad


class Window:
    """A host window onto a batched tensor that stays open until close()."""

    def __init__(self, tensor):
        self._ta = probe.probe_access(tensor._h)

    def floats(self, n):
        return np.frombuffer((C.c_float * n).from_address(probe.probe_access_data(self._ta)), np.float32)

    def close(self):
        probe.probe_access_close(self._ta)


def last_batch(tensor, n):
    """The first n floats that the last step's operations read of a batched tensor."""
    return np.frombuffer((C.c_float * n).from_address(probe.probe_last_batch(tensor._h)), np.float32).copy()
