"""The library's host code without a GPU: its sources compiled for the host alone and linked with hip_recorder.cpp, which keeps
the launches instead of making them.  `calls(name, *args)` makes a call of the C ABI and returns its launches."""
import ctypes
import functools
import os
import re
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

from conftest import ROOT

TYPES = {0: "F32", 1: "F16", 8: "Q8_0", 12: "Q4_K", 13: "Q5_K", 14: "Q6_K"}
BASE = 1 << 40  # where the made-up device buffers lie: 16-byte aligned, told apart, never followed


def ptr(k):
    return BASE + (k << 36)


class Launch:
    def __init__(self, name, shape, args):
        self.grid, self.block, self.lds, self.args = tuple(shape[:3]), shape[3], shape[6], args
        self.kernel, _, rest = name.partition("<")
        self.params = [p.strip() for p in rest.rpartition(">")[0].split(",")] if rest else []

    def __repr__(self):
        return f"{self.kernel}<{', '.join(self.params)}> grid {self.grid} block {self.block} lds {self.lds}"


class Recorder:
    def __init__(self, lib):
        self.lib = lib
        lib.rec_name.restype = ctypes.c_char_p
        lib.rec_arg.restype = ctypes.c_uint64
        assert lib.orin_fa_init(0) == 0

    def calls(self, name, *args, keep_args=0):
        self.lib.rec_start(keep_args)
        conv = [ctypes.c_float(a) if isinstance(a, float) else ctypes.c_void_p(a) if isinstance(a, int) and a >= BASE else a for a in args]
        rc = getattr(self.lib, name)(*conv)
        assert rc == 0, (name, args, rc)
        out = []
        shape = (ctypes.c_uint * 7)()
        for i in range(self.lib.rec_count()):
            self.lib.rec_shape(i, shape)
            out.append(Launch(_demangled(self.lib.rec_name(i).decode()), list(shape), [self.lib.rec_arg(i, k) for k in range(keep_args)]))
        return out


@functools.lru_cache(maxsize=None)
def _demangled(name):
    text = subprocess.run(["c++filt", name], capture_output=True, text=True, check=True).stdout.strip()
    text = re.sub(r"\(anonymous namespace\)::", "", text)
    return re.sub(r"^void ", "", text).replace("orin_fa::", "").rpartition("(")[0]


@functools.lru_cache(maxsize=None)
def recorder():
    from orin_llm_amd import build

    where = tempfile.mkdtemp(prefix="orin_recorder_")
    sources = [s for s in build.SOURCES if s.endswith(".hip")]
    objs = [os.path.join(where, os.path.basename(s) + ".o") for s in sources]
    # (-fuse-cuid=none: every object asks for the device code under the one name hip_recorder.cpp has)
    compile_one = [[build.HIPCC, "--offload-host-only", "--offload-arch=gfx950", "-O1", "-std=c++17", "-fPIC", "-fno-exceptions", "-fuse-cuid=none",
                    "-c", s, "-o", o] for s, o in zip(sources, objs)]
    with ThreadPoolExecutor(max_workers=8) as pool:
        list(pool.map(build._run, compile_one))
    lib = os.path.join(where, "liborin_recorded.so")
    build._run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wl,-Bsymbolic,-z,muldefs", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__=1", os.path.join(ROOT, "tests", "hip_recorder.cpp")]
               + objs + ["-o", lib])
    return Recorder(ctypes.CDLL(lib))
