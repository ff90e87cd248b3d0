"""Builds the library's host code against the stand-in HIP runtime
(hip_stub.cpp) and gives tests a handle on it: kernel launches as
(name, grid, block), device and pinned memory, and a memory limit."""
import ctypes as C
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
CSRC = os.path.join(ROOT, "custom-gpgpu-rasterizer_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-ffp-contract=off", "-fno-fast-math",
         "-Wno-unused-function", "-I", os.path.join(ROOT, "include"), "-I", CSRC]
SOURCES = [os.path.join(CSRC, s) for s in ("rast_kernels.hip", "rast_api.hip", "rast_mlp.hip")]


def run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, " ".join(cmd) + "\n" + r.stderr
    return r.stdout


def build(out_dir, extra=(), link=()):
    """librast_host.so in out_dir, of SOURCES, layout.hip, bounds.hip and the stub."""
    objs = []
    for src in SOURCES + [os.path.join(HERE, "layout.hip"), os.path.join(HERE, "bounds.hip")]:
        o = os.path.join(out_dir, os.path.basename(src) + ".o")
        run([HIPCC, *FLAGS, *extra, "-c", src, "-o", o])
        objs.append(o)
    # the device code that is not there: one symbol per source
    fat = os.path.join(out_dir, "fatbin.c")
    names = sorted(set(re.findall(r"__hip_fatbin_\w+", "".join(run(["nm", o]) for o in objs))))
    with open(fat, "w") as f:
        f.write("".join(f"const char {n}[8];\n" for n in names))
    stub = os.path.join(out_dir, "stub.o")
    run(["g++", "-O1", "-g", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", *extra, "-c",
         os.path.join(HERE, "hip_stub.cpp"), "-o", stub])
    out = os.path.join(out_dir, "librast_host.so")
    run(["g++", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-Wl,-z,defs", *extra, *link, "-o", out, *objs, stub, "-x", "c", fat,
         "-x", "none", "-lpthread"])
    return out


class Runtime:
    """The stub of a loaded librast_host.so; `launches` collects kernel names
    (without their mangling) and grids."""

    def __init__(self, lib):
        self.lib = lib
        for name, res, args in (("stub_fail_new", None, [C.c_long]), ("stub_fail_left", C.c_long, []),
                                ("stub_limit", None, [C.c_size_t]), ("stub_used", C.c_size_t, []),
                                ("stub_pinned", C.c_size_t, []), ("stub_mallocs", C.c_size_t, []),
                                ("stub_pinned_of", C.c_void_p, [C.c_size_t, C.c_size_t]),
                                ("layout_counters_size", C.c_size_t, []),
                                ("layout_counter", C.c_size_t, [C.c_char_p])):
            getattr(lib, name).restype, getattr(lib, name).argtypes = res, args
        self.launches = []
        self.on_launch = None
        proto = C.CFUNCTYPE(None, C.c_char_p, C.c_uint32, C.c_uint32)
        self._callback = proto(self._launched)
        lib.stub_callback.argtypes = [proto]
        lib.stub_callback(self._callback)

    def _launched(self, mangled, grid, block):
        name = re.search(r"k_[a-z_]+", mangled.decode()).group(0)
        self.launches.append((name, grid, block))
        if self.on_launch:
            self.on_launch(name)

    def names(self):
        out = [n for n, _, _ in self.launches]
        self.launches.clear()
        return out

    def limit(self, extra=None):
        """At most `extra` more bytes of device memory than now (None: no limit)."""
        self.lib.stub_limit(C.c_size_t(-1).value if extra is None else self.used() + extra)

    def used(self):
        return self.lib.stub_used()

    def pinned(self):
        return self.lib.stub_pinned()

    def mallocs(self):
        return self.lib.stub_mallocs()

    def counters(self, k=0, **values):
        """Sets words of the counters that the k-th renderer's last frame left."""
        p = self.lib.stub_pinned_of(self.lib.layout_counters_size(), k)
        for name, v in values.items():
            C.c_uint32.from_address(p + self.lib.layout_counter(name.encode())).value = v
