"""The library's host code linked against a HIP runtime without a device
(hip_stub.cpp), for tests of what it asks the runtime for."""
import ctypes as C
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
COUNTS = ("launches", "captures", "instantiated", "replays", "destroyed", "unused", "failed", "lds", "live")


def build(folder):
    """Compile the host side of every source and the stub into one library.
    Undefined behaviour that the host code meets becomes a fault of the stub."""
    from forcefieldx_amd import build as nb
    flags = ["-O1", "-std=c++17", "--offload-arch=gfx950", "-fPIC", "--cuda-host-only", "-w", "-I", nb.CSRC,
             "-Xarch_host", "-fsanitize=undefined", "-Xarch_host", "-fsanitize-minimal-runtime"]
    jobs, objs = [], []
    for src in [os.path.join(nb.CSRC, s) for s in nb.SOURCES] + [os.path.join(HERE, "hip_stub.cpp")]:
        obj = os.path.join(folder, os.path.basename(src) + ".o")
        objs.append(obj)
        jobs.append(subprocess.Popen([nb.HIPCC, *flags, "-x", "hip", "-c", src, "-o", obj]))
    assert all(j.wait() == 0 for j in jobs)
    # the device code that the host objects would carry, and the sanitizer's handlers
    missing = subprocess.check_output(["nm", "-u", *objs], text=True)
    fat = os.path.join(folder, "fatbin.c")
    with open(fat, "w") as f:
        f.write("void stub_fault(const char *);\n")
        f.writelines(f"char {n}[8];\n" for n in sorted(set(re.findall(r"__hip_fatbin_\w+", missing))))
        f.writelines(f'void {n}(void) {{ stub_fault("{n}"); }}\n'
                     for n in sorted(set(re.findall(r"__ubsan_handle_\w+", missing))))
    lib = os.path.join(folder, "libamoeba_host.so")
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", lib, fat, *objs, "-lstdc++", "-lm", "-Wl,-Bsymbolic"])
    return lib


class Stub:
    def __init__(self, lib):
        from forcefieldx_amd import ffi
        self.ffi, self.L = ffi, ffi.load(lib)
        self.L.stub_set.argtypes = [C.c_long, C.c_int, C.c_int, C.c_int]
        self.L.stub_free.argtypes = [C.c_long]
        self.L.stub_faults.restype = C.c_char_p

    def set(self, fail_bytes=0, moved=0, reject=0, iterations=1, free_bytes=1 << 38):
        self.L.stub_set(fail_bytes, moved, reject, iterations)
        self.L.stub_free(free_bytes)

    def reset(self):
        self.L.stub_reset_counts()

    def counts(self):
        v = (C.c_long * len(COUNTS))()
        self.L.stub_counts(v)
        return dict(zip(COUNTS, v))

    def allocations(self):
        """Bytes of each allocation made since the last reset."""
        v = (C.c_long * 4096)()
        return v[:self.L.stub_allocations(v, C.c_long(4096))]

    def faults(self):
        return self.L.stub_faults().decode().splitlines()

    def taken_faults(self):
        """The faults so far, which are then forgotten."""
        f = self.faults()
        self.L.stub_forget()
        return f
