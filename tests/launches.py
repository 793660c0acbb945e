"""What the library launches, observed on the CPU.

A small stand-in for the HIP runtime (compiled here, loaded ahead of the real one)
answers for a device of 256 compute units, writes down every launch (kernel, grid,
workgroup) instead of running it, and refuses what HIP refuses: a grid dimension of
2^32 work-items or more.  The calls run in a process of their own, so that no other
test sees the stand-in.
"""

import json
import re
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
LIBRARY = ROOT / "vflash_amd" / "libvflash_amd.so"

STAND_IN = r"""
#include <cstdint>
#include <cstdio>
#include <map>
#include <string>
struct Dim { uint32_t x, y, z; };
static std::map<const void*, std::string>& names() { static std::map<const void*, std::string> n; return n; }
static std::string log_;
static int last;
static Dim grid_, block_;
static size_t shared_;
static void* stream_;
extern "C" {
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipGetLastError() { int e = last; last = 0; return e; }
int hipGetSymbolAddress(void** p, const void*) { *p = (void*)4096; return 0; }
void** __hipRegisterFatBinary(const void*) { static void* module; return &module; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*,
                           void*, int*) { names()[host] = name; }
int __hipPushCallConfiguration(Dim g, Dim b, size_t s, void* t) {
  grid_ = g; block_ = b; shared_ = s; stream_ = t;
  return 0;
}
int __hipPopCallConfiguration(Dim* g, Dim* b, size_t* s, void** t) {
  *g = grid_; *b = block_; *s = shared_; *t = stream_;
  return 0;
}
int hipLaunchKernel(const void* f, Dim g, Dim b, void**, size_t, void*) {
  const uint64_t limit = uint64_t(1) << 32;
  if (!g.x || !g.y || !g.z || uint64_t(g.x) * b.x >= limit || uint64_t(g.y) * b.y >= limit) return last = 9;
  char line[2048];
  snprintf(line, sizeof line, "%s %u %u %u %u\n", names()[f].c_str(), g.x, g.y, g.z, b.x);
  log_ += line;
  return 0;
}
const char* launched() { return log_.c_str(); }
void forget() { log_.clear(); }
}
"""

RUN = r"""
import ctypes, json, sys
hip = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
hip.launched.restype = ctypes.c_char_p
results = []
for name, args in json.load(sys.stdin):
    def argument(v):
        if v is None or isinstance(v, int):
            return v if v is None else ctypes.c_int64(v)
        if isinstance(v, list):
            return (ctypes.c_float * len(v))(*v)
        return ctypes.c_void_p(int(v[1:])) if isinstance(v, str) else ctypes.c_float(v)
    hip.forget()
    status = getattr(lib, name)(*map(argument, args))
    results.append([status, hip.launched().decode().split("\n")[:-1]])
json.dump(results, sys.stdout)
"""


def kernel_name(mangled):
    """``fp8_gemm_pipe<0,64,64,4,0,1>`` of a mangled kernel of the library."""
    head = re.match(r"_ZN3vfa(\d+)", mangled)
    start, length = head.end(), int(head.group(1))
    name, rest = mangled[start : start + length], mangled[start + length :]
    arguments = re.match(r"I((?:L[ib]n?\d+E)+)E", rest)
    if arguments is None:
        return name
    values = [v.replace("n", "-") for v in re.findall(r"L[ib](n?\d+)E", arguments.group(1))]
    return f"{name}<{','.join(values)}>"


def launches(tmp_path, calls):
    """Run C-ABI calls, ``(entry, arguments)`` with integers as int64, floats as
    float, ``"@address"`` as a pointer, lists as arrays of float and None as NULL.
    Returns for each its status and its launches ``(kernel, (x, y, z), threads)``, the kernel as
    ``kernel_name`` gives it."""
    stand_in = tmp_path / "hip_stand_in.so"
    source = tmp_path / "hip_stand_in.cpp"
    if not stand_in.exists():
        source.write_text(STAND_IN)
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(source), "-o", str(stand_in)], check=True)
    done = subprocess.run([sys.executable, "-c", RUN, str(stand_in), str(LIBRARY)], input=json.dumps(calls),
                          capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stderr
    out = []
    for status, lines in json.loads(done.stdout):
        fields = [line.split() for line in lines]
        out.append((status, [(kernel_name(f[0]), tuple(map(int, f[1:4])), int(f[4])) for f in fields]))
    return out
