"""The host side of the kernel libraries without a GPU: a child process loads a stand-in for the HIP runtime (compiled
from the source below) in front of a built library, calls entries with made-up operands and gives back what they
launched. The stand-in has several devices, and refuses a launch that wants more than 64 KB of dynamic LDS on a device
on which the kernel was not allowed that much."""
import json
import os
import subprocess
import sys

from pytriton_llama_amd.ops import library

# the tiles of csrc/gemm_tile.hip in their order: rows of x, rows of W, workgroups a compute unit
TILES = [(64, 64, 2), (64, 128, 1), (128, 64, 1), (96, 128, 1), (128, 128, 1), (160, 128, 1), (192, 128, 1), (128, 192, 1),
         (96, 256, 1), (112, 256, 1), (128, 256, 1), (144, 256, 1)]

RUNTIME = r"""
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <utility>
struct dim3 { uint32_t x, y, z; };
static int device = 0, last = 0;
static std::map<const void*, std::string> names;
static std::map<std::pair<int, const void*>, int> allowed;
static std::string launches;
static struct { dim3 grid, block; size_t lds; void* stream; } config;
extern "C" {
int hipGetDevice(int* d) { *d = device; return 0; }
int hipSetDevice(int d) { device = d; return 0; }
int hipGetLastError() { int e = last; last = 0; return e; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }      // (asked for compute units only)
int hipFuncSetAttribute(const void* f, int, int v) { allowed[{device, f}] = v; return 0; }
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* s) { config = {g, b, lds, s}; return 0; }
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** s) {
  *g = config.grid; *b = config.block; *lds = config.lds; *s = config.stream;
  return 0;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t lds, void*) {
  auto at = allowed.find({device, f});
  if (lds > 65536 && (at == allowed.end() || (size_t)at->second < lds)) return last = 1;
  char text[128];
  snprintf(text, sizeof text, "\t%d\t%u\t%u\t%u\t%u\t%zu\n", device, g.x, g.y, g.z, b.x, lds);
  launches += names[f] + text;
  return 0;
}
const char* take_launches() { static std::string out; out.swap(launches); launches.clear(); return out.c_str(); }
}
"""

CHILD = r"""
import ctypes, json, sys
runtime = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)      # found before the real one
runtime.take_launches.restype = ctypes.c_char_p
lib = ctypes.CDLL(sys.argv[2])
out = []
for device, entry, args in json.load(sys.stdin):
    runtime.hipSetDevice(device)
    kinds = {"p": ctypes.c_void_p, "i": ctypes.c_int, "l": ctypes.c_long, "f": ctypes.c_float}
    code = getattr(lib, entry)(*[kinds[k](v) for k, v in args])
    took = [line.split("\t") for line in runtime.take_launches().decode().splitlines()]
    out.append({"code": code, "launches": [
        {"kernel": t[0], "device": int(t[1]), "grid": [int(v) for v in t[2:5]], "threads": int(t[5]), "lds": int(t[6])}
        for t in took]})
print(json.dumps(out))
"""


def run(folder, name, calls):
    """What the calls [(device, entry, [(kind, value), ...]), ...] of library ``name`` returned and launched; kinds: p
    (a pointer), i, l (int, long), f. ``folder``: where the stand-in is built."""
    if library.is_stale(name):
        library.build([name])
    stand_in = os.path.join(str(folder), "libstand_in.so")
    if not os.path.isfile(stand_in):
        source = os.path.join(str(folder), "stand_in.cpp")
        with open(source, "w") as f:
            f.write(RUNTIME)
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", stand_in, source], check=True)
    done = subprocess.run([sys.executable, "-c", CHILD, stand_in, library.library_path(name)], input=json.dumps(calls),
                          capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stderr
    return json.loads(done.stdout)
