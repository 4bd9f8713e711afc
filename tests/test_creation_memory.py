"""Device memory while a 3D handle is created, on the CPU: a small stand-in for
the HIP calls that atmo_create makes hands out host memory and counts it (the
kernels are not run).  The copy of the metric terms in the caller's layout, which
creation needs for a moment, may not raise the largest amount held at once above
what the finished handle holds, or a mesh that fits would be refused."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STAND_IN = r"""
#include <cstdlib>
#include <cstring>
#include <map>
static std::map<void*, size_t> sizes;
static size_t now = 0, most = 0;
extern "C" {
size_t held_now() { return now; }
size_t held_most() { return most; }
int hipMalloc(void** p, size_t n) {
  *p = std::malloc(n ? n : 1);
  sizes[*p] = n;
  now += n;
  if (now > most) most = now;
  return 0;
}
int hipFree(void* p) {
  if (!p) return 0;
  now -= sizes[p];
  sizes.erase(p);
  std::free(p);
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) { *p = std::malloc(n ? n : 1); return 0; }
int hipHostFree(void* p) { std::free(p); return 0; }
int hipHostGetDevicePointer(void** d, void* p, unsigned) { *d = p; return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { std::memcpy(d, s, n); return 0; }
int hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { *s = nullptr; return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamDestroy(void*) { return 0; }
struct dim3_ { unsigned x, y, z; };
int hipLaunchKernel(const void*, dim3_, dim3_, void**, size_t, void*) { return 0; }
int hipGetLastError() { return 0; }
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
}
"""

PROGRAM = r"""
import ctypes, os, sys
held = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # found before the HIP runtime
held.held_now.restype = held.held_most.restype = ctypes.c_size_t
sys.path.insert(0, sys.argv[2])
import trixiatmo_hip as T
mesh, eq, solver, bcs, u0 = T.workloads.periodic_cube(trees=4, polydeg=int(sys.argv[3]), seed=0,
                                                      precision=sys.argv[4])
semi = T.SemidiscretizationHyperbolic(mesh, eq, solver, bcs,
                                      metric_terms_on_device=sys.argv[5] == "device")
nodes = mesh.n_elements * mesh.nnodes ** 3
print(nodes, held.held_now(), held.held_most(), flush=True)
os._exit(0)
"""


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("stand_in")
    (d / "hip.cpp").write_text(STAND_IN)
    lib = str(d / "libheld.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(d / "hip.cpp"), "-o", lib], check=True)
    return lib


@pytest.mark.parametrize("metrics", ["device", "host"])
@pytest.mark.parametrize("polydeg,precision", [(1, "fp64"), (3, "fp64"), (4, "fp32_geometry"),
                                               (3, "fp32_kahan")])
def test_creation_holds_no_more_than_the_handle(stand_in, polydeg, precision, metrics):
    run = subprocess.run([sys.executable, "-c", PROGRAM, stand_in,
                          os.path.join(ROOT, "trixiatmo.jl_amd"), str(polydeg), precision, metrics],
                         capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stderr[-2000:]
    nodes, now, most = map(int, run.stdout.split())
    assert now >= (6 * 6 + 9 + 1) * 8 * nodes  # six states, the metric terms: all went this way
    assert most == now, (most - now) / nodes
