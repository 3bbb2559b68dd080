"""The context's allocations and its wait for a solve's progress on the CPU:
hb_context.cpp with a HIP runtime of a few functions that counts bytes, so that
running out of memory is a matter of arithmetic.  What spare() holds gives way
to every other field, and spare() itself leaves a quarter of the memory free."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "bqcd-r399-quda_amd", "csrc")
CLANG = "/opt/rocm/llvm/bin/clang++"

RUNTIME = r"""
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include "hb_internal.h"

static size_t total = 1 << 20, used = 0;
static std::map<void *, size_t> blocks;
static unsigned host_flags = ~0u;
static int queries = 0;
extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  *p = nullptr;
  if (used + n > total) return hipErrorOutOfMemory;
  used += n;
  blocks[*p = malloc(1)] = n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (p) used -= blocks.at(p);
  blocks.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) { host_flags = flags; *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = total - used; *t = total; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return ++queries < 3 ? hipErrorNotReady : hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
}
namespace hb { void noalloc_setup(int) {} }

#define EXPECT(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
  const int L[4] = {2, 2, 2, 2}, bc[4] = {1, 1, 1, -1};
  hb_context *h = nullptr;
  EXPECT(hb_init(L, bc, 0, &h) == HB_OK);
  EXPECT(host_flags & hipHostMallocCoherent);  // the words that running kernels report to
  hb::Context *c = reinterpret_cast<hb::Context *>(h);
  const size_t base = used, unit = (total - base) / 16;
  int rc = 0;
  // kept, grown, and taken back by each kind of allocation that needs the room
  void *s = hb::spare(c, 4 * unit);
  EXPECT(s && hb::spare(c, 3 * unit) == s && used == base + 4 * unit);
  EXPECT(hb::spare(c, 8 * unit) && used == base + 8 * unit);
  EXPECT(hb::scratch(c, 3, 12 * unit, &rc) && rc == HB_OK && used == base + 12 * unit);
  // a quarter of the memory has to stay free: no spare fields, and no error
  EXPECT(!hb::spare(c, unit) && used == base + 12 * unit && !*hb_last_error());
  EXPECT(!hb::scratch(c, 4, 8 * unit, &rc) && rc == HB_E_NOMEM);
  EXPECT(hb::scratch(c, 3, 12 * unit, &rc) && rc == HB_OK);
  hb_finalize(h);
  EXPECT(used == 0);
  EXPECT(hb_init(L, bc, 0, &h) == HB_OK);
  c = reinterpret_cast<hb::Context *>(h);
  EXPECT(hb::spare(c, 8 * unit) && hb::ensure_dev_stage(c, 12 * unit) == HB_OK);
  double2 *p = nullptr;
  EXPECT(hb::spare(c, unit / 2) == nullptr);
  EXPECT(hb::device_alloc(c, &p, 8 * unit) == hipErrorOutOfMemory);
  EXPECT(hb::device_alloc(c, &p, 2 * unit) == hipSuccess);
  (void)hipFree(p);
  // the wait for a report asks the runtime now and then, and ends with an error
  // when the stream is empty and nothing has been reported
  uint64_t v = 0;
  const auto t = std::chrono::steady_clock::now();
  EXPECT(hb::wait_note(c, 0, 5, &v) == HB_E_HIP && queries == 3);
  EXPECT(std::chrono::steady_clock::now() - t > std::chrono::milliseconds(100));
  c->note[0] = 5 << 2 | 1;
  EXPECT(hb::wait_note(c, 0, 5, &v) == HB_OK && v == (5 << 2 | 1) && queries == 3);
  hb_finalize(h);
  EXPECT(used == 0);
  return 0;
}
"""


@pytest.mark.skipif(not os.path.exists(CLANG), reason="no HIP compiler")
def test_allocations_and_wait(tmp_path):
    (tmp_path / "runtime.cpp").write_text(RUNTIME)
    exe = str(tmp_path / "context")
    subprocess.run([CLANG, "-O1", "-std=c++17", "-x", "hip", "--offload-host-only", "-I" + CSRC,
                    "-I" + os.path.join(REPO, "include"), "--rocm-path=/opt/rocm", "-no-hip-rt",
                    str(tmp_path / "runtime.cpp"), os.path.join(CSRC, "hb_context.cpp"), "-o", exe], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout + p.stderr
