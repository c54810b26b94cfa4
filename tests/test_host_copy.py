"""csrc/host_copy.cpp against a made-up HIP runtime on the CPU that counts its
calls: when the pinned pieces are set up, and that every byte arrives."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "combustioncodegpu_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>
typedef int hipError_t;
typedef struct Stream *hipStream_t;
typedef struct Event { int x; } *hipEvent_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1 };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
inline std::atomic<int> n_pinned{0}, n_plain{0}, n_async{0};
inline int hipHostMalloc(void **p, size_t n, unsigned) { ++n_pinned; *p = std::malloc(n); return 0; }
inline int hipHostFree(void *p) { --n_pinned; std::free(p); return 0; }
inline int hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new Event; return 0; }
inline int hipEventDestroy(hipEvent_t e) { delete e; return 0; }
inline int hipEventRecord(hipEvent_t, hipStream_t) { return 0; }
inline int hipEventSynchronize(hipEvent_t) { return 0; }
inline int hipStreamSynchronize(hipStream_t) { return 0; }
inline int hipStreamGetDevice(hipStream_t, int *d) { *d = 0; return 0; }
inline int hipGetDevice(int *d) { *d = 0; return 0; }
inline int hipSetDevice(int) { return 0; }
inline int hipGetLastError() { return 0; }
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
struct hipPointerAttribute_t { hipMemoryType type; };
inline int memory_type = 0;  // of every destination; -1: the runtime does not know the pointer
inline int hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
  if (memory_type < 0) return hipErrorInvalidValue;
  a->type = (hipMemoryType)memory_type;
  return 0;
}
inline int hipMemcpy(void *d, const void *s, size_t n, int) { ++n_plain; std::memcpy(d, s, n); return 0; }
inline int hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) { ++n_async; std::memcpy(d, s, n); return 0; }
"""

HARNESS = r"""
#include <cstdio>
#include <vector>
#include "host_copy.h"
// argv: the destinations' memory type, copies in MiB; prints for each whether it went through hipMemcpy, the pinned pieces there are, and
// whether every byte arrived
int main(int argc, char **argv) {
  {
    cfx::HostCopy c;
    memory_type = std::atoi(argv[1]);
    for (int a = 2; a < argc; ++a) {
      const size_t n = (size_t)(std::atof(argv[a]) * 1048576) + 13;
      std::vector<unsigned char> src(n), dst(n + 8, 77);
      for (size_t i = 0; i < n; ++i) src[i] = (unsigned char)(i * 2654435761u >> 13);
      const int plain = n_plain, rc = c.to_host(dst.data(), src.data(), n, nullptr);
      bool ok = rc == 0 && std::memcmp(dst.data(), src.data(), n) == 0;
      for (int i = 0; i < 8; ++i) ok = ok && dst[n + i] == 77;
      std::printf("%d %d %d\n", n_plain - plain, (int)n_pinned, ok ? 1 : 0);
    }
  }
  std::printf("left %d\n", (int)n_pinned);
  return 0;
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_copy")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (d / "main.cpp").write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(d), "-I", CSRC, str(d / "main.cpp"),
                    os.path.join(CSRC, "host_copy.cpp"), "-o", str(d / "main")], check=True)

    def run(*mib, memory=0):
        r = subprocess.run([str(d / "main"), str(memory)] + [str(m) for m in mib], capture_output=True, text=True, check=True)
        rows = r.stdout.split("\n")[:-1]
        assert rows[-1] == "left 0"
        return [tuple(map(int, x.split())) for x in rows[:-1]]
    return run


def test_few_copies_do_not_pay_for_the_pieces(exe):
    """One to three copies of 8 to 25 MB, the fields of one block: all as hipMemcpy
    would do them, nothing pinned."""
    assert exe(8.5, 24, 7) == [(1, 0, 1)] * 3
    assert exe(16, 30, 30) == [(1, 0, 1)] * 3
    assert exe(81.8) == [(1, 0, 1)]


@pytest.mark.parametrize("before,last", [([], 96), ([], 130.3), ([40, 40], 16), ([8.5] * 11, 8.5), ([3] * 40 + [90], 9)])
def test_pieces_where_they_are_worth_it(exe, before, last):
    """A large copy, or the one with which the copies so far have been worth it."""
    rows = exe(*before, last, 20, 1, 9)
    assert rows[:len(before)] == [(1, 0, 1)] * len(before)
    pinned = rows[len(before)][1]
    assert 1 <= pinned <= 8
    assert rows[len(before):] == [(0, pinned, 1), (0, pinned, 1), (1, pinned, 1), (0, pinned, 1)]


@pytest.mark.parametrize("memory", [1, 2])
def test_pinned_or_device_destination(exe, memory):
    """The runtime copies there by itself: no pieces, no store by the processor."""
    assert exe(130.3, 100, memory=memory) == [(1, 0, 1)] * 2


def test_unknown_pointer_is_ordinary_memory(exe):
    rows = exe(130.3, memory=-1)
    assert rows[0][0] == 0 and rows[0][2] == 1
