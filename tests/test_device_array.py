"""DeviceArray (host/hip_util.h) when an allocation fails: it holds no elements, says so on every later use, and
the failure is not left behind for the next launch check.  The size asked for is larger than any device, so the
allocation fails with and without a GPU.  And what scoring makes of memory it does not get (SoftmaxLayer::
LossGroupSteps, host/nmt.h): smaller groups of steps, at last one step in the buffers the model has."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "linmt_amd/host/hip_util.h"
using namespace linmt;

template <typename F>
bool Throws(F &&f) {
  try {
    f();
  } catch (const LinmtError &) {
    return true;
  }
  return false;
}

#define EXPECT(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

int main() {
  const size_t huge = size_t(1) << 55;
  int devices = 0;  // without one, every call of the runtime reports that
  const bool gpu = hipGetDeviceCount(&devices) == hipSuccess && devices > 0;
  (void)hipGetLastError();
  DeviceArray<float> a;
  float v = 0;
  EXPECT(Throws([&] { a.Alloc(huge); }));
  EXPECT(a.size() == 0 && a.get() == nullptr);
  EXPECT(!gpu || hipGetLastError() == hipSuccess);
  EXPECT(Throws([&] { a.Reserve(1000 + huge); }));  // tried again, not taken to be there
  EXPECT(Throws([&] { a.Upload(&v, 1, nullptr); }));
  EXPECT(Throws([&] { a.Download(&v, 1, nullptr); }));
  a.Zero(nullptr);                                  // nothing to clear
  EXPECT(Throws([&] { a.Alloc(SIZE_MAX / 2); }));   // the byte count must not wrap round
  EXPECT(a.size() == 0);
  EXPECT(a.TryReserve(0));
  EXPECT(!a.TryReserve(huge) && a.size() == 0 && a.get() == nullptr);
  EXPECT(!a.TryReserve(SIZE_MAX / 2));
  EXPECT(!gpu || hipGetLastError() == hipSuccess);
  return 0;
}
"""

GROUPS = r"""
#include "linmt_amd/host/nmt.h"
using namespace linmt;

int main() {
  // logits a step, steps, steps that fit, expected steps a group
  const long long cases[][4] = {{100, 7, 1000, 7},            // all at once
                                {(1 << 27) / 3, 7, 1000, 3},  // three groups of at most 2^27 logits: 3, 3, 1
                                {7680000, 41, 1000, 14},      // 17 fit: 14, 14, 13
                                {7680000, 41, 8, 7},          // 14 do not, half of them do
                                {7680000, 41, 6, 3}, {7680000, 41, 2, 1}, {7680000, 41, 0, 1},
                                {1LL << 28, 41, 1000, 1},     // one step is more than a group may have
                                {(1LL << 26) + 1, 5, 1000, 1}, {100, 1, 0, 1}, {1LL << 40, 1, 0, 1}};
  for (auto &c : cases) {
    long long asked = 0;
    const int per = SoftmaxLayer::LossGroupSteps((size_t)c[0], (int)c[1], [&](int n) {
      asked = n;
      return n <= c[2];
    });
    if (per != c[3] || (per > 1 && asked != per)) {
      printf("%lld logits, %lld steps, %lld fit: %d (expected %lld)\n", c[0], c[1], c[2], per, c[3]);
      return 1;
    }
  }
  return 0;
}
"""


def _run(source):
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "program.cc"), os.path.join(d, "program")
        with open(src, "w") as f:
            f.write(source)
        lib = os.path.join(ROOT, "linmt_amd")
        subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", ROOT, "-I", "/opt/rocm/include", src,
                        "-o", exe, "-L", lib, "-llinmt_host", "-llinmt_hip", "-Wl,-rpath," + lib,
                        "-L", "/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr


def test_failed_allocation_leaves_an_empty_array():
    _run(SOURCE)


def test_scoring_takes_smaller_groups_when_memory_is_short():
    _run(GROUPS)
