"""DeviceArray (host/hip_util.h) when an allocation fails: it holds no elements, says so on every later use, and
the failure is not left behind for the next launch check.  The size asked for is larger than any device, so the
allocation fails with and without a GPU."""
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
  return 0;
}
"""


def test_failed_allocation_leaves_an_empty_array():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "device_array.cc"), os.path.join(d, "device_array")
        with open(src, "w") as f:
            f.write(SOURCE)
        subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", ROOT, "-I", "/opt/rocm/include", src,
                        "-o", exe, "-L", "/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib",
                        "-L", os.path.join(ROOT, "linmt_amd"), "-llinmt_hip",
                        "-Wl,-rpath," + os.path.join(ROOT, "linmt_amd")], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
