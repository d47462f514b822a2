"""When a layer makes packed copies of its gate matrices (LstmLayer::PackGates, host/nmt.h)."""
from tests.test_device_array import _run

PAYS = r"""
#include "linmt_amd/host/nmt.h"
using namespace linmt;

int main() {
  const size_t one = lh_gate_pack_floats(1000, 1000);
  const struct { size_t floats; int saved_ns, steps; bool pays; } cases[] = {
      {one, 2400, 5, false}, {one, 2400, 6, true},          // 14.3 us for one matrix of 1000 hidden units
      {2 * one, 4500, 5, false}, {2 * one, 4500, 6, true},  // 24.6 us for two
      {one, 1, 1000, false}, {one, 2400, 0, false}, {one, 2400, -3, false}, {0, 1, 1, false}};
  for (const auto &c : cases)
    if (LstmLayer::PackingPays(c.floats, c.saved_ns, c.steps) != c.pays) {
      printf("%zu floats, %d ns, %d steps: expected %d\n", c.floats, c.saved_ns, c.steps, (int)c.pays);
      return 1;
    }
  return 0;
}
"""


def test_packing_pays_within_the_pass():
    _run(PAYS)

FITS = r"""
#include "linmt_amd/host/nmt.h"
using namespace linmt;

int main() {
  const size_t GB = size_t(1) << 30, total = 288 * GB;
  const struct { size_t bytes, free, total; bool fits; } cases[] = {
      {GB, 280 * GB, total, true}, {GB, 73 * GB, total, true}, {GB, 73 * GB - 1, total, false},
      {GB, GB, total, false}, {GB, GB - 1, total, false}, {GB, 0, total, false}, {80 * GB, 79 * GB, total, false},
      {SIZE_MAX, total, total, false}};
  for (const auto &c : cases)
    if (LstmLayer::PackedCopiesFit(c.bytes, c.free, c.total) != c.fits) {
      printf("%zu bytes, %zu of %zu free: expected %d\n", c.bytes, c.free, c.total, (int)c.fits);
      return 1;
    }
  // what an optional allocation may be short of, and what it must not hide
  if (!DeviceArray<float>::NoMemory(hipErrorOutOfMemory) || DeviceArray<float>::NoMemory(hipErrorIllegalAddress) ||
      DeviceArray<float>::NoMemory(hipErrorLaunchFailure))
    return 2;
  return 0;
}
"""


def test_copies_leave_a_quarter_of_the_memory():
    _run(FITS)
