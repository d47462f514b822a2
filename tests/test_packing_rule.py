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
