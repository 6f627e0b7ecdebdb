"""Division by numbers that the host knows, and the map from work-groups to XCDs that is made of it: the headers' own code, compiled for the host,
against plain division."""
import os
import shutil
import subprocess

import pytest

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CSRC = os.path.join(os.path.dirname(__file__), "..", "anchor-attention_amd", "csrc")
PROGRAM = r"""
#include "aa_common.h"
#include <cstdio>
using namespace aa;

static uint32_t by_division(uint32_t wg, uint32_t units, uint32_t per_unit, uint32_t inner, bool abreast) {
  const uint32_t total = units * per_unit, xcd = wg % 8, k = wg / 8;
  if (abreast) {
    if (total % 8 != 0 || units % 8 != 0) return wg % units * per_unit + wg / units;
    const uint32_t own = units / 8, turn = 32 % own == 0 ? k / 32 : 0;
    return ((k + turn) % own * 8 + xcd) * per_unit + k / own;
  }
  if (total % 8 != 0) return wg;
  if (units % 8 == 0) return (k / per_unit * 8 + xcd) * per_unit + k % per_unit;
  const uint32_t s = 8 / units;
  if (8 % units == 0 && (per_unit / inner) % s == 0) return (xcd / s) * per_unit + ((k / inner) * s + xcd % s) * inner + k % inner;
  return wg;
}

int main() {
  const uint32_t top = 0xffffffffu;
  uint32_t state = 1;
  auto next = [&] { return state = state * 1664525u + 1013904223u; };
  for (int i = 0; i < 200000; ++i) {
    const uint32_t d = i < 5000 ? i + 1 : i < 5032 ? 1u << (i - 5000) : i < 5064 ? top >> (i - 5032) : (next() >> next() % 32) | 1u;
    const FastDiv f = fast_div(d);
    const uint32_t q = next() >> next() % 32, some[] = {0, 1, d - 1, d, d + 1, q * d, q * d - 1, q, top, top - 1, top - d};
    for (uint32_t n : some)
      if (quotient(n, f) != n / d) return printf("%u / %u\n", n, d), 1;
  }
  for (uint32_t units : {1, 2, 3, 4, 5, 7, 8, 10, 16, 24, 40, 64})
    for (uint32_t inner : {1, 2, 3, 4, 7})
      for (uint32_t rows : {1, 2, 3, 4, 7, 8, 16, 31, 79})
        for (bool abreast : {false, true}) {
          const Deal deal = make_deal(units, inner * rows, inner, abreast);
          for (uint32_t wg = 0; wg < units * inner * rows; ++wg) {
            uint32_t unit, index;
            dealt(deal, wg, unit, index);
            if (index >= inner * rows || unit * inner * rows + index != by_division(wg, units, inner * rows, inner, abreast))
              return printf("work-group %u of %u units, %u x %u, abreast %d\n", wg, units, inner, rows, abreast), 1;
          }
        }
  return 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no compiler")
def test_quotients_and_the_map_of_work_groups(tmp_path):
    source = tmp_path / "division.hip"
    source.write_text(PROGRAM)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++17", "-O1", "-I", CSRC, str(source), "-o", str(tmp_path / "division")], check=True)
    done = subprocess.run([str(tmp_path / "division")], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
