"""Device functions that also compile for the host, run there: no GPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run_host(tmp_path, source):
    """The standard output of a host program that includes the kernels' headers."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    path = tmp_path / "host.hip"
    path.write_text(source)
    # -fwrapv: 32-bit sums wrap as on the device
    program = str(tmp_path / "host")
    subprocess.run([hipcc, "--offload-host-only", "-O2", "-fwrapv", "-std=c++17", "-ffp-contract=off",
                    f"-I{ROOT}/fastmd_amd/csrc", str(path), "-o", program], check=True, capture_output=True)
    return subprocess.run([program], check=True, capture_output=True, text=True, timeout=60).stdout


@pytest.mark.parametrize("rows", [0, 1, 1000, 2 ** 30, 2 ** 30 + 1, 1_200_000_000, 2 ** 31 - 2])
def test_segment_search_stays_within_its_rows(tmp_path, rows):
    """Runs of 1 000 rows per segment, the keys computed: every offset exact, no key read outside [0, rows)."""
    out = run_host(tmp_path, f"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include "search.h"
struct Keys {{
  mutable bool outside = false;
  uint32_t operator[](int64_t i) const {{
    if (i < 0 || i >= {rows}LL) {{ outside = true; return 0xffffffffu; }}
    return (uint32_t)(i / 1000);
  }}
}};
int main() {{
  const int64_t rows = {rows}LL, segments = (rows + 999) / 1000;
  for (int64_t k = 0; k <= 1000; ++k) {{  // the last one too
    const int64_t s = segments * k / 1000;
    Keys keys;
    const int64_t got = lower_bound(keys, (int32_t)rows, (uint32_t)s);
    if (keys.outside || got != (s * 1000 < rows ? s * 1000 : rows)) {{
      std::printf("segment %lld: %lld, outside %d", (long long)s, (long long)got, (int)keys.outside);
      return 0;
    }}
  }}
  std::printf("ok");
}}
""")
    assert out == "ok"


def test_chain_exponential_and_quotient(tmp_path):
    """exp_small over both signs against the 64-bit-mantissa exponential: within the bound its comment derives, 0.5 +
    2^-6 + 2^-9 units in the last place; div_q: the rounded quotient."""
    out = run_host(tmp_path, """
#include <hip/hip_runtime.h>
#include <cstdio>
#include <random>
#include "nhc_math.h"
int main() {
  std::mt19937_64 gen(1);
  std::uniform_real_distribution<double> uniform(-kExpSmall, kExpSmall), power(-300, 300);
  double worst[2] = {0, 0};  // below 0, above
  for (int k = 0; k < 4000000; ++k) {
    const double x = k == 0 ? -0x1.bd1823ee71d98p-6 : k % 4 == 0 ? uniform(gen) * 1e-3 : uniform(gen);
    const long double off = fabsl((long double)exp_small(x) - expl((long double)x));
    const double units = (double)(off * (x < 0 ? 0x1p53L : 0x1p52L));
    if (units > worst[x >= 0]) worst[x >= 0] = units;
  }
  int wrong = 0;
  for (int k = 0; k < 1000000; ++k) {
    const double a = exp2(power(gen)) * uniform(gen), b = exp2(power(gen) / 2);
    wrong += div_q(a, b, 1.0 / b) != a / b;
  }
  std::printf("%.6f %.6f %d", worst[0], worst[1], wrong);
}
""").split()
    below, above, wrong = float(out[0]), float(out[1]), int(out[2])
    assert 0.5 < max(below, above) <= 0.5 + 2.0 ** -6 + 2.0 ** -9 and wrong == 0
