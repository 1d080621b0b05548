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
