"""The division by the page size as a multiplication and a shift (page_magic / magic_div, which every
kernel uses): compiled for the host and compared with the division at the page edges, over the whole
range of tokens it is stated for (0 <= x < 2^31). CPU only."""
import pathlib
import subprocess
import sys

import pytest

REPO = pathlib.Path(__file__).resolve().parent.parent
sys.path.insert(0, str(REPO / "qwen-mla-vllm_amd"))

SOURCE = r"""
#include <cstdio>
#include <vector>
#include "qmla_common.h"
int main() {
  std::vector<int64_t> ds;
  for (int l = 0; l < 31; ++l)
    for (int64_t k = -3; k <= 3; ++k) ds.push_back((int64_t(1) << l) + k);
  for (int64_t d : {48LL, 784LL, 1600LL, 4095LL, 46341LL, 2147483647LL, 2147483646LL}) ds.push_back(d);
  uint64_t r = 1;
  for (int i = 0; i < 2000; ++i) {
    r = r * 6364136223846793005ULL + 1442695040888963407ULL;
    ds.push_back(int64_t(r >> 33) >> (i % 31));
  }
  const int64_t top = 2147483647;
  long n = 0;
  for (int64_t d : ds) {
    if (d < 1 || d > top) continue;
    uint32_t mul;
    int sh;
    qmla::page_magic(int(d), mul, sh);
    auto check = [&](int64_t x) {
      if (x < 0 || x > top) return true;
      ++n;
      return int64_t(qmla::magic_div(uint32_t(x), mul, sh)) == x / d;
    };
    const int64_t km = top / d;
    for (int64_t i = 0; i < 200; ++i)
      for (int64_t k : {i, km - i, km / 2 + i, km * i / 200})
        for (int64_t e = -2; e <= 2; ++e)
          if (!check(k * d + e)) return std::printf("d %lld x %lld\n", (long long)d, (long long)(k * d + e)), 1;
    for (int64_t x = top - 5; x <= top; ++x)
      if (!check(x)) return std::printf("d %lld x %lld\n", (long long)d, (long long)x), 1;
  }
  std::printf("%ld divisions\n", n);
  return 0;
}
"""


def test_page_division(tmp_path):
    import build as qbuild
    try:
        hipcc = qbuild.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    src, exe = tmp_path / "magic.hip", tmp_path / "magic"
    src.write_text(SOURCE)
    r = subprocess.run([hipcc, *qbuild.COMMON_FLAGS, f"-I{REPO / 'include'}", f"-I{qbuild.CSRC}", str(src), "-o", str(exe)],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 1_000_000
