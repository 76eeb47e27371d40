"""Bounds that the kernels test (gd_rules.h), compiled for the CPU and compared with
64-bit arithmetic."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(tmp_path, body):
    src, exe = os.path.join(tmp_path, "rules.cpp"), os.path.join(tmp_path, "rules")
    with open(src, "w") as f:
        f.write('#include <cstdio>\n#include <initializer_list>\n#include "gd_rules.h"\n'
                "int main() {\n  long bad = 0;\n" + body +
                '\n  if (bad) std::printf("%ld\\n", bad);\n  return bad != 0;\n}\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "geauxdock_amd", "csrc"), src, "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_rows_fit(tmp_path):
    """Row offsets are 32 bits: 16 rows and fewer fit at every replica count that is
    accepted (2^26), and 20 rows up to the last count whose last lane does."""
    _run(tmp_path, """
  for (long long Rp : {64ll, 1ll << 20, 53687040ll, 53687104ll, (1ll << 26) - 64, 1ll << 26})
    for (int n : {1, 2, 4, 8, 12, 16, 20}) {
      const long long last = ((n - 1) * Rp + Rp - 1) * 4 + 3;  // its last byte
      bad += gd_rows_fit(n, (int)Rp) != (last < (1ll << 32));
      bad += n <= 16 && !gd_rows_fit(n, (int)Rp);
    }
  bad += gd_rows_fit(20, 1 << 26);
""")


def test_queue_room(tmp_path):
    """Entries before the queue's start are refused also where their end wraps to
    its first ones: 8 blocks' entries queued one launch of one step late."""
    _run(tmp_path, """
  for (long long limit : {1ll, 7ll, 64ll, 257ll, 2097152ll})
    for (long long n = 1; n <= 256; ++n)
      for (long long base : {0ll, limit, limit / 2, -256ll, -2097152ll, 4294967295ll - 300})
        for (long long d = -300; d <= 300; ++d) {
          const long long at = base + d;  // what the counters' difference stands for, mod 2^32
          const long long real = at > 2147483647ll ? at - 4294967296ll : at;
          bad += gd_queue_room((uint32_t)at, (uint32_t)n, (uint32_t)limit) != (real >= 0 && real + n <= limit);
        }
  for (int k = 0; k < 8; ++k) bad += gd_queue_room(0u - 64u + 8u * k, 8, 64);
""")
