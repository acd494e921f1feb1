"""Which reads of a caller's address a kernel may do (csrc/read_route.h), compiled for the host: only words
of a live column named by its first address. Everything else (an index past the column, an address inside
one, of another owner, or stale) goes to the copy engine, which can refuse it."""
import os
import re
import shutil
import subprocess

import pytest

from hip_lib import PKG

CSRC = os.path.join(PKG, "csrc")
HARNESS = r"""
#include <cstdio>
#include "read_route.h"
using namespace sh;
int main() {
  uint32_t* const col = (uint32_t*)0x7f0000001000ull;
  LiveColumns live;
  live[col] = 4 * 1024;
  const size_t top = ~(size_t)0;
  const struct { const uint32_t* p; size_t first, words; bool kernel; } cases[] = {
      {col, 0, 0, true}, {col, 0, 1, true}, {col, 0, 1024, true}, {col, 1023, 1, true}, {col, 1015, 9, true},
      {col, 0, 1025, false}, {col, 1024, 1, false}, {col, 1016, 9, false}, {col, 1025, 0, false},
      {col, top, 1, false}, {col, top, top, false}, {col, 1, top, false}, {col, top / 4, 1, false},
      {col, top / 4 + 1, 1, false}, {col, 0, top / 4 + 2, false},
      {col + 1, 0, 1, false}, {col - 1, 1, 1, false}, {nullptr, 0, 1, false}, {(const uint32_t*)&live, 0, 1, false}};
  int bad = 0;
  for (const auto& c : cases)
    if (kernel_may_read(live, c.p, c.first, c.words) != c.kernel) {
      std::printf("%p + %zu, %zu words: not %d\n", (const void*)c.p, c.first, c.words, c.kernel);
      ++bad;
    }
  live.erase(col);  // freed
  bad += kernel_may_read(live, col, 0, 1);
  return bad;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_only_live_columns_are_read_by_a_kernel(tmp_path):
    src, exe = tmp_path / "route.cpp", tmp_path / "route"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("entry,arg", [("stwo_hip_copy_d2h", "src"), ("stwo_hip_column_at", "col"),
                                       ("stwo_hip_channel_read", "state")])
def test_reads_of_callers_addresses_take_the_checked_route(entry, arg):
    """The entries that read an address of the caller's go through read_column, whose route is the above."""
    text = open(os.path.join(CSRC, "capi.cpp")).read()
    body = re.search(r"^int %s\(.*?\n}\n" % entry, text, re.S | re.M).group(0)
    assert re.search(r"read_column\(\w+, %s, " % arg, body) and "read_own(" not in body and "d2h(" not in body.replace(entry, "")
