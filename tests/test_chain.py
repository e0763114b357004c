"""The device-side choice between the int8 and the FP32 path (dq8::Chain,
dq8_internal.h): calls that wrongly overlap may mix up their own answers, but a
call in order after them must see its own inputs only.

The state's rules are compiled from the library's own header into a host program
that runs two overlapping calls in every interleaving of their memory accesses
(the quantizer's report reads next and later stores hit; its first block copies
next into cur; the close reads hit and cur and later raises next), for every pair
of finite and non-finite inputs, and then four calls in order.  A close that only
counts on (next = cur + 1) must be caught."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "decider-engine_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include "dq8_internal.h"
#include <stdio.h>
#include <algorithm>
using dq8::Chain;
static int counted_on = 0;  // the planted fault: a plain store of cur + 1
struct Call {
  bool bad;       // reports a non-finite input
  int open_at;    // its first block's copy of next happens before (0), between (1) or after (2) the report's accesses
  int step = 0;
  uint64_t opened = 0, seen = 0, hit = 0, cur = 0;
  bool answer = false;
};
// One access of a call; false when it has ended.
static bool advance(Call& c, Chain& s) {
  const int order[3][4] = {{0, 1, 2, 3}, {2, 0, 1, 3}, {2, 3, 0, 1}};  // 0, 1: open reads, stores; 2, 3: report reads, stores
  if (c.step < 4) {
    switch (order[c.open_at][c.step++]) {
      case 0: c.opened = s.next; break;
      case 1: s.cur = c.opened; break;
      case 2: if (c.bad) c.seen = s.next; break;
      default: if (c.bad) s.hit = Chain::report(c.seen);
    }
    return true;
  }
  switch (c.step++) {
    case 4: c.answer = Chain::reported(s.hit, s.cur); break;  // the int8 launch asks
    case 5: c.hit = s.hit; c.cur = s.cur; break;              // the close reads
    case 6:
      if (counted_on) s.next = c.cur + 1;
      else s.next = std::max(s.next, Chain::closed(c.hit, c.cur));
      break;
    default: return false;
  }
  return true;
}
static int wrong = 0;
static long paths = 0;
static void later(Chain s) {
  ++paths;
  for (bool bad : {false, true, true, false}) {
    for (int at = 0; at < 3; ++at) {
      Call c;
      c.bad = bad;
      c.open_at = at;
      while (advance(c, s)) {}
      if (c.answer != bad) ++wrong;
    }
  }
}
static void interleave(Call a, Call b, Chain s) {
  if (a.step == 7 && b.step == 7) return later(s);
  if (a.step < 7) {
    Call a2 = a;
    Chain s2 = s;
    advance(a2, s2);
    interleave(a2, b, s2);
  }
  if (b.step < 7) {
    Call b2 = b;
    Chain s2 = s;
    advance(b2, s2);
    interleave(a, b2, s2);
  }
}
int main(int argc, char** argv) {
  counted_on = argc > 1;
  for (int bads = 0; bads < 4; ++bads)
    for (int at = 0; at < 9; ++at) {
      Call a, b;
      a.bad = bads & 1;
      b.bad = bads & 2;
      a.open_at = at / 3;
      b.open_at = at % 3;
      interleave(a, b, Chain{5, 4, 3});
      interleave(a, b, Chain{5, 4, 5});  // the call before them reported
      interleave(a, b, Chain{0, 0, 0});
    }
  printf("%ld interleavings, %d wrong answers\n%s\n", paths, wrong, wrong ? "FAIL" : "OK");
  return 0;
}
"""


@pytest.fixture(scope="module")
def chain_program(tmp_path_factory):
    if shutil.which(HIPCC) is None and not os.path.exists(HIPCC):
        pytest.skip("needs hipcc to compile against the HIP headers")
    d = tmp_path_factory.mktemp("chain")
    src, exe = d / "chain_check.cpp", d / "chain_check"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True,
                   capture_output=True, timeout=300)
    return str(exe)


def test_ordered_calls_after_overlapping_ones_see_their_own_inputs(chain_program):
    out = subprocess.run([chain_program], check=True, capture_output=True, text=True, timeout=300).stdout
    assert out.strip().splitlines()[-1] == "OK", out


def test_chain_check_catches_a_close_that_only_counts_on(chain_program):
    out = subprocess.run([chain_program, "planted"], check=True, capture_output=True, text=True, timeout=300).stdout
    assert out.strip().splitlines()[-1] == "FAIL", out
