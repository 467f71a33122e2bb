"""Clearing of the material-point update's pivoting list and terminally-ill
flag (csrc/response_flags.h, host code): the class is compiled with the host
compiler and driven with a model of the launches of an evaluation.  An
evaluation whose last kernels clear the list and the flag for the next one
saves that one's clearing launch, but only when it returned: after one that
threw between the update and its end, the next must clear them itself, or its
appends go on from the old count past the end of a list with room for one
update."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

DRIVER = r"""
#include <cstdio>
#include <stdexcept>
#include "response_flags.h"

struct Device {  // what the launches leave behind
  static const int N = 8;
  int count = 0, ill = 0, highest = 0, resets = 0;
  void update(bool clear) {
    if (clear) { count = 0; ill = 0; ++resets; }
    for (int c = 0; c < N; ++c) if (++count > highest) highest = count;
    ill = 1;
  }
  void finish() { count = 0; ill = 0; }
};

static void evaluate(sca::ResponseFlags& f, Device& d, bool fused, int fail) {
  f.evaluation(fused, [&](bool clear) {
    if (fail == 1) throw std::runtime_error("before the update");
    d.update(clear);
    if (fail == 2) throw std::runtime_error("after the update");
    if (fused) d.finish();
  });
}

int main() {
  // every sequence of four steps, each: fused or not, returning or throwing
  // before / after the update, or an update outside an evaluation
  for (int s = 0; s < 7 * 7 * 7 * 7; ++s) {
    sca::ResponseFlags f;
    Device d;
    d.count = 3;  // unknown contents to begin with
    bool last_fused_ok = false;
    for (int k = 0, t = s; k < 4; ++k, t /= 7) {
      const int kind = t % 7, resets = d.resets;
      if (kind == 6) {
        f.written();
        d.update(true);
        last_fused_ok = false;
      } else {
        const bool fused = kind < 3;
        try {
          evaluate(f, d, fused, kind % 3);
        } catch (const std::exception&) {
        }
        // the launch is saved exactly after a fused evaluation that returned
        if (kind % 3 != 1 && (d.resets == resets) != last_fused_ok) { std::printf("step %d of %d\n", k, s); return 1; }
        last_fused_ok = fused && kind % 3 == 0;
      }
      if (d.highest > Device::N) { std::printf("count %d in sequence %d\n", d.highest, s); return 1; }
    }
  }
  return 0;
}
"""


def test_list_is_cleared_after_an_evaluation_that_threw(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "flags.cpp", tmp_path / "flags"
    src.write_text(DRIVER)
    subprocess.check_call([cxx, "-std=c++17", "-I", os.path.join(ROOT, "solver_cpp_amd", "csrc"), str(src), "-o",
                           str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
