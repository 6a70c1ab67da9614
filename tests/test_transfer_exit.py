"""A host program whose own global gives its handle back after main (its destructor runs after those
of statics made later): the pinned slots are still there, and each allocation is freed once."""
import os
import shutil
import subprocess

import pytest

from littleharsh_amd.build import HERE
from test_transfer_host import STUB

MAIN = r"""
#include <cstdio>
#include <set>
#include <unistd.h>
static std::set<void*>& blocks() {
  static std::set<void*>* const s = new std::set<void*>;
  return *s;
}
inline void seen(void* p, bool made) {
  if (made) {
    blocks().insert(p);
  } else if (blocks().erase(p) != 1) {
    std::puts("failed: freed what was not allocated");
    std::fflush(stdout);
    _exit(1);
  }
}
#include "lh_xfer.hpp"

struct Owner {
  double* slot = nullptr;
  ~Owner() {
    lh::host_stage().release(slot);
    std::puts(blocks().empty() ? "ok" : "failed: not given back");
    std::fflush(stdout);
  }
};
static Owner owner;
int main() { owner.slot = lh::host_stage().retain(); }
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_a_handle_given_back_after_main(tmp_path):
    (tmp_path / "hip").mkdir()
    stub = STUB.replace("*p = std::malloc(n);", "*p = std::malloc(n); seen(*p, true);").replace(
        "std::free(p);", "seen(p, false); std::free(p);")
    assert stub.count("seen(") == 2
    (tmp_path / "hip" / "hip_runtime.h").write_text(stub)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "t"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-pthread", "-I", str(tmp_path), "-I", os.path.join(HERE, "csrc"),
                        str(tmp_path / "main.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    # (freed memory is overwritten, so that a use of it shows)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100, env={**os.environ, "MALLOC_PERTURB_": "90"})
    assert (r.returncode, r.stdout) == (0, "ok\n"), r.stdout + r.stderr
