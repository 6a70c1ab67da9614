"""The tile loads of the wave z assembly (lh_zw.hpp) are written as asm, where the compiler puts no
wait states of its own: in its assembly, every load into the LDS must stand at least one wait state
after the write of M0 that it reads its address from, and five after a vector instruction's write of
the scalar registers of its base (the hardware does not interlock either)."""
import os
import re
import shutil
import subprocess

import pytest

from littleharsh_amd.build import HERE, HIPCC_FLAGS

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
SOURCE = """#include <hip/hip_runtime.h>
#include "lh_zw.hpp"
namespace lh {
template __global__ void k_zw<576>(ZW, Dims);
template __global__ void k_zw<384>(ZW, Dims);
}
"""


def instructions(asm):
    out = []
    for line in asm.splitlines():
        line = line.split(";")[0].strip()
        if line and not line.startswith(".") and not line.endswith(":"):
            out.append(line)
    return out


def states_since(ins, i, writes):
    """Wait states between instruction i and the closest one above it that `writes` matches (at most 8)."""
    n = 0
    for j in range(i - 1, -1, -1):
        if n >= 8 or writes(ins[j]):
            return n
        m = re.match(r"s_nop\s+(\d+)", ins[j])
        n += int(m.group(1)) + 1 if m else 1
    return n


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which(HIPCC)), reason="no hipcc")
def test_lds_loads_wait_for_m0_and_their_base(tmp_path):
    src = tmp_path / "k.hip"
    src.write_text(SOURCE)
    flags = [f for f in HIPCC_FLAGS if f not in ("-fPIC", "-shared")]
    r = subprocess.run([HIPCC, *flags, "-I", os.path.join(HERE, "csrc"), "--offload-device-only", "-S", str(src), "-o",
                        str(tmp_path / "k.s")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    ins = instructions((tmp_path / "k.s").read_text())
    loads = [i for i, s in enumerate(ins) if s.startswith("global_load_lds")]
    # a kernel's loop and its first tile: nine loads of 72 chunks, six of 48
    assert len(loads) >= 2 * (9 + 6)
    for i in loads:
        assert states_since(ins, i, lambda s: re.match(r"s_\w+\s+m0\b", s)) >= 1, ins[i - 3:i + 1]
        a, b = map(int, re.search(r"s\[(\d+):(\d+)\]", ins[i]).groups())

        def valu_base(s):
            # the first operand of a vector instruction, where that is a scalar register of the base
            m = re.match(r"v_\w+\s+(?:s(\d+)\b|s\[(\d+):(\d+)\])", s)
            if not m:
                return False
            lo, hi = (int(m.group(1)),) * 2 if m.group(1) else (int(m.group(2)), int(m.group(3)))
            return lo <= b and hi >= a

        assert states_since(ins, i, valu_base) >= 5, ins[i - 6:i + 1]
