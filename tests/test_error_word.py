"""The error word a kernel sets is published by the iteration's last block, so
the write has to be complete before the writer's block takes its ticket.  No
call can make a kernel set it (the plan rules the states out), so this looks
at the code: every kernel of the two methods sets the word through raise_err,
and what raise_err compiles to waits for the atomic's result before the
barrier in front of the ticket."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "galp_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

KERNEL = """
#include "device_common.hpp"
using namespace galp;
__global__ void __launch_bounds__(256) k(int32_t *err, unsigned long long *counter, IterEnd e) {
    __shared__ uint32_t scratch[4];
    if (threadIdx.x == 192) raise_err(err, 8);
    block_count_end<4>(1u, counter, scratch, e);
}
"""


@pytest.mark.parametrize("name", ["lp_hash.hip", "lp_sort.hip"])
def test_kernels_set_the_error_word_through_raise_err(name):
    with open(os.path.join(CSRC, name)) as f:
        src = re.sub(r"//[^\n]*", "", f.read())
    assert "raise_err(err," in src
    assert not re.search(r"atomic\w*\(\s*err\b", src) and not re.search(r"\*\s*err\s*=[^=]", src)


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_raise_err_waits_before_the_ticket(tmp_path):
    (tmp_path / "k.hip").write_text(KERNEL)
    out = tmp_path / "k.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-device-only", "-O3", "-std=c++17", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + CSRC, "-S", "-o", str(out),
                    str(tmp_path / "k.hip")], check=True, capture_output=True)
    ops = [ln.strip() for ln in out.read_text().splitlines()]
    at = next(i for i, ln in enumerate(ops) if ln.startswith("global_atomic_or"))
    assert "sc0" in ops[at].split()[-2:], ops[at]   # returns its result
    wait = next(i for i in range(at, len(ops)) if ops[i].startswith("s_waitcnt") and "vmcnt(0)" in ops[i])
    barrier = next(i for i in range(at, len(ops)) if ops[i].startswith("s_barrier"))
    assert wait < barrier
