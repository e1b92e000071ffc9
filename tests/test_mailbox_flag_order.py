"""The kernel that moves words to the host raises the host's flag from one wave: the stores of
every wave have to be complete before the barrier ahead of it.  Checked in the assembly that
the compiler makes of whir_amd/csrc/runtime.hip, since a run shows it only now and then."""
import os
import re
import subprocess

import pytest

from whir_amd import build as B


def kernel_body(asm, name):
    m = re.search(rf"^(_Z\S*{name}\S*):.*?^\.Lfunc_end", asm, re.S | re.M)
    assert m, f"no kernel {name} in the assembly"
    return [line.split(";")[0].strip() for line in m.group(0).splitlines()]


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
def test_every_wave_waits_for_its_stores_before_the_flag(tmp_path):
    out = tmp_path / "runtime.s"
    subprocess.run([B.HIPCC, *B.COMMON, "-w", "--offload-device-only", "-S", os.path.join(B.CSRC, "runtime.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    body = kernel_body(out.read_text(), "k_move")
    barrier = max(i for i, line in enumerate(body) if line.startswith("s_barrier"))
    stores = [i for i, line in enumerate(body) if re.match(r"(global|flat)_store", line)]
    copy, flag = [i for i in stores if i < barrier], [i for i in stores if i > barrier]
    assert copy and flag
    assert any(re.match(r"s_waitcnt\b.*vmcnt\(0\)", line) for line in body[max(copy):barrier])
