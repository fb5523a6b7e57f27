"""CPU checks of the built library's gfx950 code: wait states that only the
writer of an inline assembly block can add."""
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin",
                       "llvm-objdump")


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    import sam3_hip
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    so = shutil.copy(sam3_hip.LIB_PATH, d)
    subprocess.run([OBJDUMP, "--offloading", so], check=True, cwd=d,
                   stdout=subprocess.DEVNULL)
    out = []
    for f in sorted(os.listdir(d)):
        if f.endswith("gfx950"):
            out.append(subprocess.run(
                [OBJDUMP, "-d", "--no-show-raw-insn", f], check=True, cwd=d,
                stdout=subprocess.PIPE, text=True).stdout.splitlines())
    assert out
    return out


def test_m0_write_before_lds_load_has_its_wait_state(listings):
    """A scalar write of M0 needs one wait state before a global load to LDS
    that reads it (gfx9 hazard table): some other instruction lies between
    the two."""
    writes_m0 = re.compile(r"\bs_\w+ m0\b")
    loads = bad = 0
    for lines in listings:
        prev = ""
        for line in lines:
            ins = line.split("//")[0].strip()
            if not ins or ins.endswith(":"):
                continue
            if "_load_lds_" in ins or re.search(r"\bbuffer_load.* lds\b", ins):
                loads += 1
                bad += writes_m0.search(prev) is not None
            prev = ins
    assert loads > 0
    assert bad == 0, "%d of %d copies" % (bad, loads)
