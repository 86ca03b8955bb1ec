"""CPU: the layout in LDS of structures that kernels read and write with wide accesses.

Compiled for the host only, as the device compiles it: the alignment is the type's own."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("claim", [
    # work_open and find_slot_fold access the offsets as int4
    "alignof(dba::FoldLds) >= 16 && offsetof(dba::FoldLds, o) % 16 == 0",
])
def test_alignment_of_wide_lds_accesses(claim, tmp_path):
    src = tmp_path / "layout.hip"
    src.write_text(f'#include <cstddef>\n#include "common.h"\nstatic_assert({claim}, "layout");\n')
    r = subprocess.run(["hipcc", "--offload-host-only", "-fsyntax-only", "-std=c++17", "-I",
                        os.path.join(ROOT, "dba_amd", "csrc"), str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
