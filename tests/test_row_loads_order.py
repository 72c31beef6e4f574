"""The row-owned backward kernel requests its own rows, the statistics and the first stage copies one behind the other: nothing
it requests may be awaited in between.  Read off the assembly of single instances, compiled here (no GPU): the cotangent on TO
alone at full and padded head dimensions, both cotangents where D ends in an earlier tile."""
import re
import subprocess

import pytest

from semicat_amd import build

UNIT = "sjvp_tu_pair16.hip"


def _assembly(tmp_path, instance):
    src = tmp_path / "one.hip"
    src.write_text('#include "sjvp_pair16.hpp"\nnamespace sjvp { template __global__ void bwd_row16_kernel<%s>(const BwdParams); }\n' % instance)
    out = tmp_path / "one.s"
    subprocess.run([build.hipcc_path(), *build.HIPCC_FLAGS, *build.UNIT_FLAGS[UNIT], "-I" + build.CSRC, "--cuda-device-only", "-w", "-S",
                    str(src), "-o", str(out)], check=True, capture_output=True)
    return [line.split(";")[0].strip() for line in out.read_text().splitlines()]


@pytest.mark.parametrize("instance", ["Bf16, 128, 2, false, true, 2, 0, kIoDma, 1, 1, 8", "Bf16, 64, 3, false, true, 3, 0, kIoDma, 1, 1, 4",
                                      "Fp16, 128, 2, true, true, 2, 0, kIoDma, 1, 1, 6", "Bf16, 64, 4, false, true, 2, 0, kIoDma, 1, 2, 3"])
def test_no_wait_between_the_requests(tmp_path, instance):
    lines = _assembly(tmp_path, instance)
    rows = [i for i, s in enumerate(lines) if s.startswith("global_load_dwordx4 ")]
    stats = next(i for i, s in enumerate(lines) if s.startswith("global_load_dword "))
    rows = [i for i in rows if i < stats]
    assert len(rows) >= 10  # the own rows of the general path (with predicates) and of the path of whole rows
    waits = [i for i in range(rows[0], stats) if lines[i].startswith("s_waitcnt") and "vmcnt" in lines[i]]
    # a wait that no row load of its own path precedes waits for nothing: the one at the head of the path of whole rows
    whole = [i for i in rows if re.match(r"global_load_dwordx4 v\[\d+:\d+\], v\d+, s\[", lines[i])]
    labels = [i for i, s in enumerate(lines) if s.startswith(".LBB")]
    head = max(i for i in labels if i < whole[0])
    assert [i for i in waits if not head < i < whole[0]] == []
