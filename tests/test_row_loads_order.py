"""What the 16-bit kernels request ahead is not awaited ahead.  Read off the assembly of single instances, compiled here (no GPU)."""
import re
import subprocess

import pytest

from semicat_amd import build


def _assembly(tmp_path, unit, instance):
    src = tmp_path / "one.hip"
    header = {"sjvp_tu_pair16.hip": "sjvp_pair16.hpp", "sjvp_tu_fwd_staged16.hip": "sjvp_fwd16_staged.hpp"}[unit]
    params = "FwdParams" if "fwd" in unit else "BwdParams"
    src.write_text(f'#include "{header}"\nnamespace sjvp {{ template __global__ void {instance}(const {params}); }}\n')
    out = tmp_path / "one.s"
    subprocess.run([build.hipcc_path(), *build.HIPCC_FLAGS, *build.UNIT_FLAGS.get(unit, []), "-I" + build.CSRC, "--cuda-device-only", "-w", "-S",
                    str(src), "-o", str(out)], check=True, capture_output=True)
    return [line.split(";")[0].strip() for line in out.read_text().splitlines()]


@pytest.mark.parametrize("instance", ["Bf16, 128, 2, false, true, 2, 0, kIoDma, 1, 1, 8", "Bf16, 64, 3, false, true, 3, 0, kIoDma, 1, 1, 4",
                                      "Fp16, 128, 2, true, true, 2, 0, kIoDma, 1, 1, 6", "Bf16, 64, 4, false, true, 2, 0, kIoDma, 1, 2, 3"])
def test_no_wait_between_the_requests(tmp_path, instance):
    """The row-owned backward requests its own rows, the statistics and the first stage copies one behind the other.  The
    cotangent on TO alone at full and padded head dimensions, both cotangents where D ends in an earlier tile."""
    lines = _assembly(tmp_path, "sjvp_tu_pair16.hip", f"bwd_row16_kernel<{instance}>")
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


@pytest.mark.parametrize("instance", ["Bf16, 32, 2, true, 4, 1, false, kIoAny, 1, 1, 2", "Bf16, 64, 4, false, 4, 1, false, kIoAny, 1, 1, 3",
                                      "Fp16, 128, 2, true, 2, 1, false, kIoAny, 1, 1, 8", "Bf16, 64, 4, true, 4, 2, false, kIoAny, 1, 2, 3"])
def test_no_wait_for_the_next_stage_ahead_of_the_products(tmp_path, instance):
    """The forward over rows of any alignment requests the next stage ahead of the products of this one; what the products take
    from global memory, the own rows, has to be there before the loop."""
    lines = [s for s in _assembly(tmp_path, "sjvp_tu_fwd_staged16.hip", f"fwd16_kernel<{instance}>") if s]
    products = [i for i, s in enumerate(lines) if "mfma" in s and s.startswith("v_")]
    assert len(products) > 8
    waits = []
    for i in products:  # the last wait since the product before, if it stands with the product's operands
        before = [s for s in lines[max(0, i - 3):i] if s.startswith("s_waitcnt") and "vmcnt" in s]
        waits += [(i, s) for s in before]
    assert waits == []
