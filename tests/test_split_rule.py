"""How many waves share a group of rows: by the compute units that the device has, a whole chip or a partition of one.  (Host code
alone, compiled and run here.)"""
import subprocess

import pytest

from semicat_amd import build


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    where = tmp_path_factory.mktemp("rule")
    (where / "rule.hip").write_text('#include <cstdio>\n#include <cstdlib>\n#include "sjvp_launch.hpp"\nint main(int, char** a) {\n'
                                    "  std::printf(\"%d\", sjvp::split_rows(atoi(a[1]), atoi(a[2]), atoi(a[3]), atoi(a[4]), atoi(a[5])));\n}\n")
    subprocess.run([build.hipcc_path(), "-std=c++20", "-O0", "-w", "--cuda-host-only", "-I" + build.CSRC, "-x", "hip", str(where / "rule.hip"),
                    "-o", str(where / "rule")], check=True, capture_output=True)
    return lambda *a: int(subprocess.run([str(where / "rule"), *map(str, map(int, a))], check=True, capture_output=True).stdout)


@pytest.mark.parametrize("units", [256, 64, 32])
def test_split_rows(rule, units):
    assert rule(units // 4, 5, 4, False, units) == 4 and rule(units // 4, 4, 4, False, units) == 2  # a unit for each
    assert rule(units // 4 + 1, 16, 4, False, units) == 2 and rule(units // 4, 5, 2, False, units) == 2
    assert rule(units // 2, 4, 4, False, units) == 2 and rule(units // 2, 3, 4, True, units) == 1
    assert rule(units // 2 + 1, 99, 4, False, units) == 1
    assert rule(units, 12, 4, True, units) == 2 and rule(units, 11, 4, True, units) == 1  # two to a unit
    assert rule(units + 1, 99, 4, True, units) == 1
