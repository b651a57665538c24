"""The device plans of the packed attention calls stay within what the host
provides (CPU): tests/plan_bounds.hip takes random calls through the library's
own host code and the plan's arithmetic."""

from __future__ import annotations

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def broken(tmp_path_factory):
    binary = str(tmp_path_factory.mktemp("plans") / "plan_bounds")
    # The kernels' launches are not linked: nothing here calls them.
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "residualquant_amd", "csrc"), "-Wl,--unresolved-symbols=ignore-all",
                    os.path.join(HERE, "plan_bounds.hip"), "-o", binary], check=True)
    out = subprocess.run([binary], check=True, capture_output=True, text=True, timeout=300).stdout
    return {line.split()[0]: int(line.split()[1]) for line in out.splitlines()}


@pytest.mark.parametrize("name", [
    "rows_required_within_total", "rows_entries", "rows_entries_in_workspace", "rows_items", "rows_arrivals",
    "rows_split_pages", "rows_scratch", "decode_items_in_workspace", "decode_items", "decode_items_by_pages",
    "decode_arrivals"])
def test_plan_stays_within(broken, name):
    assert broken[name] == 0
