"""Host rules that need no device (invdft_amd/csrc/host_rules.h)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "..", "invdft_amd", "csrc")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("host compiler missing")
    out = tmp_path_factory.mktemp("rules") / "host_rules"
    subprocess.run([gxx, "-std=c++17", "-O1", f"-I{SRC}", os.path.join(HERE, "host_rules.cpp"),
                    "-o", str(out)], check=True, capture_output=True)
    txt = subprocess.run([str(out)], check=True, capture_output=True, text=True).stdout
    return [line.split() for line in txt.splitlines()]


def test_optional_workspace_is_whole_or_absent(rules):
    """An allocation that fails leaves none of the buffers and no exception."""
    seen = {int(f[1]): (int(f[2]), [int(v) for v in f[3:]]) for f in rules if f[0] == "alloc"}
    assert sorted(seen) == list(range(6))
    for room, (ok, sizes) in seen.items():
        if room < 4:  # four of the five need an allocation
            assert not ok and sizes == [0] * 5
        else:
            assert ok and sizes == [64, 64, 64, 70, 64]


def test_column_slices_start_at_even_columns(rules):
    """Slices of an even block start at even columns, so that 16-byte accesses stay
    aligned, and fit the scratch; a block that fits is one slice."""
    n = 0
    for f in rules:
        if f[0] != "slice":
            continue
        b, fit, w = (int(v) for v in f[1:])
        n += 1
        assert 1 <= w <= min(b, max(fit, 1))
        if b <= fit:
            assert w == b
        elif b % 2 == 0 and w > 1:
            assert all(j % 2 == 0 for j in range(0, b, w)), (b, fit, w)
    assert n == 800
