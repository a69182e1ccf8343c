"""Properties of the compiled gfx950 code that no result shows, without a GPU."""

import re
import subprocess

import pytest

from diffrast_amd import _build


def kernels(source, name):
    """The assembly of the kernels of csrc/``source`` whose mangled names match ``name``."""
    try:
        compiler = _build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc was not found")
    result = subprocess.run([compiler, *_build.FLAGS, "-S", "--cuda-device-only", "-o", "-",
                             str(_build.SOURCES / source)], capture_output=True, text=True)
    assert result.returncode == 0, result.stderr[-2000:]
    found = re.findall(r"\n(_Z\w+):.*?\n(.*?)\n\.Lfunc_end", result.stdout, re.S)
    return {symbol: body for symbol, body in found if re.search(name, symbol)}


def test_mip_stages_take_three_channels_in_one_access():
    bodies = kernels("texture.hip", r"mip_(down|up)_stageI.*3RgbELi1E")
    assert len(bodies) == 2
    for symbol, body in bodies.items():
        for access in ("load", "store"):
            assert re.search(rf"global_{access}_dwordx3\b", body), symbol
            assert not re.search(rf"global_{access}_dword(x2)?\b", body), symbol


def test_antialias_reads_groups_of_four_channels_in_one_access():
    # More than four channels go in fours, 16 bytes an access (a path for fewer channels beside it
    # made the compiler split them into 12 and 4 bytes: a third slower at 8 channels).
    bodies = kernels("antialias.hip", r"aa_(blend|bwd)_kernelILi0E")
    assert len(bodies) == 4
    for symbol, body in bodies.items():
        assert not re.search(r"global_(load|store)_dwordx3\b", body), symbol
        assert re.search(r"global_store_dwordx4\b", body), symbol
