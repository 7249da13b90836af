"""Properties of the device code that no result shows, read from the assembly
that the build's own flags give."""
import re
import subprocess

import pytest

from mcvslam_amd import build


@pytest.fixture(scope="module")
def match_kernels(tmp_path_factory):
    """Kernel name -> assembly of mcv_match.hip."""
    out = tmp_path_factory.mktemp("asm") / "match.s"
    flags = [f for f in build.HIP_FLAGS if f != "-shared"]
    subprocess.run([build.hipcc(), *flags, "--cuda-device-only", "-S", "-o", str(out),
                    str(build.PKG / "csrc" / "mcv_match.hip")], check=True, capture_output=True)
    text = out.read_text()
    return {m.group(1): m.group(2) for m in re.finditer(r"^(_Z\w+):(.*?)^\.Lfunc_end", text, re.M | re.S)}


@pytest.mark.parametrize("per_lane,rows", [(1, 4), (2, 2), (2, 4), (2, 8), (1, 8), (4, 2)])
def test_popcount_top2_loads_trains_by_the_scalar_unit(match_kernels, per_lane, rows):
    """k_knn2_s: a wave's train rows are the same for all its lanes and come
    through scalar loads, 32 bytes a row; the vector loads are the queries'
    alone, two of 16 bytes for each query of a lane (and the counts')."""
    names = [k for k in match_kernels if f"k_knn2_sILi{per_lane}ELi{rows}E" in k]
    assert names
    for name in names:
        scalar = re.findall(r"\bs_load_dwordx(8|16)\b", match_kernels[name])
        assert sum(int(n) // 8 for n in scalar) >= rows
        vector = re.findall(r"\b(?:global|flat)_load_dwordx4\b", match_kernels[name])
        assert len(vector) == 2 * per_lane
