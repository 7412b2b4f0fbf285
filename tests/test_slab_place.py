"""The places of the K-split slab GEMM's workgroups (csrc/slab_place.h),
compiled for the CPU: every part of every slab is taken by one workgroup, and a
slab's parts share an XCD from whichever XCD a launch starts."""

import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "hawkpoint-npu-llm_amd" / "csrc"


@pytest.mark.parametrize("slabs", [1, 8, 36, 56, 61])
@pytest.mark.parametrize("parts", [2, 4])
def test_every_part_of_every_slab_has_a_workgroup(tmp_path, slabs, parts):
    source = tmp_path / "places.cpp"
    source.write_text('#include "slab_place.h"\n#include <cstdio>\n'
                      "int main() {\n"
                      f"  for (int b = 0; b < hk::slab_places({slabs}, {parts}); ++b) {{\n"
                      f"    const hk::SlabPlace p = hk::slab_place(b, {parts});\n"
                      '    std::printf("%d %d\\n", p.slab, p.part);\n  }\n}\n')
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", str(source), "-o", str(tmp_path / "places")], check=True)
    lines = subprocess.run([str(tmp_path / "places")], check=True, capture_output=True, text=True).stdout.split("\n")
    places = [tuple(map(int, line.split())) for line in lines if line]
    taken = [p for p in places if p[0] < slabs]
    assert sorted(taken) == [(s, q) for s in range(slabs) for q in range(parts)]
    for first in range(8):  # workgroup b runs on XCD (first + b) % 8
        xcds = {}
        for b, (slab, _) in enumerate(places):
            xcds.setdefault(slab, set()).add((first + b) % 8)
        assert all(len(x) == 1 for x in xcds.values())
