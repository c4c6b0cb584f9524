"""Registers and scratch of the tile kernels, read from the gfx950 assembly metadata: those that the
public entry points run wherever the caller leaves the tiling to the library, the benchmark's workloads
included.  A workgroup of 16 wavefronts leaves 128 VGPRs per lane, one of 12 168 and one of 8 256; every
variant fits its launch bound, and but for the ones named spills none to scratch.  Host-only: hipcc
cross-compiles the device code, no GPU is needed.
"""
import os
import shutil

import pytest

from adfwi_amd import build
from test_kernel_resources import _kernels

# variants (mangled) that spill, and how many VGPRs at most
SPILLING = {
    "ac_adj_tileILi4ELi16ELi2ELb0ELb0E": 9,     # 64 x 128 points, pressure records
    "ac_adj_tileILi4ELi16ELi2ELb0ELb1E": 27,    # 64 x 128 points, all records
    "el_fwd_tileILi3ELi4E": 2,                  # three-term differences
}
COUNT = {"acoustic.hip": 28, "elastic.hip": 20}   # tile kernels per file


@pytest.mark.skipif(shutil.which(build.hipcc()) is None and not os.path.exists(build.hipcc()),
                    reason="hipcc not available")
@pytest.mark.parametrize("source", sorted(COUNT))
def test_tile_kernels_fit_their_workgroups(source, tmp_path):
    kernels = _kernels(open(build.device_asm(source, str(tmp_path / (source + ".s")))).read())
    tiles = {n: k for n, k in kernels.items() if "_tileILi" in n}
    assert len(tiles) == COUNT[source], sorted(tiles)
    for name, k in tiles.items():
        waves = int(name.split("_tileILi")[1].split("ELi")[2 if source == "elastic.hip" else 1].split("E")[0])
        assert k["vgpr_count"] <= {16: 128, 12: 168}.get(waves, 256), (name, k)
        allowed = max([n for f, n in SPILLING.items() if f in name], default=0)
        assert k["vgpr_spill_count"] <= allowed, (name, k)
        assert allowed or k["private_segment_fixed_size"] == 0, (name, k)
