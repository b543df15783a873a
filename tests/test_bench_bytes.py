"""The algorithmic bytes that bench.py divides by a kernel's time: a block
without a wet cell, which the fine kernels leave at once, counts with its zeros
alone."""
import numpy as np
import pytest

import bench
from fluidisim_amd import workloads as W


@pytest.mark.parametrize("kernel,wet_layers,per_cell,per_dry_cell", [
    ("k_q_brick<0>", 24, 13, 4),      # 17 wet layers: three bricks of 8 of the four
    ("k_q_gs_first", 17, 13, 4),      # blocks of one layer
    ("k_q_restrict", 18, 9.5, 0.5),   # of two
    ("k_q_spmv_dir", 17, 17, 0),
    ("k_q_update", 17, 32, 0),
    ("k_q_gs<0>", 32, 13, 0),         # no block left out
])
def test_bytes_of_a_launch_leave_dry_blocks_out(kernel, wet_layers, per_cell, per_dry_cell):
    wl = W.tank(64, 32, 48, seed=1)
    d = wl.domain
    wl.solid = None
    wl.eta = np.full(d.columns, 17.2, np.float32)
    got, share = bench.bytes_per_launch(kernel, wl, 4)
    layer = d.nx * d.ny
    assert got == layer * (wet_layers * per_cell + (32 - wet_layers) * per_dry_cell)
    assert share == wet_layers / 32
