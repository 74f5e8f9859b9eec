"""Workgroups of a device Newton pass: one a CU for a 4-state tree of up to four
tiles a CU, else two, and as many as PLK_SWEEP_BLOCKS_PER_CU says where it is
set, whatever the size; the lengths are those of the default."""
import os
import re
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

# 8 categories: tiles of 32 patterns, about 400 of them (1.6 a CU)
PROGRAM = """
import sys
sys.path.insert(0, %r)
import iqtree2_amd as ia
w = ia.Workload(seq_type=ia.DNA, ntaxa=20, nsite=13000, ncat=8, mean_len=0.3, seed=4)
ctx = ia.Context(0)
tree = ia.PhyloTree(ctx, w)
lnl, _ = tree.optimize_all_branches(iterations=1, tolerance=1e-3, max_nr=100)
print("tiles", -(-w.npatterns // 256) * 8, repr(lnl), *[repr(tree.get_length(a, b)) for a, b in tree.branches()])
tree.close()
ctx.close()
"""


def sweep(blocks):
    env = dict(os.environ, PLK_SWEEP_TIMING="1")
    env.pop("PLK_SWEEP_BLOCKS_PER_CU", None)
    if blocks:
        env["PLK_SWEEP_BLOCKS_PER_CU"] = str(blocks)
    p = subprocess.run([sys.executable, "-c", PROGRAM % ROOT], env=env, capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stderr
    words = next(line for line in p.stdout.splitlines() if line.startswith("tiles")).split()
    return (int(re.search(r"grid (\d+)", p.stderr).group(1)), int(words[1]), np.array([float(x) for x in words[2:]]))


def test_workgroups_per_cu():
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    grid, tiles, values = sweep(None)
    assert cus < tiles < 2 * cus
    assert grid == cus
    for blocks, expected in ((1, cus), (2, tiles)):
        grid, _, other = sweep(blocks)
        assert grid == expected, blocks
        np.testing.assert_allclose(other, values, rtol=1e-9, atol=1e-12)
