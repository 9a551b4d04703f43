"""Muon calls around the choice between 64x64 and 256x256 tiles of the products (all three fine, only the symmetric ones, one
K chunk more or less than the waves of a tile, padding to either size, several matrices), against the fp32 restatement."""
import pytest
import torch

from test_gpu_muon import _run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shapes", [
    [(129, 130)], [(200, 800), (801, 199)], [(1, 66000)], [(64, 1088), (1100, 60)],      # 64x64 for all three products
    [(256, 2048)] * 8,                                     # the symmetric products only
    [(512, 260), (129, 129), (20, 3000)],                  # matrices of different kinds in one call
], ids=["one", "both", "row", "chunks", "apply256", "mixed"])
def test_tile_choice(shapes, dtype):
    _run_case(shapes, dtype, 1, seed=7, ns=3 if shapes[0] != (129, 130) else 2)
