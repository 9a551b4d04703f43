"""Muon calls whose matrices all fit one workgroup's LDS (the whole iteration in one launch) at the edges of that rule and of
its tiles, and the same matrices beside one that does not fit (the products' path), against the fp32 restatement."""
import pytest
import torch

from test_gpu_muon import _run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shapes", [
    [(128, 512), (512, 128), (64, 1024), (1, 1)],          # the largest that fit, and the smallest
    [(65, 129), (65, 65), (33, 961), (127, 448), (64, 64)],        # both paddings, odd multiples of 64 and even ones
    [(129, 130), (30, 50)], [(128, 513), (40, 30)],        # just beyond it
], ids=["largest", "ragged", "taller", "longer"])
def test_small_matrices(shapes, dtype):
    _run_case(shapes, dtype, 1, seed=5, ns=2 if shapes[0] == (65, 129) else 3)
