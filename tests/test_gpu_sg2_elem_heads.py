"""The per-element kernel with a wave per head (small calls) against the form that records the routing, which takes a lane
per element at every size: the same sums in the same order, so the same bits.  The debug form is compared with the checker
elsewhere."""
import pytest
import torch

import workloads as wl
from sg2_harness import Sg2Case, per_tensor_scalars, shared_scalars

pytestmark = pytest.mark.gpu

LARGE = dict(wl.DEFAULT_DIMS, d_model=16, d_state=32, d_inner=32)
EH4 = dict(wl.DEFAULT_DIMS, expert_hidden=4)


@pytest.mark.parametrize("dims", [None, LARGE, EH4], ids=["default", "large", "narrow experts"])
@pytest.mark.parametrize("shapes", [
    [(1,), (63,), (64,), (65,), (129,), (1023,), (1024,), (1025,)],
    [(1024,)] * 15 + [(7,)],            # 16 tiles of 1024: the largest such call
    [(1024,)] * 16 + [(7,)],            # one more
], ids=["edges", "largest", "beyond"])
def test_same_bits_as_a_lane_per_element(shapes, dims):
    cases = [Sg2Case(shapes, seed=6, random_state=True, dims=dims) for _ in range(2)]
    cases[1].step_fn.debug.expert_idx = None
    for t in (1, 2):
        grads = wl.make_grads(shapes, seed=30 + t, std=0.05)
        sharps = [g.abs() * 0.5 for g in wl.make_grads(shapes, seed=530 + t, std=0.05)]
        for case in cases:
            case.gpu_step(grads, sharps, per_tensor_scalars(case.P, t, 2.0), shared_scalars(4.5))
    for a, b in zip(cases[0].gpu, cases[1].gpu):
        for k in a:
            assert torch.equal(a[k], b[k]), k
    assert torch.equal(cases[0].counts_gpu, cases[1].counts_gpu)
