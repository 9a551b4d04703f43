"""The scan kernels of both geometries at the edges of their tiles, blocks and chunks, in the forms that inputs of different
size take (products with linear parts, products, lane polynomials, general recurrence): against the CPU checker, which
makes the same choices, bit for bit."""
import numpy as np
import pytest
import torch

import workloads as wl
from sg2_harness import Sg2Case, per_tensor_scalars, shared_scalars

pytestmark = pytest.mark.gpu

LARGE = dict(wl.DEFAULT_DIMS, d_model=16, d_state=32, d_inner=32)
# partial blocks and tiles at the end of a tensor; one chunk of 512 steps and a little more; several chunks
SHAPES = [(1,), (7,), (8,), (9,), (63,), (64,), (65,), (71,), (127,), (512,), (513,), (577,), (1200,)]


@pytest.mark.parametrize("sharp", [False, True])
@pytest.mark.parametrize("std", [1e-4, 3e-3, 0.05, 2.0])
@pytest.mark.parametrize("dims", [None, LARGE], ids=["default", "large"])
def test_bit_identical_to_the_checker(dims, std, sharp):
    _compare(SHAPES, dims, std, sharp)


@pytest.mark.parametrize("std", [1e-3, 0.3])
@pytest.mark.parametrize("dims,more", [(None, [(13000,)] * 24), (LARGE, [(5003,)] * 16)], ids=["default", "large"])
def test_bit_identical_with_chunks_that_fill_the_chip(dims, more, std):
    """Enough chunks for two columns per lane (the sets above take one)."""
    _compare(SHAPES + more, dims, std, True)


def _compare(shapes, dims, std, sharp):
    case = Sg2Case(shapes, seed=4, random_state=True, dims=dims)
    for t in (1, 2):
        grads = wl.make_grads(case.shapes, seed=20 + t, std=std)
        sharps = [g.abs() * 0.5 for g in wl.make_grads(case.shapes, seed=520 + t, std=std)] if sharp else [torch.zeros_like(g) for g in grads]
        pt, sh = per_tensor_scalars(case.P, t, 2.0), shared_scalars(4.5)
        case.gpu_step(grads, sharps, pt, sh)
        dbg = case.oracle_step(grads, sharps, pt, sh, chunk_len=None)
        case.compare(dbg, 1e-4, 1e-7)
        ctx = case.step_fn.ctx.cpu().numpy()
        for i in range(case.P):
            a, b = int(case.offsets[i]), int(case.offsets[i + 1])
            for d in range(2):
                assert np.array_equal(ctx[d, a:b], dbg[i]["ctx"][d]), (t, i, d)
            for k in ("gru", "mamba_fwd", "mamba_bwd"):
                assert np.array_equal(case.gpu[i][k].cpu().numpy().reshape(case.np[i][k].shape), case.np[i][k]), (t, i, k)
