"""The two-pass sort of calls whose gradients are all 16-bit: the permutation against a stable argsort of the magnitudes, over
every form of the sort (a workgroup per tensor, merged runs, small tiles, large tiles with and without scan kernels) and the whole range of
the types (subnormals, zeros of either sign, the largest values, non-finite entries, ties)."""
import numpy as np
import pytest
import torch

import workloads as wl
from sg2_harness import Sg2Case, per_tensor_scalars, shared_scalars

pytestmark = pytest.mark.gpu

# name: (shapes, form of the sort where all gradients are 16-bit, form where some are fp32)
SHAPES = {"tensors": ([(1,), (511,), (513,), (2048,), (2047,)], "tensors", "tensors"),
          "large_tensors": ([(8192,), (8191,), (4097,), (2049,), (513,)] + [(8192,)] * 255, "tensors", "tensors"),
          "runs": ([(1,), (511,), (513,), (2049,), (8192,)], "runs", "runs"),
          "small": ([(8193,), (2048,), (4097,), (5,)], "small passes", "runs"),
          "small_wide": ([(300001,), (8191,), (16384,)], "small passes", "small passes"),
          "large": ([(70001,), (2200000 // 16,), (250000,), (1900000 // 8,)] * 4, "passes", "passes"),
          "scan": ([(300001,), (8191,), (250000,)], "scanned passes", "scanned passes")}


def _values(n, dtype, seed):
    r = np.random.RandomState(seed)
    lo, hi = (-24.0, 15.9) if dtype == torch.float16 else (-133.0, 120.0)
    v = np.exp2(r.uniform(lo, hi, n)) * r.choice([-1.0, 1.0], n)
    v[r.rand(n) < 0.05] = 0.0
    v[r.rand(n) < 0.02] = -0.0
    if n > 100:
        v[3], v[50], v[70] = np.inf, np.nan, -np.inf
        v[60:64] = 5.9604644775390625e-08          # the smallest float16 there is
    return torch.from_numpy(v).to(dtype)


@pytest.mark.parametrize("form", sorted(SHAPES))
@pytest.mark.parametrize("types", ["bf16", "fp16", "both", "with_fp32"])
def test_permutation(form, types):
    from grokking_optimizers import _cabi
    shapes, of_16bit, of_mixed = SHAPES[form]
    assert _cabi.sort_form_for([wl.numel(s) for s in shapes], types != "with_fp32") == (of_mixed if types == "with_fp32" else of_16bit)
    of = {"bf16": [torch.bfloat16], "fp16": [torch.float16], "both": [torch.float16, torch.bfloat16],
          "with_fp32": [torch.bfloat16, torch.float32, torch.float16]}[types]
    dtypes = [of[i % len(of)] for i in range(len(shapes))]
    case = Sg2Case(shapes, dtypes=dtypes, seed=1)
    grads = [_values(wl.numel(s), dt, 7 + i) for i, (s, dt) in enumerate(zip(shapes, dtypes))]
    sharps = [torch.zeros(wl.numel(s)) for s in shapes]
    case.gpu_step(grads, sharps, per_tensor_scalars(case.P, 1), shared_scalars())
    perm = case.step_fn.perm.cpu().numpy()
    for i, g in enumerate(grads):
        a, b = int(case.offsets[i]), int(case.offsets[i + 1])
        v = g.float().numpy()
        want = np.argsort(np.abs(np.where(np.isfinite(v), v, 0.0)), kind="stable")
        assert np.array_equal(perm[a:b], want), (form, types, i)
