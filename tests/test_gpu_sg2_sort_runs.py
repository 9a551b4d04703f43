"""The sort of small calls (runs of 4096 keys in LDS, merged) and the limits at which it gives way to one workgroup per tensor
and to the radix passes: the permutation against a stable argsort of the magnitudes."""
import numpy as np
import pytest
import torch

import workloads as wl
from sg2_harness import Sg2Case, per_tensor_scalars, shared_scalars

pytestmark = pytest.mark.gpu

# (both sides of the limits on the work are in test_gpu_sg2_paths.py)
SHAPES = {"one run": [(2049,), (1,), (4095,), (4096,), (2048,)], "two": [(4097,), (6145,), (8192,), (3,)], "more": [(8193,), (12288,), (12289,), (40000,)],
          "most": [(81920,), (5,), (65537,)], "passes": [(81921,), (2500,)], "beyond": [(300000,), (230000,), (2049,)]}
FORMS = {"passes": "small passes", "beyond": "scanned passes"}       # the others are merged
WIDE = ("more", "most", "passes")                                    # ... as fp32 only: 16-bit tensors above 8192 elements are not
VALUES = ["random", "ties", "equal", "ascending", "descending", "not finite"]


def _values(kind, n, r):
    if kind == "ties":
        return r.choice([-1.0, 1.0], n) * r.randint(0, 40, n) / 8.0
    if kind == "equal":
        return r.choice([-0.5, 0.5], n)
    v = r.randn(n) * 1e-3
    if kind in ("ascending", "descending"):
        v = np.sort(np.abs(v)) * r.choice([-1.0, 1.0], n)
        return v if kind == "ascending" else v[::-1].copy()
    if kind == "not finite":
        v[r.rand(n) < 0.3] = np.inf
        v[r.rand(n) < 0.1] = np.nan
        v[r.rand(n) < 0.05] = -np.finfo(np.float32).max
    return v


@pytest.mark.parametrize("form", sorted(SHAPES))
@pytest.mark.parametrize("kind", VALUES)
def test_permutation(form, kind):
    from grokking_optimizers import _cabi
    sizes = [wl.numel(s) for s in SHAPES[form]]
    assert _cabi.sort_form_for(sizes) == FORMS.get(form, "runs")
    assert _cabi.sort_form_for(sizes, True) == ("small passes" if form in WIDE else FORMS.get(form, "runs"))
    for dtype in ([torch.float32, torch.bfloat16] if kind in ("random", "ties") else [torch.float32]):
        shapes, r = SHAPES[form], np.random.RandomState(len(form) + len(kind))
        case = Sg2Case(shapes, dtypes=[dtype] * len(shapes), seed=1)
        grads = [torch.from_numpy(_values(kind, wl.numel(s), r)).to(dtype) for s in shapes]
        sharps = [torch.rand(wl.numel(s)).to(dtype) if i % 2 else torch.zeros(wl.numel(s), dtype=dtype) for i, s in enumerate(shapes)]
        case.gpu_step(grads, sharps, per_tensor_scalars(case.P, 1), shared_scalars())
        perm = case.step_fn.perm.cpu().numpy()
        for i, g in enumerate(grads):
            a, b = int(case.offsets[i]), int(case.offsets[i + 1])
            v = g.float().numpy()
            want = np.argsort(np.abs(np.where(np.isfinite(v), v, 0.0)), kind="stable")
            assert np.array_equal(perm[a:b], want), (form, kind, dtype, i)
