"""The forms that the scan's kernels and the fp32 checker share (products with and without their quadratic parts, in whole tiles,
in the ragged one at the end of a tensor and in the first attempt of a chunk summary; lane polynomials; the general
recurrence) against the float64 policy's sequential recurrence, which has none of them.  That kernel and checker agree bit
for bit says nothing about a form that both take; this does, and two mistakes planted in the checker show that it would."""
import os
import subprocess

import numpy as np
import pytest

import workloads as wl
from helpers import copy_state, default_scalars, random_state_np
from oracle import oracle as orc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LARGE = dict(wl.DEFAULT_DIMS, d_model=16, d_state=32, d_inner=32)
NETS = {"bench": (wl.DEFAULT_DIMS, lambda: wl.meta_weights(7)), "module": (wl.DEFAULT_DIMS, lambda: wl.module_weights(3)),
        "large": (LARGE, lambda: wl.meta_weights(7, LARGE))}
SIZES = (7, 9, 65, 71, 513, 577, 1200, 3000)      # a partial block alone, after a block, a tile, a chunk; several chunks
# 2-norm of the difference over the 2-norm of the result.  A context is a sum over 16 (32) columns of products of three rounded
# factors, each within a few units of 2^-24: the general recurrence alone (gradients of size 2) shows 0.9e-7 to 1.6e-7 over
# the three nets, and no form is allowed half as much again.  A state is a sum of up to 240 rounded updates: 2e-7 to 1e-6.
CTX, STATE = 4 * 2.0 ** -24, 2.0 ** -19


def _errors(net, n, std, sharp, chunk):
    dims, weights = NETS[net]
    W = [w.numpy() for w in weights()]
    r = np.random.RandomState(n)
    g = (r.randn(n) * std).astype(np.float32)
    s = (np.abs(r.randn(n)) * (0.5 * std if sharp else 0.0)).astype(np.float32)
    st, out = random_state_np(n, n, dims), []
    for precision, chunk_len, window in ((32, chunk, 64), (64, 0, 0)):
        x = copy_state(st)
        dbg = orc.sg2_step(W, x, g, s, default_scalars(), dims=dims, precision=precision, chunk_len=chunk_len, window=window, debug=True)
        out.append((dbg["ctx"][0], dbg["ctx"][1], x["mamba_fwd"], x["mamba_bwd"]))
    rel = [float(np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)) for a, b in zip(*out)]
    return max(rel[:2]), max(rel[2:])


def _check(net, std, sizes=SIZES):
    for n in sizes:
        for chunk in (256, 512):
            for sharp in (False, True):
                ctx, state = _errors(net, n, std, sharp, chunk)
                assert ctx <= CTX and state <= STATE, (net, std, n, chunk, sharp, ctx, state)


@pytest.mark.parametrize("std", [1e-4, 1e-3, 3e-3, 0.05, 2.0])
@pytest.mark.parametrize("net", sorted(NETS))
def test_contexts_and_states_against_float64(net, std):
    _check(net, std)


MUTANTS = [
    # (name, text in sg2_oracle.cpp, replacement, sizes that show it)
    ("partial_block_of_another_pair", "const float* k = &w.lane_prod[(size_t)l * 12];",
     "const float* k = &w.lane_prod[(size_t)(len < ORC_BLOCK ? 0 : l) * 12];", (7, 9, 65, 71, 513)),
    ("summary_products_without_rotation", "m[4] = O::fma(ae, ve, O::fma(sn, vo, be));", "m[4] = O::fma(ae, ve, be);", (577, 1200, 3000)),
]


@pytest.mark.parametrize("name,old,new,sizes", MUTANTS, ids=[m[0] for m in MUTANTS])
def test_notices_a_mistake_in_a_shared_form(name, old, new, sizes, tmp_path):
    src = open(os.path.join(ROOT, "oracle", "sg2_oracle.cpp")).read()
    assert src.count(old) == 1, "the text to mutate must occur exactly once: " + name
    path, so = str(tmp_path / (name + ".cpp")), str(tmp_path / (name + ".so"))
    with open(path, "w") as f:
        f.write(src.replace(old, new).replace('"../include/', '"%s/include/' % ROOT))
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-ffp-contract=off", "-mfma", "-shared", "-o", so, path,
                           os.path.join(ROOT, "oracle", "elem_oracle.cpp")])
    good = orc.lib()
    try:
        orc._lib = orc.load(so)
        for n in sizes:
            with pytest.raises(AssertionError):
                _check("module", 1e-4, (n,))
    finally:
        orc._lib = good
