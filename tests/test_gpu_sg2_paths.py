"""The v2 step at the edges of its sort and clip dispatch: tensor sizes on both sides of what one LDS sort holds, of the
small sort tile (by the widest tensor and by the total), of what is merged from runs, and of what a scatter workgroup adds up itself - each
in the form of the sort that it is there for, as the library reports it; and the clipping step of the class (factor applied as
the gradients are read, fp32 sharpness beside 16-bit gradients) against clipped copies through the list functions."""
import pytest
import torch

import workloads as wl
from sg2_harness import Sg2Case, per_tensor_scalars, shared_scalars

pytestmark = pytest.mark.gpu

# name: (tensor sizes, form of the sort)
SIZES = {"a workgroup each": ([2048, 1, 512, 513, 2047, 65], "tensors"), "one above": ([2049, 2048, 1, 512], "runs"),
         "a large tile at most": ([8192, 1, 512, 513, 2048], "runs"), "one above a large tile": ([8193, 2047, 2049], "runs"),
         "most merged by work": ([65536] * 19 + [17 * 2048], "runs"), "one above the work": ([65536] * 19 + [17 * 2048, 1], "small passes"),
         "32 small tiles": ([65536, 70], "runs"), "one above 32": ([65537, 3], "runs"),
         "128 small tiles": ([262144, 9], "small passes"), "one above 128": ([262145, 8191], "small passes"),
         "one below a large tile for every fourth CU": ([262144, 262143], "small passes"), "a large tile for every fourth CU": ([262144, 262144], "passes"),
         "narrow beyond that": ([65536] * 9, "runs"), "not narrow": ([65537] + [65536] * 8, "passes"),
         "most tiles of a self scan": ([262144, 9, 262144], "passes"), "one above that": ([262145, 262144, 8191], "scanned passes"),
         "one below a large tile per CU": ([65536] * 31 + [65535], "small passes"), "a large tile per CU": ([65536] * 32, "passes"),
         "a large tile each": ([8192, 8191, 2049, 4097, 513] + [8192] * 255, "tensors")}


@pytest.mark.parametrize("sizes", list(SIZES), ids=lambda s: s.replace(" ", "_"))
@pytest.mark.parametrize("sharpness", [False, True])
def test_sort_paths(sizes, sharpness):
    from grokking_optimizers import _cabi
    assert _cabi.sort_form_for(SIZES[sizes][0]) == SIZES[sizes][1]
    shapes = [(n,) for n in SIZES[sizes][0]]
    case = Sg2Case(shapes, seed=3, random_state=True)
    grads = wl.make_grads(shapes, seed=4, tail_frac=0.01)
    grads[0][::7] = 0.0                                   # runs of equal keys
    grads[0][1::13] = float("nan")
    sharps = [g.abs() if sharpness else torch.zeros_like(g) for g in wl.make_grads(shapes, seed=5)]
    pt, sh = per_tensor_scalars(len(shapes), 1, lamb_eff=2.0), shared_scalars()
    case.gpu_step(grads, sharps, pt, sh)
    dbg = case.oracle_step(grads, sharps, pt, sh, chunk_len=None)
    case.compare(dbg, 1e-4, 1e-7)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_clipping_step_equals_clipped_copies(dtype):
    from grokking_optimizers import SuperGrok2
    shapes = [(300,), (70, 130), (64, 1100), (5,)]

    def run(lists):
        torch.manual_seed(1)
        params = [torch.nn.Parameter((p * 1.0).to(dtype).cuda()) for p in wl.make_params(shapes, seed=0)]
        opt = SuperGrok2(params, warmup_steps=0, warmup_ramp=1, gradient_clipping=0.05, recycle_interval=0)
        opt._ensure_state()
        for i, s in enumerate(wl.make_grads(shapes, seed=9)):
            opt._flat_sharpness[i].copy_(s.abs().reshape(-1))
        for t in range(3):
            for p, g in zip(params, wl.make_grads(shapes, seed=20 + t, std=1e-3, tail_frac=0.01)):
                p.grad = g.to(dtype).cuda()
            params[3].grad[0] = float("inf")
            params[0].grad[1] = float("nan")
            if lists:
                opt._global_step += 1
                opt._cached_weights = opt.meta_net.flat_weights()
                lamb = opt.lamb * opt._get_ramp_factor() * opt._get_gate_signal()
                with torch.no_grad():
                    opt._step_lists(1e-3, 0.999, 1e-8, opt._get_effective_wd(1.0), lamb)
            else:
                opt.step()
        return params, opt
    (pa, a), (pb, b) = run(True), run(False)
    assert a._flat_steps == b._flat_steps == [3] * 4
    for x, y in zip(pa, pb):
        assert torch.equal(x, y)
    for k in ("_flat_exp_avgs", "_flat_exp_avg_sqs", "_flat_mus", "_flat_gru_states", "_flat_mamba_fwd_states", "_flat_mamba_bwd_states"):
        for x, y in zip(getattr(a, k), getattr(b, k)):
            assert torch.equal(x, y), k
    assert torch.equal(a.meta_net.expert_counts, b.meta_net.expert_counts)
