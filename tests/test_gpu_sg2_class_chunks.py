"""The class's step at the chunk lengths that it chooses for itself (`sg2_clipped_step`: 256 in small calls of the default geometry,
lengths that fill the chip in whole rounds for the large one), and the batched step at such lengths pinned: bit for bit
against the CPU checker, which is handed the length that the library reports."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

import workloads as wl
from oracle import oracle as orc
from sg2_harness import Sg2Case, per_tensor_scalars, shared_scalars

pytestmark = pytest.mark.gpu

LARGE = dict(wl.DEFAULT_DIMS, d_model=16, d_state=32, d_inner=32)
STATE = dict(exp_avg="_flat_exp_avgs", exp_avg_sq="_flat_exp_avg_sqs", mu="_flat_mus", gru="_flat_gru_states",
             mamba_fwd="_flat_mamba_fwd_states", mamba_bwd="_flat_mamba_bwd_states")
# dimensions, tensor sizes, the length that the class takes there
CALLS = {"small": (None, [3000, 700, 513, 40], 256), "largest small": (None, [8192, 8191, 257], 256), "just beyond": (None, [8193, 700], 512), "as the batched step": (None, [70001, 512, 5], 512),
         "large, all at once": (LARGE, [20000, 9000, 513, 77], 512), "large, just beyond": (LARGE, [131073, 300], 640),
         "large, transformer": (LARGE, [wl.numel(s) for s in wl.shared14_shapes()], 1792),
         "large, one long round": (LARGE, [63400] * 15 + [63488], 3968)}


@pytest.mark.parametrize("call", sorted(CALLS))
def test_class_step_is_the_checkers(call):
    from grokking_optimizers import SuperGrok2, _cabi
    dims, sizes, expected = CALLS[call]
    d = dims or wl.DEFAULT_DIMS
    chunk_len = _cabi.clipped_chunk_len_for(sizes, dims)
    assert chunk_len == expected
    shapes = [(n,) for n in sizes]
    p0 = wl.make_params(shapes, seed=0)
    params = [torch.nn.Parameter(p.clone().cuda()) for p in p0]
    opt = SuperGrok2(params, warmup_steps=0, warmup_ramp=1, recycle_interval=0, d_model=d["d_model"], d_state=d["d_state"])
    opt.meta_net.load_flat_weights([w.cuda() for w in wl.meta_weights(7, dims)])
    opt._ensure_state()
    sharp = [(s.abs() * 0.5 if i % 2 else torch.zeros_like(s)).reshape(-1) for i, s in enumerate(wl.make_grads(shapes, seed=31))]
    for dst, s in zip(opt._flat_sharpness, sharp):
        dst.copy_(s)
    f32 = lambda v: float(np.float32(v))
    ref = [dict(param=p.numpy().reshape(-1).copy(), exp_avg=np.zeros(p.numel(), np.float32), exp_avg_sq=np.zeros(p.numel(), np.float32),
                mu=np.zeros(p.numel(), np.float32), gru=np.zeros((p.numel(), 4), np.float32),
                mamba_fwd=np.zeros((d["d_inner"], d["d_state"]), np.float32), mamba_bwd=np.zeros((d["d_inner"], d["d_state"]), np.float32))
           for p in p0]
    W = [w.numpy() for w in wl.meta_weights(7, dims)]
    counts = np.zeros(144, np.int32)
    for t in (1, 2):
        grads = wl.make_grads(shapes, seed=1 + t)
        for p, g in zip(params, grads):
            p.grad = g.clone().cuda()
            assert float(g.norm()) < opt.gradient_clipping        # the clip multiplies by exactly 1
        opt.step(train_acc=0.85)
        sig = lambda v, th: 1.0 / (1.0 + np.exp(-20.0 * (v - th)))
        each = [np.zeros(144, np.int32) for _ in sizes]

        def one(i):
            b1 = 0.9 * (0.9 ** i)
            sc = dict(alpha=f32(0.98), lamb_eff=f32(2.0 * sig(0.85, 0.8)), beta1=f32(b1), bc1=f32(1.0 - b1 ** t), bc2=f32(1.0 - 0.999 ** t),
                      rescale=f32(0.1), beta2=f32(0.999), lr=f32(1e-3), wd_eff=f32(1.0 * (1.0 + 4.0 * sig(0.85, 0.9))), eps=f32(1e-8))
            orc.sg2_step(W, ref[i], np.ascontiguousarray(grads[i].numpy().reshape(-1)), sharp[i].numpy(), sc, dims=d, chunk_len=chunk_len,
                         window=_cabi.lib().sg2_get_scan_window(), expert_counts=each[i])
        with ThreadPoolExecutor(8) as ex:
            list(ex.map(one, range(len(sizes))))
        counts += sum(each)
        for i in range(len(sizes)):
            assert np.array_equal(params[i].detach().cpu().numpy(), ref[i]["param"]), (t, i)
            for k, attr in STATE.items():
                assert np.array_equal(getattr(opt, attr)[i].cpu().numpy().reshape(ref[i][k].shape), ref[i][k]), (t, i, k)
        assert np.array_equal(opt.meta_net.expert_counts.cpu().numpy(), counts), t


@pytest.mark.parametrize("chunk_len", [640, 1792, 3968])
def test_pinned_lengths_of_the_large_geometry(chunk_len):
    shapes = [(n,) for n in (chunk_len - 1, chunk_len, chunk_len + 1, 2 * chunk_len + 65, 3 * chunk_len, 3 * chunk_len + 1, 7)]
    case = Sg2Case(shapes, seed=9, random_state=True, dims=LARGE, chunk_len=chunk_len)
    for t in (1, 2):
        grads = wl.make_grads(shapes, seed=60 + t, tail_frac=0.01)
        sharps = [g.abs() * 0.5 if i % 2 else torch.zeros_like(g) for i, g in enumerate(wl.make_grads(shapes, seed=70 + t))]
        pt, sh = per_tensor_scalars(case.P, t, 2.0), shared_scalars(4.5)
        case.gpu_step(grads, sharps, pt, sh)
        dbg = case.oracle_step(grads, sharps, pt, sh, chunk_len)
        case.compare(dbg, 1e-4, 1e-7)
        ctx = case.step_fn.ctx.cpu().numpy()
        for i in range(case.P):
            a, b = int(case.offsets[i]), int(case.offsets[i + 1])
            for d in range(2):
                assert np.array_equal(ctx[d, a:b], dbg[i]["ctx"][d]), (t, i, d)
