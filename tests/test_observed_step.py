"""The optimizers' step with listeners (hooks of the instance, global hooks, a profiler) and without: the base class's wrapper
is in the call exactly while there is one."""
import pytest
import torch
from torch.optim import optimizer as base

import grokking_optimizers as go

CLASSES = [go.Grokfast, go.Lion, go.GrokAdamW, go.Prodigy, go.NeuralGrok, go.LookSAM, go.SuperGrok15, go.SuperGrok11, go.SuperGrok2,
           lambda params: go.Muon(params, [])]


@pytest.mark.parametrize("make", CLASSES)
def test_listeners_are_served(make):
    opt = make([torch.nn.Parameter(torch.zeros(4, 4))])           # no gradient: nothing to step, no GPU needed
    cls, seen = type(opt), []
    name = "Optimizer.step#%s.step" % cls.__name__

    def recorded():
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
            opt.step()
        return name in [e.name for e in prof.events()]
    opt.step()
    assert seen == [] and recorded()
    handles = [opt.register_step_pre_hook(lambda o, args, kwargs: seen.append("pre")),
               opt.register_step_post_hook(lambda o, args, kwargs: seen.append("post")),
               base.register_optimizer_step_pre_hook(lambda o, args, kwargs: seen.append("global pre")),
               base.register_optimizer_step_post_hook(lambda o, args, kwargs: seen.append("global post"))]
    try:
        assert opt.step(closure=lambda: 2.0) == 2.0
        assert sorted(seen) == ["global post", "global pre", "post", "pre"]
    finally:
        for h in handles:
            h.remove()
    opt.step()
    assert len(seen) == 4
    # a pre hook's new arguments reach the step
    h = opt.register_step_pre_hook(lambda o, args, kwargs: ((o,), {"closure": lambda: 3.0}))
    assert opt.step() == 3.0
    h.remove()
    # schedulers patch the instance's step
    sched = torch.optim.lr_scheduler.StepLR(opt, 1)
    opt.step()
    sched.step()
