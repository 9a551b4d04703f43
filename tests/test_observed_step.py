"""The optimizers' step with listeners (hooks of the instance and of a subclass's instance, global hooks, a profiler, an observer
without one, dispatch and function modes) and without: every listener sees what it sees of an optimizer of torch's own."""
import json
import os
import subprocess
import sys

import pytest
import torch
from torch.optim import optimizer as base
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

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


SUBCLASSES = """
import json, torch
import grokking_optimizers as go
made = {"Muon": lambda cls, p: cls([p], [])}
def hooks_seen(parent, name, construct_parent):
    class Mine(parent):
        def step(self, closure=None):
            return super().step(closure)
    make = made.get(name, lambda cls, p: cls([p]))
    if construct_parent:
        make(parent, torch.nn.Parameter(torch.zeros(4, 4)))
    opt, seen = make(Mine, torch.nn.Parameter(torch.zeros(4, 4))), []
    opt.register_step_pre_hook(lambda o, args, kwargs: seen.append("pre"))
    opt.register_step_post_hook(lambda o, args, kwargs: seen.append("post"))
    opt.step()
    return seen
classes = {n: getattr(go, n) for n in ("Grokfast", "Lion", "GrokAdamW", "Prodigy", "NeuralGrok", "LookSAM", "SuperGrok15", "SuperGrok11",
                                       "SuperGrok2", "Muon")}
classes["torch"] = torch.optim.Rprop
print(json.dumps({n: [hooks_seen(c, n, False), hooks_seen(c, n, True)] for n, c in classes.items()}))
"""


def test_hooks_of_a_subclass_that_calls_the_parents_step():
    """In a process of its own: whether a class has been constructed before is part of what is compared."""
    out = subprocess.run([sys.executable, "-c", SUBCLASSES], capture_output=True, text=True, check=True,
                         env=dict(os.environ, PYTHONPATH=os.pathsep.join(p for p in sys.path if p)))
    seen = json.loads(out.stdout.strip().splitlines()[-1])
    expected = seen.pop("torch")
    assert expected[0] == ["pre", "post"]
    for name, s in seen.items():
        assert s == expected, name


@pytest.mark.parametrize("make", CLASSES)
def test_observers_without_a_profiler(make, tmp_path):
    opt = make([torch.nn.Parameter(torch.zeros(4, 4))])
    name = "Optimizer.step#%s.step" % type(opt).__name__
    path = str(tmp_path / "trace.json")
    observer = torch.profiler.ExecutionTraceObserver().register_callback(path)
    observer.start()
    opt.step()
    observer.stop()
    observer.unregister_callback()
    with open(path) as f:
        assert name in [n["name"] for n in json.load(f)["nodes"]]
    seen = []

    class Dispatched(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append((str(func), args))
            return func(*args, **(kwargs or {}))

    class Called(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append((str(func), args))
            return func(*args, **(kwargs or {}))
    for mode in (Dispatched, Called):
        seen.clear()
        with mode():
            opt.step()
        assert [a for f, a in seen if "record_function_enter" in f and a and a[0] == name], mode.__name__
    seen.clear()
    opt.step()
    assert not seen


@pytest.mark.parametrize("make", CLASSES)
def test_what_the_base_class_calls_in_a_step_without_listeners(make):
    opt, sgd = make([torch.nn.Parameter(torch.zeros(4, 4))]), torch.optim.SGD([torch.nn.Parameter(torch.zeros(4, 4))])

    def order(o):
        seen, handles = [], []
        o._optimizer_step_code = lambda: seen.append("code")

        def closure():         # a closure may register a hook of the step that it is part of
            seen.append("closure")
            handles.append(o.register_step_post_hook(lambda *a: seen.append("post")))
            handles.append(base.register_optimizer_step_post_hook(lambda *a: seen.append("global post")))
            return torch.zeros(())
        o.step(closure)
        for h in handles:
            h.remove()
        o.step()
        del o._optimizer_step_code
        return seen
    assert order(opt) == order(sgd)
