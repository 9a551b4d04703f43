"""Argument checks, per-parameter state and the base class shared by the optimizer classes."""
import functools
import itertools

import torch
import torch.optim.optimizer as _base

from grokking_optimizers import _ops


class FusedOptimizer(_base.Optimizer):
    """torch's Optimizer with a cheaper wrapper around `step`.  At construction the base class replaces the `step` of the
    instance's class by what `profile_hook_step` makes of it: a record for profilers and the step hooks around every call,
    6 us where nobody listens, as much as the rest of the call of a step whose kernels take 5.  Here the record is left
    out of the calls that nothing can see it in (Grokfast on 14 tensors, 0.42 M elements: 15.6 -> 9.5 us with the
    gradient's arrival).  What is wrapped, and when, stays the base class's affair, subclasses included."""

    @staticmethod
    def profile_hook_step(func):
        listened = _base.Optimizer.profile_hook_step(func)
        before, after = (getattr(_base, "_global_optimizer_%s_hooks" % k, None) for k in ("pre", "post"))
        if before is None or after is None:
            return listened             # another base class: as it sees fit

        @functools.wraps(func)
        def step(*args, **kwargs):
            self = args[0]
            if before or self._optimizer_step_pre_hooks or torch.compiler.is_compiling() or _ops.calls_are_observed():
                return listened(*args, **kwargs)
            out = func(*args, **kwargs)
            self._optimizer_step_code()
            if after or self._optimizer_step_post_hooks:       # (also those that the step itself registered)
                for hook in itertools.chain(self._optimizer_step_post_hooks.values(), after.values()):
                    hook(self, args, kwargs)
            return out
        return step


def check_hyper(lr=None, eps=None, betas=None):
    if lr is not None and lr < 0.0:
        raise ValueError(f"Invalid learning rate: {lr}")
    if eps is not None and eps < 0.0:
        raise ValueError(f"Invalid epsilon value: {eps}")
    if betas is not None:
        for k in (0, 1):
            if not 0.0 <= betas[k] < 1.0:
                raise ValueError(f"Invalid beta parameter at index {k}: {betas[k]}")


def check_ranges(checks):
    """checks: (name, value, lowest, upper bound or None); lowest <= value (< upper) or ValueError("Invalid <name>: <value>")."""
    for name, value, low, high in checks:
        if value < low or (high is not None and not value < high):
            raise ValueError(f"Invalid {name}: {value}")


def run_closure(closure):
    if closure is None:
        return None
    with torch.enable_grad():
        return closure()


def gather(optimizer, group, buffers, count_steps=True, extra_init=None):
    """Parameters of `group` that have a gradient, with their fp32 state buffers (created as zeros on
    first use) and step counters (incremented here when count_steps)."""
    out = {"params": [], "grads": [], "steps": []}
    for b in buffers:
        out[b] = []
    for p in group["params"]:
        if p.grad is None:
            continue
        st = optimizer.state[p]
        if len(st) == 0:
            st["step"] = 0
            for b in buffers:
                st[b] = torch.zeros_like(p, dtype=torch.float32)
            if extra_init is not None:
                extra_init(p, st)
        if count_steps:
            st["step"] += 1
        out["params"].append(p)
        out["grads"].append(p.grad)
        out["steps"].append(st["step"])
        for b in buffers:
            out[b].append(st[b])
    return out
