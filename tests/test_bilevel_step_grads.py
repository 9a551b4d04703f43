"""SuperGrok2.bilevel_step keeps the training gradients apart from the validation pass, also where a backward pass returns
the same buffer every time: the pass works on them and .grad holds them afterwards."""
import pytest
import torch

from grokking_optimizers import SuperGrok2, _bilevel

SHAPES = [(40, 30), (300,), (1,)]


class _GivenGradients(torch.autograd.Function):
    """A loss whose gradients are `grads`, handed out in the memory where they lie."""

    @staticmethod
    def forward(ctx, grads, *params):
        ctx.grads = grads
        return params[0].new_ones(())

    @staticmethod
    def backward(ctx, _):
        return (None, *(g.detach() for g in ctx.grads))


class _Network(torch.nn.Module):
    """Its input is (train, validation) gradients' index; the gradients pass through one persistent buffer per parameter, or
    through a new tensor each time."""

    def __init__(self, shapes, device, static):
        super().__init__()
        gen = torch.Generator().manual_seed(5)
        make = lambda: [(torch.randn(s, generator=gen) * 1e-3).to(device) for s in shapes]      # noqa: E731
        self.params = torch.nn.ParameterList(make())
        self.sets = [make(), make()]
        self.buffers = [torch.zeros(s, device=device) for s in shapes] if static else None

    def forward(self, which):
        grads = [g.clone() for g in self.sets[which]]
        if self.buffers is not None:
            grads = [b.copy_(g) for b, g in zip(self.buffers, grads)]
        return _GivenGradients.apply(grads, *self.params)


def _bilevel_step(device, static):
    net = _Network(SHAPES, device, static)
    torch.manual_seed(2)
    opt = SuperGrok2(net.parameters())
    opt._ensure_state()
    gen = torch.Generator().manual_seed(6)
    for i, p in enumerate(net.params):
        opt._flat_mamba_fwd_states[i] = (torch.randn(16, 16, generator=gen) * 0.1).to(device)
        opt._flat_mamba_bwd_states[i] = (torch.randn(16, 16, generator=gen) * 0.1).to(device)
        opt._flat_gru_states[i].copy_(torch.randn(p.numel(), 4, generator=gen) * 0.1)
    net(0).backward()
    if static:
        assert all(p.grad.data_ptr() == b.data_ptr() for p, b in zip(net.params, net.buffers))
    opt.bilevel_step(net, 0, None, 1, None, lambda out, _: out, torch.optim.SGD(opt.meta_net.parameters(), lr=0.0))
    for p, g in zip(net.params, net.sets[0]):
        assert torch.equal(p.grad, g)
    return opt


@pytest.mark.parametrize("static", [False, True])
def test_training_gradients_reach_the_pass_and_stay(static, monkeypatch):
    seen = {}
    monkeypatch.setattr(_bilevel, "begin_pass", lambda mn, grads, *a, **kw: None)
    monkeypatch.setattr(_bilevel, "accumulate_meta_gradients", lambda mn, grads, s, h, f, b, cots, **kw: seen.update(
        grads=[g.clone() for g in grads], cots=[c.clone() for c in cots]))
    _bilevel_step("cpu", static)
    ref = _Network(SHAPES, "cpu", False)
    for k, name in enumerate(("grads", "cots")):
        assert all(torch.equal(a, b) for a, b in zip(seen[name], ref.sets[k])), name


@pytest.mark.parametrize("over,order", [(0, ["begin", "network", "finish"]), (1, ["network", "finish"])])
def test_a_large_pass_takes_its_workspace_after_the_validation_pass(over, order, monkeypatch):
    """Up to EARLY_ELEMENTS the sort and scan are enqueued first; beyond, the pass begins inside the accumulation, when the
    validation pass has given its activations back."""
    calls = []
    forward = _Network.forward
    monkeypatch.setattr(_Network, "forward", lambda self, which: calls.append("network") or forward(self, which))
    monkeypatch.setattr(_bilevel, "EARLY_ELEMENTS", sum(torch.Size(s).numel() for s in SHAPES) - over)
    monkeypatch.setattr(_bilevel, "begin_pass", lambda *a, **kw: calls.append("begin"))
    monkeypatch.setattr(_bilevel, "accumulate_meta_gradients", lambda *a, **kw: calls.append("finish"))
    _bilevel_step("cpu", False)
    assert calls == ["network"] + order               # the first one is the training pass


@pytest.mark.gpu
def test_static_gradient_buffers_give_the_same_meta_gradients():
    a, b = (_bilevel_step("cuda", static).meta_net for static in (False, True))
    for (name, p), q in zip(a.named_parameters(), b.parameters()):
        # same kernels on the same values; the experts' sums are atomics in varying order
        assert float((p.grad - q.grad).abs().max()) <= 1e-5 * float(p.grad.abs().max()), name
