"""Elements whose |gradient| lies beyond neighbouring unit thresholds of their experts, from none of a tile's picks to all
of them (64 elements, 16 picks of each head: 1024 jobs dealt to the lanes), against the float64 statement."""
import copy

import pytest
import torch

from test_gpu_sg2_bilevel import _grad_ratios, _meta_net, _ref_forward_for_bilevel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("numel", [1, 64, 65, 200])
@pytest.mark.parametrize("decades,far", [(0.0, 0), (0.0, 1), (0.0, 5), (4.0, 0)], ids=["none", "one element", "five", "nearly all"])
def test_picks_in_other_intervals(numel, decades, far):
    from grokking_optimizers import _bilevel
    dev = torch.device("cuda:0")
    mn, gen = _meta_net(31, dev), torch.Generator().manual_seed(32)
    E, EH = mn.num_experts, mn.expert_W1.shape[1]
    sign = lambda *s: torch.randint(0, 2, s, generator=gen) * 2.0 - 1.0
    with torch.no_grad():
        w1 = torch.randn(E, EH, 1, generator=gen) * 0.5
        theta = sign(E, EH) * 10.0 ** (-4.0 * torch.rand(E, EH, generator=gen))      # thresholds from 1e-4 to 1, either sign
        mn.expert_W1.copy_(w1.to(dev))
        mn.expert_b1.copy_((-theta * w1[:, :, 0]).to(dev))
    g = sign(numel) * 1e-2 * 10.0 ** (decades * (torch.rand(numel, generator=gen) - 0.5))
    g[:far] *= 100.0
    d = dict(g=g, s=torch.rand(numel, generator=gen) * 1e-2, h=torch.randn(numel, 4, generator=gen) * 0.5,
             hf=torch.randn(16, 16, generator=gen) * 0.3, hb=torch.randn(16, 16, generator=gen) * 0.3, R=torch.randn(numel, generator=gen))
    mn64 = copy.deepcopy(mn).double().cpu()
    ref, _, _, _ = _ref_forward_for_bilevel(mn64, *(d[k].double() for k in ("g", "s", "h", "hf", "hb")))
    (ref * d["R"].double()).sum().backward()
    mn.zero_grad()
    got = _bilevel.accumulate_meta_gradients(mn, *([d[k].to(dev)] for k in ("g", "s", "h", "hf", "hb", "R"))).double().cpu()
    # the bounds of the test of the thresholds at the gradients' scale
    err, tol = (got - ref.detach()).abs(), 1e-4 * torch.maximum(got.abs(), ref.detach().abs()) + 1e-7
    assert bool((err <= tol).all()), float((err / tol).max())
    w = _grad_ratios([(n, p.grad) for n, p in mn.named_parameters()], [(n, p.grad) for n, p in mn64.named_parameters()], 2e-4)
    assert max(w.values()) <= 1.0, w
