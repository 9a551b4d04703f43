"""Expert recycling in two launches against the loop of single draws that defines its sequence: same values to rounding, same
generator state afterwards; and the way through the framework's own draws, which is taken where its generator draws otherwise
than the kernels."""
import pytest
import torch


def _loop(experts, keys_a, keys_b, dead, pk, top):
    n = experts[0].shape[0]
    for i in dead:
        for t in experts:
            t[i] = t[top] + 0.01 * torch.randn_like(t[i])
        for keys, sharers, row in ((keys_a, range(i // pk * pk, min(n, i // pk * pk + pk)), i // pk), (keys_b, range(i % pk, n, pk), i % pk)):
            if all(j in dead for j in sharers):
                for k in keys:
                    k[row] = torch.randn_like(k[row]) * 0.02


@pytest.mark.gpu
@pytest.mark.parametrize("n,pk,hidden,dead,top", [
    (144, 12, 16, [i for i in range(144) if i % 7], 0),          # most dead, no key
    (144, 12, 4, [i for i in range(144) if i % 12 != 5], 41),    # all columns of keys but one, no row
    (144, 12, 17, list(range(24, 60)) + [100], 30),              # whole rows; the sampled expert is dead, rows above a group of 16
    (10, 4, 1, [1, 2, 3, 5, 6, 7, 8, 9], 0),                     # ragged last row of keys
    (9, 3, 300, list(range(9)), 8),                              # all dead, the sampled one last
    (16, 4, 16, [6], 3),
])
def test_recycling_equals_the_loop(n, pk, hidden, dead, top):
    from grokking_optimizers import _ops

    def tensors():
        gen = torch.Generator().manual_seed(3)
        make = lambda *s: torch.randn(*s, generator=gen).cuda()     # noqa: E731
        return ([make(n, hidden, 1), make(n, hidden), make(n, 1, hidden), make(n, 1)], [make(pk, 4) for _ in range(4)],
                [make(pk, 4) for _ in range(4)])

    want, got = tensors(), tensors()
    gen = torch.cuda.default_generators[0]
    torch.manual_seed(11)
    torch.randn(3, device="cuda")
    _loop(*want, dead, pk, top)
    offset = gen.get_offset()
    torch.manual_seed(11)
    torch.randn(3, device="cuda")
    rows = [all(i in dead for i in range(a * pk, min(n, (a + 1) * pk))) for a in range(pk)]
    cols = [all(i in dead for i in range(b, n, pk)) for b in range(pk)]
    assert _ops.recycle_experts(*got, dead, rows, cols, pk, n, top)
    assert gen.get_offset() == offset
    for w, g in zip([t for group in want for t in group], [t for group in got for t in group]):
        assert (w - g).abs().max().item() < 1e-6


def test_draws_of_another_generator_are_noticed():
    from grokking_optimizers import _ops
    rows = [0.02 * torch.randn(n) for n in (1, 301, 4096)]
    same = [r + 1e-8 * torch.randn_like(r) for r in rows]
    assert _ops.draws_agree(rows, same)
    for k, row in enumerate(rows):
        other = [r.clone() for r in same]
        other[k][-1] += 1e-4
        assert not _ops.draws_agree(rows, other)
        other[k][-1] = float("nan")
        assert not _ops.draws_agree(rows, other)


@pytest.mark.gpu
def test_recycling_by_the_frameworks_draws_gives_the_same_net(monkeypatch):
    from grokking_optimizers import Mamba3PEERMetaNet, _ops

    def run():
        torch.manual_seed(7)
        mn = Mamba3PEERMetaNet().cuda()
        mn.expert_counts.copy_((torch.arange(144) % 12 < 2) * (torch.arange(144) < 60) * 100)      # rows and columns of keys with no live expert
        assert mn._recycle_dead_experts() and int(mn.expert_counts.sum()) == 0
        return list(mn.parameters()), torch.cuda.default_generators[0].get_offset()
    got, offset = run()
    monkeypatch.setattr(_ops, "recycle_experts", lambda *a: False)
    want, want_offset = run()
    assert offset == want_offset
    for a, b in zip(got, want):
        assert (a - b).abs().max().item() < 1e-6
