"""Expert recycling after counts have run past 2^31: entries of the 32-bit counter read as negative."""
import torch

from grokking_optimizers import Mamba3PEERMetaNet


def _recycled(counts):
    torch.manual_seed(3)
    net = Mamba3PEERMetaNet()
    net.expert_counts.copy_(counts)
    torch.manual_seed(4)
    assert net._recycle_dead_experts()
    assert int(net.expert_counts.sum()) == 0
    return [p.clone() for p in net.parameters()]


def test_counts_past_two_to_the_31_recycle_as_counts():
    small = torch.zeros(144, dtype=torch.int32)
    small[5], small[9] = 3, 1
    large = torch.zeros(144, dtype=torch.int32)
    large[5], large[9] = 3 * 2 ** 30 - 2 ** 32, 2 ** 30          # 3 * 2^30 as the counter holds it
    for a, b in zip(_recycled(small), _recycled(large)):
        assert torch.equal(a, b)
