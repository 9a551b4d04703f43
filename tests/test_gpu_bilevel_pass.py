"""The bilevel pass in one call (elements in the order of the sort, expert sums around a moving reference) against the
same net through the separate entry points (element order, packed copies): tensor sizes around the 64-element tiles and the
1024-element tiles of the sorted walk, unit thresholds all at zero, among the gradients and beyond them, storage types,
expert widths, sharpness absent or not finite."""
import pytest
import torch

from grokking_optimizers import _bilevel
from grokking_optimizers.mamba3_peer_metanet import Mamba3PEERMetaNet

pytestmark = pytest.mark.gpu

# "rests": every number of tiles that a tensor's last 1024 elements can hold
SIZES = {"rests": [64 * k - 31 for k in range(1, 17)] + [1024 + 64 * 3], "tiles": [1, 63, 64, 65, 1023, 1024, 1025], "one_element": [1], "many": [7] * 70 + [200_003]}


@pytest.mark.parametrize("validation", [False, True])
@pytest.mark.parametrize("sizes,dtype,eh,theta,sharp", [
    ("tiles", torch.float32, 16, 0.0, "none"), ("tiles", torch.bfloat16, 4, 1e-3, "some"), ("one_element", torch.float32, 16, 1e-3, "some"),
    ("rests", torch.float32, 16, 1e-3, "some"),
    ("many", torch.float32, 16, 1e-3, "nan"), ("many", torch.float16, 16, 1.0, "none")])
def test_pass_equals_separate_calls(sizes, dtype, eh, theta, sharp, validation, monkeypatch):
    torch.manual_seed(3)
    mn = Mamba3PEERMetaNet(expert_hidden=eh).cuda()
    gen = torch.Generator(device="cuda").manual_seed(4)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    with torch.no_grad():
        mn.expert_b1.copy_(-theta * rand(144, eh) * mn.expert_W1[:, :, 0])
    ns = SIZES[sizes]
    grads = [(rand(n) * 1e-3).to(dtype) for n in ns]
    grads[-1][::5] = 0.0
    sharps = [(rand(n).abs() * 1e-3 * (sharp != "none")).to(torch.float32 if validation else dtype) for n in ns]
    if sharp == "nan":                                    # a tensor whose sharpness holds nothing but zeros and a NaN comes out NaN where it is
        sharps[0].zero_()
        sharps[0][-1] = float("nan")
    grus = [rand(n, 4) * 0.1 for n in ns]
    mf, mb = ([rand(16, 16) * 0.1 for _ in ns] for _ in range(2))
    cots = [rand(n).to(dtype) for n in ns]
    keep = [m.clone() for m in mf + mb]

    def run():
        mn.zero_grad()
        smart = _bilevel.accumulate_meta_gradients(mn, grads, sharps, grus, mf, mb, cots, validation=validation)
        return smart, [p.grad.clone() for p in mn.parameters()]
    smart, got = run()
    assert all(torch.equal(a, b) for a, b in zip(keep, mf + mb))
    monkeypatch.setattr(_bilevel, "_pass_fits", lambda mn: False)
    ref_smart, ref = run()
    torch.testing.assert_close(smart, ref_smart, rtol=1e-5, atol=1e-9, equal_nan=True)
    assert sharp == "nan" or torch.isfinite(smart).all()
    for (name, _), a, b in zip(mn.named_parameters(), got, ref):
        scale = float(b.abs().max())
        assert torch.equal(a.isnan(), b.isnan()) if sharp == "nan" else float((a - b).abs().max()) <= 1e-4 * scale, name
