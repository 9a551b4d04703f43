"""The elementwise kernels at the edges of their dispatch: amplifier tables of every width class with units that have no
threshold and its rounding far from zero, gradients on both sides of the meta-net polynomial's reach, tensor counts on both sides of what travels
as kernel arguments, and pointers that do not allow four elements per access."""
import numpy as np
import pytest
import torch

from helpers import rel_close
from oracle import family_oracle as fo

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ops():
    from grokking_optimizers import _ops
    return _ops


def _dev(arrs, shift=0):
    """device copies; shift: element offset from an aligned address"""
    out = []
    for a in arrs:
        buf = torch.zeros(a.size + shift, device=DEV)
        buf[shift:].copy_(torch.from_numpy(a))
        out.append(buf[shift:])
    return out


def _check(got, want, tag):
    for k in got:
        for i, (a, b) in enumerate(zip(got[k], want[k])):
            ok, worst = rel_close(a.cpu().numpy(), b, 1e-4, 1e-7)
            assert ok, (tag, k, i, worst)


def _state(r, sizes, gstd):
    f = lambda std: [(r.randn(n) * std).astype(np.float32) for n in sizes]
    return dict(p=f(0.02), g=f(gstd), ea=f(1e-3), easq=[np.abs(x) * 1e-3 for x in f(1e-3)], aux=f(1e-3), sh=[np.abs(x) for x in f(gstd)])


@pytest.mark.parametrize("H", [1, 2, 3, 127, 128, 255, 256])
@pytest.mark.parametrize("shift", [0, 1])
def test_amplifier_table(H, shift):
    r = np.random.RandomState(H)
    w1, b1, w2, b2 = (r.randn(H, 1)).astype(np.float32), (r.randn(H) * 0.5).astype(np.float32), (r.randn(1, H) * 0.1).astype(np.float32), \
        np.float32([0.05])
    w1[::5] = 0.0                      # units that do not look at the gradient
    b1[::7] = 0.0                      # thresholds at 0
    st = _state(r, [5000, 3], 0.7)     # gradients on every side of the thresholds
    st["g"][1][0] = 0.0
    want = {k: [x.copy() for x in v] for k, v in st.items()}
    got = {k: _dev(v, shift) for k, v in st.items()}
    sc = (10.0, 4.0, 0.9, 0.98, 1e-3, 1.0, 1e-8, 0.0)
    W = [torch.from_numpy(x).to(DEV) for x in (w1, b1, w2, b2)]
    _ops().neuralgrok_fused_step(got["p"], got["g"], got["ea"], got["easq"], [3, 3], *W, sc[0], sc[1], H, *sc[2:])
    fo.neuralgrok_step(want["p"], want["g"], want["ea"], want["easq"], [3, 3], w1, b1, w2, b2, *sc)
    _check({k: got[k] for k in ("p", "g", "ea", "easq")}, want, H)


@pytest.mark.parametrize("spread", [1e-3, 1.0, 300.0])
def test_amplifier_table_stays_within_its_rounding(spread):
    """The line A g + B of an interval against float64, for gradients up to and far beyond the thresholds: A and B are rounded
    once (2^-24 each), the fused multiply-add and the product with g once more."""
    r, H = np.random.RandomState(5), 128
    w1, b1, w2 = (r.uniform(-1, 1, s).astype(np.float32) for s in ((H, 1), (H,), (1, H)))
    g = (r.randn(40_000) * spread).astype(np.float32)
    got = {k: _dev([x]) for k, x in dict(p=np.zeros_like(g), g=g, ea=np.zeros_like(g), easq=np.zeros_like(g)).items()}
    W = [torch.from_numpy(x).to(DEV) for x in (w1, b1, w2, np.float32([0.0]))]
    _ops().neuralgrok_fused_step(got["p"], got["g"], got["ea"], got["easq"], [3], *W, 1.0, 0.0, H, 0.0, 0.98, 1e-3, 1.0, 1e-8, 0.0)      # beta1 = 0: exp_avg is the amplified gradient
    x, w1, b1, w2 = (a.astype(np.float64).reshape(-1) for a in (g, w1, b1, w2))
    active = w1[:, None] * x + b1[:, None] > 0
    A, B = ((active * (w2 * c)[:, None]).sum(0) for c in (w1, b1))
    value = A * x + B
    err = np.abs(got["ea"][0].cpu().numpy() / x - value)
    assert (err <= 2.0 ** -24 * 1.01 * (np.abs(A * x) + np.abs(B) + 2 * np.abs(value)) + 1e-30).all(), float(err.max())


@pytest.mark.parametrize("H", [63, 64, 65, 128, 129, 193, 256])
def test_amplifier_table_across_waves(H):
    """Widths at which the running sums cross a wave, with equal thresholds, thresholds that overflow to either infinity and units
    that do not look at the gradient, against float64: the line's rounding as above, and each of H float64 additions 2^-53."""
    r = np.random.RandomState(H)
    w1, b1, w2 = (r.uniform(-1, 1, s).astype(np.float32) for s in ((H, 1), (H,), (1, H)))
    w1[1::6], b1[1::6] = 0.5, -0.25                    # all at 0.5, rising
    w1[2::6], b1[2::6] = -0.5, 0.25                    # all at 0.5, falling
    w1[3::12], b1[3::12] = 1e-39, 0.75                 # -inf
    w1[9::12], b1[9::12] = -1e-39, 0.75                # +inf, always active
    w1[4::6] = 0.0
    g = np.concatenate([r.randn(20_000), np.float32([0.5, -0.5, 3e38, -3e38, 1e-30])]).astype(np.float32)
    got = {k: _dev([x]) for k, x in dict(p=np.zeros_like(g), g=g, ea=np.zeros_like(g), easq=np.zeros_like(g)).items()}
    W = [torch.from_numpy(x).to(DEV) for x in (w1, b1, w2, np.float32([0.0]))]
    _ops().neuralgrok_fused_step(got["p"], got["g"], got["ea"], got["easq"], [3], *W, 1.0, 0.0, H, 0.0, 0.98, 1e-3, 1.0, 1e-8, 0.0)
    x, w1, b1, w2 = (a.astype(np.float64).reshape(-1) for a in (g, w1, b1, w2))
    active = w1[:, None] * x + b1[:, None] > 0
    A, B = ((active * (w2 * c)[:, None]).sum(0) for c in (w1, b1))
    sA, sB = ((active * np.abs(w2 * c)[:, None]).sum(0) for c in (w1, b1))
    value = A * x + B
    sel = np.abs(x) < 1e4                              # the product with g overflows for the largest
    err = np.abs(got["ea"][0].cpu().numpy() / x - value)
    bound = 2.0 ** -24 * 1.01 * (np.abs(A * x) + np.abs(B) + 2 * np.abs(value)) + H * 2.0 ** -53 * (sA * np.abs(x) + sB) + 1e-30
    assert (err <= bound)[sel].all(), float((err / bound)[sel].max())


@pytest.mark.parametrize("H", [1, 32, 256])
@pytest.mark.parametrize("gstd", [1e-3, 0.03, 1.0])
def test_meta_net_polynomial(H, gstd):
    r = np.random.RandomState(int(H + 1000 * gstd))
    W = [(r.randn(H, 2) * 0.5).astype(np.float32), (r.randn(H) * 0.5).astype(np.float32), (r.randn(1, H) * 0.5).astype(np.float32), np.float32([0.1])]
    st = _state(r, [4099, 700], gstd)
    want = {k: [x.copy() for x in v] for k, v in st.items()}
    got = {k: _dev(v) for k, v in st.items()}
    sc = (0.1, 0.999, 1e-3, 1.0, 1e-8, 5.0, 0.7, 5.0, 1.0)
    al, be = [0.98, 0.97], [0.9, 0.81]
    Wd = [torch.from_numpy(x).to(DEV) for x in W]
    _ops().supergrok11_fused_step(got["p"], got["g"], got["ea"], got["easq"], got["aux"], got["sh"], [4, 4], al, be, *Wd, sc[0], H, *sc[1:])
    fo.sg11_step(want["p"], want["g"], want["ea"], want["easq"], want["aux"], want["sh"], [4, 4], al, be, *W, *sc)
    _check({k: got[k] for k in ("p", "g", "ea", "easq", "aux")}, want, (H, gstd))


@pytest.mark.parametrize("P", [49, 50, 51, 70])
def test_tensor_counts(P):
    r = np.random.RandomState(P)
    sizes = [1 + 37 * i for i in range(P)]
    st = _state(r, sizes, 0.05)
    want = {k: [x.copy() for x in v] for k, v in st.items()}
    got = {k: _dev(v) for k, v in st.items()}
    sc = (0.98, 5.0, 0.9, 0.98, 1e-3, 1.0, 1e-8, 1.0)
    _ops().grokadamw_fused_step(got["p"], got["g"], got["ea"], got["easq"], got["aux"], [2] * P, *sc)
    fo.grokadamw_step(want["p"], want["g"], want["ea"], want["easq"], want["aux"], [2] * P, *sc)
    _check({k: got[k] for k in ("p", "g", "ea", "easq", "aux")}, want, P)
    clipped = _ops().supergrok2_clip_grads(got["sh"], 1e-3)
    _check({"c": clipped}, {"c": fo.sg2_clip(want["sh"], 1e-3)}, P)
