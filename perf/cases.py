"""Timed work of this package: optimizer steps and meta-training passes as a training program calls them.

Every case is one call of a public class method on parameters, gradients and optimizer state that already live on the
GPU, as they do in the middle of a run: `SuperGrok2.step`, `SuperGrok2.bilevel_step`, `Muon.step` and the `step` of
the elementwise optimizers.  Parameter sets are the ones of `workloads.py` (the two-layer transformer for modular
addition, the 50-tensor set of 25 M elements, the tensors below 256 elements) and ladders of ragged sizes between
their extremes.
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "supergrok1.5_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import grokking_optimizers as go  # noqa: E402
import workloads  # noqa: E402

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
ELEMENTWISE = ("grokfast", "supergrok15", "supergrok11", "grokadamw", "neuralgrok", "prodigy", "lion")
MAX_ELEMENTS = 25_000_000


def listed():
    return [
        # SuperGrok v2 step of a model with nothing but biases and norms left to it (every tensor below 256 elements):
        # launches and host work are all there is
        dict(name="v2_step_tiny", path="v2_step", shapes="small8", dtype="float32", sharpness=False, d_model=8, d_state=16,
             expert_hidden=16),
        # SuperGrok v2 step of the modular-addition transformer with the sharpness cache filled, as step_full keeps it
        dict(name="v2_step_transformer", path="v2_step", shapes="shared14", dtype="float32", sharpness=True, d_model=8,
             d_state=16, expert_hidden=16),
        # SuperGrok v2 step of a bf16 model of a few million parameters with ragged sizes, sharpness cache filled, and the
        # narrower experts that the reference's training harness constructs the optimizer with
        dict(name="v2_step_ragged_bf16", path="v2_step", shapes="ladder", tensors=23, elements=3_141_593, dtype="bfloat16",
             sharpness=True, d_model=8, d_state=16, expert_hidden=4),
        # SuperGrok v2 step at scale, the headline configuration: 50 tensors, 25 M elements, no sharpness probe yet
        dict(name="v2_step_scale50", path="v2_step", shapes="scale50", dtype="float32", sharpness=False, d_model=8, d_state=16,
             expert_hidden=16),
        # SuperGrok v2 step of the transformer under the wider meta-net (d_model 16, d_state 32)
        dict(name="v2_step_wide_meta_net", path="v2_step", shapes="shared14", dtype="float32", sharpness=True, d_model=16,
             d_state=32, expert_hidden=16),
        # Meta-training of v2 on the transformer: the bilevel update that a run makes every 5 to 30 steps
        dict(name="bilevel_transformer", path="bilevel", shapes="shared14", dtype="float32", expert_hidden=16),
        # The same on the 25 M-element set
        dict(name="bilevel_scale50", path="bilevel", shapes="scale50", dtype="float32", expert_hidden=16),
        # Muon on the transformer: its matrices through Newton-Schulz, its vectors through AdamW
        dict(name="muon_transformer", path="muon", shapes="shared14", dtype="float32"),
        # Muon on 24 bf16 matrices of a transformer with width 1024
        dict(name="muon_24_bf16", path="muon", shapes="matrices", matrices=24, rows=1024, cols=4096, dtype="bfloat16"),
        # The elementwise optimizers on the transformer, where a step is a launch or three
        dict(name="grokfast_transformer", path="elementwise", optimizer="grokfast", shapes="shared14", dtype="float32"),
        dict(name="supergrok15_transformer", path="elementwise", optimizer="supergrok15", shapes="shared14", dtype="float32"),
        # An elementwise optimizer at scale (learned amplifier of width 128)
        dict(name="neuralgrok_scale50", path="elementwise", optimizer="neuralgrok", shapes="scale50", dtype="float32"),
    ]


def draw(rng):
    """One more case: a path, then sizes over the logarithm of its range."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def ladder(lo):
        elements = log_int(lo, MAX_ELEMENTS)
        return dict(shapes="ladder", tensors=min(log_int(1, 60), max(1, elements // 8)), elements=elements)

    path = rng.choice(("v2_step", "v2_step", "v2_step", "bilevel", "muon", "elementwise", "elementwise", "elementwise"))
    if path == "v2_step":
        d_model, d_state, expert_hidden = rng.choice(((8, 16, 16), (8, 16, 16), (8, 16, 4), (16, 32, 16)))
        case = dict(path=path, **ladder(300), dtype=rng.choice(("float32", "float32", "bfloat16", "float16")),
                    sharpness=rng.random() < 0.5, d_model=d_model, d_state=d_state, expert_hidden=expert_hidden)
    elif path == "bilevel":
        case = dict(path=path, **ladder(3000), dtype=rng.choice(("float32", "float32", "bfloat16")),
                    expert_hidden=rng.choice((16, 16, 4)))
    elif path == "muon":
        case = dict(path=path, shapes="matrices", matrices=log_int(1, 24), rows=log_int(32, 1024), cols=log_int(32, 4096),
                    dtype=rng.choice(("bfloat16", "float32")))
    else:
        case = dict(path=path, optimizer=rng.choice(ELEMENTWISE), **ladder(1000),
                    dtype=rng.choice(("float32", "float32", "bfloat16")))
    return case


def _shapes(case):
    kind = case["shapes"]
    if kind == "small8":
        return workloads.small8_shapes()
    if kind == "shared14":
        return workloads.shared14_shapes()
    if kind == "scale50":
        return workloads.scale50_shapes()
    if kind == "matrices":       # every other one transposed, as the two projections of an MLP are
        r, c = case["rows"], case["cols"]
        return [(r, c) if i % 2 == 0 else (c, r) for i in range(case["matrices"])]
    # sizes log-uniform over three decades (fewer where the tensors are few), vectors, together case["elements"]
    n = case["tensors"]
    weights = [1000.0 ** ((i + 0.5) / n) for i in range(n)]
    scale = case["elements"] / sum(weights)
    sizes = [max(1, int(w * scale)) for w in weights]
    sizes[-1] = max(1, sizes[-1] + case["elements"] - sum(sizes))
    return [(s,) for s in sizes]


def _numels(case):
    return [math.prod(s) for s in _shapes(case)]


class _Packed:
    """Tensors of one kind as views of a single buffer, each at a multiple of 512 bytes as the caching allocator
    places them, so that all of a kind can be handed back as one tensor."""

    def __init__(self, shapes, dtype, fill=None):
        step = 512 // torch.empty(0, dtype=dtype).element_size()
        offsets, end = [], 0
        for s in shapes:
            offsets.append(end)
            end += -(-math.prod(s) // step) * step
        self.flat = torch.zeros(end, dtype=dtype, device="cuda")
        self.views = [self.flat[o:o + math.prod(s)].view(s) for o, s in zip(offsets, shapes)]
        if fill is not None:
            src, o = fill(sum(math.prod(s) for s in shapes)), 0
            for v in self.views:
                v.copy_(src[o:o + v.numel()].view(v.shape))
                o += v.numel()


class _Source:
    """Random values on the GPU from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, std):
        return lambda n: torch.randn(n, generator=self.gen, device="cuda").mul_(std)

    def positive(self, scale):
        return lambda n: torch.rand(n, generator=self.gen, device="cuda").add_(0.01).mul_(scale)

    def gradient(self, std=1e-3, tail=0.005):
        """N(0, std) with a Student-t(3) tail on a share of the entries."""
        def make(n):
            g = torch.randn(n, generator=self.gen, device="cuda").mul_(std)
            k, block = int(n * tail), int(1 / tail)        # one entry of each block, at a random place
            if k:
                z = torch.randn(4, k, generator=self.gen, device="cuda")
                at = torch.arange(k, device="cuda") * block + torch.randint(block, (k,), generator=self.gen, device="cuda")
                g[at] = std * z[0] / torch.sqrt(z[1:].square().sum(0) / 3)
            return g
        return make


class _KnownGradient(torch.autograd.Function):
    """A loss whose gradient is given: stands for the user's network and its validation batch."""

    @staticmethod
    def forward(ctx, grads, *params):
        ctx.grads = grads
        return params[0].new_zeros(())

    @staticmethod
    def backward(ctx, _):
        return (None, *ctx.grads)


class _Network(torch.nn.Module):
    def __init__(self, params, val_grads):
        super().__init__()
        self.params = torch.nn.ParameterList(params)
        self.val_grads = val_grads

    def forward(self, x):
        return _KnownGradient.apply(self.val_grads, *self.params)


class _State:
    pass


def _parameters(st, case, src):
    dtype, shapes = DTYPES[case["dtype"]], _shapes(case)
    st.param_store = _Packed(shapes, dtype, src.normal(0.02))
    st.grad_store = _Packed(shapes, dtype, src.gradient())
    st.params = [torch.nn.Parameter(v) for v in st.param_store.views]
    for p, g in zip(st.params, st.grad_store.views):
        p.grad = g


def _flat_lists(st, opt, kinds):
    """Optimizer state of a run in progress in the class's per-parameter lists, restored as from a checkpoint."""
    opt._ensure_state()
    out = {}
    for attr, (shapes, fill) in kinds.items():
        out[attr] = _Packed(shapes, torch.float32, fill)
        setattr(opt, attr, list(out[attr].views))
    opt._global_step = 250
    return {k: v.flat for k, v in out.items()}


def _supergrok2(st, case, src, seed, sharpness):
    torch.manual_seed(seed)
    d_model, d_state, eh = case.get("d_model", 8), case.get("d_state", 16), case["expert_hidden"]
    opt = go.SuperGrok2(st.params, d_model=d_model, d_state=d_state, expert_hidden=eh)
    flat = [(p.numel(),) for p in st.params]
    gru = [(p.numel(), opt.gru_hidden) for p in st.params]
    mamba = [(opt.meta_net.mamba_fwd.d_inner, d_state)] * len(flat)
    st.buffers = _flat_lists(st, opt, {
        "_flat_exp_avgs": (flat, src.normal(3e-4)), "_flat_exp_avg_sqs": (flat, src.positive(1e-6)),
        "_flat_mus": (flat, src.normal(3e-4)), "_flat_gru_states": (gru, src.normal(0.05)),
        "_flat_mamba_fwd_states": (mamba, src.normal(1e-3)), "_flat_mamba_bwd_states": (mamba, src.normal(1e-3)),
        "_flat_sharpness": (flat, src.positive(1e-3) if sharpness else None)})
    del st.buffers["_flat_sharpness"]            # an input
    opt._flat_steps = [250] * len(flat)
    return opt


def _prepare_v2_step(st, case, src, seed):
    _parameters(st, case, src)
    st.opt = _supergrok2(st, case, src, seed, case["sharpness"])


def _run_v2_step(st):
    st.opt.step()
    return dict(st.buffers, params=st.param_store.flat, expert_counts=st.opt.meta_net.expert_counts)


def _prepare_bilevel(st, case, src, seed):
    _parameters(st, case, src)
    st.opt = _supergrok2(st, case, src, seed, True)
    val = _Packed(_shapes(case), DTYPES[case["dtype"]], src.gradient())
    st.model = _Network(st.params, val.views)
    # a small rate: the meta-net stays the one that the case describes over many passes
    st.meta_opt = torch.optim.Adam(st.opt.meta_net.parameters(), lr=1e-6)
    st.batch = torch.zeros(1, device="cuda")


def _run_bilevel(st):
    loss = st.opt.bilevel_step(st.model, st.batch, st.batch, st.batch, st.batch, lambda out, y: out, st.meta_opt)
    return {"val_loss": loss, "meta_gradients": [p.grad for p in st.opt.meta_net.parameters()]}


def _prepare_muon(st, case, src, seed):
    _parameters(st, case, src)
    two = [p for p in st.params if p.dim() == 2]
    one = [p for p in st.params if p.dim() != 2]
    st.opt = go.Muon(two, one)
    shapes = [tuple(p.shape) for p in two]
    st.buffers = {"momentum": _Packed(shapes, torch.float32, src.normal(1e-3))}
    for p, m in zip(two, st.buffers["momentum"].views):
        st.opt.state[p] = {"momentum_buffer": m}
    if one:
        shapes = [tuple(p.shape) for p in one]
        st.buffers.update(exp_avg=_Packed(shapes, torch.float32, src.normal(3e-4)),
                          exp_avg_sq=_Packed(shapes, torch.float32, src.positive(1e-6)))
        for i, p in enumerate(one):
            st.opt.state[p] = {"step": 250, "exp_avg": st.buffers["exp_avg"].views[i], "exp_avg_sq": st.buffers["exp_avg_sq"].views[i]}


def _run_muon(st):
    st.opt.step()
    return dict({k: b.flat for k, b in st.buffers.items()}, params=st.param_store.flat)


_CLASSES = dict(grokfast=go.Grokfast, supergrok15=go.SuperGrok15, supergrok11=go.SuperGrok11, grokadamw=go.GrokAdamW,
                neuralgrok=go.NeuralGrok, prodigy=go.Prodigy, lion=go.Lion)
_PER_PARAMETER = dict(grokfast=("ema", "exp_avg", "exp_avg_sq"), grokadamw=("ema", "exp_avg", "exp_avg_sq"),
                      neuralgrok=("exp_avg", "exp_avg_sq"), prodigy=("exp_avg", "exp_avg_sq", "s", "param_init"), lion=("exp_avg",))


def _prepare_elementwise(st, case, src, seed):
    _parameters(st, case, src)
    torch.manual_seed(seed)
    name = case["optimizer"]
    # the step clips or amplifies the gradients where they lie; a backward pass brings new ones before each
    st.incoming = st.grad_store.flat.clone()
    if name == "neuralgrok":
        st.opt = go.NeuralGrok(st.params, num_layers=2)
    else:
        st.opt = _CLASSES[name](st.params)
    shapes = [tuple(p.shape) for p in st.params]
    if name in ("supergrok15", "supergrok11"):
        with torch.no_grad():
            st.opt.meta_net.rescale.fill_(0.1)           # a trained meta-net: the module starts at 0
        flat = [(p.numel(),) for p in st.params]
        st.buffers = _flat_lists(st, st.opt, {
            "_flat_exp_avgs": (flat, src.normal(3e-4)), "_flat_exp_avg_sqs": (flat, src.positive(1e-6)),
            "_flat_mus": (flat, src.normal(3e-4)), "_flat_sharpness": (flat, src.positive(1e-3))})
        del st.buffers["_flat_sharpness"]
        return
    fills = dict(ema=src.normal(3e-4), exp_avg=src.normal(3e-4), exp_avg_sq=src.positive(1e-6), s=src.positive(1e-6),
                 param_init=src.normal(0.02))
    packed = {k: _Packed(shapes, torch.float32, fills[k]) for k in _PER_PARAMETER[name]}
    for i, p in enumerate(st.params):
        st.opt.state[p] = dict({k: b.views[i] for k, b in packed.items()}, **({} if name == "lion" else {"step": 250}))
    packed.pop("param_init", None)                       # an input
    st.buffers = {k: b.flat for k, b in packed.items()}


def _run_elementwise(st):
    st.grad_store.flat.copy_(st.incoming)
    st.opt.step()
    return dict(st.buffers, params=st.param_store.flat, grads=st.grad_store.flat)


_PREPARE = dict(v2_step=_prepare_v2_step, bilevel=_prepare_bilevel, muon=_prepare_muon, elementwise=_prepare_elementwise)
_RUN = dict(v2_step=_run_v2_step, bilevel=_run_bilevel, muon=_run_muon, elementwise=_run_elementwise)


def prepare(case, seed):
    st = _State()
    st.path = case["path"]
    _PREPARE[st.path](st, case, _Source(seed), seed)
    return st


def run(state):
    return _RUN[state.path](state)


def work(case):
    """Bytes that have to be moved and operations that have to be done, per pass."""
    n = sum(_numels(case))
    e = torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
    path = case["path"]
    if path in ("v2_step", "bilevel"):
        dm, ds = case.get("d_model", 8), case.get("d_state", 16)
        di, gh, heads, keys = 2 * dm, 4, 4, 12
        # both directions: projections of the two-number input, 2x2 state update with its drive and output, gate, out_proj
        scan = 2 * (2 * 2 * (3 * di + 2 * ds) + di * ds * 8 + 2 * di * dm)
        gru = 2 * 3 * gh * (2 + 2 * dm + gh)
        peer = heads * 2 * (dm * (gh + 2 * dm + 2) + keys * dm)
        experts = heads * 4 * case["expert_hidden"]
        if path == "v2_step":
            # param, grad, sharpness in their type; exp_avg, exp_avg_sq, mu and the four GRU entries in fp32; the first
            # and the last five written back
            moved = n * (3 * e + 4 * (3 + gh) + e + 4 * (3 + gh))
            if not case["sharpness"]:
                moved -= n * e
            return {"bytes": moved, "flops": n * (scan + gru + peer + experts)}
        # gradient, validation gradient, sharpness and GRU state read once; forward and twice as much backward,
        # 16 experts a head
        return {"bytes": n * (2 * e + 4 + 4 * gh), "flops": 3 * n * (scan + gru + peer + 16 * experts)}
    if path == "muon":
        shapes = [s for s in _shapes(case) if len(s) == 2]
        n2 = sum(math.prod(s) for s in shapes)
        # parameter and gradient in their type, momentum in fp32; five quintic iterations on the smaller side
        return {"bytes": n2 * (3 * e + 8) + (n - n2) * (3 * e + 16),
                "flops": 5 * sum(6 * min(s) ** 2 * max(s) for s in shapes)}
    reads, writes, flops = {"grokfast": (3, 3, 20), "supergrok15": (4, 3, 20 + 32 * 12), "supergrok11": (4, 3, 30 + 32 * 12),
                            "grokadamw": (3, 3, 20), "neuralgrok": (2, 2, 20 + 128 * 4), "prodigy": (4, 3, 24),
                            "lion": (1, 1, 8)}[case["optimizer"]]
    # the gradient's arrival (a copy) and the step: parameter and gradient in their type, the rest in fp32
    return {"bytes": n * (2 * e + 3 * e + 4 * (reads + writes)), "flops": n * flops}


def tolerance(case):
    if case["path"] == "muon":
        return {"rel": 1e-2}               # the iteration runs in bf16
    if case["dtype"] != "float32" and case["path"] != "bilevel":
        # parameters (and clipped gradients) rounded to 8 bits, fp16 ones to 11; expert counts at ties
        return {"rel": 4e-3, "differ": 0.01} if case["path"] == "v2_step" else {"rel": 4e-3}
    if case["path"] == "bilevel":
        return {"rel": 1e-4}               # 32-bit sums over all elements of terms of either sign
    if case["path"] == "v2_step":
        return {"rel": 1e-4, "differ": 0.01}      # a chain of 32-bit transcendental functions; expert counts at ties
    return {"rel": 1e-5}
