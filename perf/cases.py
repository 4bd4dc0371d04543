"""Timed workloads of the FP8 linear path, through the module API a training program uses.

Sizes are the text layer of the model this path serves (hidden 2560, intermediate 10240, query
2048, key and value 1024 each), with the row counts its training meets: one decoder branch of 64
tokens, a branch batch of 512, micro-batches of 2,000 to 8,192 packed tokens and a packed
encoder batch of 18,494. Every recipe of the converted modules is covered, forward and
backward (the recipes are the module attribute a user chooses in ``enable_float8`` and
``enable_te_linear`` / ``enable_fused_mlp``).

A training case returns the layer's output and every gradient a step needs; a forward case
is what a frozen or checkpointed region runs under ``no_grad``. ``fresh``: the pass is the
first after an optimizer step, so the module quantizes its weights again; otherwise a later
micro-batch of the step, on the cached FP8 weights (the torchao recipes and the functional MLP
quantize them on every call by design).
"""

import math
import types

import torch
from torch import nn
from torch.nn import functional as F

from bongard_amd import float8_training, fused_mlp, linear, state_kv, te_linear

HIDDEN, INTER = 2560, 10240
EPS = 1e-6
DELAYED_WARM_STEPS = 20  # fills the amax history (16) with steady values

# (in, out) of the text layer's projections
PROJECTIONS = ((2560, 2048), (2560, 1024), (2048, 2560), (2560, 10240), (10240, 2560), (2560, 4096))
TORCHAO_RECIPES = ("tensorwise", "rowwise", "rowwise_with_gw_hp")
TE_RECIPES = ("fp8", "fp8_delayed", "mxfp8", "nvfp4")


def listed():
    return [
        # One decoder branch of 64 tokens through a query projection whose FP8 weight is
        # cached: the smallest call, launches and host time count most.
        dict(name="branch_query_fwd", kind="te_linear", recipe="fp8", rows=64, k=2560, n=2048,
             train=False),
        # A query projection trained on a short batch (torchao tensorwise; 500 rows are not a
        # multiple of the 16 the weight-gradient GEMM wants).
        dict(name="query_tensorwise", kind="linear", recipe="tensorwise", rows=500, k=2560,
             n=2048, train=True),
        # A gate projection trained with one scale per row (torchao rowwise).
        dict(name="gate_rowwise", kind="linear", recipe="rowwise", rows=4096, k=2560, n=10240,
             train=True),
        # A fused query/key/value projection trained with row scales and a bf16 weight
        # gradient, on a ragged batch.
        dict(name="qkv_rowwise_gw_hp", kind="linear", recipe="rowwise_with_gw_hp", rows=2001,
             k=2560, n=4096, train=True),
        # A query projection of the branch batch trained in MXFP8 blocks.
        dict(name="query_mxfp8", kind="te_linear", recipe="mxfp8", rows=512, k=2560, n=2048,
             train=True),
        # The decoder branches' MLP forward on cached weights.
        dict(name="branch_mlp_fwd", kind="te_mlp", recipe="fp8", rows=512, hidden=HIDDEN,
             inter=INTER, train=False),
        # The MLP forward with its weights quantized in the call (a first micro-batch).
        dict(name="mlp_first_fwd", kind="geglu_mlp", recipe="fp8", rows=4096, hidden=HIDDEN,
             inter=INTER, train=False),
        # Norm and MLP trained as one module on a ragged micro-batch (current scaling).
        dict(name="fused_mlp_fp8", kind="fused_mlp", recipe="fp8", rows=3001, hidden=HIDDEN,
             inter=INTER, train=True),
        # The MLP's training step at the largest micro-batch, delayed scaling, the weights new
        # from the optimizer.
        dict(name="mlp_fp8_delayed", kind="te_mlp", recipe="fp8_delayed", rows=8192,
             hidden=HIDDEN, inter=INTER, train=True, fresh=True),
        # The MLP's training step in MXFP8 blocks, the weights new from the optimizer.
        dict(name="mlp_mxfp8", kind="te_mlp", recipe="mxfp8", rows=4096, hidden=HIDDEN,
             inter=INTER, train=True, fresh=True),
        # Norm and MLP trained in NVFP4 blocks.
        dict(name="fused_mlp_nvfp4", kind="fused_mlp", recipe="nvfp4", rows=2048, hidden=HIDDEN,
             inter=INTER, train=True),
        # The decoder's key/value projection of the whole packed encoder batch, trained.
        dict(name="state_kv_fp8", kind="state_kv", recipe="fp8", rows=18494, hidden=HIDDEN,
             kv=1024, train=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "te_linear", "te_linear", "te_mlp", "te_mlp",
                       "fused_mlp", "geglu_mlp", "state_kv"))
    if kind in ("linear", "te_linear"):
        if rng.random() < 0.6:
            k, n = rng.choice(PROJECTIONS)
        else:  # other layers: widths in steps of 32
            k, n = 32 * _log_int(rng, 8, 128), 32 * _log_int(rng, 8, 128)
        recipe = rng.choice(TORCHAO_RECIPES if kind == "linear" else TE_RECIPES)
        return dict(kind=kind, recipe=recipe, rows=_log_int(rng, 33, 8192), k=k, n=n,
                    train=kind == "linear" or rng.random() < 0.75, fresh=rng.random() < 0.5)
    if kind == "state_kv":
        return dict(kind=kind, recipe="fp8", rows=_log_int(rng, 512, 18494),
                    hidden=rng.choice((1024, 1536, 2048, 2560)), kv=rng.choice((512, 1024)),
                    train=True)
    hidden = rng.choice((640, 1024, 1536, 2048, 2560))
    recipe = "fp8" if kind == "geglu_mlp" else rng.choice(TE_RECIPES)
    # NVFP4 multiplies on the half-rate bf16 MFMA: half the rows keep the cost below the
    # largest listed case
    most = 4096 if recipe == "nvfp4" else 8192
    train = kind == "fused_mlp" or (kind == "te_mlp" and rng.random() < 0.75)
    return dict(kind=kind, recipe=recipe, rows=_log_int(rng, 64, most), hidden=hidden,
                inter=4 * hidden, train=train, fresh=rng.random() < 0.5)


# ---- inputs --------------------------------------------------------------------------------
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def __call__(self, *shape, std=1.0):
        t = torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32)
        return (t * std).to(torch.bfloat16)

    def activations(self, rows, cols):
        """N(0, 1) with 8 outlier columns, as hidden states have."""
        t = torch.randn(rows, cols, generator=self.g, device="cuda", dtype=torch.float32)
        t[:, torch.randperm(cols, generator=self.g, device="cuda")[:8]] *= 20.0
        return t.to(torch.bfloat16)


def _inputs(case, seed):
    r = _Rand(seed)
    kind = case["kind"]
    if kind in ("linear", "te_linear"):
        t = dict(x=r.activations(case["rows"], case["k"]), w=r(case["n"], case["k"], std=0.02))
        if case["train"]:
            t["dy"] = r(case["rows"], case["n"], std=1e-3)
        return t
    if kind == "state_kv":
        rows, kv = case["rows"], case["kv"]
        return dict(x=r.activations(rows, case["hidden"]), wk=r(kv, case["hidden"], std=0.02),
                    wv=r(kv, case["hidden"], std=0.02), dk=r(rows, kv, std=1e-3),
                    dv=r(rows, kv, std=1e-3))
    rows, hidden, inter = case["rows"], case["hidden"], case["inter"]
    x = r(rows, hidden) if kind != "fused_mlp" else r.activations(rows, hidden)
    t = dict(x=x, w_gate=r(inter, hidden, std=0.02), w_up=r(inter, hidden, std=0.02),
             w_down=r(hidden, inter, std=0.014))
    if kind == "fused_mlp":
        t["gamma"] = r(hidden, std=0.1)
    if case["train"]:
        t["dy"] = r(rows, hidden, std=1e-3)
    return t


def _linear_of(w):
    m = nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta")
    m.weight = nn.Parameter(w)
    return m


class _HfMlp(nn.Module):
    """The attributes of the model's gated MLP that the conversions read."""

    def __init__(self, t):
        super().__init__()
        self.config = types.SimpleNamespace(hidden_activation="gelu_pytorch_tanh")
        self.intermediate_size, self.hidden_size = t["w_gate"].shape
        self.gate_proj, self.up_proj = _linear_of(t["w_gate"]), _linear_of(t["w_up"])
        self.down_proj = _linear_of(t["w_down"])
        self.dropout = nn.Dropout(0.0)


def _converted_linear(w, recipe):
    """enable_float8 on a model whose one text layer holds the projection."""
    layer = nn.Module()
    layer.proj = _linear_of(w)
    model = nn.Module()
    model.backbone = nn.Module()
    model.backbone.decoder = nn.Module()
    model.backbone.decoder.layers = nn.ModuleList([layer])
    model.device = w.device
    float8_training.enable_float8(model, recipe)
    return layer.proj


def prepare(case, seed):
    t = _inputs(case, seed)
    kind, recipe, train = case["kind"], case["recipe"], case["train"]
    if kind == "geglu_mlp":
        return dict(case=case, x=t["x"], w_gu=torch.cat([t["w_gate"], t["w_up"]]),
                    w_down=t["w_down"])
    x = t["x"].requires_grad_(train)
    if kind == "state_kv":
        att = types.SimpleNamespace(
            k_proj=te_linear.TELinear([_linear_of(t["wk"])], recipe).train(),
            v_proj=te_linear.TELinear([_linear_of(t["wv"])], recipe).train(),
            k_norm=nn.Identity(),  # the model's own norm, not part of this path
            head_dim=256)
        heads = lambda d: d.view(1, case["rows"], -1, 256).transpose(1, 2)  # noqa: E731
        return dict(case=case, att=att, x=x, params=[att.k_proj.weight, att.v_proj.weight],
                    dys=[heads(t["dk"]), heads(t["dv"])])
    if kind == "linear":
        module = _converted_linear(t["w"], recipe)
        params = [module.weight]
    elif kind == "te_linear":
        module = te_linear.TELinear([_linear_of(t["w"])], recipe)
        params = [module.weight]
    elif kind == "te_mlp":
        module = te_linear.TEMLP(_HfMlp(t), recipe)
        params = [module.gate_up.weight, module.down.weight]
    else:
        norm = types.SimpleNamespace(weight=nn.Parameter(t["gamma"]), eps=EPS,
                                     eval=lambda: types.SimpleNamespace())
        module = fused_mlp.FusedMLP(_HfMlp(t), norm, recipe)
        params = [module.layer_norm_weight, module.fc1_weight, module.fc2_weight]
    module.train()
    state = dict(case=case, module=module, x=x, params=params, dys=[t["dy"]] if train else None)
    if recipe == "fp8_delayed":  # a running training job's amax histories
        for _ in range(DELAYED_WARM_STEPS):
            _optimizer_step(params)
            run(state)
    return state


def _optimizer_step(params):
    """The weights count as changed in place (their values stay)."""
    torch.autograd.graph.increment_version(params)


def run(state):
    case = state["case"]
    if case.get("fresh") and case["kind"] in ("te_linear", "te_mlp", "fused_mlp"):
        _optimizer_step(state["params"])
    if case["kind"] == "geglu_mlp":
        with torch.no_grad():
            return linear.Fp8GegluMlpFunction.apply(state["x"], state["w_gu"], state["w_down"],
                                                    None, None, case["inter"], False)
    if not case["train"]:
        with torch.no_grad():
            return state["module"](state["x"])
    if case["kind"] == "state_kv":
        ys = list(state_kv.project_state_kv(state["att"], state["x"][None]))
    else:
        ys = [state["module"](state["x"])]
    grads = torch.autograd.grad(ys, [state["x"], *state["params"]], state["dys"])
    return dict(y=[y.detach() for y in ys], grads=list(grads))


# ---- the work a pass cannot do without -------------------------------------------------------
def work(case):
    """Each input read once, each output written once (bf16); the multiplications' flops."""
    rows, train = case["rows"], case["train"]
    if case["kind"] in ("linear", "te_linear"):
        weight = case["k"] * case["n"]
        ins, outs = rows * case["k"], rows * case["n"]
    elif case["kind"] == "state_kv":
        weight = 2 * case["kv"] * case["hidden"]
        ins, outs = rows * case["hidden"], 2 * rows * case["kv"]
    else:
        weight = 3 * case["hidden"] * case["inter"]
        ins = outs = rows * case["hidden"]
    values = ins + weight + outs
    # the step also reads dy and writes dx and every weight gradient
    return {"bytes": 2 * values * (2 if train else 1), "flops": 2 * rows * weight * (3 if train else 1)}


def tolerance(case):
    """About four times what the path is off the 64-bit results (measured over the listed
    and drawn cases). One multiplication: the bf16 rounding of its output (0.0017 in norm,
    half a bf16 step at most); the key/value input gradient is a bf16 sum of two rounded
    products (0.0024, 0.015). The gated MLP quantizes H and dGU between its multiplications:
    where two correct sums differ by a bf16 step, a value can move by a whole fp8 step
    (0.0021 to 0.0037; 0.03 to 0.86). In NVFP4 such a step of a tensor's largest value
    moves the scale of all its blocks, and every fp4 rounding with it (0.0017 to 0.067)."""
    if case["kind"] in ("linear", "te_linear"):
        return {"rel": 7e-3, "max": 1.6e-2}
    if case["kind"] == "state_kv":
        return {"rel": 1e-2, "max": 6e-2}
    return {"rel": 3e-2 if case["recipe"] == "nvfp4" else 1.5e-2, "max": 0.9}


# ---- the same results in 64 bits ---------------------------------------------------------------
FP8 = {"e4m3": (torch.float8_e4m3fn, 448.0), "e5m2": (torch.float8_e5m2, 57344.0)}


def _scale(amax, top, pow2=False):
    s = (top / amax.double().clamp(min=1e-12)).float()
    return torch.exp2(torch.floor(torch.log2(s))) if pow2 else s


def _cast(x, scale, fmt):
    """The values of the fp8 copy of x under ``scale``, in 64 bits."""
    dt, top = FP8[fmt]
    return (x.float() * scale).clamp(-top, top).to(dt).double() / scale.double()


def _tensorwise(x, fmt, pow2=False):
    return _cast(x, _scale(x.abs().amax(), FP8[fmt][1], pow2), fmt)


def _axiswise(x, dim):
    return _cast(x, _scale(x.abs().amax(dim, keepdim=True), 448.0, True), "e4m3")


def _mx(x):
    """Blocks of 32 along the last dimension, e4m3 values, power-of-two scales."""
    b = x.reshape(x.shape[0], -1, 32)
    val = b.abs().amax(-1, keepdim=True).float() * torch.tensor(1.0 / 448.0, device=x.device)
    bits = val.view(torch.int32)
    e = (bits >> 23) + ((bits & 0x7FFFFF) > 0).int()
    e = torch.where(((bits >> 23) == 0) & ((bits & 0x7FFFFF) <= 0x400000), 0, e)
    return _cast(b, torch.exp2((127 - e).double()).float(), "e4m3").reshape(x.shape)


def _nvfp4(x, amax):
    """Blocks of 16 along the last dimension: e2m1 values, e4m3 scales, one tensor scale."""
    s_enc = _scale(amax, 448.0 * 6.0)
    b = x.float().reshape(x.shape[0], -1, 16)
    v = (b.abs().amax(-1, keepdim=True) / 6.0) * s_enc
    s = v.clamp(max=448.0).to(torch.float8_e4m3fn).float()
    p = b * torch.where(s == 0, 0.0, s_enc / s)
    a = p.abs()
    grid = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=x.device)
    code = ((a > 0.25).int() + (a >= 0.75).int() + (a > 1.25).int() + (a >= 1.75).int()
            + (a > 2.5).int() + (a >= 3.5).int() + (a > 5.0).int())
    q = torch.copysign(grid[code.long()], p.double()) * s.double()
    return q.reshape(x.shape) * s_enc.reciprocal().double()


class _Exact:
    """One multiplication y = x w^T of a recipe, forward and backward, in 64 bits."""

    def __init__(self, recipe):
        self.recipe = {"fp8": "tensorwise", "fp8_delayed": "tensorwise"}.get(recipe, recipe)

    def _q(self, t, axis, grad=False):
        """``t`` as the multiplication that sums over ``axis`` reads it."""
        if self.recipe == "tensorwise":
            return _tensorwise(t, "e5m2" if grad else "e4m3")
        if self.recipe in TORCHAO_RECIPES:
            return _axiswise(t, axis)
        s = t if axis == 1 else t.t().contiguous()
        short = (-s.shape[1]) % 32  # rows are padded with zeros to a multiple of 32
        s = F.pad(s, (0, short))
        q = _mx(s) if self.recipe == "mxfp8" else _nvfp4(s, t.abs().amax())
        q = q[:, :q.shape[1] - short]
        return q if axis == 1 else q.t()

    def forward(self, x, w):
        return self._q(x, 1) @ self._q(w, 1).t()

    def backward(self, dy, x, w):
        d = self._q(dy, 1, True)
        if self.recipe == "rowwise_with_gw_hp":
            return d @ _tensorwise(w, "e4m3", True), dy.double().t() @ x.double()
        return d @ self._q(w, 0), self._q(dy, 0, True).t() @ self._q(x, 0)


def _gelu(g):
    return F.gelu(g.double(), approximate="tanh").to(torch.bfloat16)


def _gelu_grad(g):
    x = g.double()
    c = math.sqrt(2.0 / math.pi)
    th = torch.tanh(c * (x + 0.044715 * x ** 3))
    return 0.5 * (1 + th) + 0.5 * x * (1 - th * th) * c * (1 + 3 * 0.044715 * x * x)


def exact(case, seed):
    t = _inputs(case, seed)
    mm = _Exact(case["recipe"])
    b16 = torch.bfloat16
    kind, train = case["kind"], case["train"]
    if kind in ("linear", "te_linear"):
        y = mm.forward(t["x"], t["w"])
        return dict(y=[y], grads=list(mm.backward(t["dy"], t["x"], t["w"]))) if train else y
    if kind == "state_kv":
        ys, dx, dws = [], 0, []
        for w, dy in ((t["wk"], t["dk"]), (t["wv"], t["dv"])):
            y = mm.forward(t["x"], w)
            ys.append(y.view(1, case["rows"], -1, 256).transpose(1, 2))
            part, dw = mm.backward(dy, t["x"], w)
            dx = dx + part
            dws.append(dw)
        return dict(y=ys, grads=[dx, *dws])
    x = t["x"]
    if kind == "fused_mlp":
        xd, gain = x.double(), 1.0 + t["gamma"].double()
        r = torch.rsqrt(xd.square().mean(-1, keepdim=True) + EPS)
        x = (xd * r * gain).to(b16)
    w_gu = torch.cat([t["w_gate"], t["w_up"]])
    g, u = mm.forward(x, w_gu).to(b16).chunk(2, 1)
    act = _gelu(g)
    h = act * u
    y = mm.forward(h, t["w_down"])
    if not train:
        return y
    dh, dw_down = mm.backward(t["dy"], h, t["w_down"])
    dh = dh.to(b16)
    dg = ((dh * u).double() * _gelu_grad(g)).to(b16)
    dx, dw_gu = mm.backward(torch.cat([dg, dh * act], 1), x, w_gu)
    if kind != "fused_mlp":
        return dict(y=[y], grads=[dx, dw_gu, dw_down])
    dn = dx.to(b16).double()
    dgamma = (dn * xd * r).sum(0)
    a = dn * gain
    dx = a * r - xd * r ** 3 * (a * xd).mean(-1, keepdim=True)
    return dict(y=[y], grads=[dx, dgamma, dw_gu, dw_down])
