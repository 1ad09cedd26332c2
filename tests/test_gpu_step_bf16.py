"""mtl_decode_step_batched_bf16 on a bfloat16 model (weights, activations and conv
history in bf16; fp32 residual, SSM state and partial sums): MambaLM.step
(model.py:343-353) at 1-32 rows against the float64 oracle and the per-op
step, and captured; the models and states that keep it, and a long fp32
prompt's one call, on the per-op path; models copied and saved after calls."""
import copy
import io

import numpy as np
import pytest
import torch

import _golden as G
from _util import assert_rel
from mamba_lite import ops
from mamba_lite.cuda_graph import GraphedStepper
from mamba_lite.model import MambaCache, MambaConfig, MambaLM
from oracle import mixer as om

pytestmark = pytest.mark.gpu


# d_model, d_inner / d_model, batch, d_conv, bias: fp32-ineligible widths too (d_inner 1280 and 1792, not a multiple
# of 512; wavefronts with unequal stage counts), one row, fold edge (16 / 17 rows), 32 rows on 32-row tiles (d 2048)
BF16_SHAPES = [(512, 2, 1, 4, False), (640, 2, 3, 4, True), (896, 2, 16, 3, False), (512, 3, 17, 2, True),
               (768, 2, 32, 4, False), (2048, 2, 5, 4, False), (2048, 2, 32, 4, False)]


@pytest.mark.parametrize("dm,expand,b,d_conv,bias", BF16_SHAPES)
def test_bf16_one_call_step_matches_oracle_and_per_op(dm, expand, b, d_conv, bias, monkeypatch):
    """A bfloat16 model's one-call step against the float64 oracle on the same
    bf16-rounded weights and caches (1e-2, the bf16 gate), and no further
    from it than the per-op step; graph replays equal eager."""
    import mamba_lite.model as mm
    torch.manual_seed(dm + b)
    cfg = MambaConfig(d_model=dm, n_layer=2, vocab_size=200, d_state=16, d_conv=d_conv, expand=expand, bias=bias)
    with torch.device("cuda"):
        m = MambaLM(cfg).eval()
    with torch.no_grad():
        for blk in m.layers:
            blk.mixer.dt_proj.bias.uniform_(-6.0, -2.0)
    m = m.to(torch.bfloat16)
    cache = MambaCache.allocate(cfg, b, "cuda", torch.bfloat16)
    for lc in cache.layers:
        lc.conv_state.normal_(0, 0.6)
        lc.ssm_state.normal_(0, 0.1)
    clone = lambda: MambaCache([type(lc)(lc.conv_state.clone(), lc.ssm_state.clone()) for lc in cache.layers])
    ids = torch.randint(0, cfg.vocab_size, (b, 1), device="cuda")
    calls = []
    real = ops.decode_step_batched
    monkeypatch.setattr(ops, "decode_step_batched", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    with torch.no_grad():
        one, per_op = clone(), clone()
        got = [m.step(ids, one) for _ in range(2)]
        assert len(calls) == 2 and got[0].dtype == torch.bfloat16
        monkeypatch.setattr(mm, "BATCHED_STEP_NATIVE", False)
        old = [m.step(ids, per_op) for _ in range(2)]
        monkeypatch.setattr(mm, "BATCHED_STEP_NATIVE", True)
        W = G.oracle_lm_dict({k: v.double().cpu().numpy() for k, v in m.state_dict().items()}, cfg.n_layer)
        f64 = lambda t: t.double().cpu().numpy()
        oc = [(f64(lc.conv_state), f64(lc.ssm_state)) for lc in cache.layers]
        for g, o in zip(got, old):
            ref = om.lm_step(W, ids.cpu().numpy(), oc, dtype=np.float64)
            assert_rel(f64(g), ref, 1e-2, "one call vs oracle")
            e_g, e_o = np.linalg.norm(f64(g) - ref), np.linalg.norm(f64(o) - ref)
            assert e_g <= 1.02 * e_o, (e_g, e_o)      # measured 0.989 to 1.004
        for a_, b_ in zip(one.layers, per_op.layers):
            assert_rel(f64(a_.ssm_state), f64(b_.ssm_state), 1e-2, "ssm_state")
            assert_rel(f64(a_.conv_state), f64(b_.conv_state), 2e-2, "conv_state")
        st = GraphedStepper(m, clone(), b, "cuda")
        st.capture()
        for g in got:
            assert torch.equal(st.replay(ids), g)


@pytest.mark.parametrize("dtype,b,l", [(torch.bfloat16, 3, 1), (torch.float32, 2, 1024)])
def test_a_hooked_stack_keeps_the_per_op_path(dtype, b, l):
    """The bf16 step and an fp32 prompt of more than 2^21 token-channels run op by op where a module has a hook or
    autocast is on, and in one call otherwise."""
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=640, n_layer=2, vocab_size=300)).eval().to(dtype)
    cache = MambaCache.allocate(lm.cfg, b, torch.device("cuda"), dtype)
    ids, x = torch.zeros(b, l, dtype=torch.long, device="cuda"), torch.zeros(b, 640, dtype=dtype, device="cuda")

    def one_call():
        with torch.no_grad():
            return (lm._batched_step_layers(x, cache) if l == 1 else lm._prefill_native(ids, None, None)) is not None
    assert one_call()
    handle = lm.layers[1].mixer.out_proj.register_forward_hook(lambda *_: None)
    assert not one_call()
    handle.remove()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not one_call()
    assert one_call()


def test_a_norm_f_cast_between_steps():
    """norm_f kept in float32 on a bf16 model, before the first step or after one: the per-op path, as if it had been
    so from the start."""
    torch.manual_seed(5)
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=640, n_layer=2, vocab_size=300)).eval().to(torch.bfloat16)
    ids = torch.zeros(3, 1, dtype=torch.long, device="cuda")

    def step():
        with torch.no_grad():
            return lm.step(ids, MambaCache.allocate(lm.cfg, 3, "cuda", torch.bfloat16)).double()

    before = step()
    lm.norm_f.float()
    after = step()
    lm._batched_tmpl = None
    assert torch.equal(after, step())
    assert float((after - before).norm() / before.norm()) < 1e-2


@pytest.mark.parametrize("dtype,b,l", [(torch.bfloat16, 3, 1), (torch.float32, 2, 1024), (torch.float32, 1, 1),
                                       (torch.float32, 1, 20)])
def test_a_model_is_copied_and_saved_after_its_calls(dtype, b, l):
    """copy.deepcopy and torch.save of a model that has stepped or prefilled: its call plans stay behind, and the copy
    gives the same bits from its own weights."""
    torch.manual_seed(6)
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=640, n_layer=2, vocab_size=300)).eval().to(dtype)
        ids = torch.randint(0, 300, (b, l))

    def logits(m):
        with torch.no_grad():
            return m.step(ids, MambaCache.allocate(m.cfg, b, "cuda", dtype)) if l == 1 else m.prefill(ids)[0]

    want = logits(lm)
    twin = copy.deepcopy(lm)
    buf = io.BytesIO()
    torch.save(lm, buf)
    buf.seek(0)
    with torch.no_grad():
        lm.layers[0].mixer.out_proj.weight.zero_()
    assert torch.equal(logits(twin), want)
    assert torch.equal(logits(torch.load(buf, weights_only=False)), want)
    assert not torch.equal(logits(lm), want)


@pytest.mark.parametrize("l", [1, 40])
def test_a_model_made_in_inference_mode(l):
    """Its parameters are inference tensors, which have no version counter: it steps and prefills, and a
    weight changed in place counts."""
    torch.manual_seed(8)
    with torch.inference_mode(), torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=640, n_layer=2, vocab_size=300)).eval().to(torch.bfloat16)
    ids = torch.zeros(3, l, dtype=torch.long, device="cuda")
    with torch.inference_mode():
        cache = MambaCache.allocate(lm.cfg, 3, "cuda", torch.bfloat16)
        got = lm.step(ids, cache) if l == 1 else lm.prefill(ids)[0]
        assert bool(torch.isfinite(got).all())
        lm.layers[0].mixer.x_proj.weight.mul_(3)
        cache = MambaCache.allocate(lm.cfg, 3, "cuda", torch.bfloat16)
        assert not torch.equal(lm.step(ids, cache) if l == 1 else lm.prefill(ids)[0], got)


def test_a_step_the_sizes_rule_out_walks_no_modules(monkeypatch):
    """A bf16 step of a model too narrow for the one call is bound by the host: its modules are not looked through."""
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=256, n_layer=2, vocab_size=300)).eval().to(torch.bfloat16)
    walked = []
    monkeypatch.setattr(MambaLM, "_plain_stack", lambda self: walked.append(1))
    with torch.no_grad():
        lm.step(torch.zeros(3, 1, dtype=torch.long, device="cuda"),
                MambaCache.allocate(lm.cfg, 3, "cuda", torch.bfloat16))
    assert not walked


class _Negating(torch.nn.Linear):
    def forward(self, x):
        return -super().forward(x)


class _Adapter(torch.nn.Module):
    """A projection inside another module, which shows its weight and bias."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    weight = property(lambda self: self.inner.weight)
    bias = property(lambda self: self.inner.bias)

    def forward(self, x):
        return -self.inner(x)


class _Negated(torch.nn.Module):
    def forward(self, w):
        return -w


@pytest.mark.parametrize("kind,dtype,b,l", [("subclass", torch.bfloat16, 3, 1), ("subclass", torch.float32, 2, 1024),
                                            ("adapter", torch.float32, 2, 1024),
                                            ("parametrization", torch.float32, 2, 1024)])
def test_a_replaced_projection_is_called(kind, dtype, b, l):
    """An out_proj of another class is called as a module, not read past, by the bf16 step and by an fp32 prompt of
    more than 2^21 token-channels: here each negates what nn.Linear gives."""
    torch.manual_seed(3)
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=640, n_layer=1, vocab_size=300)).eval().to(dtype)
        ids = torch.randint(0, 300, (b, l))
    mx = lm.layers[0].mixer

    def logits():
        with torch.no_grad():
            cache = MambaCache.allocate(lm.cfg, b, "cuda", dtype)
            return (lm.step(ids, cache) if l == 1 else lm.prefill(ids)[0]).double()

    with torch.no_grad():
        mx.out_proj.weight.mul_(-50)            # the block outweighs the embedding it is added to
        want = logits()
        mx.out_proj.weight.neg_()
    if kind == "subclass":
        mx.out_proj.__class__ = _Negating
    elif kind == "adapter":
        mx.out_proj = _Adapter(mx.out_proj)
    else:
        torch.nn.utils.parametrize.register_parametrization(mx.out_proj, "weight", _Negated())
    assert float((logits() - want).norm() / want.norm()) < (1e-2 if dtype == torch.bfloat16 else 1e-5)


class _Halved(torch.Tensor):
    """A weight whose values are half of those it holds, as a quantized weight's are not the ones in memory."""

    @staticmethod
    def __new__(cls, held):
        return torch.Tensor._make_wrapper_subclass(cls, held.shape, strides=held.stride(), dtype=held.dtype,
                                                   device=held.device)

    def __init__(self, held):
        self.held = held

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        real = lambda t: t.held * 0.5 if isinstance(t, cls) else t
        if func is torch.ops.aten.detach.default:
            return cls(args[0].held)
        return func(*torch.utils._pytree.tree_map(real, args), **(kwargs or {}))


@pytest.mark.parametrize("dtype,b,l", [(torch.bfloat16, 3, 1), (torch.float32, 2, 1024), (torch.bfloat16, 2, 40)])
def test_a_subclass_weight_is_read_through_torch(dtype, b, l):
    """An out_proj weight (a bf16 prompt: dt_proj's bias) of a tensor subclass keeps torch's product, or float copy, of
    it: the bf16 step, an fp32 prompt of more than 2^21 token-channels, the bf16 scan's parameters."""
    torch.manual_seed(3)
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=640, n_layer=1, vocab_size=300)).eval().to(dtype)
        ids = torch.randint(0, 300, (b, l))
    mx = lm.layers[0].mixer
    mod, name = (mx.dt_proj, "bias") if l == 40 else (mx.out_proj, "weight")

    def logits():
        with torch.no_grad():
            cache = MambaCache.allocate(lm.cfg, b, "cuda", dtype)
            return (lm.step(ids, cache) if l == 1 else lm.prefill(ids)[0]).double()

    with torch.no_grad():
        mx.out_proj.weight.mul_(50)
        mx.dt_proj.bias.normal_(0, 4)
        held = getattr(mod, name).detach().clone()
        setattr(mod, name, torch.nn.Parameter(held * 0.5))
        want = logits()
        setattr(mod, name, torch.nn.Parameter(_Halved(held), requires_grad=False))
        assert type(getattr(mod, name)) is _Halved
    assert float((logits() - want).norm() / want.norm()) < (1e-2 if dtype == torch.bfloat16 else 1e-5)
