"""Scans that run in parallel segments (mtl_selective_scan_fwd_ws) against the
step-by-step kernel on the same inputs (segment boundaries, remainders,
layouts, state counts, h0, types, the optional operands, final states over the
initial ones, zero and infinite states) and the float64 oracle; bf16
parameters against their float copies."""
import numpy as np
import pytest
import torch

from mamba_lite import _lib, ops
from mamba_lite.model import MambaCache, MambaConfig, MambaLM
from oracle import mixer as om

pytestmark = pytest.mark.gpu


def _case(b, D, L, N, dtype, cm, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s, k=1.0: (k * torch.randn(*s, device="cuda", generator=g)).to(dtype)
    lay = (lambda t: t) if cm else (lambda t: t.transpose(1, 2).contiguous().transpose(1, 2))
    return dict(u=lay(r(b, D, L)), delta=lay(r(b, D, L, k=0.5)), z=lay(r(b, D, L)), B=r(b, N, L), C=r(b, N, L),
                A=-torch.arange(1, N + 1, device="cuda", dtype=torch.float32).repeat(D, 1).contiguous(),
                D=torch.ones(D, device="cuda"), bias=-2 - 3 * torch.rand(D, device="cuda", generator=g),
                h0=torch.randn(b, D, N, device="cuda", generator=g))


# b, D, L, N: the smallest segmented length, one step past whole segments, a last segment of 1 step, tail channels,
# the fewest and most workgroups of the range, 1-32 states
SHAPES = [(1, 3072, 320, 16), (3, 1536, 333, 16), (1, 4096, 1025, 16), (2, 4090, 385, 5), (3, 5000, 500, 1),
          (2, 2048, 640, 32), (1, 3080, 2000, 8)]


@pytest.mark.parametrize("b,D,L,N", SHAPES)
@pytest.mark.parametrize("dtype,cm", [(torch.float32, True), (torch.float32, False), (torch.bfloat16, False)])
def test_segments_match_the_sequential_scan(b, D, L, N, dtype, cm):
    assert _lib.load().mtl_selective_scan_ws_bytes(b, D, N, L) > 0
    c = _case(b, D, L, N, dtype, cm)
    # fp32: the decay over a segment is exp(A sum dt) for a product of exps, and the carried state is rounded once more
    # per segment: some 2^-23; bf16 y: one rounding of the output, 2^-9
    tol = 1e-6 if dtype == torch.float32 else 2.0 ** -8
    rel = lambda a, r: float((a.double() - r.double()).norm() / r.double().norm())
    for kw in (dict(z=c["z"], h0=c["h0"], delta_bias=c["bias"], D=c["D"]), dict(delta_bias=c["bias"]),
               dict(z=c["z"], delta_softplus=False, delta_bias=None)):
        d = c["delta"] if kw.get("delta_softplus", True) else 0.01 * c["delta"].abs()
        y, h = ops.selective_scan(c["u"], d, c["A"], c["B"], c["C"], **kw)
        yr, hr = ops.selective_scan(c["u"], d, c["A"], c["B"], c["C"], algo="tiled", **kw)
        assert rel(y, yr) < tol and rel(h, hr) < 1e-6


@pytest.mark.parametrize("b,D,L,N", [(1, 3072, 320, 16), (2, 4090, 385, 5)])
@pytest.mark.parametrize("cm", [True, False])
def test_segments_against_float64(b, D, L, N, cm):
    """fp32 with h0, and with a last segment of one step: no further from the float64 oracle than the
    step-by-step kernel (measured 0.88 to 0.97 of its 1.0e-7 for y and 1.5e-7 for the states, 2-norm)."""
    c = _case(b, D, L, N, torch.float32, cm)
    f64 = lambda t: t.double().cpu().numpy()
    ref = om.selective_scan_bnl(*(f64(c[k]) for k in ("u", "delta", "A", "B", "C", "D", "z", "bias", "h0")),
                                dtype=np.float64)
    def errors(algo):
        got = ops.selective_scan(c["u"], c["delta"], c["A"], c["B"], c["C"], D=c["D"], z=c["z"],
                                 delta_bias=c["bias"], h0=c["h0"], algo=algo)
        return [np.linalg.norm(f64(g) - r) / np.linalg.norm(r) for g, r in zip(got, ref)]

    for seg, step in zip(errors("auto"), errors("tiled")):
        assert seg <= step < 3e-7, (seg, step)


@pytest.mark.parametrize("b,D,L,N", SHAPES)
@pytest.mark.parametrize("dtype,cm", [(torch.float32, True), (torch.bfloat16, False)])
def test_final_states_over_the_initial_ones(b, D, L, N, dtype, cm):
    """h_out may be h0: every segment starts from h0 while the last one writes h_out, so the bits have to be those of
    separate buffers."""
    c = _case(b, D, L, N, dtype, cm)
    run = lambda h0, **kw: ops.selective_scan(c["u"], c["delta"], c["A"], c["B"], c["C"], D=c["D"], z=c["z"],
                                              delta_bias=c["bias"], h0=h0, **kw)
    y, h = run(c["h0"])
    kept = c["h0"].clone()
    y2, h2 = run(kept, h_out=kept)
    assert h2 is kept and torch.equal(h, h2) and torch.equal(y, y2)


@pytest.mark.parametrize("d_model,b,l", [(768, 3, 333), (768, 7, 400), (2048, 1, 420), (768, 10, 700)])
def test_a_prompt_that_continues_its_cache_in_place(d_model, b, l):
    """MambaLM.prefill with out_cache = cache, in one call and op by op (10 x 700), at segmented sizes."""
    torch.manual_seed(b)
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=d_model, n_layer=2, vocab_size=300)).eval()
        ids = torch.randint(0, 300, (b, l))
    assert _lib.load().mtl_selective_scan_ws_bytes(b, 2 * d_model, 16, l) > 0
    cache = MambaCache.allocate(lm.cfg, b, "cuda", torch.float32)
    for lc in cache.layers:
        lc.conv_state.normal_(0, 0.6)
        lc.ssm_state.normal_()
    with torch.no_grad():
        logits, new = lm.prefill(ids, cache)
        logits2, got = lm.prefill(ids, cache, out_cache=cache)
    assert got is cache and torch.equal(logits, logits2)
    for p, q in zip(new.layers, cache.layers):
        assert torch.equal(p.ssm_state, q.ssm_state) and torch.equal(p.conv_state, q.conv_state)


@pytest.mark.parametrize("b,D,L,N", SHAPES)
@pytest.mark.parametrize("cm", [True, False])
def test_zero_and_infinite_states_as_step_by_step(b, D, L, N, cm):
    """The product of a segment's decays overflows (A > 0) or underflows (A = -16) where each step's is in range: a
    state that is zero until the last steps stays zero, an infinite one stays infinite."""
    c = _case(b, D, L, N, torch.float32, cm)
    zero = torch.zeros_like(c["u"])
    zero[..., -5:] = c["u"][..., -5:]
    h0 = c["h0"].clone()
    h0[:, ::2] = float("inf")
    h0[:, 1::4] = 0
    for A, u, start in ((2.0, zero, None), (2.0, zero, torch.zeros_like(h0)), (-16.0, c["u"], h0)):
        run = lambda **kw: ops.selective_scan(u, torch.full_like(c["delta"], 1.0 if A > 0 else 0.2),
                                              torch.full_like(c["A"], A), c["B"], c["C"], h0=start,
                                              delta_softplus=False, **kw)
        for got, ref in zip(run(), run(algo="tiled")):
            assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
            ok = torch.isfinite(ref)
            assert bool(ok.any()) and float((got[ok] - ref[ok]).norm()) <= 1e-6 * float(ref[ok].norm())


def test_outside_the_rule_nothing_changes():
    ws = _lib.load().mtl_selective_scan_ws_bytes
    assert ws(1, 1536, 16, 1024) == 0 and ws(32, 1536, 16, 1024) == 0 and ws(1, 4096, 16, 300) == 0


@pytest.mark.parametrize("b,D,L", [(1, 70, 5), (2, 256, 100), (1, 4096, 500), (8, 1536, 64)])
def test_bf16_parameters_equal_their_float_copies(b, D, L):
    """A bf16 model's scan and conv read its parameters as stored: the bits
    that float copies of them give, on every scan kernel (chunked, segmented,
    tiled) and with 4-channel and single-channel conv threads."""
    c = _case(b, D, L, 16, torch.bfloat16, False)
    A, Dv, bias = (-c["A"]).log().bfloat16(), c["D"].bfloat16(), c["bias"].bfloat16()
    for algo in ("auto", "tiled", "chunked"):
        kw = dict(z=c["z"], a_is_log=True, algo=algo)
        got = ops.selective_scan(c["u"], c["delta"], A, c["B"], c["C"], D=Dv, delta_bias=bias, bf16_params=True, **kw)
        ref = ops.selective_scan(c["u"], c["delta"], A.float(), c["B"], c["C"], D=Dv.float(),
                                 delta_bias=bias.float(), **kw)
        assert all(torch.equal(p, q) for p, q in zip(got, ref))
    for K in (1, 3, 4):
        w, wb = torch.randn(D, 1, K, device="cuda").bfloat16(), torch.randn(D, device="cuda").bfloat16()
        got = ops.causal_conv1d(c["u"], w, wb, bf16_params=True)
        ref = ops.causal_conv1d(c["u"], w.float(), wb.float())
        assert all(torch.equal(p, q) for p, q in zip(got, ref))
    with pytest.raises(ValueError):
        ops.selective_scan(c["u"], c["delta"], A, c["B"], c["C"])          # bf16 parameters only on request
