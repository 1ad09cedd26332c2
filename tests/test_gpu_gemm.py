"""mtl_linear_f32: the fp32 product on split f16 operands against the float64
product, at tile edges and remainders, and its handling of extreme rows."""
import ctypes
import math

import pytest
import torch
import torch.nn.functional as F

from mamba_lite import _lib, ops

pytestmark = pytest.mark.gpu

# M, N, K: below, at and past the 64, 128 and 256 tiles, K not a multiple of 16 or 32, one and several K stages
SHAPES = [(1, 1, 1), (63, 33, 15), (64, 64, 16), (65, 129, 33), (257, 96, 100), (100, 1000, 48), (999, 768, 1536),
          (1500, 2500, 130), (4100, 8200, 64), (16500, 1100, 96)]


def _inputs(M, N, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K, device="cuda", generator=g)
    w = torch.randn(N, K, device="cuda", generator=g) * 0.02
    b = torch.randn(N, device="cuda", generator=g)
    return x, w, b


def _err(got, x, w, b=None):
    ref = x.double() @ w.double().t()
    if b is not None:
        ref = ref + b.double()
    return float((got.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_product_matches_float64(M, N, K):
    x, w, b = _inputs(M, N, K)
    # operand parts: two roundings and the dropped lo.lo term, each under 2^-22 of a product; the fp32 sum of K
    # products rounds 3 K / 16 times, a random walk: under 2^-24 sqrt(3 K / 16) of the result
    tol = 3 * 2.0 ** -22 + 2.0 ** -24 * math.sqrt(3 * K / 16 + 4)
    assert _err(ops.linear_f32(x, w), x, w) < tol
    assert _err(ops.linear_f32(x, w, b), x, w, b) < tol


@pytest.mark.parametrize("K", [992, 1024, 1025, 2047, 2056, 4096, 4100])
def test_split_widths(K):
    """Either side of each width up to which the split holds a row in
    registers (1024, 2048, 4096; past it two passes), with a row whose last
    column is infinite; the bound of the products above."""
    x, w, _ = _inputs(130, 70, K)
    x[77, -1] = math.inf
    got, rows = ops.linear_f32(x, w), torch.arange(130, device="cuda") != 77
    assert torch.equal(got[77], torch.sign(w[:, -1]) * math.inf)
    tol = 3 * 2.0 ** -22 + 2.0 ** -24 * math.sqrt(3 * K / 16 + 4)
    assert _err(got[rows], x[rows], w) < tol


@pytest.mark.parametrize("M,N,K", [(1024, 2048, 4096), (4096, 3072, 768), (512, 4096, 2048)])
def test_error_not_above_the_fp32_product(M, N, K):
    x, w, _ = _inputs(M, N, K)
    assert _err(ops.linear_f32(x, w), x, w) <= _err(F.linear(x, w), x, w)


@pytest.mark.parametrize("M,N,K", [(999, 3072, 768), (600, 4096, 2500), (512, 2048, 4500), (1000, 8200, 1030)])
@pytest.mark.parametrize("power", [12, 17, 18, 20, 23, 30])
def test_spread_rows_keep_the_fp32_error(M, N, K, power):
    """One value 2^power times the rest of its row against a zero in the other operand: what is left of the row
    counts.  In every third row of x, and in every third row of W."""
    x, w, _ = _inputs(M, N, K)
    x[::3, 5] *= 2.0 ** power
    w[::3, 9] *= 2.0 ** power
    x[:, 9] = w[:, 5] = 0
    assert _err(ops.linear_f32(x, w), x, w) <= _err(F.linear(x, w), x, w)


@pytest.mark.parametrize("K", [32, 768, 2500, 4500])
def test_selecting_rows_are_exact(K):
    """A row of W (or x) that picks one column gives that column's bits, as an fp32 product does."""
    x, _, _ = _inputs(200, 1, K)
    x[::7] = 0
    pick = torch.randint(0, K, (300,), generator=torch.Generator().manual_seed(K)).cuda()
    w = F.one_hot(pick, K).float()
    assert torch.equal(ops.linear_f32(x, w), x[:, pick])
    assert torch.equal(ops.linear_f32(w, x), x[:, pick].t())


def test_split_output_and_strided_weight():
    x, w, b = _inputs(300, 192, 80)
    y0, y1 = ops.linear_f32(x, w, b, n_split=96)
    y = ops.linear_f32(x, w, b)
    assert torch.equal(torch.cat([y0, y1], 1), y)
    wide = torch.randn(192, 200, device="cuda")
    sub = wide[:, 3:83]                       # rows off a 16-byte boundary
    assert torch.equal(ops.linear_f32(x, sub, b), ops.linear_f32(x, sub.contiguous(), b))
    with pytest.raises(ValueError):
        ops.linear_f32(x, w, b, n_split=50)


@pytest.mark.parametrize("M,N,K", [(1, 40, 32), (65, 129, 33), (257, 96, 100), (100, 1000, 48), (1793, 2049, 32),
                                   (1000, 3001, 32), (4100, 8200, 32), (16500, 1100, 32)])
def test_nothing_is_written_outside_the_outputs(M, N, K):
    """y0 and y1 inside a larger filled buffer, 256 rows before and behind each and columns past N in every row
    (the 64 x 64 tiles, the 128 x 128 and the 256 x 128 ones): what lies around them stays."""
    x, w, b = _inputs(M, N, K)
    lib = _lib.load()
    for n0 in (N, 32):
        widths = [n0, N - n0] if n0 < N else [N]
        bufs = [torch.full((M + 512, n + 3), 7.25, device="cuda") for n in widths]
        ws = torch.empty(lib.mtl_linear_f32_ws_bytes(M, N, K), dtype=torch.uint8, device="cuda")
        a = _lib.LinearF32Args()
        a.x, a.W, a.bias, a.ws, a.ws_bytes = x.data_ptr(), w.data_ptr(), b.data_ptr(), ws.data_ptr(), ws.numel()
        a.ldx, a.ldw, a.M, a.N, a.K, a.n_split = K, K, M, N, K, n0
        a.y0, a.ldy0 = bufs[0][256:].data_ptr(), n0 + 3
        if n0 < N:
            a.y1, a.ldy1 = bufs[1][256:].data_ptr(), N - n0 + 3
        _lib.check(lib.mtl_linear_f32(ctypes.byref(a), torch.cuda.current_stream().cuda_stream), "linear_f32")
        y = ops.linear_f32(x, w, b)
        for buf, ref in zip(bufs, y.split(widths, 1)):
            assert torch.equal(buf[256:256 + M, :ref.shape[1]], ref)
            assert bool((buf[:256] == 7.25).all()) and bool((buf[256 + M:] == 7.25).all())
            assert bool((buf[:, ref.shape[1]:] == 7.25).all())


def test_rows_of_very_different_magnitude():
    """Each row's split is relative to its own largest value: rows 1e-30 to 1e30 keep their relative error, and
    rows whose values spread from 1 to 1e-12 are not split."""
    x, w, _ = _inputs(128, 96, 256)
    s = torch.logspace(-30, 30, 128, device="cuda")[:, None]
    a, b = ops.linear_f32(x * s, w).double() / s.double(), ops.linear_f32(x, w).double()
    assert float((a - b).norm() / b.norm()) < 4 * 2.0 ** -24 * math.sqrt(256)
    spread = x * torch.logspace(0, -12, 256, device="cuda")
    assert _err(ops.linear_f32(spread, w), spread, w) < 1e-6
    z = ops.linear_f32(torch.zeros(70, 64, device="cuda"), w[:, :64].contiguous())
    assert torch.equal(z, torch.zeros_like(z))


@pytest.mark.parametrize("M,N,K", [(70, 90, 40), (300, 500, 64), (1300, 12800, 32), (200, 300, 129),
                                   (130, 260, 96)])
def test_infinities_and_nan_as_in_fp32(M, N, K):
    x, w, b = _inputs(M, N, K)
    x[3, 5], x[17, 0], x[17, 2], x[-1, -1] = math.inf, math.inf, -math.inf, -math.inf
    x[40, 1] = math.nan
    w[7, 5], w[11, 3], w[-2, 0] = 0.0, math.inf, math.nan
    x[50, K // 2], w[60, K // 2] = math.inf, -math.inf
    got, ref = ops.linear_f32(x, w, b), (x.double() @ w.double().t() + b.double()).float()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(torch.isinf(got), torch.isinf(ref))
    inf = torch.isinf(ref)
    assert torch.equal(got[inf], ref[inf])
    ok = torch.isfinite(ref)
    assert float((got[ok] - ref[ok]).norm() / ref[ok].norm()) < 1e-6


def test_non_finite_rows_stay_within_a_few_products_time():
    """Every row of x marked (one NaN each): the outputs come from fp32 matrix products in the epilogue, measured at
    2.2 times the fp32 library product's time; 10 times is the bound."""
    x, w, _ = _inputs(4096, 3072, 768)
    x[:, 5] = math.nan

    def us(f):
        for _ in range(3):
            f()
        t = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        t[0].record()
        for _ in range(5):
            f()
        t[1].record()
        t[1].synchronize()
        return t[0].elapsed_time(t[1]) * 200
    ours, lib = us(lambda: ops.linear_f32(x, w)), us(lambda: F.linear(x, w))
    assert bool(torch.isnan(ops.linear_f32(x, w)).all())
    assert ours < 10 * lib, (ours, lib)


def test_route_keeps_autograd_and_autocast():
    x, w, _ = _inputs(1024, 4096, 768)
    assert ops.linear_f32_ok(x, w)
    wp = torch.nn.Parameter(w)
    assert not ops.linear_f32_ok(x, wp)
    with torch.no_grad():
        assert ops.linear_f32_ok(x, wp)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not ops.linear_f32_ok(x, wp)
    assert not ops.linear_f32_ok(x.bfloat16(), w.bfloat16())
    assert not ops.linear_f32_ok(x[:128], w)


@pytest.mark.parametrize("d_model,b,l,kw", [(768, 3, 333, dict(bias=True)), (768, 1, 2000, {}), (2048, 1, 420, {}),
                                            (1000, 1, 1100, {})])
def test_one_call_prefill_with_split_projections(d_model, b, l, kw, monkeypatch):
    """A one-call prefill whose in_proj (and, from 1909 rows at d_model 768,
    out_proj) run split, the in_proj's operand written by the norm before it
    (d_model 1000 is no multiple of 32: a split of its own there), against the
    per-op path: the two differ by fp32 rounding only (1e-5, the bound the
    long prefill's other forms are held to)."""
    import mamba_lite.model as mm
    from mamba_lite.model import MambaConfig, MambaLM
    torch.manual_seed(l)
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=d_model, n_layer=2, vocab_size=300, **kw)).eval()
    ids = torch.randint(0, 300, (b, l), device="cuda")
    assert lm._native_prefill_kind(b, l) == "long"
    with torch.no_grad():
        got, cache = lm.prefill(ids)
        monkeypatch.setattr(mm, "LONG_PREFILL_NATIVE", False)
        monkeypatch.setattr(ops, "linear_f32_ok", lambda *a, **k: False)
        ref, rcache = lm.prefill(ids)
    rel = lambda a, r: float((a.double() - r.double()).norm() / r.double().norm())
    assert rel(got, ref) < 1e-5
    for a, r in zip(cache.layers, rcache.layers):
        assert rel(a.ssm_state, r.ssm_state) < 1e-5 and rel(a.conv_state, r.conv_state) < 1e-5


@pytest.mark.parametrize("d_model", [512, 768, 2048])
def test_one_call_prefill_with_spread_norm_rows(d_model, monkeypatch):
    """A norm weight of 2^27 on a column that the in_proj ignores: the rows that the norm writes are not split, and
    the one call agrees with the per-op path on fp32 products (1e-5, as above; split, the rows would keep 2^-13)."""
    import mamba_lite.model as mm
    from mamba_lite.model import MambaConfig, MambaLM
    torch.manual_seed(d_model)
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=d_model, n_layer=2, vocab_size=300)).eval()
        ids = torch.randint(0, 300, (1, 2600))
    with torch.no_grad():
        for blk in lm.layers:
            blk.norm.weight[3] = 2.0 ** 27
            blk.mixer.in_proj.weight[:, 3] = 0
        assert ops.linear_f32_pays(2600, 4 * d_model, d_model)
        got, _ = lm.prefill(ids)
        monkeypatch.setattr(mm, "LONG_PREFILL_NATIVE", False)
        monkeypatch.setattr(ops, "linear_f32_ok", lambda *a, **k: False)
        ref, _ = lm.prefill(ids)
    assert float((got.double() - ref.double()).norm() / ref.double().norm()) < 1e-5


@pytest.mark.parametrize("d_model,l", [(2560, 1024), (1000, 1100)])
def test_one_call_in_proj_is_split_past_the_norms_widths(d_model, l):
    """Where the norm does not write the split (more than 2048 columns, or no multiple of 32), the in_proj of the one
    call is the split product all the same: the conv state it leaves has that product's bits."""
    from mamba_lite.model import MambaConfig, MambaLM
    torch.manual_seed(d_model)
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=d_model, n_layer=1, vocab_size=300)).eval()
        ids = torch.randint(0, 300, (1, l))
    assert lm._native_prefill_kind(1, l) == "long"
    mx, D = lm.layers[0].mixer, 2 * d_model
    with torch.no_grad():
        _, cache = lm.prefill(ids)
        xn = ops.add_rmsnorm(lm.embedding(ids), lm.layers[0].norm.weight, lm.layers[0].norm.eps)
        xz = ops.linear_f32(xn, mx.in_proj.weight, mx.in_proj.bias)
    assert torch.equal(cache.layers[0].conv_state, xz[:, -3:, :D].transpose(1, 2))


def test_small_calls_ask_for_the_sizes_only(monkeypatch):
    """A small eager mixer is bound by the host: where the sizes rule the split product out, nothing else about the
    call is looked at (9 us of 124 at 633 x 512 otherwise)."""
    import mamba_lite.model as mm
    with torch.device("cuda"):
        m = mm.MambaMixer(mm.MambaConfig(d_model=512, n_layer=1, vocab_size=8), 0).eval()
        x = torch.randn(3, 211, 512)
    asked = []
    monkeypatch.setattr(mm, "_plain_modules", lambda *a: asked.append(a))
    monkeypatch.setattr(ops, "linear_f32_ok", lambda *a: asked.append(a))
    with torch.no_grad():
        m.prefill(x)
        assert not asked
        m.prefill(torch.randn(8, 1024, 512, device="cuda"))
        assert asked


def _no_more_than(mp, most):
    """torch.empty of more than `most` bytes is out of memory, as far as Python's calls go."""
    real = torch.empty

    def empty(*size, **kw):
        t = real(*size, **{**kw, "device": "meta"})
        if t.numel() * t.element_size() > most:
            raise torch.OutOfMemoryError(f"{t.numel() * t.element_size()} bytes")
        return real(*size, **kw)
    mp.setattr(torch, "empty", empty)


def test_without_room_for_the_split_operands_the_library_takes_the_product(monkeypatch):
    x, w, b = _inputs(1024, 2048, 4096)
    ref = F.linear(x, w, b)
    _no_more_than(monkeypatch, 16 << 20)         # the output's 8 MB; the operands take 48 MB
    with pytest.raises(torch.OutOfMemoryError):
        torch.empty(x.numel() + w.numel(), device="cuda")
    assert torch.equal(ops.linear_f32(x, w, b), ref)
    halves = ops.linear_f32(x, w, b, n_split=1024)
    assert float((torch.cat(halves, 1) - ref).norm() / ref.norm()) < 2e-6


def test_without_room_for_its_workspace_a_prompt_runs_as_it_fits(monkeypatch):
    """A prompt of over 2^21 token-channels with no room for the one call's workspace runs op by op; with room for that
    but not for the split operands, in one call on library products."""
    import mamba_lite.model as mm
    from mamba_lite.model import MambaConfig, MambaLM
    torch.manual_seed(4)
    with torch.device("cuda"):
        lm = MambaLM(MambaConfig(d_model=768, n_layer=2, vocab_size=300)).eval()
        ids = torch.randint(0, 300, (1, 5000))
    calls = []
    real = ops.prefill_long
    monkeypatch.setattr(ops, "prefill_long", lambda *a, **k: (calls.append(1), real(*a, **k), calls.append(2))[1])
    rows, M, D = 5000, 768, 1536
    one_call = 4 * rows * (4 * M + 5 * D + 80) + (33 << 20)
    with torch.no_grad():
        with monkeypatch.context() as mp:
            mp.setattr(mm, "LONG_PREFILL_NATIVE", False)
            mp.setattr(ops, "linear_f32_ok", lambda *a, **k: False)
            ref, _ = lm.prefill(ids)
        for most, path in ((1 << 40, [1, 2]), (one_call, [1, 2]), (one_call - (40 << 20), [1])):
            calls.clear()
            with monkeypatch.context() as mp:
                _no_more_than(mp, most)
                got, _ = lm.prefill(ids)
            assert calls == path
            assert float((got - ref).norm() / ref.norm()) < 1e-5


def test_without_room_for_the_summaries_a_scan_is_not_segmented(monkeypatch):
    b, D, L, N = 1, 4096, 1024, 16
    u, z = (torch.randn(b, D, L, device="cuda") for _ in range(2))
    B, C = (torch.randn(b, N, L, device="cuda") for _ in range(2))
    A = -torch.arange(1, N + 1, device="cuda", dtype=torch.float32).repeat(D, 1).contiguous()
    y, h = torch.empty_like(u), torch.empty(b, D, N, device="cuda")
    run = lambda **kw: ops.selective_scan(u, u, A, B, C, z=z, **kw)
    ref = run(algo="chunked")
    _no_more_than(monkeypatch, 1 << 10)
    got = run(y=y, h_out=h)
    assert all(torch.equal(p, q) for p, q in zip(got, ref))
