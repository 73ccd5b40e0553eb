"""The fp32 fused sweep on split operands (gptq2d_sweep_split_f32): values before rounding against the fp64 sweep under
the same codes, at the edges of tiles, outer blocks and flush blocks; batches with shared and own factors; and inputs
that are not finite, against the sweep on fp32 operands (gptq2d_sweep_fused_f32)."""

import functools

import pytest
import torch

import _hip
import gptq_2d as G
import quantizer_int as QI
from oracle import sweep as S

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _layer(m, n, seed, batch=()):
    g = torch.Generator().manual_seed(seed)
    x = 4. * torch.randn(*batch, m, n, generator=g)
    lo = S.unit_triangular(.5 / m ** .5 * torch.randn(m, m, generator=g), upper=False)
    up = S.unit_triangular(.5 / n ** .5 * torch.randn(n, n, generator=g), upper=True)
    # what the sweep must not read
    lo = lo.masked_fill(torch.ones(m, m, dtype=torch.bool).triu(), torch.nan)
    up = up.masked_fill(torch.ones(n, n, dtype=torch.bool).tril(), torch.nan)
    return x.to(DEV), lo.to(DEV), up.to(DEV)


SIZES = [(1, 1), (1, 40), (33, 1), (31, 33), (32, 32), (64, 65), (95, 129), (257, 130), (130, 515), (640, 353)]


@pytest.mark.parametrize("m,n", SIZES)
@pytest.mark.parametrize("outer", [32, 96, 512])
def test_values_before_rounding(m, n, outer):
    """Each fp32 sum of up to m + n products errs by at most (m + n + 4) 2^-23 times the sum of the products' magnitudes
    (the piece products left out are below 2^-22.9 of their product together)."""
    print(f"split sweep {m}x{n} outer={outer}", flush=True)
    x, lo, up = _layer(m, n, m + 3 * n)
    z = torch.round(x)
    pre = torch.full_like(x, torch.nan)
    got = G.gptq_2d(x, lo, up, quantizer=QI.teacher_forced_quantizer, quantizer_inputs=(z, pre), outer_block_size=outer,
                    fused=True)
    pre64 = torch.full_like(x, torch.nan, dtype=torch.float64)
    G.gptq_2d(x.double(), lo.double(), up.double(), quantizer=QI.teacher_forced_quantizer,
              quantizer_inputs=(z.double(), pre64), outer_block_size=outer, fused=True)
    assert got.equal(z) and not pre.isnan().any()
    l64, u64 = lo.double().tril(-1), up.double().triu(1)
    e = z.double() - pre64
    c = e + l64 @ e
    size = x.double().abs() + l64.abs() @ e.abs() + c.abs() @ u64.abs() + (l64.abs() @ e.abs()) @ u64.abs()
    assert ((pre.double() - pre64).abs() <= (m + n + 4) * 2. ** -23 * size).all()


@pytest.mark.parametrize("zero_zp", [True, False])
@pytest.mark.parametrize("m,n", [(31, 33), (96, 161)])
def test_affine_outputs_are_the_quantizer_of_their_values(m, n, zero_zp):
    """Both affine loops (zero points all 0, and not): the outputs are the plug-in's of the values that the same sweep
    reports under these codes, bit for bit."""
    print(f"split affine {m}x{n} zero_zp={zero_zp}", flush=True)
    x, lo, up = _layer(m, n, 5 * m + n)
    g = torch.Generator().manual_seed(1)
    s = (0.3 + torch.rand(m, n, generator=g)).to(DEV)
    zp = torch.zeros_like(s) if zero_zp else torch.randint(-3, 4, (m, n), generator=g).float().to(DEV)
    q = functools.partial(QI.affine_quantizer_hip, qmin=-8, qmax=7)
    z = G.gptq_2d(x, lo, up, quantizer=q, quantizer_inputs=(s, zp), outer_block_size=64, fused=True)
    pre = torch.full_like(x, torch.nan)
    assert G.gptq_2d(x, lo, up, quantizer=QI.teacher_forced_quantizer, quantizer_inputs=(z, pre), outer_block_size=64,
                     fused=True).equal(z)
    assert torch.equal((torch.clamp(torch.round(pre / s + zp), -8, 7) - zp) * s, z)


def test_batches_equal_single_matrices():
    """A batch whose matrices share L, or have factors and scales of their own (a two-dimensional batch: general
    strides), equals one call per matrix bit for bit."""
    m, n = 70, 130
    print("split batches", flush=True)
    x, lo, up = _layer(m, n, 3, (2, 3))
    g = torch.Generator().manual_seed(2)
    ups = torch.stack([_layer(m, n, 10 + i)[2] for i in range(3)])
    s = (0.3 + torch.rand(2, 1, m, n, generator=g)).to(DEV)
    zp = torch.zeros_like(s)
    q = functools.partial(QI.affine_quantizer_hip, qmin=-8, qmax=7)
    z = G.gptq_2d(x, lo, ups, quantizer=q, quantizer_inputs=(s, zp), outer_block_size=64, fused=True)
    for a in range(2):
        for b in range(3):
            one = G.gptq_2d(x[a, b], lo, ups[b], quantizer=q, quantizer_inputs=(s[a, 0], zp[a, 0]), outer_block_size=64,
                            fused=True)
            assert z[a, b].equal(one)


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3e38])
@pytest.mark.parametrize("at", [(3, 5), (40, 70), (90, 10)])
def test_values_that_are_not_finite(value, at):
    """One entry infinite, NaN or close to overflow: the entries it reaches come out as in the sweep on fp32 operands
    (the same infinities and NaN before rounding), the others as ever."""
    m, n = 100, 140
    print(f"split sweep with {value} at {at}", flush=True)
    x, lo, up = _layer(m, n, 17)
    x[at] = value
    z = torch.zeros_like(x)
    pre = torch.full_like(x, 7.)
    G.gptq_2d(x, lo, up, quantizer=QI.teacher_forced_quantizer, quantizer_inputs=(z, pre), outer_block_size=64, fused=True)
    y, c, e, want = x.clone(), torch.empty_like(x), torch.empty_like(x), torch.full_like(x, 7.)
    one = _hip.i64_array([])
    _hip.call("sweep_fused", x.dtype, _hip.ptr(y), _hip.ptr(c), _hip.ptr(e), _hip.ptr(lo), _hip.ptr(up), m, n, 0, one, one,
              one, 2, _hip.ptr(z), one, None, None, 0., 0., _hip.ptr(want), 2, 0, -1, _hip.stream(x.device))
    assert torch.equal(pre.isnan(), want.isnan()) and torch.equal(pre.isinf(), want.isinf())
    ok = want.isfinite()
    assert torch.equal(pre[pre.isinf()], want[want.isinf()])
    # a finite value's rounding errors reach what lies below and right of it: (m + n + 4) 2^-23 of the products' size
    tol = 1e-4 * (1. + want.abs())
    if abs(value) < float("inf"):
        tol[at[0]:, at[1]:] += (m + n + 4) * 2. ** -23 * value
    assert ((pre - want).abs() <= tol)[ok].all()


def _sums(run, monkeypatch):
    """What `run` reports before rounding on split operands, and with the same call on fp32 operands."""
    pre = run()
    with monkeypatch.context() as mp:
        mp.setattr(G, "_run_split", lambda *a, **k: False)
        want = run()
    return pre, want


@pytest.mark.parametrize("m,n,outer", [(64, 65, 32), (640, 353, 64), (353, 640, 512), (1500, 1100, 256)])
def test_error_is_that_of_fp32_sums(m, n, outer, monkeypatch):
    """Feedback alone (X = 0, normal values forced), against 64 bits: in norm no further off than the sweep on fp32
    operands, but for 1.25 for the two engines' different summation orders.  Without the third piece of an operand, or
    with one product of the pieces wrong, the sums are 2^-18 off, eight times that and more."""
    print(f"split sweep error {m}x{n} outer={outer}", flush=True)
    x, lo, up = _layer(m, n, m + n)
    z, x = torch.round(x) / 4, torch.zeros_like(x)

    def run(dt=torch.float32):
        pre = torch.full_like(x, torch.nan, dtype=dt)
        G.gptq_2d(x.to(dt), lo.to(dt), up.to(dt), quantizer=QI.teacher_forced_quantizer, quantizer_inputs=(z.to(dt), pre),
                  outer_block_size=outer, fused=True)
        return pre

    ref = run(torch.float64)
    split, fp32 = (((p.double() - ref).norm() / ref.norm()).item() for p in _sums(run, monkeypatch))
    print(f"relative error {split:.2e}, on fp32 operands {fp32:.2e}", flush=True)
    assert split <= 1.25 * fp32


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3e38])
@pytest.mark.parametrize("form", ["flush of 4 x 4 tiles", "batch", "rows", "kronecker", "kronecker rows"])
def test_values_that_are_not_finite_elsewhere(form, value, monkeypatch):
    """The sums formed again in the flush of 4 x 4 tiles (a batch of 600 blocks of them), in a batch with factors of
    its own, in 1 x 32 rows and with a Kronecker U: the infinities and NaN of the sweep on fp32 operands."""
    print(f"split sweep with {value}, {form}", flush=True)
    m, n, batch = {"flush of 4 x 4 tiles": (640, 640, (24,)), "batch": (100, 140, (3,))}.get(form, (100, 192, ()))
    x, lo, up = _layer(m, n, 19, batch)
    rows = "rows" in form
    if form == "batch":
        lo = torch.stack([_layer(m, n, 20 + i)[1] for i in range(3)])
    if "kronecker" in form:
        g = torch.Generator().manual_seed(23)
        p, q = (torch.eye(k) + .5 / k ** .5 * torch.randn(k, k, generator=g).triu(1) for k in (3, 64))
        if rows:
            q = torch.block_diag(*[torch.eye(32)] * 2) + torch.nn.functional.pad(q[:32, 32:], (32, 0, 0, 32))
        up = G.KroneckerU(p.to(DEV), q.to(DEV))
    at = (2, 40, 70) if batch else (40, 70)
    x[at] = value
    z = torch.zeros_like(x)

    def run():
        pre = torch.full_like(x, 7.)
        kw = dict(quantizer=QI.teacher_forced_quantizer, quantizer_inputs=(z, pre), outer_block_size=64, fused=True)
        G.gptq_2d_super_entry(x, lo, up, super_entry_shape=(1, 32), **kw) if rows else G.gptq_2d(x, lo, up, **kw)
        return pre

    pre, want = _sums(run, monkeypatch)
    assert torch.equal(pre.isnan(), want.isnan()) and torch.equal(pre.isinf(), want.isinf())
    assert torch.equal(pre[pre.isinf()], want[want.isinf()])
    ok = want.isfinite()
    assert not ok.all() or abs(value) < float("inf")
    tol = 1e-4 * (1. + want.abs())
    if abs(value) < float("inf"):
        tol[..., at[-2]:, at[-1]:] += (m + n + 4) * 2. ** -23 * value
    assert ((pre - want).abs() <= tol)[ok].all()


@pytest.mark.parametrize("m,n,outer", [(1, 32, 64), (32, 32, 64), (31, 64, 64), (96, 32, 512), (130, 96, 32), (257, 640, 512),
                                       (700, 320, 4096)])
def test_rows_before_rounding(m, n, outer):
    """1 x 32 rows: single tiles, the last tile row and column (whose split blocks nobody reads), and preps that pull
    more halves than are in flight at once (44 of them a product in blocks of 4096 antidiagonals).  The bound of
    test_values_before_rounding."""
    print(f"split rows {m}x{n} outer={outer}", flush=True)
    x, lo, up = _layer(m, n, m + 5 * n)
    z = torch.round(x)

    def run(dt):
        pre = torch.full_like(x, torch.nan, dtype=dt)
        got = G.gptq_2d_super_entry(x.to(dt), lo.to(dt), up.to(dt), super_entry_shape=(1, 32),
                                    quantizer=QI.teacher_forced_quantizer, quantizer_inputs=(z.to(dt), pre),
                                    outer_block_size=outer, fused=True)
        assert got.equal(z.to(dt))
        return pre.double()

    pre, pre64 = run(torch.float32), run(torch.float64)
    block = torch.arange(n, device=DEV) // 32
    l64, u64 = lo.double().tril(-1), torch.where(block[:, None] < block[None], up.double(), 0.)
    e = z.double() - pre64
    c = e + l64 @ e
    size = x.double().abs() + l64.abs() @ e.abs() + c.abs() @ u64.abs() + (l64.abs() @ e.abs()) @ u64.abs()
    assert ((pre - pre64).abs() <= (m + n + 4) * 2. ** -23 * size).all()
