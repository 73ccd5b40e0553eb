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
    (six piece products each: 2^-25 for the three left out)."""
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
