"""Products of the factorisation and of the triangular inverse on split bf16 operands: sizes at the edges of their
128 x 128 blocks, 16-deep k-tiles, bands of 8 block rows and strips, against the definition in fp64; and values outside
the pieces' range, whose sums must be what fp32 products give."""

import pytest
import torch

import gptq_2d_ldl as LDL
import instances
from oracle import algorithms as A

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = torch.finfo(torch.float32).eps


@pytest.mark.parametrize("k", [128, 132, 192, 196, 252, 260, 508, 512, 516, 640, 644, 1020, 1024, 1152, 1156, 1924,
                               2048, 2052])
def test_factor_edges(k):
    m = instances.wishart_factor(k, .5, 21).float()
    for fn, of in ((LDL.ldl_of_inverse, A.ldl_of_inverse), (LDL.ldl, A.ldl)):
        ref = of(m.double())
        got = fn(m.to(DEV)).double().cpu()
        # entries bounded by the condition number (alpha .5: below 100) times the fp32 sums' error, sqrt(k) eps
        # for k terms of random rounding: 100 sqrt(k) eps, which a dropped or doubled k-tile exceeds by far
        assert (got - ref).abs().max() <= 100 * k ** .5 * EPS * ref.abs().max(), (fn.__name__, k)


def test_error_no_larger_than_fp32_sums():
    """Factor error of 3072 at the level of one fp32 rounding per stored entry: the split products add less."""
    k = 3072
    m = instances.wishart_factor(k, .5, 22, device=DEV).float()
    ref = LDL.ldl_of_inverse(m.double())
    err = ((LDL.ldl_of_inverse(m).double() - ref).norm() / ref.norm()).item()
    print(f"relative error {err:.1e}")
    assert err < 4 * EPS


def _arrow(k, head, at):
    """I plus a symmetric row and column `head` at index `at`: its factor is known in closed form."""
    m = torch.eye(k, dtype=torch.float64)
    m[at, :at] = head
    m[:at, at] = head
    m[at, at] = 1 + head * head * at
    return m


@pytest.mark.parametrize("head", [1e-30, 1e-20, 3.0, 1e15])
def test_range(head):
    """Entries whose lower pieces are denormal, and ones near the square root of the largest float."""
    k, at = 1024, 900
    got = LDL.ldl(_arrow(k, head, at).float().to(DEV), check=False).double().cpu()
    ref = torch.eye(k, dtype=torch.float64)
    ref[at, :at] = head
    if head <= 3:  # above, 1 + head^2 at loses the 1 in fp32 and the last pivot is not positive
        assert torch.allclose(got, ref, rtol=1e-5, atol=0)
    else:
        assert torch.allclose(got[at, :at], ref[at, :at], rtol=1e-5, atol=0)


@pytest.mark.parametrize("value", [float("inf"), float("nan"), -1.0])
def test_not_positive_definite(value):
    """The first pivot that is not positive is reported, and nothing before it is touched by what follows."""
    k, at = 1280, 700
    m = torch.eye(k, device=DEV)
    m[at, at] = value
    m[at, :at] = m[:at, at] = 0.
    if value == float("inf"):
        m[at + 1, at] = m[at, at + 1] = value  # inf / inf in the column below
    with pytest.raises(torch.linalg.LinAlgError):
        LDL.ldl(m)
    out = LDL.ldl(m, check=False)
    assert out[:at, :at].equal(torch.eye(at, device=DEV))


def test_inverse_past_the_largest_float():
    """A chain of 17 links whose inverse doubles 5 times a link from 2^60: 14 links and more overflow fp32 in the last
    level's product and are infinite, neither NaN nor finite, everything else as the definition gives it.  The pivots
    cancel 10 bits a link: 2^10 eps each, under 1 % over the chain."""
    k, step, d = 2048, 120, 2.0 ** -60
    c = torch.eye(k, dtype=torch.float64) * d
    inv = torch.eye(k, dtype=torch.float64) / d
    at = list(range(0, k, step))
    for a, b in zip(at, at[1:]):
        c[b, a] = 32 * d
    for i, b in enumerate(at):
        for j, a in enumerate(at[:i]):
            inv[b, a] = (-32.0) ** (i - j) / d
    # ldl_of_inverse factors the reversed matrix: C is its Cholesky factor
    got = LDL.ldl_of_inverse((c @ c.t()).flip(0, 1).float().to(DEV), check=False).cpu()
    raw = inv.flip(0, 1).t()
    want = raw.float().double() * d  # each diagonal entry of raw is 1 / d
    assert got.isinf().equal(want.isinf()) and got.isinf().sum() == sum(len(at) - n for n in range(14, len(at)))
    assert torch.allclose(got.double(), want, rtol=1e-2, atol=0)
