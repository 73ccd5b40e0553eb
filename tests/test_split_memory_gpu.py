"""An fp32 fused sweep whose split operands the device has no room for runs on fp32 operands: plain entries, a
batch, a Kronecker U and 1 x 32 rows, against the fp64 sweep under the same codes; and an allocator whose
limit holds C and E but not the pieces."""

import functools
import gc

import pytest
import torch

import gptq_2d as G
import quantizer_int as QI
from test_kron_gpu import _instance
from test_split_sweep_gpu import _layer

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture
def no_room(monkeypatch):
    """Every allocation in bytes (the sweep's workspace) fails; the list of what was asked for."""
    asked, empty = [], torch.empty

    def refuse(*args, dtype=None, **kw):
        if dtype is torch.uint8:
            asked.append(args[0])
            raise torch.OutOfMemoryError("no room")
        return empty(*args, dtype=dtype, **kw)

    monkeypatch.setattr(torch, "empty", refuse)
    return asked


def _close(pre, pre64, x, z, lo, up):
    """The bound of test_split_sweep_gpu.py: (m + n + 4) 2^-23 times the sum of the products' magnitudes."""
    l64, u64 = lo.double().tril(-1), up.double().triu(1)
    e = z.double() - pre64
    c = e + l64 @ e
    size = x.double().abs() + l64.abs() @ e.abs() + c.abs() @ u64.abs() + (l64.abs() @ e.abs()) @ u64.abs()
    return ((pre.double() - pre64).abs() <= sum(x.shape[-2:], 4) * 2. ** -23 * size).all()


def _forced(run, x, lo, u, z, pre):
    return run(x, lo, u, quantizer=QI.teacher_forced_quantizer, quantizer_inputs=(z, pre), outer_block_size=64, fused=True)


@pytest.mark.parametrize("m,n,batch", [(31, 33, ()), (100, 140, ()), (257, 130, ()), (64, 96, (3,))])
def test_plain(m, n, batch, no_room):
    print(f"no room {m}x{n} batch={batch}", flush=True)
    x, lo, up = _layer(m, n, m + n, batch)
    z, pre, pre64 = torch.round(x), torch.full_like(x, torch.nan), torch.full_like(x, torch.nan, dtype=torch.float64)
    assert _forced(G.gptq_2d, x, lo, up, z, pre).equal(z) and len(no_room) == 1
    _forced(G.gptq_2d, x.double(), lo.double(), up.double(), z.double(), pre64)
    assert len(no_room) == 1 and _close(pre, pre64, x, z, lo, up)


@pytest.mark.parametrize("m,np_,nq,rows", [(64, 3, 48, False), (96, 3, 112, False), (64, 3, 64, True)])
def test_kronecker(m, np_, nq, rows, no_room):
    print(f"no room kron {m}x({np_}x{nq}) rows={rows}", flush=True)
    x, lo, p, q = _instance(m, np_, nq, m + nq)
    up = torch.kron(p, q)
    run = functools.partial(G.gptq_2d_super_entry, super_entry_shape=(1, 32)) if rows else G.gptq_2d
    z, pre, pre_d = torch.round(x), torch.full_like(x, torch.nan), torch.full_like(x, torch.nan)
    pre64 = torch.full_like(x, torch.nan, dtype=torch.float64)
    assert _forced(run, x, lo, G.KroneckerU(p, q), z, pre).equal(z)
    assert _forced(run, x, lo, up, z, pre_d).equal(z) and len(no_room) == 2
    _forced(run, x.double(), lo.double(), up.double(), z.double(), pre64)
    assert pre.equal(pre_d) and _close(pre, pre64, x, z, lo, up)


@pytest.mark.parametrize("quant", ["absmax", "affine"])
def test_rows(quant, no_room):
    """The outputs are the quantizer's of the values that the sweep along them reports."""
    print(f"no room rows {quant}", flush=True)
    m, n = 70, 160
    x, lo, up = _layer(m, n, 9)
    run = functools.partial(G.gptq_2d_super_entry, super_entry_shape=(1, 32))
    s = torch.full_like(x, .7)
    if quant == "absmax":
        q, qi = functools.partial(QI.int_abs_max_quantizer_hip, qmin=-8, qmax=7, dtype=torch.bfloat16), (s,)
    else:
        q, qi = functools.partial(QI.affine_quantizer_super_entry_hip, qmin=-8, qmax=7), (s, torch.zeros_like(x))
    z = run(x, lo, up, quantizer=q, quantizer_inputs=qi, outer_block_size=64, fused=True)
    pre = torch.full_like(x, torch.nan)
    assert _forced(run, x, lo, up, z, pre).equal(z) and len(no_room) == 2
    assert torch.equal(torch.clamp(torch.round(pre / s), -8, 7) * s, z)


def test_allocator_limit():
    """A limit that holds the work matrix, C and E of 4096 x 4096 (192 MiB) but not the pieces (288 MiB more)."""
    print("allocator limit", flush=True)
    m = n = 4096
    x, lo, up = (torch.randn(m, n, device=DEV) for _ in range(3))
    lo, up = (.3 / n ** .5 * lo).tril_(-1), (.3 / n ** .5 * up).triu_(1)
    want, pre_want = torch.round(x), torch.empty_like(x)
    pre = torch.empty_like(x)
    _forced(G.gptq_2d, x, lo, up, want, pre_want)
    torch.cuda.synchronize()
    gc.collect()
    torch.cuda.empty_cache()
    total, hold, size = torch.cuda.mem_get_info()[1], [], 1 << 30
    try:
        # what other tensors' segments have free, so that only the room left below counts
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
        while size >= 1 << 20:
            try:
                hold.append(torch.empty(size, dtype=torch.uint8, device=DEV))
            except torch.OutOfMemoryError:
                size >>= 1
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (256 << 20)) / total)
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(480 << 20, dtype=torch.uint8, device=DEV)
        _forced(G.gptq_2d, x, lo, up, want, pre)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.)
    # the two engines' sums differ by rounding only: 8192 products of size up to 0.02 each
    assert (pre - pre_want).abs().max() < 1e-3 and not pre.equal(pre_want)
