"""INT packing of long and unaligned rows: a row by a wave or by a workgroup (256 words and more), units cut off by the
row's end, rows that do not start on 16 bytes, per-entry scales; words, counts and values equal the CPU oracle's."""

import numpy as np
import pytest
import torch

import _hip
import packing as PK
from oracle import packing as P

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("per_entry", [False, True])
@pytest.mark.parametrize("qmin,qmax", [(-8, 7), (-128, 127), (-4, 3), (0, 1), (-16384, 16383)])
@pytest.mark.parametrize("n", [1, 31, 2040, 2048, 2049, 8195])
def test_rows_equal_oracle(n, qmin, qmax, per_entry):
    print(f"pack rows n={n} [{qmin}, {qmax}] per_entry={per_entry}", flush=True)
    g = torch.Generator().manual_seed(n + qmax)
    m = 3
    s = (0.5 + torch.rand(m, n if per_entry else 1, generator=g)).to(torch.bfloat16).float()
    z = torch.randint(qmin, qmax + 1, (m, n), generator=g).float() * s
    z[1, n // 2] += 0.25 * float(s[1, n // 2 if per_entry else 0])  # off the grid
    zp = torch.zeros(())
    # the matrix one element into its buffer: rows aligned to 4 bytes only
    zd = torch.empty(m * n + 1, device=DEV)[1:].view(m, n).copy_(z)
    words, bad = PK.pack_int(zd, s.to(DEV), zp.to(DEV), qmin=qmin, qmax=qmax, check=False, return_bad=True)
    u, ok = P.int_codes(z.numpy(), s.numpy(), zp.numpy(), qmin, qmax)
    assert np.array_equal(words.cpu().numpy().view(np.uint32), P.pack_lsb(u, P.int_bits(qmin, qmax)))
    assert np.array_equal(bad.cpu().numpy(), (~ok).sum(-1))
    back = PK.unpack_int(words, s.to(DEV), zp.to(DEV), n=n, qmin=qmin, qmax=qmax).cpu()
    good = torch.from_numpy(ok)
    assert torch.equal(back[good], z[good])


def _fields(form, m, n, dtype, g):
    """(scale, zero point) of a form, on the CPU: powers of two, so that every z = (q - zp) s is exact."""
    one = lambda *shape: (2. ** torch.randint(-3, 4, shape, generator=g)).to(dtype)
    whole = lambda *shape: torch.randint(-2, 3, shape, generator=g).to(dtype)
    return {"row": lambda: (one(m, 1), None), "row+row": lambda: (one(m, 1), whole(m, 1)),
            "entry": lambda: (one(m, n), None), "entry+entry": lambda: (one(m, n), whole(m, n)),
            "row+entry": lambda: (one(m, 1), whole(m, n)), "entry+scalar": lambda: (one(m, n), whole(1, 1)),
            "column+row": lambda: (one(1, n), whole(m, 1)), "transposed": lambda: (one(n, m).t(), whole(n, m).t())}[form]()


@pytest.mark.parametrize("form", ["row", "row+row", "entry", "entry+entry", "row+entry", "entry+scalar", "column+row",
                                  "transposed"])
@pytest.mark.parametrize("m,n", [(70, 1), (33, 24), (31, 64), (5, 128), (5, 129), (4, 255), (5, 256), (6, 300), (2, 2047), (3, 2050)])
def test_forms_equal_oracle(m, n, form):
    """Every width and both types: rows by eight threads, a wave and a workgroup at the edges of their ranges, rows past
    the last workgroup's share, and scales and zero points that vary along the row, or lie in other orders."""
    print(f"pack forms {m}x{n} {form}", flush=True)
    g = torch.Generator().manual_seed(m + n)
    for dtype in (torch.float32, torch.float64):
        for bits in range(1, 17):
            s, zp = _fields(form, m, n, dtype, g)
            qmin, qmax = -(1 << bits >> 1), (1 << bits) - 1 - (1 << bits >> 1)
            zero = torch.zeros(1, 1, dtype=dtype) if zp is None else zp
            z = (torch.randint(qmin, qmax + 1, (m, n), generator=g).to(dtype) - zero) * s
            z[m // 2, n - 1] += 0.25 * (s.expand(m, n))[m // 2, n - 1]  # off the grid
            dev = lambda t: None if t is None else t.to(DEV)
            words, bad = PK.pack_int(dev(z), dev(s), dev(zp), qmin=qmin, qmax=qmax, check=False, return_bad=True)
            full = lambda t: t.expand(m, n).contiguous().numpy()
            u, ok = P.int_codes(z.numpy(), full(s), full(zero), qmin, qmax)
            assert np.array_equal(words.cpu().numpy().view(np.uint32), P.pack_lsb(u, P.int_bits(qmin, qmax))), (dtype, bits)
            assert np.array_equal(bad.cpu().numpy(), (~ok).sum(-1)) and (~ok).sum() == 1, (dtype, bits)
            back = PK.unpack_int(words, dev(s), dev(zp), n=n, qmin=qmin, qmax=qmax, dtype=dtype).cpu()
            good = torch.from_numpy(ok)
            assert torch.equal(back[good], z[good]), (dtype, bits)


def test_more_rows_than_a_grid_has_workgroups():
    """2^24 + 1 rows of 256 words: a workgroup per row would be more threads than a grid can have."""
    rows, n, row_words = (1 << 24) + 1, 256, 256
    print(f"pack {rows} rows", flush=True)
    z = torch.zeros(rows, n, device=DEV)
    z[-1, 1::2] = 7.
    z[-1, -1] = .5
    s = torch.ones(1, 1, device=DEV)
    words = torch.full((rows, row_words), -1, dtype=torch.int32, device=DEV)
    bad = torch.full((rows,), -1, dtype=torch.int32, device=DEV)
    stride = _hip.i64_array([0, 0, 0])
    _hip.call("pack_int", z.dtype, _hip.ptr(z), 1, rows, n, _hip.ptr(s), stride, None, None, 0., 15., 4, _hip.ptr(words),
              row_words, _hip.ptr(bad), _hip.stream(z.device))
    assert not words[:-1].any() and not bad[:-1].any()
    last = [0x70707070] * 31 + [0x00707070] + [0] * (row_words - 32)
    assert words[-1].tolist() == last and bad[-1].item() == 1
