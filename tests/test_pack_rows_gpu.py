"""INT packing of long and unaligned rows: a row by a wave or by a workgroup (256 words and more), units cut off by the
row's end, rows that do not start on 16 bytes, per-entry scales; words, counts and values equal the CPU oracle's."""

import numpy as np
import pytest
import torch

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
