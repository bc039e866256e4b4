"""Operand preparation at the sizes where the sort changes its form: one
workgroup in LDS (up to one tile of 6144 nonzeros), one-launch look-back passes
above, reduce-then-scan passes on X's free bits alone above 2^21 (pairs of 10- and
11-bit digits above 2^18 and 2^16).  The plan's contraction with a permutation returns the operand in key
order, so the sorted keys and values are checked exactly."""
import ctypes

import numpy as np
import pytest

from gsparc_amd import sptc
from gsparc_amd.coo import COOTensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 511, 512, 6143, 6144, 6145, 12287, 12289, 70_001, 2_200_000])
@pytest.mark.parametrize("wide", [False, True])
def test_operand_order_and_values(gpu, n, wide):
    """X contracted with the identity over its last mode: the output is X in
    (row, column) order with its values unchanged.  wide: 64-bit indices and a
    key of 60 bits; else modes whose high digits all keys share."""
    rng = np.random.default_rng(n + wide)
    d0, d1, c = (1 << 24, 1 << 24, 4096) if wide else (40_000, 30, 77)
    i0 = rng.integers(0, d0, n) if wide else rng.integers(39_000 if n < 100_000 else 0, 39_900, n)
    lin = np.unique((i0 * d1 + rng.integers(0, d1, n)) * c + rng.integers(0, c, n))
    lin = rng.permutation(lin)
    dt = np.uint64 if wide else np.uint32
    X = COOTensor((d0, d1, c), [(lin // (d1 * c)).astype(dt), (lin // c % d1).astype(dt),
                                (lin % c).astype(dt)], rng.random(len(lin)).astype(np.float32) + 1)
    assert n < 2_200_000 or len(lin) > 1 << 21
    eye = COOTensor((c, c), [np.arange(c, dtype=dt)] * 2, np.ones(c, np.float32))
    idx, v = sptc.SpTC(X, eye, [2], [0]).decode()
    o = np.argsort(lin, kind="stable")
    for a, b in zip(idx, X.idx):
        np.testing.assert_array_equal(a.astype(np.int64), b[o].astype(np.int64))
    np.testing.assert_array_equal(v, X.val[o])


@pytest.mark.parametrize("n,rb", [(1 << 18, 10), ((1 << 18) + 1, 10), (1 << 16, 11),
                                  ((1 << 16) + 1, 11), (3073, 10), (3073, 11)])
def test_wide_digits_on_both_sides_of_their_line(gpu, n, rb):
    import torch
    rng = np.random.default_rng(n)
    keys = rng.integers(0, 1 << 33, n).astype(np.int64) >> rng.integers(0, 30, n)
    k = torch.from_numpy(keys).cuda()
    v = torch.arange(n, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    sptc.check(sptc.lib().sptc_sort_pairs(ctypes.c_void_p(k.data_ptr()),
                                          ctypes.c_void_p(v.data_ptr()), n, 33, rb, None))
    o = np.argsort(keys, kind="stable")
    np.testing.assert_array_equal(k.cpu().numpy(), keys[o])
    np.testing.assert_array_equal(v.cpu().numpy(), o.astype(np.float32))
