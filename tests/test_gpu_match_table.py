"""The index match's table over the top contract bits: ranges of one contract
value and of many, against searches over the whole sorted Y."""
import ctypes

import numpy as np
import pytest

from gsparc_amd import sptc

pytestmark = pytest.mark.gpu


def _dev(torch, a):
    return torch.from_numpy(a.view(np.int64)).cuda()


# name: contract bits, Y's free bits, and the contract values of n keys
def _uniform(rng, n, nb):
    return rng.integers(0, 1 << nb, n, dtype=np.uint64)


def _one_range(rng, n, nb):  # every value below 1000: one entry of the table
    return rng.integers(0, min(1000, 1 << nb), n, dtype=np.uint64)


def _few(rng, n, nb):  # long segments at both ends of the field and inside a range
    return rng.choice(np.array([0, 1, 2, (1 << nb) // 2, (1 << nb) - 2, (1 << nb) - 1], np.uint64), n)


@pytest.mark.parametrize("dist", [_uniform, _one_range, _few])
@pytest.mark.parametrize("ncb,ynf", [(9, 11), (14, 3), (15, 10), (23, 5), (40, 24), (50, 0)])
@pytest.mark.parametrize("nx,ny", [(1, 1), (3, 2), (4096, 4095), (4097, 70_000), (70_001, 3),
                                   (200_000, 131_072)])
def test_match_equals_search(gpu, dist, ncb, ynf, nx, ny):
    import torch
    L = sptc.lib()
    L.sptc_index_match_noalloc.argtypes = L.sptc_index_match.argtypes
    rng = np.random.default_rng(ncb * 1000 + nx)
    cy = dist(rng, ny, ncb)
    y = np.sort(cy << np.uint64(ynf) | rng.integers(0, 1 << ynf, ny, dtype=np.uint64))
    if ncb + ynf < 64:  # the largest key lies outside the field: it matches nothing
        y[-1] |= np.uint64(1) << np.uint64(ncb + ynf)
    c = np.concatenate([rng.choice(cy, nx // 2), dist(rng, nx - nx // 2, ncb)])
    x = np.sort(rng.integers(0, 1 << 13, nx, dtype=np.uint64) << np.uint64(ncb) | c)
    c = x & np.uint64((1 << ncb) - 1)
    yc = y >> np.uint64(ynf)
    pos, end = np.searchsorted(yc, c, "left"), np.searchsorted(yc, c, "right")
    cnt = end - pos
    want = [np.where(cnt, pos, 0), cnt, np.concatenate([[0], np.cumsum(cnt)])]
    dx, dy = _dev(torch, x), _dev(torch, y)
    for fn in (L.sptc_index_match, L.sptc_index_match_noalloc):
        out = [torch.full((n,), -1, dtype=torch.int64, device="cuda") for n in (nx, nx, nx + 1)]
        ir = ctypes.c_uint64()
        sptc.check(fn(ctypes.c_void_p(dx.data_ptr()), nx, ctypes.c_void_p(dy.data_ptr()), ny, ncb,
                      ynf, *[ctypes.c_void_p(o.data_ptr()) for o in out], ctypes.byref(ir),
                      ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        assert ir.value == int(cnt.sum())
        for g, w in zip(out, want):
            np.testing.assert_array_equal(g.cpu().numpy(), w.astype(np.int64))
