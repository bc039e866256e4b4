"""Dense accumulation of many rows, a wave per row: rows of one owner, of
several, of none, and rows left to the whole workgroup (over 4096 products, or
under 8 products per owner), on both sides of the row count where waves take
over (16384), over column spaces at the edges of its two LDS row widths."""
import numpy as np
import pytest
import scipy.sparse as sp

from gsparc_amd import sptc
from gsparc_amd.coo import COOTensor
from helpers import REL_TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,R", [(1, 16384), (2, 16384), (63, 16384), (65, 16383), (65, 16384),
                                 (65, 16417), (65, 70_001), (255, 16384), (256, 16384),
                                 (257, 16384), (1023, 16383), (1023, 16384), (1024, 16389)])
def test_rows_by_waves(gpu, K, R):
    rng = np.random.default_rng(K * 10 + R % 10)
    # contract values: 40 with segments of random length, one of every column, one unused by Y
    segs = [int(x) for x in rng.integers(1, K + 1, 40)] + [K]
    C = len(segs) + 1
    yc = np.concatenate([np.full(n, c, np.uint32) for c, n in enumerate(segs)])
    yj = np.concatenate([rng.choice(K, size=n, replace=False) for n in segs]).astype(np.uint32)
    own = rng.choice([1, 1, 1, 1, 1, 2, 5], R)
    own[[5, 6, R // 2, R - 1]] = C  # with K near 1024: over 4096 products
    xr = np.repeat(np.arange(R, dtype=np.uint32), own)
    xc = np.concatenate([rng.choice(C, size=n, replace=False) for n in own]).astype(np.uint32)
    vx = (rng.standard_normal(len(xr))).astype(np.float32)
    vy = (rng.standard_normal(len(yc))).astype(np.float32)
    vx[::7] *= 0.0  # signed zeros among the products
    X = COOTensor((R, C), [xr, xc], vx)
    Y = COOTensor((C, K), [yc, yj], vy)
    res = sptc.SpTC(X, Y, [1], [0], dense_accumulator=1)
    assert res.info.accumulator == 1
    # (signed zeros: a relative error of the helper's kind would divide by zero)
    mk = lambda t, v: sp.csr_matrix((v, (t.idx[0], t.idx[1])), shape=t.dims)
    pat = (mk(X, np.ones(len(vx))) @ mk(Y, np.ones(len(vy)))).tocsr()
    pat.sort_indices()
    (i, j), v = res.decode()
    np.testing.assert_array_equal(i, np.repeat(np.arange(R), np.diff(pat.indptr)))
    np.testing.assert_array_equal(j, pat.indices)
    want = (mk(X, vx.astype(np.float64)) @ mk(Y, vy.astype(np.float64))).tocsr()
    scale = (mk(X, np.abs(vx.astype(np.float64))) @ mk(Y, np.abs(vy.astype(np.float64)))).tocsr()
    at = lambda m: np.asarray(m[i, j]).ravel()
    assert (np.abs(v - at(want)) <= REL_TOL * at(scale)).all()
    assert not np.signbit(v[v == 0]).any()
    esc = sptc.SpTC(X, Y, [1], [0], dense_accumulator=-1)
    assert abs(esc.info.value_sum - res.info.value_sum) <= 1e-12 * len(xr) * K
