"""Calls in a row, from several threads and after the caches were given back:
what one call leaves behind (pinned words, events) must not show in the next."""
import threading

import numpy as np
import pytest

from gsparc_amd import sptc
from gsparc_amd.coo import COOTensor
from helpers import random_coo

pytestmark = pytest.mark.gpu


def test_calls_share_nothing_visible(gpu):
    rng = np.random.default_rng(5)
    pairs = []
    for n in (1, 40, 3000, 20_000):  # with and without duplicate Y coordinates, dense and not
        X, Y = random_coo(rng, (60, 70, 50), n), random_coo(rng, (50, 900), n)
        D = COOTensor(Y.dims, [np.concatenate([i, i[:1]]) for i in Y.idx],
                      np.concatenate([Y.val, Y.val[:1]]))
        pairs += [(X, Y), (X, D)]

    def run(X, Y):
        r = sptc.SpTC(X, Y, [2], [0])
        idx, v = r.decode()
        return r.info.ir_nnz, r.info.accumulator, idx, v

    want = [run(X, Y) for X, Y in pairs]
    bad = []

    def worker(seed):
        order = np.random.default_rng(seed).permutation(len(pairs))
        for k in order:
            got = run(*pairs[k])
            if got[:2] != want[k][:2] or not all(np.array_equal(a, b)
                                                 for a, b in zip(got[2], want[k][2])):
                bad.append(k)
            elif not np.allclose(got[3], want[k][3], rtol=1e-5, atol=0):
                bad.append(k)

    for _ in range(2):
        ts = [threading.Thread(target=worker, args=(s,)) for s in range(4)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        sptc.lib().sptc_trim_cache()
    worker(9)
    assert not bad
