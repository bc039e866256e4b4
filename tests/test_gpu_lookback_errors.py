"""A look-back sort pass that gives up must fail every call that used it: its
output is not sorted.  SPTC_LOOKBACK_FAILS=1 sets the pass's error word though no
wait failed, so every kernel runs as always; each call form runs with and without
it in a process of its own."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
SCRIPT = r"""
import sys
sys.path[:0] = [sys.argv[1], sys.argv[2]]
import ctypes
import numpy as np
import torch
from gsparc_amd import sptc
from helpers import random_coo

rng = np.random.default_rng(1)
X = random_coo(rng, (300, 80, 50), 30_000)   # more than one sort tile, look-back sizes
Y = random_coo(rng, (50, 900), 20_000)
small = random_coo(rng, (30, 20, 50), 3000)  # operands of one tile: no look-back pass
v = random_coo(rng, (50,), 50)

def serve():
    srv = sptc.Server(budget_bytes=4 << 30)
    try:
        a, b = srv.add_tensor(X), srv.add_tensor(Y)
        srv.wait(srv.submit(a, b, [2], [0]))
    finally:
        srv.close()

def pairs():
    k = torch.randint(0, 1 << 40, (50_000,), dtype=torch.int64, device="cuda")
    f = torch.rand(50_000, device="cuda")
    sptc.check(sptc.lib().sptc_sort_pairs(ctypes.c_void_p(k.data_ptr()),
                                          ctypes.c_void_p(f.data_ptr()), 50_000, 40, 0, None))

forms = {
    "call": lambda: sptc.SpTC(X, Y, [2], [0]),
    "esc": lambda: sptc.SpTC(X, Y, [2], [0], dense_accumulator=-1),
    "count": lambda: sptc.SpTC(X, Y, [2], [0], dense_accumulator=-1, count_only=True),
    "plan": lambda: sptc.Plan(X, Y, [2], [0]),
    "batch": lambda: sptc.Batch([(X, v, [2], [0])], dense_accumulator=-1),
    "server": serve,
    "pairs": pairs,
    "small": lambda: sptc.SpTC(small, small, [2], [2]),
}
for name, f in forms.items():
    try:
        f()
        print("form", name, "ok", flush=True)
    except sptc.SpTCError as e:
        print("form", name, e.status, flush=True)
print("end", flush=True)
"""


def _forms(**env):
    p = subprocess.run([sys.executable, "-u", "-c", SCRIPT, os.path.dirname(HERE), HERE],
                       env=dict(os.environ, **env), stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=100)
    assert p.returncode == 0 and p.stdout.rstrip().endswith("end"), p.stdout[-3000:]
    return {ln.split()[1]: ln.split()[2] for ln in p.stdout.splitlines()
            if ln.startswith("form ")}


@pytest.mark.parametrize("product_sort", [False, True])
def test_failed_look_back_is_reported(gpu, product_sort):
    from gsparc_amd import sptc
    env = {"SPTC_PROD_SORT": "rows"} if product_sort else {}
    print(f"[look-back] {env}", flush=True)
    good = _forms(**env)
    assert set(good.values()) == {"ok"} and len(good) == 8
    bad = _forms(SPTC_LOOKBACK_FAILS="1", **env)
    assert bad.pop("small") == "ok"
    assert bad == {k: str(sptc.ERR_INTERNAL) for k in bad}
