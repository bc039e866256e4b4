"""sptc_exclusive_scan_u64 at the sizes where the scan changes its launches: one
workgroup (up to 4096 items), workgroups that add up the tile
sums before their own (up to 512 tiles of 2048), a separate tile-sum scan
above.  Whole numbers: equal to numpy's."""
import ctypes

import numpy as np
import pytest

from gsparc_amd import sptc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 2, 63, 1024, 4095, 4096, 4097, 16383, 16384, 16385, 18432,
                               18433, 512 * 2048 - 1, 512 * 2048, 512 * 2048 + 1, 3_000_001])
def test_exclusive_scan_sizes(gpu, n):
    import torch
    rng = np.random.default_rng(n)
    a = rng.integers(0, 1 << 40, size=n, dtype=np.int64)
    d = torch.from_numpy(a).cuda()
    out = torch.full((n + 1,), -1, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    sptc.check(sptc.lib().sptc_exclusive_scan_u64(ctypes.c_void_p(d.data_ptr() if n else 0),
                                                  ctypes.c_void_p(out.data_ptr()), n, None))
    np.testing.assert_array_equal(out.cpu().numpy(), np.concatenate([[0], np.cumsum(a)]))
