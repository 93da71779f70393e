"""Shot sampling at the limits of its kernels, against the oracle's sampler."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import sampling as S
from tests.gpu_util import to_gpu

pytestmark = pytest.mark.gpu


# 4096-amplitude blocks: one to 33 shots in one block (wave and dense kernel),
# groups of four, few distinct states; 131072 and one more shot (one and two
# copies); 5 blocks of 8192; a scan of 8192 counters
@pytest.mark.parametrize("n,shots,distinct", [
    (12, 1, 0), (12, 8, 0), (12, 9, 3), (12, 32, 2), (12, 32, 0), (12, 33, 0), (13, 64, 5),
    (11, 131072, 0), (18, 131072, 0), (18, 131073, 0), (25, 40000, 0)])
def test_counts_equal_oracle_at_limits(gpu, n, shots, distinct):
    from tyxonq_amd import _native as nat

    rng = np.random.default_rng(n + shots)
    v = (rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)).astype(np.complex64)
    if distinct:
        keep = rng.choice(1 << n, distinct, replace=False)
        w = np.zeros_like(v)
        w[keep] = v[keep]
        v = w
    s = nat.Sampler(n, shots)
    for seed in (1, 2):  # the sampler's buffers are used again
        idx, cnt = s.sample(to_gpu(v), shots, seed)
        widx, wcnt = S.sample_counts(v, shots, seed)
        np.testing.assert_array_equal(idx, widx)
        np.testing.assert_array_equal(cnt, wcnt)
    s.close()
