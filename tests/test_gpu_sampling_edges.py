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


# both sides of 131072 shots; results of a few states and of every state
@pytest.mark.parametrize("n,shots,distinct", [(12, 5000, 2), (18, 140000, 3), (6, 4000, 64)])
def test_only_the_results_are_written(gpu, n, shots, distinct):
    """Entries of the caller's arrays beyond the distinct states stay as they are."""
    import ctypes

    from tyxonq_amd import _native as nat

    rng = np.random.default_rng(n)
    v = np.zeros(1 << n, dtype=np.complex64)
    v[rng.choice(1 << n, distinct, replace=False)] = 1.0
    psi, s = to_gpu(v), nat.Sampler(n, shots)
    size = min(shots, 1 << n)
    idx = np.full(size, 2 ** 64 - 3, dtype=np.uint64)
    cnt = np.full(size, -7, dtype=np.int64)
    nu = ctypes.c_int64(0)
    for seed in (1, 2):
        nat._check(nat.load().tqsv_sampler_run(s._h, nat._ptr(psi), shots, seed, idx.ctypes.data,
                                               cnt.ctypes.data, ctypes.byref(nu), nat.stream_ptr()))
        widx, wcnt = S.sample_counts(v, shots, seed)
        assert nu.value == len(widx) == distinct
        np.testing.assert_array_equal(idx[:distinct], widx)
        np.testing.assert_array_equal(cnt[:distinct], wcnt)
        assert (idx[distinct:] == 2 ** 64 - 3).all() and (cnt[distinct:] == -7).all()
    s.close()
