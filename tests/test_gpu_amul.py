"""unap_hip_ldu_spmv and its allocation-free form against the oracle bit for
bit: host and device vectors, in place, and on partly overlapping vectors."""
import numpy as np
import pytest

from unap_amd import hip, meshgen

pytestmark = pytest.mark.gpu


class _At:
    """n doubles at an address inside another device array."""

    def __init__(self, a, first, n):
        self.base, self.ptr, self.n = a, a.data_ptr() + 8 * first, n

    def data_ptr(self):
        return self.ptr


@pytest.mark.parametrize("c,N", [(2, 1), (2, 24), (3, 17)])
def test_amul_vectors(oracle, c, N):
    s = meshgen.config_system(c, N)
    A = hip.LduMatrix.from_system(s)
    x = np.random.default_rng(5).uniform(-1, 1, s.n)
    want = oracle.matrix(s).spmv(x)
    assert np.array_equal(A.spmv(x), want)
    for call in (lambda a, b: A.spmv(a, out=b), A.spmv_noalloc):
        xd, out = hip.DeviceArray.from_numpy(x), hip.DeviceArray(s.n)
        call(xd, out)
        assert np.array_equal(out.numpy(), want) and np.array_equal(xd.numpy(), x)
        call(xd, xd)
        assert np.array_equal(xd.numpy(), want)
        both = hip.DeviceArray.from_numpy(np.concatenate([x, np.zeros(3)]))
        call(_At(both, 0, s.n), _At(both, 3, s.n))  # y three doubles after x
        assert np.array_equal(both.numpy()[3:], want)
