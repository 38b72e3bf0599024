"""Observables and samples on both sides of the sizes where their kernels change
(direct sums up to 20 qubits, block walks above; block prefix by waves from
2^13 blocks), against numpy on the same amplitudes."""
import numpy as np
import pytest

from damavand_amd import StateVector

pytestmark = pytest.mark.gpu


def random_state(n, seed, dtype="complex128"):
    rng = np.random.default_rng(seed)
    amp = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    amp[: 1 << (n - 3)] *= 0.0  # blocks without mass too
    amp /= np.linalg.norm(amp)
    s = StateVector(n, dtype)
    s.load(amp)
    return s, np.abs(amp if dtype == "complex128" else amp.astype(np.complex64).astype(complex)) ** 2


def signs(n, q):
    return 1.0 - 2.0 * ((np.arange(1 << n) >> q) & 1)


@pytest.mark.parametrize("n,n_pairs,dtype", [(3, 2, "complex128"), (9, 9, "complex64"), (11, 20, "complex128"),
                                             (20, 128, "complex128"), (21, 0, "complex128"), (21, 128, "complex64"),
                                             (22, 70, "complex128")])
def test_pair_observable(n, n_pairs, dtype):
    """Pairs inside the low 12 qubits, above them, across, in either order and of a qubit with itself."""
    s, p = random_state(n, n)
    if dtype == "complex64":
        s, p = random_state(n, n, dtype)
    rng = np.random.default_rng(7 + n)
    a, b = rng.standard_normal(n), rng.standard_normal(n_pairs)
    pairs = [tuple(int(x) for x in rng.integers(0, n, 2)) for _ in range(n_pairs)]
    z = [signs(n, q) for q in range(n)]
    h = sum(c * zq for c, zq in zip(a, z)) + sum(c * z[i] * z[j] for c, (i, j) in zip(b, pairs))
    # |error| <= (terms + log of the sum's length) roundings of at most sum |coefficients|
    tol = (n + n_pairs + 64) * 2.0 ** -52 * (np.abs(a).sum() + np.abs(b).sum())
    assert abs(s.expect_zz(a, pairs, b) - float(h @ p)) <= tol
    np.testing.assert_allclose(s.expect_z(), [float(zq @ p) for zq in z], atol=64 * 2.0 ** -52, rtol=0)


@pytest.mark.parametrize("n,wires", [(6, [5, 0]), (20, [19, 3, 11]), (21, [20, 0, 5, 6, 11, 12]),
                                     (22, [1, 21, 13, 7, 12, 0, 10, 9, 8, 4, 17, 2])])
def test_table_observable(n, wires):
    s, p = random_state(n, 50 + n)
    table = np.random.default_rng(n).standard_normal(1 << len(wires))
    idx = np.zeros(1 << n, dtype=np.int64)
    for j, q in enumerate(wires):
        idx |= ((np.arange(1 << n) >> q) & 1) << j
    assert abs(s.expect_diag(wires, table) - float(table[idx] @ p)) <= 64 * 2.0 ** -52 * np.abs(table).max()


@pytest.mark.parametrize("n", [12, 24, 25])
def test_samples_by_inverse_cdf(n):
    """2^0, 2^12 and 2^13 blocks.  A draw may differ from numpy's cumulative sum only where u lies within
    the sums' rounding (2^n terms in pieces, so below 1e-11) of an outcome's edge."""
    s, p = random_state(n, 90 + n)
    u = np.concatenate([np.random.default_rng(n).uniform(1e-9, 1, 400), [1.0, 1e-12]])
    got = s.sample_uniforms(u)
    cum = np.cumsum(p)
    want = np.searchsorted(cum, u * cum[-1], side="left")
    off = got != want
    edge = np.abs(cum[np.minimum(got[off], want[off])] - u[off] * cum[-1])
    assert np.all(p[got] > 0) and np.all(edge <= 1e-11), (off.sum(), edge.max(initial=0.0))


@pytest.mark.parametrize("n", [4, 13])
def test_a_zero_state_is_refused(n):
    s = StateVector(n)
    s.load(np.zeros(1 << n))
    with pytest.raises(Exception, match="could not sample"):
        s.sample(10, 1)
