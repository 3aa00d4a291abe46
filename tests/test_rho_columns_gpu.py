"""rho_k of a whole path by columns of k-vectors (and by single k-vectors where a list
has them sparse or twice) against the direct sum in numpy: 4 eps a particle and step of
the phase recurrences, from particle tiles' edges to k-vectors beyond one tile's LDS."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def lists():
    shell = system.config_c1(n_part=4, n_bead=4).k_n
    far = np.array([[n0, n1, n2] for n0 in (0, 1, 20) for n1 in (-18, 1) for n2 in range(-40, 41)], dtype=np.int32)
    sparse = np.array([[1, j, 11 + j] for j in range(12)] + [[0, 0, 1]], dtype=np.int32)
    return {"shell": shell, "far": far, "sparse": sparse, "twice": np.concatenate([shell[:9], shell[:3]])}


@pytest.mark.parametrize("n,m", [(1, 4), (63, 5), (64, 4), (66, 7), (130, 4)])
@pytest.mark.parametrize("kind", ["shell", "far", "sparse", "twice"])
def test_rho_of_a_path_is_the_direct_sum(n, m, kind):
    s = system.config_c1(n_part=n, n_bead=m, n_level=1)
    k = np.ascontiguousarray(lists()[kind])
    s.k_n = k
    s.v_long_k = np.full(len(k), 0.01)
    pos = system.random_path(s, seed=n, spread=0.2)
    with abi.Engine([s], seed=1) as e:
        e.upload(pos)
        rho = np.asarray(e.rho_k()).reshape(m, len(k))
    phi = np.einsum("kd,dmn->kmn", k.astype(np.float64), pos * (2 * np.pi / s.L))
    want = np.exp(1j * phi).sum(axis=2).T
    steps = np.abs(k).sum(axis=1).max() + 4
    assert np.abs(rho - want).max() <= 4 * np.finfo(float).eps * n * steps * max(1.0, np.abs(phi).max() / steps)
