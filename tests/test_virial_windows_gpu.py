"""Kinetic::VirialEnergy over windows longer than the path, which go on around it:
just past it, whole turns, several turns and a part, more than 2^31 links; with and
without a permutation, whose cycles close after several turns.  Every bead is drawn
anywhere in the box, so the paths wind.  Against the CPU oracle's walk and, for the
longest window, the sums formed from a turn's: 1e-11 of the terms' size."""
import numpy as np
import pytest

from oracle_ffi import Oracle
from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def closed_form(s, pos, sigma, window):
    """(value, size of its terms) with a cycle's links laid out once and whole turns counted."""
    m, n = s.n_bead, s.n_part
    const, tot, size = n * m * 3 / (2.0 * s.tau) / window, 0.0, 0.0
    for p in range(n):
        labels = [p]
        while sigma[labels[-1]] != p:
            labels.append(int(sigma[labels[-1]]))
        x = np.concatenate([pos[:, :, q] for q in labels], axis=1).T
        d = np.roll(x, -1, axis=0) - x
        d -= np.rint(d / s.L) * s.L
        turns, rest = divmod(window, len(d))
        for b in range(m):
            whole = turns * d.sum(axis=0) + np.roll(d, -b, axis=0)[:rest].sum(axis=0)
            tot += whole @ d[b]
            size += np.abs(whole * d[b]).sum()
    f = 1.0 / (4.0 * s.lam * s.tau) / (window * s.tau)
    return const - f * tot, const + f * size


@pytest.mark.parametrize("n,m,cycle", [(1, 2, 1), (3, 5, 1), (3, 5, 3), (70, 5, 1), (70, 5, 4), (9, 33, 2)])
def test_windows_past_the_path(n, m, cycle):
    s = system.config_c1(n_part=n, n_bead=m, n_level=1)
    pos = np.random.default_rng(n + m).uniform(-s.L / 2, s.L / 2, (3, m, n))
    sigma = np.arange(n)
    sigma[:cycle] = np.roll(sigma[:cycle], -1)
    o = Oracle(s, seed=1)
    o.upload(pos)
    with abi.Engine(s, seed=1) as e:
        e.upload(pos)
        if cycle > 1:
            o.set_perm(sigma)
            e.set_perm(sigma)
        for w in (m - 1, m, m + 1, m + 2, 2 * m - 1, 2 * m, 3 * m + 1, cycle * m, cycle * m + 1, 2 * cycle * m + m, 2**31 + 3):
            want, size = closed_form(s, pos, sigma, w)
            if w < 2**31:
                assert abs(o.kinetic_virial_energy(w) - want) <= 1e-11 * size
            assert abs(e.kinetic_virial_energy(w) - want) <= 1e-11 * size, w
