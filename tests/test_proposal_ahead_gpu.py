"""Bisections whose proposal is made while the one before it is decided: the chain is
the one of rounds that propose after the decision, bit for bit (flags, positions and
rho_k; the action terms to 1e-12 of their size, whose partner sums associate
differently).  Few particles make the next attempt move the particle that the
decision just committed (always, for one), windows from one moved slice to the
longest, stages of one attempt, and a changed level of one replica."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,level,replicas", [(1, 8, 2, 2), (2, 8, 1, 3), (2, 64, 6, 1), (3, 16, 3, 40), (33, 12, 3, 2),
                                                (65, 70, 5, 1)])
@pytest.mark.parametrize("pair", ["bare", "ilkka", "david"])
def test_proposals_ahead_keep_the_chain(monkeypatch, n, m, level, replicas, pair):
    make = {"bare": system.config_c1, "ilkka": system.config_ilkka,
            "david": lambda **k: system.config_c2(k_shell=20.5, n_grid=400, **k)}[pair]
    s = make(n_part=n, n_bead=m, n_level=level)
    got = []
    for launches in ("2", "0"):
        monkeypatch.setenv("SPIMC_ONE_LAUNCH", launches)
        with abi.Engine([s] * replicas, seed=23) as e:
            for r in range(replicas):
                e.upload(system.random_path(s, seed=r, spread=0.1), r=r)
            e.trace(True)
            out = []
            for fn, k in ((e.bisect, 1), (e.bisect, 25), (e.displace, 3), (e.bisect, 2)):
                out.append(fn(k))
                out += [e.trace_read(k, r=r) for r in (0, replicas - 1)]
            if level > 1:
                e.set_bisect_level(level - 1)
                out.append(e.bisect(9))
            out += [e.download(r) for r in (0, replicas - 1)]
            out += [e.rho_k(r=r) for r in (0, replicas - 1)]
            got.append(out)
    for a, b in zip(*got):
        if a.shape[-1] == abi.TRACE_WORDS and a.ndim == 2 and a.dtype == np.float64:
            assert np.array_equal(np.isnan(a), np.isnan(b))
            a, b = np.nan_to_num(a), np.nan_to_num(b)
            assert np.abs(a - b).max() <= 1e-12 * max(1.0, np.abs(b).max())
        else:
            assert np.array_equal(a, b)
