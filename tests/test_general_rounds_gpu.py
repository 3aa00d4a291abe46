"""One-launch rounds on tables in global memory (tabulated Ilkka actions, and every
action where the tables are not staged in LDS) against three launches: the same
draws, accept flags and, bit for bit, positions; the action terms to 1e-12 of their
size (partner sums associate differently).  Sizes at the edges of the partner
ranges (64 a wavefront, two ranges a link), axes that fit the LDS and axes that are
searched in global memory, and a batch with two rho_k items a workgroup and more."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def wide(n, m):
    s = system.config_ilkka(n_part=n, n_bead=m, n_level=2)
    return system.ilkka_ewald(s, alpha=5.0 / s.L, n_x=700, n_y=500)


CASES = {
    "ilkka_2x4": ([lambda: system.config_ilkka(n_part=2, n_bead=4, n_level=1)], 1, True),
    "ilkka_64x9": ([lambda: system.config_ilkka(n_part=64, n_bead=9)], 2, True),
    "ilkka_65x16": ([lambda: system.config_ilkka(n_part=65, n_bead=16)], 3, True),
    "ilkka_129x8": ([lambda: system.config_ilkka(n_part=129, n_bead=8)], 2, True),
    "ilkka_16x32_100": ([lambda: system.config_ilkka(n_part=16, n_bead=32)], 100, True),
    "ilkka_wide": ([lambda: wide(31, 12)], 2, True),
    "ilkka_and_bare": ([lambda: system.config_ilkka(n_part=33, n_bead=8), lambda: system.config_c1(n_part=70, n_bead=12)], 5,
                       True),
    "david_global": ([lambda: system.config_c2(n_part=130, n_bead=16, n_level=2, k_shell=20.5, n_grid=400)], 2, False),
    "bare_1_global": ([lambda: system.config_c1(n_part=1, n_bead=8, n_level=2)], 2, False),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_one_launch_from_global_tables_keeps_the_chain(monkeypatch, name):
    kinds, replicas, staged = CASES[name]
    if not staged:
        monkeypatch.setenv("SPIMC_PAIR_LDS", "0")
    base = [k() for k in kinds]
    systems = [base[r % len(base)] for r in range(replicas)]
    got = []
    for launches in ("2", "0"):
        monkeypatch.setenv("SPIMC_ONE_LAUNCH", launches)
        with abi.Engine(systems, seed=22) as e:
            for r, s in enumerate(systems):
                e.upload(system.random_path(s, seed=r, spread=0.1), r=r)
            e.trace(True)
            out = []
            for fn, n in ((e.bisect, 12), (e.displace, 5), (e.bisect, 7)):
                out.append(fn(n))
                out += [e.trace_read(n, r=r) for r in (0, replicas - 1)]
            out += [e.download(r) for r in (0, replicas // 2, replicas - 1)]
            got.append(out)
    for a, b in zip(*got):
        if a.shape[-1] == abi.TRACE_WORDS and a.ndim == 2 and a.dtype == np.float64:
            assert np.array_equal(np.isnan(a), np.isnan(b))
            a, b = np.nan_to_num(a), np.nan_to_num(b)
            assert np.abs(a - b).max() <= 1e-12 * max(1.0, np.abs(b).max())
        else:
            assert np.array_equal(a, b)
