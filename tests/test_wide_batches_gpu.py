"""Wide batches take other launch shapes than narrow ones (wavefronts of the bisection's
decision, pair workgroup sizes, splits of the whole-path sums, the long-range adjoint by
runs, no proposals ahead past their bound): a replica's chain depends on its own index
and seed only, so the first replicas of a wide context have the flags and paths
of a narrow one, bit for bit, and its estimators to rounding (1e-9: sums of the same
terms in another order)."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def david(n, m, level, n_grid=400):
    return system.config_c2(n_part=n, n_bead=m, n_level=level, k_shell=20.5, n_grid=n_grid)


CASES = {
    "two_wavefronts": (lambda: system.config_c1(n_part=4, n_bead=8, n_level=3), 1025),
    "four_wavefronts": (lambda: system.config_c1(n_part=4, n_bead=8, n_level=3), 1024),
    "two_links": (lambda: system.config_c1(n_part=5, n_bead=6, n_level=1), 700),
    "large_tables": (lambda: david(20, 8, 2, 2000), 300),
    "three_workgroups": (lambda: system.config_c1(n_part=149, n_bead=11, n_level=2), 70),
    "runs": (lambda: david(3, 64, 2), 260),
    "ahead_past_bound": (lambda: system.config_c1(n_part=2, n_bead=64, n_level=6), 4600),
}


def run(s, replicas):
    with abi.Engine([s] * replicas, seed=17) as e:
        for r in range(replicas):
            e.upload(system.random_path(s, seed=r % 5, spread=0.2), r=r)
        out = [[fn(n)[:3] for fn, n in ((e.bisect, 9), (e.displace, 4), (e.bisect, 5))], [e.download(r) for r in range(3)]]
        est = []
        for energy in (abi.ENERGY_THERMAL, abi.ENERGY_VIRIAL_ADJOINT, abi.ENERGY_VIRIAL_COMPAT):
            e.obs_configure(energy=energy, gr_n_r=32)
            e.obs_accumulate(abi.OBS_ENERGY | abi.OBS_SK | abi.OBS_GR)
            est += [e.obs_read(o, r)[0] for o in (abi.OBS_ENERGY, abi.OBS_SK, abi.OBS_GR) for r in range(3)]
        return out, est


@pytest.mark.parametrize("name", sorted(CASES))
def test_wide_and_narrow(name):
    make, replicas = CASES[name]
    s = make()
    (wide, est_w), (narrow, est_n) = run(s, replicas), run(s, 3)
    for a, b in zip(wide, narrow):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
    for a, b in zip(est_w, est_n):
        assert np.abs(a - b).max() <= 1e-9 * max(1.0, np.abs(b).max())
