"""The whole-path estimators' workgroup splits against the global-table kernels and
the CPU oracle: odd and even N (the last partner distance counts half), one and
two particles, fewer pairs than threads, more slice ranges than slices, paths
whose pairs change image between slices, and replicas of very different sizes in
one launch.  Sums of the same terms in another order: 1e-11 relative."""
import numpy as np
import pytest

from oracle_ffi import Oracle
from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def david(n, m, n_order=2):
    s = system.config_c2(n_part=n, n_bead=m, n_level=1, k_shell=20.5, n_grid=400)
    return system.david_ewald(s, alpha=7.0 / s.L, n_grid=400, n_order=n_order)


CASES = {
    "bare_1x3": lambda: [system.config_c1(n_part=1, n_bead=3, n_level=1)],
    "bare_2x2": lambda: [system.config_c1(n_part=2, n_bead=2, n_level=1)],
    "bare_33x200": lambda: [system.config_c1(n_part=33, n_bead=200, n_level=1)],
    "bare_70x9": lambda: [system.config_c1(n_part=70, n_bead=9, n_level=1)],
    "david_64x16": lambda: [david(64, 16)],
    "david_65x7_order3": lambda: [david(65, 7, 3)],
    "mixed": lambda: [system.config_c1(n_part=130, n_bead=40, n_level=1), david(3, 2), david(40, 11, 1)],
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_whole_path_sums(monkeypatch, name):
    systems = CASES[name]()
    paths = []
    for i, s in enumerate(systems):
        p = system.random_path(s, seed=40 + i, spread=0.1)
        if s.n_part > 1:
            p[0, ::2, 1] = p[0, ::2, 0] + 0.49 * s.L  # changes image from slice to slice
            p[0, 1::2, 1] = p[0, 1::2, 0] + 0.51 * s.L
        paths.append(p)
    out = []
    for lds in ("1", "0"):
        monkeypatch.setenv("SPIMC_PAIR_LDS", lds)
        with abi.Engine(systems) as e:
            for i, p in enumerate(paths):
                e.upload(p, r=i)
            e.obs_configure(energy=abi.ENERGY_THERMAL, gr_n_r=64)
            which = abi.OBS_ENERGY | abi.OBS_SK | abi.OBS_GR
            e.obs_accumulate(which)
            e.obs_accumulate(which)
            ids = range(len(systems))
            out.append([np.concatenate([[e.d_action_d_beta(abi.ACTION_PAIR, r=i), e.potential(abi.ACTION_PAIR, r=i)],
                                        [e.kinetic_virial_energy(w, r=i) for w in (0, 1, systems[i].n_bead - 1)],
                                        *[e.obs_read(o, i)[0] for o in (abi.OBS_ENERGY, abi.OBS_SK, abi.OBS_GR)]])
                        for i in ids])
            e.obs_reset(which)
            assert all(e.obs_read(o, i)[1] == 0 and not e.obs_read(o, i)[0].any()
                       for i in ids for o in (abi.OBS_ENERGY, abi.OBS_SK, abi.OBS_GR))
    for i, s in enumerate(systems):
        o = Oracle(s, seed=1)
        o.upload(paths[i])
        vir = [o.kinetic_virial_energy(w) for w in (0, 1, s.n_bead - 1)]
        for got in (out[0][i], out[1][i]):
            assert np.allclose(got[2:5], vir, rtol=1e-11, atol=1e-11 * abs(vir[0]))
        assert np.allclose(out[0][i], out[1][i], rtol=1e-11, atol=1e-9 if s.n_part == 1 else 0)
