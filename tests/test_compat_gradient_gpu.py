"""The reference's finite-difference gradient with a bead's partners shared by a
workgroup against the kernel with a thread per bead, which forms every link action
whole.  Both are central
differences of the same actions at the same points; terms that cancel in the
difference leave rounding of a few 1e-16 of a link action over 2 eps = 2e-4, far
below 1e-9 of the largest component.  Sizes at the edges of the particle tiles
and partner groups, paths whose pairs cross half the box within eps, and a
replica of every pair action in one context; the virial energy built on it."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def david(n, m, n_order=2):
    s = system.config_c2(n_part=n, n_bead=m, n_level=1, k_shell=20.5, n_grid=400)
    return system.david_ewald(s, alpha=7.0 / s.L, n_grid=400, n_order=n_order)


CASES = {
    "bare_1x2": lambda: [system.config_c1(n_part=1, n_bead=2, n_level=1)],
    "bare_2x2": lambda: [system.config_c1(n_part=2, n_bead=2, n_level=1)],
    "bare_65x7": lambda: [system.config_c1(n_part=65, n_bead=7, n_level=1)],
    "bare_130x40": lambda: [system.config_c1(n_part=130, n_bead=40, n_level=1)],
    "bare_1030x2": lambda: [system.config_c1(n_part=1030, n_bead=2, n_level=1)],
    "david_64x6": lambda: [david(64, 6)],
    "david_33x5_order1": lambda: [david(33, 5, 1)],
    "david_33x5_order3": lambda: [david(33, 5, 3)],
    "mixed": lambda: [system.config_c1(n_part=20, n_bead=6, n_level=2), david(31, 9)],
}


def run(monkeypatch, systems, paths, lds):
    monkeypatch.setenv("SPIMC_PAIR_LDS", lds)
    with abi.Engine(systems) as e:
        for i, p in enumerate(paths):
            e.upload(p, r=i)
        e.obs_configure(energy=abi.ENERGY_VIRIAL_COMPAT)
        e.obs_accumulate(abi.OBS_ENERGY)
        ids = range(len(systems))
        return [e.gradient(abi.GRAD_PAIR_SHORT, compat=True, r=i) for i in ids], [e.obs_read(abi.OBS_ENERGY, i)[0] for i in ids]


@pytest.mark.parametrize("edge", [False, True])
@pytest.mark.parametrize("name", sorted(CASES))
def test_lds_differences_match_global(monkeypatch, name, edge):
    systems = CASES[name]()
    paths = [system.random_path(s, seed=80 + i, spread=0.2) for i, s in enumerate(systems)]
    if edge:
        # the first particles' separations straddle half the box, at one slice and between two
        for s, p in zip(systems, paths):
            if s.n_part > 1:
                p[0, :, 1] = p[0, :, 0] + 0.5 * s.L + 3e-5
                p[1, ::2, 1] = p[1, ::2, 0] + 0.5 * s.L - 6e-5
    print(f"case {name} edge {edge}", flush=True)
    got, e_got = run(monkeypatch, systems, paths, "1")
    ref, e_ref = run(monkeypatch, systems, paths, "0")
    for a, b in zip(got, ref):
        assert np.abs(a - b).max() <= 1e-9 * max(1.0, np.abs(b).max())
    for a, b in zip(e_got, e_ref):
        assert np.allclose(a, b, rtol=1e-9, atol=0)
