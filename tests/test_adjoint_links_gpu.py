"""The adjoint with a workgroup per link and the long range by columns, against the
per-particle kernel (each link evaluated from both of its beads) and the walk of
the runs: at the edges of the 64-particle tiles, with one and several workgroups
per link and segments per column set, the fewest slices and k-vectors, the
largest column the registers take and one past it, and replicas of different
sizes and pair actions in one launch.  The sums associate differently: 1e-10 of the largest component, as for
the other forms; repeated calls are equal bit for bit."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def david(n, m, k_shell=20.5):
    return system.config_c2(n_part=n, n_bead=m, n_level=1, k_shell=k_shell, n_grid=400)


CASES = {
    "bare_1x2": lambda: [system.config_c1(n_part=1, n_bead=2, n_level=1)],
    "bare_2x2": lambda: [system.config_c1(n_part=2, n_bead=2, n_level=1)],
    "bare_63x3": lambda: [system.config_c1(n_part=63, n_bead=3, n_level=1)],
    "bare_64x64": lambda: [system.config_c1(n_part=64, n_bead=64, n_level=1)],
    "david_65x5": lambda: [david(65, 5)],
    "david_129x2_k2": lambda: [david(129, 2, 2.5)],
    "david_257x130": lambda: [david(257, 130)],
    "bare_300x300": lambda: [system.config_c1(n_part=300, n_bead=300, n_level=1)],
    "david_7x2_k15": lambda: [david(7, 2, 230.5)],
    "david_7x2_k16": lambda: [david(7, 2, 260.5)],
    "mixed": lambda: [system.config_c1(n_part=70, n_bead=6, n_level=2), david(16, 9), system.config_c1(n_part=3, n_bead=40)],
}


def gradients(monkeypatch, systems, form, terms):
    monkeypatch.setenv("SPIMC_ADJ_PAIRS", form)
    if form == "0":
        monkeypatch.setenv("SPIMC_ADJ_RUNS", "1")
    else:
        monkeypatch.delenv("SPIMC_ADJ_RUNS", raising=False)
    with abi.Engine(systems) as e:
        for i, s in enumerate(systems):
            e.upload(system.random_path(s, seed=60 + i, spread=0.1), r=i)
        return [[e.gradient(terms, r=i) for i in range(len(systems))] for _ in range(2)]


@pytest.mark.parametrize("terms", [abi.GRAD_PAIR_SHORT, abi.GRAD_PAIR_LONG, abi.GRAD_ALL])
@pytest.mark.parametrize("name", sorted(CASES))
def test_links_match_per_particle(monkeypatch, name, terms):
    systems = CASES[name]()
    print(f"case {name} terms {terms}", flush=True)
    got = gradients(monkeypatch, systems, "2", terms)
    ref = gradients(monkeypatch, systems, "0", terms)[0]
    for a, b, r in zip(got[0], got[1], ref):
        assert np.array_equal(a, b)
        assert np.abs(a - r).max() <= 1e-10 * max(1.0, np.abs(r).max())
