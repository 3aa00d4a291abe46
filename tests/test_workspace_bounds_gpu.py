"""Gradients, the virial estimator of several replicas and rho_k downloads where the
workspaces hold every replica, one or two at a time, some of the rows only, and
nothing (the kernels that need none): the same rho_k bit for bit, the gradients to
1e-10 of the largest component (the sums associate differently, as between the
adjoint's forms), the energies formed from them to 1e-9."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def david(n, m):
    return system.config_c2(n_part=n, n_bead=m, n_level=1, k_shell=20.5, n_grid=400)


def results(monkeypatch, systems, limit):
    if limit is None:
        monkeypatch.delenv("SPIMC_WORK_BYTES", raising=False)
    else:
        monkeypatch.setenv("SPIMC_WORK_BYTES", str(limit))
    with abi.Engine(systems) as e:
        for i, s in enumerate(systems):
            e.upload(system.random_path(s, seed=80 + i, spread=0.1), r=i)
        ids = range(len(systems))
        e.obs_configure(energy=abi.ENERGY_VIRIAL_ADJOINT)
        e.obs_accumulate(abi.OBS_ENERGY)
        return ([e.gradient(t, r=i) for i in ids for t in (abi.GRAD_ALL, abi.GRAD_PAIR_LONG)], [e.rho_k(i) for i in ids],
                [e.obs_read(abi.OBS_ENERGY, i)[0] for i in ids])


# (of a replica of the first case the column weights take 129 kB, the link shares 225 kB
# and a row of its rho_k 3.1 kB)
@pytest.mark.parametrize("limit", [500_000, 250_000, 140_000, 10_000, 0])
@pytest.mark.parametrize("name", ["three", "mixed"])
def test_bounded_workspaces(monkeypatch, name, limit):
    systems = [david(65, 24)] * 3 if name == "three" else [david(65, 24), david(5, 3), david(130, 7)]
    want = results(monkeypatch, systems, None)
    got = results(monkeypatch, systems, limit)
    for a, b in zip(got[0], want[0]):
        assert np.abs(a - b).max() <= 1e-10 * max(1.0, np.abs(b).max())
    for a, b in zip(got[1], want[1]):
        assert np.array_equal(a, b)
    for a, b in zip(got[2], want[2]):
        assert np.allclose(a, b, rtol=1e-9)
