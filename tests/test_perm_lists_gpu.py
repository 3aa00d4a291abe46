"""The permuting rounds' list kernels in one launch (few replicas) and one after the
other (many, where every proposal is listed: tables in global memory, cycle tables of
two): a replica's chain depends on its own index and seed only, so the first replicas
of a large context have the flags, permutations and paths of a small one, bit for bit."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def run(s, replicas, k):
    with abi.Engine([s] * replicas, seed=31) as e:
        for r in range(replicas):
            e.upload(system.random_path(s, seed=r, spread=0.2), r=r)
            e.perm_configure(2, r=r)
            if k:
                e.perm_table_configure(k, 0, r=r)
        acc = (e.perm_table if k else e.perm_bisect)(30)
        return [acc[:3]] + [f(r) for r in range(3) for f in (e.perm, e.download, e.rho_k)]


@pytest.mark.parametrize("name,k", [("ilkka", 0), ("bare", 2), ("bare", 1), ("bare", 0)])
def test_few_and_many_replicas(name, k):
    make = system.config_ilkka if name == "ilkka" else system.config_c1
    s = make(n_part=9, n_bead=8, n_level=2)
    few, at, past = run(s, 3, k), run(s, 40, k), run(s, 41, k)
    for a, b, c in zip(few, at, past):
        assert np.array_equal(a, b) and np.array_equal(a, c)
