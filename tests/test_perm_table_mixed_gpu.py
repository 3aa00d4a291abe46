"""The cycle-table move of a small replica in a context that also holds a replica of
thousands of particles without a table: the same accept flags, permutation and path,
bit for bit, as in a context of its own; and a table configured later, larger than
the first, is taken up by the next stage."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def run(systems):
    with abi.Engine(systems, seed=9) as e:
        for r, s in enumerate(systems):
            e.upload(system.random_path(s, seed=r, spread=0.3), r=r)
        out = []
        e.perm_configure(2, r=0)
        e.perm_table_configure(3, 0, r=0)
        out.append(e.perm_table([24] + [0] * (len(systems) - 1))[0])
        e.perm_configure(2, r=1)
        e.perm_table_configure(2, 1, r=1)
        out += list(e.perm_table([12, 16] + [0] * (len(systems) - 2))[:2])
        for r in (0, 1):
            out += [e.perm(r), e.download(r)]
        return out


@pytest.mark.parametrize("n_large", [2000, 3600, 4096])
def test_table_beside_a_large_replica(n_large):
    small = [system.config_c1(n_part=8, n_bead=8, r_s=0.6, n_level=2), system.config_c1(n_part=120, n_bead=8, n_level=2)]
    large = system.config_c1(n_part=n_large, n_bead=2, n_level=1)
    for a, b in zip(run(small), run(small + [large])):
        assert np.array_equal(a, b)
