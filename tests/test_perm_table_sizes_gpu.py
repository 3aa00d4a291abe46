"""The cycle table at the edges of its forms, replayed from the CPU oracle's draws:
every n_perm_part (all types of a subset at once up to 4, a type at a time
above), fewer subsets than threads, one subset, the largest replica whose table
sits in LDS and one past it.  Accept flags, positions and the wrap permutation
must match bit for bit: the table's sums only choose entries and decide."""
import numpy as np
import pytest

from oracle_ffi import Oracle
from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu

SIZES = [(2, 1, 0), (2, 2, 1), (3, 3, 0), (4, 4, 1), (5, 5, 0), (6, 6, 1), (7, 4, 0), (8, 5, 1), (7, 6, 0), (13, 4, 1),
         (33, 3, 0), (120, 2, 1), (140, 2, 0)]


@pytest.mark.parametrize("n,k,balance", SIZES)
def test_table_sizes_replay_bit_exact(n, k, balance):
    s = system.config_c1(n_part=n, n_bead=8, r_s=0.6, n_level=2)
    pos = system.random_path(s, seed=n, spread=0.3)
    o = Oracle(s, seed=3 + k)
    o.upload(pos)
    o.perm_configure(2)
    o.perm_table_configure(k, balance)
    o.record(True)
    ref = o.perm_table(24)
    tape = o.recorded()
    print(f"n={n} k={k}: {int(ref.sum())} accepted, sigma {o.perm().tolist()[:16]}", flush=True)
    with abi.Engine(s, seed=1) as e:
        e.upload(pos)
        e.perm_configure(2)
        e.perm_table_configure(k, balance)
        e.tape_set(tape)
        got = e.perm_table(24)[0]
        assert e.tape_cursor() == len(tape)
        assert np.array_equal(got, ref)
        assert np.array_equal(e.perm(), o.perm())
        assert np.array_equal(e.download(), o.download())
