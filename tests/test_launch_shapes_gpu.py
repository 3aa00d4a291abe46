"""The launch shapes chosen by rule (one-launch rounds with a link's partners split
over wavefronts, the pair workgroup size, rho_k beside or after the pair kernel)
against a fixed shape of three launches: the same draws, so the same accept flags
and, bit for bit, the same positions; the action terms of every attempt to 1e-12
of their size (their partner sums associate differently).  Sizes at the edges of
the splits: 64, 128 and 256 partners a wavefront, odd ones, and replicas that
exceed one residency wave."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def david(n, m):
    return system.config_c2(n_part=n, n_bead=m, n_level=2, k_shell=20.5, n_grid=400)


CASES = {
    "bare_1x4": ([lambda: system.config_c1(n_part=1, n_bead=4, n_level=1)], 1),
    "bare_64x9": ([lambda: system.config_c1(n_part=64, n_bead=9, n_level=3)], 2),
    "david_65x16": ([lambda: david(65, 16)], 1),
    "david_129x8": ([lambda: david(129, 8)], 3),
    "david_257x8": ([lambda: david(257, 8)], 2),
    "bare_16x16_300": ([lambda: system.config_c1(n_part=16, n_bead=16)], 300),
    "mixed": ([lambda: system.config_c1(n_part=130, n_bead=8), lambda: david(17, 12)], 5),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_shapes_by_rule_keep_the_chain(monkeypatch, name):
    kinds, replicas = CASES[name]
    base = [k() for k in kinds]
    systems = [base[r % len(base)] for r in range(replicas)]
    got = []
    for fixed in (False, True):
        for k, v in (("SPIMC_ONE_LAUNCH", "0"), ("SPIMC_FORK", "0"), ("SPIMC_PAIR_BLOCK", "1024")):
            if fixed:
                monkeypatch.setenv(k, v)
        with abi.Engine(systems, seed=21) as e:
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
