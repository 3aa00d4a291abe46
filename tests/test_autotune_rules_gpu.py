"""The autotuner measures the shape that the context chooses by rule beside its fixed
ones, so that a tuned context can keep it, also when it is tuned again; with the whole
shape fixed by the environment there is none to add."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu

FIXED = (("SPIMC_FORK", "0"), ("SPIMC_PAIR_BLOCK", "1024"), ("SPIMC_ONE_LAUNCH", "0"))


@pytest.mark.parametrize("make", [system.config_c1, system.config_ilkka])
def test_rules_are_a_candidate(monkeypatch, make):
    s = make(n_part=8, n_bead=8, n_level=2)
    tried = []
    for env in (FIXED[:0], FIXED[:2], FIXED):
        for k, v in env:
            monkeypatch.setenv(k, v)
        with abi.Engine([s] * 3, seed=4) as e:
            for r in range(3):
                e.upload(system.random_path(s, seed=r, spread=0.2), r=r)
            tried.append([e.autotune(3)["shapes_tried"] for _ in range(2)])
            e.bisect(5)
            assert np.isfinite(e.download(0)).all()
    assert tried[0] == tried[1] == [n + 1 for n in tried[2]]
