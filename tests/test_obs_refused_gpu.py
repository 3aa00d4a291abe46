"""A refused obs_configure leaves the observables as they were, also the size of the
g(r) histogram that obs_read returns."""
import numpy as np
import pytest

from simpimc_amd import abi, system

pytestmark = pytest.mark.gpu


def test_refused_configuration_keeps_the_histogram():
    s = system.config_c1(n_part=8, n_bead=8, n_level=2)
    with abi.Engine(s) as e:
        e.upload(system.random_path(s, seed=1, spread=0.2))
        e.obs_configure(gr_n_r=200)
        e.obs_accumulate(abi.OBS_GR)
        want = e.obs_read(abi.OBS_GR)
        for bad in (dict(virial_window=9), dict(gr_n_r=1), dict(energy=7)):
            with pytest.raises(abi.SpimcError):
                e.obs_configure(**bad)
            assert e.gr_n_r == 200
        got = e.obs_read(abi.OBS_GR)
        assert got[1] == want[1] == 1 and got[0].shape == (200,) and np.array_equal(got[0], want[0])
