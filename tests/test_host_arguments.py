"""Argument checks of the host entry's Python form (no GPU: a refused call
does not reach the library)."""
import numpy as np
import pytest

from simc_gfortran_amd import api
from simc_gfortran_amd import workloads as W


@pytest.mark.parametrize("column", ["x", "y", "z", "dxdz", "dydz", "fry"])
def test_run_host_refuses_a_short_input_column(column):
    """The library reads as many elements of every column as dpp has."""
    n = 1000
    ev = dict(W.generate(W.SHMS_C1, n, seed=1), fry=np.zeros(n))
    ev[column] = ev[column][: n - 1]
    ctx = api.Spectrometers.__new__(api.Spectrometers)
    ctx._h = None
    with pytest.raises(TypeError, match=column):
        ctx.run_host(5, ev, p_spec=6000.0, m2=W.ME ** 2)
