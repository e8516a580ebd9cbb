"""Grid.to_c: the packed write gives the bytes of the field-by-field one, takes the values it takes
and raises what it raises (no GPU needed)."""
import numpy as np
import pytest

from asteriy_2d_amd import grid as G

STATE = [[1.2, 0.9, 0.8, 0.1], [0.7, 1.4, -0.6, -0.2], [1.1, 0.8, 0.2, 0.5], [0.9, 1.2, -0.1, -0.4]]
BASE = G.Grid.from_extent(300, 70, -1.0, 2.0, 1.0, gamma=1.4, krit=0.3, bc=(1, 2, 3, 0),
                          bc_state=STATE, bc_vclamp=(-0.2, 0.3, 0.1, -0.1), frozen_x0=0.1,
                          frozen_ax=0.2, frozen_ay=0.3)


@pytest.mark.parametrize("kw", [
    {}, dict(N=np.int64(40), M=np.int32(9)), dict(bc_state=np.array(STATE)),
    dict(bc_state=np.array(STATE, dtype=np.float32)), dict(gamma=np.float64(1.3), krit=1),
    dict(bc_state=[["1", "2", "-3e-1", "4"]] * 4), dict(bc_vclamp=("0.1", "0", "0", "0")),
    dict(bc_state={k: STATE[k] for k in range(4)}), dict(ho_lo=-np.inf, ho_hi=0.25),
    dict(bc_pulse=(0.3, 2.0, -1e30, 1e30))])
def test_same_bytes(kw):
    g = BASE.replace(**kw)
    assert bytes(g.to_c()) == bytes(g._fields_to_c())


@pytest.mark.parametrize("kw,error", [
    (dict(N=64.0), TypeError), (dict(M=None), TypeError), (dict(krit="0.3"), TypeError),
    (dict(gamma=None), TypeError), (dict(bc=(0, 1)), IndexError),
    (dict(bc_state=[[1.0, 2.0, 3.0]] * 4), IndexError), (dict(bc_vclamp=(0.0, 0.0)), IndexError),
    (dict(bc_state=[["one", 1, 0, 0]] * 4), ValueError)])
def test_same_errors(kw, error):
    with pytest.raises(error):
        BASE.replace(**kw).to_c()
