"""The wave step's boundary forms: the one-launch extrapolation of a box, and the stages that form
the ghost values they read, on the smallest boxes (three interior points a
side) and on tiles with remainders."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(3, 3, 3), (5, 4, 3), (3, 67, 4), (64, 4, 3), (67, 9, 5)]


def _pair(oracle_lib, Nxx, seed):
    from nrpy_amd.runtime import CARTESIAN, SYSTEM_WAVE, Patch, PatchConfig

    P = Patch(PatchConfig(system=SYSTEM_WAVE, coord=CARTESIAN, Nxx=Nxx, fd_order=4, symmetry_axes=0,
                          grid_physical_size=10.0, wavespeed=1.0))
    O = oracle_lib.OracleGrid(0, Nxx, 4, 10.0)
    y = np.random.default_rng(seed).standard_normal((2, *P.Nx[::-1]))
    return P, O, np.ascontiguousarray(y)


@pytest.mark.parametrize("Nxx", SIZES)
def test_extrapolation_of_a_box_is_the_oracles(hip, oracle_lib, Nxx):
    """Same operations in the same order, none contracted: the same bits."""
    import torch

    P, O, y = _pair(oracle_lib, Nxx, 1)
    yd = torch.from_numpy(y).cuda()
    P.wave_apply_bcs(yd)
    O.wave_apply_bcs(y)
    assert np.array_equal(yd.cpu().numpy(), y)


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("Nxx", SIZES)
def test_wave_steps_match_oracle(hip, oracle_lib, Nxx, use_graph):
    """Three steps of random data (its ghost zones too, which only the first stage reads): each
    stage's rounding is within a few ulp of its largest value, which extrapolation (weights 3, 3,
    1 twice) and the stencil amplify by at most 50 a stage: 12 * 50 * 4 * 1.1e-16 < 1e-12."""
    import torch
    from nrpy_amd.runtime import MoLState

    P, O, y = _pair(oracle_lib, Nxx, 2)
    S = MoLState(P, torch.from_numpy(y.copy()).cuda())
    st = O.new_state(y, 2)
    for _ in range(3):
        O.wave_mol_step(st, P.dt)
    S.steps(3, P.dt, use_graph=use_graph)
    torch.cuda.synchronize()
    a, b = S.y_n.cpu().numpy(), st["y_n"]
    assert (np.abs(a - b).reshape(2, -1).max(1) / np.abs(b).reshape(2, -1).max(1)).max() < 1e-12
