"""Schedules that were replaced stay selectable by name, on the grids they took, and run the schedule
that took their place."""

import numpy as np
import pytest

from nrpy_amd import initial_data as ID

pytestmark = pytest.mark.gpu

RHS, RICCI = 0, 1
FD4_RHS = ["p1_lb1_sl_lf_pf16_u32_w2", "p1_lb1_sj_L16x8x2x1_d3_dma_rb1", "p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8",
           "p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub", "p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub_mi"]
FD4_RICCI = ["r1_lb1_pf16_u32", "r1_lb1_sj_L16x4x4x1_d2_dma_xcd", "r1_lb1_sj_L16x8x2x1_d3_dma_rb1",
             "r1_lb1_sj_L16x8x2x1_d3_dma_rb1_mi"]
RETIRED = {
    (1, 4, 4, False): {RHS: ["p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub_mi"],
                       RICCI: ["r1_lb1_sj_L16x4x4x1_d2_dma_xcd", "r1_lb1_sj_L16x8x2x1_d3_dma_rb1_mi"]},
    (2, 6, 0, True): {RHS: ["p1_lb1_sj_L16x4x4x1_d4_dma_rb1_io_pg_ub_sa_lr40_di_mi_xcd_blk",
                            "p1_lb1_sj_L16x4x4x1_d3_dma_rb1_io_pg_ub_mi_xcd"],
                      RICCI: ["r1_lb1_sj_L16x4x4x1_d3_dma_rb1_io_pg2_mi_xcd",
                              "r1_lb1_sj_L16x4x4x1_d3_dma_rb1_io_pg_lr40_mi_xcd"]},
    (2, 4, 0, True): {RHS: FD4_RHS, RICCI: FD4_RICCI},
}


def _cfg(build, Nxx):
    from nrpy_amd.runtime import PatchConfig

    coord, order, sym, ko = build
    return PatchConfig(coord=coord, Nxx=Nxx, fd_order=order, symmetry_axes=sym, enable_KO=ko, grid_physical_size=10.0,
                       SINHW=0.4, eta=2.0)


@pytest.mark.parametrize("build", list(RETIRED))
def test_retired_names_run_the_preferred_schedule(hip, build):
    from nrpy_amd.runtime import BHaHError, Patch

    P = Patch(_cfg(build, (18, 8, 4)), tuned=False)
    odd = Patch(_cfg(build, (17, 8, 4)), tuned=False)
    for kind, names in RETIRED[build].items():
        preferred = P.schedule(kind)
        for name in names:
            assert name not in P.schedules(kind)
            P.select_schedule(kind, 0)
            P.select_schedule(kind, name)
            assert P.schedule(kind) == preferred
            before = odd.schedule(kind)
            if "_dma" in name:  # refused on odd rows, as the schedule itself was
                with pytest.raises(BHaHError, match="even Nx0"):
                    odd.select_schedule(kind, name)
            else:
                odd.select_schedule(kind, name)
            assert odd.schedule(kind) == before
        with pytest.raises(ValueError, match="no schedule"):
            P.select_schedule(kind, "r9_lb1")


def test_retired_names_in_an_ensemble(hip):
    import torch
    from nrpy_amd.runtime import Ensemble

    build = (1, 4, 4, False)
    got = []
    for names in (None, RETIRED[build]):
        E = Ensemble([_cfg(build, N) for N in [(24, 6, 2), (16, 8, 2)]])
        for kind in (RHS, RICCI):
            E.select_schedule(kind, names[kind][-1] if names else E.schedules(kind)[-1])
            assert E.choice[kind] == len(E.schedules(kind)) - 1
        for P, st in zip(E.members, E.states):
            y = ID.brill_lindquist(1, P.xx(), 10.0, 0.4, (0.5, 0.5), (0, 0, 0.5), (0, 0, -0.5))
            st.y_n.copy_(torch.from_numpy(np.ascontiguousarray(y)))
            P.apply_bcs_outerextrap_and_inner(st.y_n)
        E.steps(2)
        torch.cuda.synchronize()
        got.append([st.y_n.clone() for st in E.states])
    assert [torch.equal(a, b) for a, b in zip(*got)] == [True, True]


def test_stored_table_with_an_unknown_name_warns(hip, monkeypatch):
    from nrpy_amd import autotune
    from nrpy_amd.runtime import Patch

    build = (1, 4, 4, False)
    P = Patch(_cfg(build, (24, 6, 2)), tuned=False)
    table = {"rhs": "p9_lb1", "ricci": RETIRED[build][RICCI][0], "tile": [64, 4]}
    monkeypatch.setattr(autotune, "load_choice", lambda cfg: table)
    before = P.schedule(RHS), P.schedule(RICCI)
    P.select_schedule(RICCI, 0)
    with pytest.warns(UserWarning, match="p9_lb1"):
        autotune.apply_tuned(P)
    assert (P.schedule(RHS), P.schedule(RICCI)) == before


def test_refusals_keep_their_errors(hip):
    from nrpy_amd.runtime import CARTESIAN, SYSTEM_WAVE, BHaHError, Patch, PatchConfig

    W = Patch(PatchConfig(system=SYSTEM_WAVE, coord=CARTESIAN, Nxx=(4, 4, 4), fd_order=4, symmetry_axes=0,
                          grid_physical_size=10.0, wavespeed=1.0))
    with pytest.raises(BHaHError, match="not a BSSN patch"):
        W.select_schedule(RHS, "p1_lb1")
    P = Patch(_cfg((1, 4, 4, False), (24, 6, 2)), tuned=False)
    with pytest.raises(BHaHError, match="unknown kernel kind"):
        P.select_schedule(7, "p1_lb1")
    with pytest.raises(BHaHError, match="out of range"):
        P.select_schedule(RHS, len(P.schedules(RHS)))
