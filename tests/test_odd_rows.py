"""The staged schedules that take rows of any length (``_dmo``), at the sizes where their boxes
can go wrong: odd and even Nx0 and Nx1, partial tiles in every direction, the smallest grids,
and, on the CPU, the bounds of every access."""

import shutil

import numpy as np
import pytest

from nrpy_amd import initial_data as ID
from nrpy_amd.codegen.hip_gen import CONSTRAINTS_STAGED
from tests.test_kernels_on_cpu import _check, build, interior, rel_err, run, schedules

BUILDS = {
    "Spherical_sym2_KO0_fd4": dict(coord=1, fd_order=4, sym=4, KO=False, size=7.5, variant=0),
    "SinhSpherical_symnone_KO1_fd4": dict(coord=2, fd_order=4, sym=0, KO=True, size=64.0, variant=1),
    "SinhSpherical_symnone_KO1_fd6": dict(coord=2, fd_order=6, sym=0, KO=True, size=64.0, variant=1),
}
SIZES = {
    "Spherical_sym2_KO0_fd4": [(16, 4, 2), (17, 9, 2), (33, 12, 4), (18, 5, 6)],
    "SinhSpherical_symnone_KO1_fd4": [(16, 4, 4), (17, 9, 8), (21, 8, 10), (18, 11, 4)],
    "SinhSpherical_symnone_KO1_fd6": [(16, 4, 8), (19, 9, 10), (17, 12, 8), (18, 11, 10)],
}
CASES = [(t, n) for t in BUILDS for n in SIZES[t]]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("tag,Nxx", [(t, SIZES[t][1]) for t in BUILDS] + [("SinhSpherical_symnone_KO1_fd4", (18, 11, 4))])
def test_odd_row_schedules_on_cpu(oracle_lib, tag, Nxx):
    cands = [kc for kc in schedules(tag) if "_dmo_" in kc[1]]
    assert {k for k, _ in cands} == {"rhs", "ricci"}
    _check(oracle_lib, tag, cands, [(64, 4)], Nxx=Nxx)


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("tag,Nxx", [(t, n) for t in BUILDS for n in SIZES[t][:2]])
def test_staged_constraints_on_cpu(oracle_lib, tag, Nxx, tmp_path):
    """Bounds of every access, and H, M^i, M^2 and |Lambda| against the oracle: each is a sum that
    cancels to the constraint violation of the data (here of the order of its terms), so 1e-11 of
    the largest value, the bound of the GPU parity test."""
    b = BUILDS[tag]
    O = oracle_lib.OracleGrid(b["coord"], Nxx, b["fd_order"], b["size"], 0.2, variant=b["variant"])
    y = ID.smooth_perturbation(ID.brill_lindquist(b["coord"], O.xx, b["size"], 0.2), O.xx, 5)
    y = np.ascontiguousarray(y)
    O.apply_bcs_outerextrap_and_inner(y)
    aux = O.ricci(y)
    exe = build(tag, "constraints", CONSTRAINTS_STAGED, str(tmp_path))
    out = run(exe, O, "rhs", y, aux, (64, 4), str(tmp_path))[:6]
    assert rel_err(interior(out, O.NG), interior(O.constraints(y, aux), O.NG)).max() < 1e-11


@pytest.mark.gpu
@pytest.mark.parametrize("tag,Nxx", CASES)
def test_default_schedule_takes_every_size(hip, oracle_lib, tag, Nxx):
    """A new patch runs a staged schedule at any size and agrees with the oracle to 1e-12, the
    bound of every other schedule (max over the points relative to the gridfunction's maximum)."""
    import torch
    from nrpy_amd.runtime import KERNEL_RHS, KERNEL_RICCI, Patch, PatchConfig

    b = BUILDS[tag]
    P = Patch(PatchConfig(coord=b["coord"], Nxx=Nxx, fd_order=b["fd_order"], symmetry_axes=b["sym"], enable_KO=b["KO"],
                          grid_physical_size=b["size"], SINHW=0.2, eta=2.0))
    want = "_dmo_" if (P.Nx[0] & 1 or b["fd_order"] == 4) else "_dma_"
    assert want in P.schedule(KERNEL_RHS) and want in P.schedule(KERNEL_RICCI)
    O = oracle_lib.OracleGrid(b["coord"], Nxx, b["fd_order"], b["size"], 0.2, variant=b["variant"])
    y = ID.smooth_perturbation(ID.brill_lindquist(b["coord"], O.xx, b["size"], 0.2), O.xx, 5)
    y = np.ascontiguousarray(y)
    O.apply_bcs_outerextrap_and_inner(y)
    aux = O.ricci(y)
    yd, a, r = torch.from_numpy(y).cuda(), P.new_gfs(6), P.new_gfs()
    P.Ricci_eval(yd, a)
    P.rhs_eval(torch.from_numpy(aux).cuda(), yd, r)
    for got, ref in ((a, aux), (r, O.rhs(y, aux, O.params()))):
        s = (slice(None),) + (slice(O.NG, -O.NG),) * 3
        d, m = np.abs(got.cpu().numpy() - ref)[s], np.abs(ref)[s]
        assert (d.max((1, 2, 3)) / np.maximum(m.max((1, 2, 3)), 1e-300)).max() < 1e-12
