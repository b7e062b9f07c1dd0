"""The RK pass and the radiation condition at the forms their dispatch has: points and pairs of
points, sources of a pair together or apart, every ghost-zone count and stencil radius."""

import os

import numpy as np
import pytest

from nrpy_amd import initial_data as ID

pytestmark = pytest.mark.gpu

FORMS = {
    # pairs, sources together / apart (odd rows, three ghost zones); single points (arrays that
    # are 8 bytes past a 16-byte boundary)
    "fd6_even": dict(coord=2, Nxx=(20, 12, 10), fd_order=6, sym=0, KO=True, off=0),
    "fd6_odd": dict(coord=2, Nxx=(21, 11, 10), fd_order=6, sym=0, KO=True, off=0),
    "fd4": dict(coord=2, Nxx=(18, 9, 8), fd_order=4, sym=0, KO=True, off=0),
    "fd6_even_unaligned": dict(coord=2, Nxx=(20, 12, 10), fd_order=6, sym=0, KO=True, off=1),
    "fd4_odd_unaligned": dict(coord=1, Nxx=(17, 7, 2), fd_order=4, sym=4, KO=False, off=1),
}


def _patch(c, separate, **kw):
    from nrpy_amd.runtime import Patch, PatchConfig

    cfg = PatchConfig(coord=c["coord"], Nxx=c["Nxx"], fd_order=c["fd_order"], symmetry_axes=c["sym"], enable_KO=c["KO"],
                      grid_physical_size=10.0, SINHW=0.4, eta=2.0, **kw)
    if separate:
        os.environ["BHAH_HIP_SEPARATE_INNER_BC"] = "1"
    try:
        return Patch(cfg)
    finally:
        os.environ.pop("BHAH_HIP_SEPARATE_INNER_BC", None)


def _state(P, y, off):
    """A MoLState whose arrays start ``off`` doubles past a 16-byte boundary."""
    import torch
    from nrpy_amd.runtime import MoLGridfunctions, MoLState

    S = MoLState(P, y.clone())
    if off:
        def moved(t):
            flat = torch.zeros(t.numel() + off, dtype=t.dtype, device=t.device)
            flat[off:].copy_(t.reshape(-1))
            return flat[off:].view(t.shape)

        S.y_n, S.y_run, S.k_odd, S.k_even, S.aux = (moved(t) for t in (S.y_n, S.y_run, S.k_odd, S.k_even, S.aux))
        assert S.y_n.data_ptr() % 16 == 8
        S.c = MoLGridfunctions(*(t.data_ptr() for t in (S.y_n, S.y_run, S.k_odd, S.k_even, S.aux)))
    return S


def _initial(P, seed=7):
    import torch

    xx = P.xx()
    y = ID.brill_lindquist(P.cfg.coord, xx, 10.0, 0.4, (0.5, 0.4), (0.1, 0.2, 0.5), (-0.1, 0, -0.6))
    yd = torch.from_numpy(np.ascontiguousarray(ID.smooth_perturbation(y, xx, seed, amplitude=2e-2))).cuda()
    P.apply_bcs_outerextrap_and_inner(yd)
    return yd


@pytest.mark.parametrize("name", list(FORMS))
def test_folded_pass_equals_the_separate_copy(hip, name):
    """The pass with the inner-parity condition folded in gives the state of the separate copy bit
    for bit: it takes the same values of k, and an inner ghost point's running sum is its
    source's with the parity sign."""
    import torch

    c = FORMS[name]
    PF, PS = _patch(c, False), _patch(c, True)
    y0 = _initial(PF)
    SF, SS = _state(PF, y0, c["off"]), _state(PS, y0, c["off"])
    SF.steps(3, PF.dt)
    SS.steps(3, PS.dt)
    torch.cuda.synchronize()
    assert torch.isfinite(SF.y_n).all() and not torch.equal(SF.y_n, y0)
    assert torch.equal(SF.y_n, SS.y_n)


@pytest.mark.parametrize("Nxx", [(24, 6, 2), (17, 7, 2), (18, 5, 4)])
@pytest.mark.parametrize("off", [0, 1])
def test_taped_step_keeps_inner_ghosts_of_k(hip, Nxx, off):
    """The tape of a step whose RK pass takes the inner-parity condition with it equals, bit for
    bit and inner ghost points of every k included, that of the separate copy."""
    import torch

    c = dict(coord=1, Nxx=Nxx, fd_order=4, sym=4, KO=False)
    PF, PS = _patch(c, False), _patch(c, True)
    y0 = _initial(PF)
    tapes, ends = [], []
    for P in (PF, PS):
        flat = torch.zeros(P.tape_doubles + off, dtype=torch.float64, device="cuda")
        y = y0.clone()
        P.MoL_step_forward_taped(y, PF.dt, flat[off:])
        torch.cuda.synchronize()
        tapes.append(flat)
        ends.append(y)
    assert torch.isfinite(tapes[0]).all() and torch.equal(*tapes) and torch.equal(*ends)


@pytest.mark.parametrize("name", ["fd6_odd", "fd4_odd_unaligned"])
@pytest.mark.parametrize("order", [2, 4, 6])
def test_radiation_lines_match_oracle(hip, oracle_lib, name, order):
    """Every ghost-zone count (3, 4) and stencil radius (1, 2, 3) of the line form, to the 1e-12
    the per-call boundary tests use (max over the points, relative to the gridfunction's)."""
    import torch

    c = FORMS[name]
    P = _patch(c, False, radiation_bc_fd_order=order)
    O = oracle_lib.OracleGrid(c["coord"], c["Nxx"], c["fd_order"], 10.0, 0.4, variant=0 if c["coord"] == 1 else 1)
    y = _initial(P)
    k = torch.randn(y.shape, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    ref = k.cpu().numpy().copy()
    O.apply_bcs_outerradiation_and_inner(np.ascontiguousarray(y.cpu().numpy()), ref, order)
    P.apply_bcs_outerradiation_and_inner(y, k)
    d = np.abs(k.cpu().numpy() - ref).reshape(24, -1).max(1) / np.abs(ref).reshape(24, -1).max(1)
    assert d.max() < 1e-12


# The forms that stream every array (more than 470,000 interior points): pairs whose sources lie apart
# (odd rows, three ghost zones) and together, single points, and without the folded inner condition
# (extrapolation boundary, separate copy).
STREAMED = {
    "fd6_odd": dict(coord=2, Nxx=(121, 65, 62), fd_order=6, sym=0, KO=True, off=0),
    "fd6_odd_unaligned": dict(coord=2, Nxx=(121, 65, 62), fd_order=6, sym=0, KO=True, off=1),
    "fd6_even": dict(coord=2, Nxx=(122, 64, 62), fd_order=6, sym=0, KO=True, off=0),
    "sym2_separate": dict(coord=1, Nxx=(480, 124, 8), fd_order=4, sym=4, KO=False, off=0, separate=True),
    "fd4_extrapolation": dict(coord=2, Nxx=(122, 64, 62), fd_order=4, sym=0, KO=True, off=0, outer_bc=1),
    "fd4_odd_extrapolation_unaligned": dict(coord=2, Nxx=(123, 65, 60), fd_order=4, sym=0, KO=True, off=1, outer_bc=1),
}


@pytest.mark.parametrize("name", list(STREAMED))
def test_streamed_pass_equals_the_single_calls(hip, name):
    """A step at the sizes where the pass streams, against the per-call functions with the RK4
    combinations in torch.  Each stage then differs by the rounding of a fused multiply-add (an
    ulp or two of its largest value), which a stage's right-hand side amplifies no further than the
    whole steps the parity tests compare to 1e-10; same bound."""
    import torch
    from nrpy_amd.runtime import OUTER_BC_EXTRAPOLATION

    c = STREAMED[name]
    kw = {"outer_bc": c["outer_bc"]} if "outer_bc" in c else {}
    assert not kw or kw["outer_bc"] == OUTER_BC_EXTRAPOLATION
    assert c["Nxx"][0] * c["Nxx"][1] * c["Nxx"][2] > 470000
    P = _patch(c, c.get("separate", False), setup_on_device=True, **kw)
    y = P.new_gfs()
    P.initial_data_brill_lindquist(y, 0.5, (0.1, 0.2, 0.5), 0.4, (-0.1, 0.0, -0.6))
    # terms of every kind alive: smooth waves over the grid, different in each gridfunction
    x = [torch.linspace(0.0, 1.0, n, dtype=torch.float64, device="cuda") for n in P.Nx]
    for g in range(24):
        y[g] += 1e-2 * torch.sin((2 + g % 3) * x[0] + g) * torch.cos((1 + g % 4) * x[1] + g)[:, None] \
            * torch.cos(2 * x[2] + g)[:, None, None]
    P.apply_bcs_outerextrap_and_inner(y)
    P.enforce_detgammabar_equals_detgammahat(y)
    S = _state(P, y, c["off"])
    S.steps(1, P.dt, use_graph=False)

    aux, k, stage, total = P.new_gfs(6), P.new_gfs(), y, y
    for w, a in ((1, 0.5), (2, 0.5), (2, 1.0), (1, None)):
        P.Ricci_eval(stage, aux)
        P.rhs_eval(aux, stage, k)
        if not kw:
            P.apply_bcs_outerradiation_and_inner(stage, k)
        total = total + (w * P.dt / 6.0) * k
        stage = total if a is None else y + (a * P.dt) * k
        P.enforce_detgammabar_equals_detgammahat(stage)
        if kw:
            P.apply_bcs_outerextrap_and_inner(stage)
            P.enforce_detgammabar_equals_detgammahat(stage)
    torch.cuda.synchronize()
    d = (S.y_n - stage).abs().reshape(24, -1).amax(1) / stage.abs().reshape(24, -1).amax(1)
    moved = (stage - y).abs().reshape(24, -1).amax(1) / stage.abs().reshape(24, -1).amax(1)
    print(name, "step against single calls", d.max().item(), "step against its start", moved.min().item())
    assert torch.isfinite(S.y_n).all() and moved.min() > 1e-8
    assert d.max() < 1e-10
