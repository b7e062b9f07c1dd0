"""The stored autotuner tables: what they time and choose is what the build has, and the choice is
the fastest of what was timed."""

import json
import os

import pytest

from nrpy_amd import autotune
from nrpy_amd.codegen import hip_gen

TABLES = sorted(f for f in os.listdir(autotune.TABLE_DIR) if f.endswith(".json"))
BUILDS = {hip_gen.kernel_name_tag(v, order): cands for v, order, cands, _ in hip_gen.BSSN_BUILDS}


@pytest.mark.parametrize("name", TABLES)
def test_table_holds_the_build_and_its_fastest_choice(name):
    with open(os.path.join(autotune.TABLE_DIR, name)) as f:
        d = json.load(f)
    t = {}
    for k, ms in d["timings_ms"].items():
        kind, _, what = k.partition(":")
        t.setdefault(kind, {})[what] = ms
    for kind in ("rhs", "ricci"):
        assert sorted(t[kind]) == sorted(BUILDS[d["build"]][kind])
        assert d[kind] == min(t[kind], key=t[kind].get)
    shape, chosen = ("launch", "{0}x{1}:{2}") if "launch" in d else ("tile", "{0}x{1}")
    assert chosen.format(*d[shape]) == min(t[shape], key=t[shape].get)


@pytest.mark.gpu
def test_tuner_times_tiles_on_the_schedules_that_run_in_them(hip, monkeypatch):
    from nrpy_amd.runtime import KERNEL_RHS, KERNEL_RICCI, Patch, PatchConfig

    at_tile = []
    set_tile = Patch.set_tile

    def noted(P, x, y):
        at_tile.append((P.schedule(KERNEL_RHS), P.schedule(KERNEL_RICCI)))
        set_tile(P, x, y)

    monkeypatch.setattr(autotune, "apply_tuned", lambda P: None)
    monkeypatch.setattr(Patch, "set_tile", noted)
    out = autotune.tune(PatchConfig(coord=2, Nxx=(16, 8, 8), fd_order=6, symmetry_axes=0, enable_KO=True,
                                    grid_physical_size=10.0, SINHW=0.4, eta=2.0), reps=1, write=False,
                        log=lambda s: None)
    assert at_tile == [("p1_lb1", "r1_lb1")] * len(autotune.TILES)
    assert out["tile"] in [list(t) for t in autotune.TILES]


@pytest.mark.parametrize("Nxx", [(72, 12, 2), (151, 33, 10), (256, 64, 16)])
def test_phi_symmetric_plain_schedules_run_in_the_tile_their_table_chose(Nxx):
    """32x8: rows of 151 points fill 5 x 5 x 10 workgroups, one round of the 256 CUs; 64x4 takes 3 x 9
    x 10, two rounds (Ricci and right-hand side 80 against 136 us there; never slower elsewhere)."""
    from nrpy_amd.runtime import PatchConfig

    assert autotune.load_choice(PatchConfig(coord=1, Nxx=Nxx, fd_order=4, symmetry_axes=4))["tile"] == [32, 8]
