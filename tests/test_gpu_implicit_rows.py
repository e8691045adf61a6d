"""The implicit solve's rows (colours, slices of twelve rows, padded slots, the relaxations a sweep
leaves out) where they can go wrong: one solve on meshes of two to six colours, with colours that end
inside a slice, colours of fewer rows than one slice, rows of unlike lengths in a slice and runs of
small colours, bit for bit the oracle's."""

from __future__ import annotations

import numpy as np
import pytest

import cases
from autan_amd import mesh as meshes
from autan_amd.stepper import DeviceStepper
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

STATE = [meshes.STATE] * 6
# name: colours come from the mesh; tets1 has six cells, vortex7's odd period needs a third colour
MESHES = {
    "tets1": lambda: cases.tets_case(1),
    "tets2": lambda: cases.tets_case(2),
    "tets9": lambda: cases.tets_case(9),
    "vortex6": lambda: cases.vortex_case(6),
    "vortex7": lambda: cases.vortex_case(7),
    "hex": lambda: cases.fixture_case("hex", flux="hllc", kinds_by_zone=STATE),
    "hybrid": lambda: cases.fixture_case("hybrid", flux="hllc", kinds_by_zone=STATE),
    "tet-gmsh": lambda: cases.fixture_case("tet-gmsh", flux="hllc", kinds_by_zone=STATE),
}


@pytest.mark.parametrize("policy", ["fp64", "fp32+acc64"])
@pytest.mark.parametrize("name", list(MESHES))
def test_one_solve_on_uneven_colours_is_the_oracles(name, policy):
    c = MESHES[name]()
    print(f"implicit rows {name} {c.mesh.n_cells} cells {policy}", flush=True)
    second = bool(c.scheme.second_order)
    with DeviceStepper(c.mesh, c.scheme, policy, c.bc_kind, c.bc, c.source) as dev:
        dev.upload(c.u)
        dev.implicit_evaluate()
        rep = dev.implicit_solve(100.0)
        u_dev, colours = dev.download(), dev.implicit_colours()
    ora = orc.Oracle(c.mesh, c.scheme, policy, c.bc_kind, c.bc, c.source)
    parts = ora.residual_and_jacobian(c.u)
    u_ora, _, want, col = orc.implicit_solve(c.mesh, parts, ora.spectral_radius(), 100.0, c.scheme.gamma, c.u, oracle=ora,
                                             second=second)
    np.testing.assert_array_equal(colours, col)
    assert rep == want
    np.testing.assert_array_equal(u_dev, u_ora)
