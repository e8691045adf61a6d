"""A steady run's first-order start, whose iterations evaluate the second-order norms and step in one
call, by the routes its ordinary test does not take: with the step replayed from a graph, and on a mesh
whose largest cell has too many faces for the fused face kernel; against the oracle's run, bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

import cases
from autan_amd import mesh as meshes
from autan_amd import steady
from oracle.oracle import Oracle

N, BLOCK = 22, 20  # cells along an edge, and of the block in its middle that is one cell


def write_mesh(path) -> None:
    """An N^3 grid of the unit cube whose inner BLOCK^3 cells are one: 6 BLOCK^2 = 2400 faces, of which
    the fused kernel's LDS holds neither fp64's nor fp32's fluxes."""
    lo = (N - BLOCK) // 2
    ids = np.arange(N**3).reshape(N, N, N)
    inner = (slice(lo, lo + BLOCK),) * 3
    ids[inner] = ids[lo, lo, lo]
    _, ids = np.unique(ids, return_inverse=True)
    ids = ids.reshape(N, N, N)
    point = lambda i, j, k: i + (N + 1) * (j + (N + 1) * k)  # noqa: E731
    inside, outside = [], []
    for axis in range(3):
        a, b = (axis + 1) % 3, (axis + 2) % 3
        for at in np.ndindex(*[N + 1 if d == axis else N for d in range(3)]):
            corners = []
            for da, db in ((0, 0), (1, 0), (1, 1), (0, 1)):  # normal along +axis
                p = list(at)
                p[a] += da
                p[b] += db
                corners.append(point(*p))
            right = at
            left = tuple(v - (d == axis) for d, v in enumerate(at))
            if at[axis] == 0:
                outside.append((int(ids[right]), corners[::-1]))
            elif at[axis] == N:
                outside.append((int(ids[left]), corners))
            elif ids[left] != ids[right]:
                lc, rc = int(ids[left]), int(ids[right])
                inside.append((lc, rc, corners) if lc < rc else (rc, lc, corners[::-1]))
    inside.sort(key=lambda f: f[:2])
    head = "FoamFile\n{{\n version 2.0;\n format ascii;\n class {};\n object {};\n}}\n"

    def put(name, cls, rows):
        (path / name).write_text(head.format(cls, name) + f"{len(rows)}\n(\n" + "\n".join(rows) + "\n)\n")

    x = np.linspace(0.0, 1.0, N + 1)
    used = sorted({p for f in inside for p in f[2]} | {p for f in outside for p in f[1]})
    new = {p: q for q, p in enumerate(used)}
    xyz = [(p % (N + 1), p // (N + 1) % (N + 1), p // (N + 1) ** 2) for p in used]
    put("points", "vectorField", ["({:.17g} {:.17g} {:.17g})".format(*(x[i] for i in q)) for q in xyz])
    faces = [f[2] for f in inside] + [f[1] for f in outside]
    put("faces", "faceList", ["4(" + " ".join(str(new[p]) for p in f) + ")" for f in faces])
    put("owner", "labelList", [str(f[0]) for f in inside] + [str(f[0]) for f in outside])
    put("neighbour", "labelList", [str(f[1]) for f in inside])
    (path / "boundary").write_text(head.format("polyBoundaryMesh", "boundary") + "1\n(\n all\n {\n type patch;\n"
                                   f" nFaces {len(outside)};\n startFace {len(inside)};\n }}\n)\n")


def block_case(path) -> cases.Case:
    write_mesh(path)
    c = cases.tets_case(1, flux="hllc")
    m = meshes.read_polymesh(path)
    kinds = np.full(m.n_boundary, meshes.STATE, np.int32)
    meshes.set_boundary_kinds(m, kinds)
    field = lambda x: cases.smooth_state(x, vel=(0.3, 0.05, -0.02))  # noqa: E731
    bc = cases._prim(field(m.face_centroids()[m.n_interior :]))
    return cases.Case("block", m, c.scheme, field(m.centroids()).reshape(-1), kinds.astype(np.float64), bc)


def test_the_block_is_one_cell(tmp_path):
    m = block_case(tmp_path).mesh
    assert m.n_cells == N**3 - BLOCK**3 + 1
    assert np.diff(m.cell_face_offsets).max() == 6 * BLOCK**2
    assert m.cell_volume.max() == pytest.approx((BLOCK / N) ** 3)


@pytest.mark.gpu
@pytest.mark.parametrize("policy", ["fp64", "fp32+acc64"])
@pytest.mark.parametrize("route", ["graph", "unfused"])
def test_a_first_order_start_is_the_oracles(route, policy, tmp_path):
    from autan_amd.stepper import DeviceStepper

    case = cases.tets_case(4) if route == "graph" else block_case(tmp_path)
    kw = dict(max_iterations=20 if route == "graph" else 6, level_rule=False)
    ora = Oracle(case.mesh, case.scheme, policy, case.bc_kind, case.bc, case.source)
    target = cases.OracleTarget(ora, case.u)
    with DeviceStepper(case.mesh, case.scheme, policy, case.bc_kind, case.bc, case.source) as dev:
        if route == "graph":
            dev.tune("graph", 1)
        elif policy == "fp32+acc64":
            with pytest.raises(RuntimeError, match="fused face kernel"):
                dev.tune("face_stage", 1)
        dev.upload(case.u)
        got = steady.solve(dev, **kw)
        want = steady.solve_with(target, **kw)
        assert got.iterations == want.iterations and got.first_order_steps == want.first_order_steps > 0
        np.testing.assert_array_equal(got.history, want.history)
        np.testing.assert_array_equal(got.provisional, want.provisional)
        np.testing.assert_array_equal(dev.download(), target.u)
        # The stepper's order and boundary values are the run's last step's.
        np.testing.assert_array_equal(dev.residual(target.u).reshape(-1), ora.residual(target.u).reshape(-1))
        names = dev.profile(1, 0.5, True)["kernels"]
        assert ("gather" in names) == (route == "unfused")
