"""Faces whose moments are zero on a mesh with warped ones: the device leaves out their warp term where
zero_warp (autan_amd/csrc/device/kernels.hpp) finds it zero. That finding, restated here, against the
term itself (the oracle's body) over ordinary, extreme, infinite and NaN factors; and the device's residual
of states that hold such values against the oracle's."""

from __future__ import annotations

import numpy as np
import pytest

import cases
from autan_amd import mesh as meshes
from oracle import oracle as orc

MAX = np.finfo(np.float64).max


def zero_warp(w, gl, gr, gamma, pref) -> bool:
    """The device's test: every factor that the term multiplies by a zero, times zero, is zero."""
    vv = w[1] * w[1] + w[2] * w[2] + w[3] * w[3]
    rh = gamma / (gamma - 1.0) * (w[4] + pref) + 0.5 * w[0] * vv
    factors = np.concatenate([[vv, rh], w, gl, gr])
    return not np.isnan(factors * 0.0).any()


@pytest.mark.parametrize("seed", range(4))
def test_a_term_found_zero_is_zero(seed):
    """The momentum rho v_i is among the term's factors and not among the test's: the mean state's
    density is at most half the largest number, so for |v_i| <= 2 the product is finite, and beyond it is
    at most rho v_i^2 / 2, which is in the enthalpy density."""
    rng = np.random.default_rng(seed)
    pool = np.array([0.0, -0.0, 1e-320, 1e-3, 1.0, -1.4, 1.9999999, 2.0, -2.0000001, 3.0, 1e100, np.sqrt(MAX), -1e160,
                     MAX / 4, MAX / 2, np.nextafter(MAX / 2, 0.0), MAX, -MAX, np.inf, -np.inf, np.nan])
    found = 0
    with np.errstate(all="ignore"):
        for k in range(4000):
            top = [7, 10, 18, 21][k % 4]  # ordinary factors only, up to large ones, up to every one
            sides = rng.choice(pool[:top], (2, 5))
            if k % 3 == 0:
                sides[:, 0] = rng.choice([MAX / 2, MAX, 0.9 * MAX], 2)
            w = 0.5 * (sides[0] + sides[1])
            gl, gr = rng.choice(pool[: max(10, top - 3)], (2, 20))
            pref = rng.choice([0.0, 0.7])
            if not zero_warp(w, gl, gr, 1.4, pref):
                continue
            found += 1
            out = orc.warp(w, gl[:15], gl[15:], gr[:15], gr[15:], np.zeros(9), 1.4, pref)
            np.testing.assert_array_equal(out, 0.0, err_msg=f"{w} {gl} {gr}")
    assert found > 1000  # every ordinary draw, and the large ones that stay finite


@pytest.mark.gpu
@pytest.mark.parametrize("policy", ["fp64", "fp32+acc64"])
@pytest.mark.parametrize("second", [False, True])
@pytest.mark.parametrize("flux", ["roe", "hllc", "ausm+up"])
def test_residuals_beside_infinities_and_nan(flux, second, policy):
    from autan_amd.stepper import DeviceStepper

    case = cases.bump_case(16, 12, 8, flux=flux, second_order=second, limiter=second, hybrid=True)
    m = case.mesh
    kinds = np.full(m.n_boundary, meshes.STATE, np.int32)
    meshes.set_boundary_kinds(m, kinds)
    w = np.array([1.0, 0.5, 0.0, 0.0, 1.0 / 1.4])
    case.bc = cases.boundary_data(kinds, w)
    moment = m.face_moment.reshape(9, -1)[:, : m.n_interior]
    warped = moment.any(axis=0)
    assert warped.any() and not m.all_planar
    big = 1e300 if policy == "fp64" else 1e37
    dev = DeviceStepper(m, case.scheme, policy, kinds.astype(np.float64), case.bc, None)
    ora = orc.Oracle(m, case.scheme, policy, kinds.astype(np.float64), case.bc, None)
    # A cell with a warped face and a flat one, and a cell of flat ones alone.
    touched = np.zeros(m.n_cells, bool)
    touched[m.owner[: m.n_interior][warped]] = touched[m.neighbour[warped]] = True
    bad = [int(np.nonzero(touched)[0][0]), int(np.nonzero(~touched)[0][m.n_cells // 4])]
    for name, value in (("nan", np.full(5, np.nan)), ("inf density", [np.inf, 0.5, 0.0, 0.0, 2.0]),
                        ("inf energy", [1.0, 0.5, 0.0, 0.0, np.inf]), ("negative", [-1.0, 0.5, 0.0, 0.0, -2.0]),
                        ("large", [big, 1.4 * big, 0.0, 0.0, 3.0 * big]), ("fast", [1.0, np.sqrt(big), 0.0, 0.0, 3.0 * big])):
        u = case.u.reshape(5, -1).copy()
        u[:, bad] = np.asarray(value)[:, None]
        with np.errstate(all="ignore"):
            got, want = dev.residual(u.reshape(-1)), ora.residual(u.reshape(-1))
        np.testing.assert_array_equal(got, want, err_msg=name)
    dev.close()
