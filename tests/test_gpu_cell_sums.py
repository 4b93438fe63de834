"""The transfers that sum a cell's particles together (P2G's matrix products,
the gradient scatters of the implicit and ADMM steps) where their splits can
go wrong: cells of one to nine particles (a product takes four at a time),
cells that a chunk of particles cuts, pages at and past a chunk of 256 and of
304 particles, one cell with a whole page's particles, a page past the 2,048
keys that a block sorts in one piece, and pages on both sides of the line where
cells are shared by more threads."""
import numpy as np
import pytest

import oracle
from ziran2019_amd.engine import (ZR_FP32_REFINED, ZR_MODEL_STVK_HENCKY, admm_opts, implicit_opts,
                                  phase_field_opts)
from _helpers import make_pair, perturbed, rel_err

pytestmark = pytest.mark.gpu

# particles in each cell of one page (x 2, y 4, z 4), the page's total in the name
COUNTS = {
    "1-9": [1 + k % 9 for k in range(32)],
    "255": [8] * 31 + [7],
    "256": [8] * 32,
    "257": [8] * 31 + [9],
    "303": [9] * 31 + [24],
    "304": [9] * 31 + [25],
    "305": [9] * 31 + [26],
    "one cell 300": [0] * 13 + [300] + [0] * 18,
    "one cell 700": [0] * 31 + [700],
    "cut cells": [40, 0, 250, 0, 20, 3, 0, 300] + [0] * 23 + [1],
    "2300": [72] * 31 + [68],
    # past 1,216 particles, the empty cells' threads take parts of the others
    "one cell 1216": [0] * 9 + [1216] + [0] * 22,
    "one cell 1217": [0] * 9 + [1217] + [0] * 22,
    "three cells 2600": [700] + [0] * 20 + [1890] + [0] * 9 + [10],
    "16 cells 1300": [81, 0] * 15 + [85, 0],
    "17 cells 1300": [80, 0] * 14 + [80, 50, 50, 80],
}


def _scene(counts):
    s = perturbed(5, n_cells=5, F_noise=0.03, C_noise=0.2, E=2e4)
    rng = np.random.default_rng(5)
    n = int(np.sum(counts))
    dx = s["dx"]
    cell = np.repeat(np.arange(32), counts)
    lo = np.floor(s["X"].mean(axis=0) / dx).astype(np.int64) // np.array([2, 4, 4]) * np.array([2, 4, 4])
    at = lo + np.stack([cell >> 4, (cell >> 2) & 3, cell & 3], axis=1)
    # base node at + 1/2: the particle lies within the cell from there, ends left out
    s["X"] = np.ascontiguousarray((at + 0.5 + 0.001 + 0.998 * rng.random((n, 3))) * dx)
    src = rng.integers(0, len(s["mass"]), n)
    for k in ("V", "C", "F", "mass", "vol", "mu", "lam"):
        s[k] = np.ascontiguousarray(np.asarray(s[k])[src])
    p = rng.permutation(n)
    s["X"] = np.ascontiguousarray(s["X"][p])
    return s


@pytest.mark.parametrize("counts", COUNTS.values(), ids=COUNTS.keys())
def test_transfers(counts):
    s = _scene(counts)
    eng, ora = make_pair(s)
    # explicit, force and momentum in fields of their own
    eng.sortParticlesAndPolluteGrid()
    eng.particlesToGrid()
    ora.sort_and_pollute()
    ora.update_stress()
    ora.p2g()
    g = ora.grid()
    # the explicit parity tests' bounds; a cell of 700 sums 700 terms
    assert rel_err(eng.dump("grid_m"), g["m"]) < 1e-12
    assert rel_err(eng.dump("grid_v"), g["v"]) < 1e-12
    assert rel_err(eng.dump("grid_f"), g["new_v"]) < 1e-12
    eng.close()
    # APIC, the Newton residual's scatter and the operator (the implicit parity
    # tests' bounds)
    for precision, tol in ((0, 1e-11), (1, 2e-5)):
        eng, ora = make_pair(s)
        eng.sortParticlesAndPolluteGrid()
        eng.particlesToGridApic()
        eng.backwardEulerStep(1e-3, implicit_opts(newton_max_iterations=1, precision=precision))
        ora.sort_and_pollute()
        ora.p2g_apic()
        ora.backward_euler(1e-3, oracle.implicit_opts(newton_max_iterations=1))
        active = ora.grid()["idx"] >= 0
        rng = np.random.default_rng(3)
        dv = 0.001 * rng.normal(size=(len(active), 3))
        dv[~active] = 0.0
        assert rel_err(eng.implicit_residual(dv), ora.implicit_residual(dv)) < 1e-11
        x = rng.normal(size=(len(active), 3))
        x[~active] = 0.0
        assert rel_err(eng.implicit_multiply(x), ora.implicit_multiply(x)) < tol
        eng.close()
    # the fused explicit step
    eng, ora = make_pair(s)
    for _ in range(2):
        eng.advanceOneTimeStep(1e-5)
        ora.step(1e-5)
    out = eng.download()
    for k, r in zip("XVCF", ora.get_particles()):
        assert rel_err(out[k], r) < 1e-10, k
    eng.close()


@pytest.mark.parametrize("counts", COUNTS.values(), ids=COUNTS.keys())
@pytest.mark.parametrize("precision", [0, ZR_FP32_REFINED])
def test_admm_step(counts, precision):
    """The ADMM operator and right side; the ground touches the page, so that
    the dual update meets nodes that the collision changes.  FP32: the
    operator's rounding leaves the solution within the solve's tolerance, and
    1e-4 of dv holds with a margin of ten over 2^-24 times the 27 x 8 terms."""
    s = _scene(counts)
    s["V"][:, 1] -= 0.5
    y0 = float(s["X"][:, 1].min() + 0.5 * s["dx"])
    eng, ora = make_pair(s, colliders=[dict(shape=0, type=1, origin=(0.0, y0, 0.0), normal=(0.0, 1.0, 0.0))])
    eng.set_materials(model=ZR_MODEL_STVK_HENCKY, plasticity=0, plastic_param=(0, 0, 0, 0), plastic_state=0.0)
    ora.set_materials(model=ZR_MODEL_STVK_HENCKY, plastic=0, pparam=(0, 0, 0, 0), pstate=0.0)
    o = dict(admm_iterations=3)
    for _ in range(2):
        eng.advanceOneTimeStepAdmm(1e-4, admm_opts(precision=precision, **o))
        ora.step_admm(1e-4, oracle.admm_opts(**o))
    out, st, ref = eng.download(), eng.get_admm_state(), ora.get_admm()
    tol = 1e-8 if precision == 0 else 1e-4  # FP64: the ADMM parity tests' bound
    for k, r in zip("XVCF", ora.get_particles()):
        assert rel_err(out[k], r) < tol, k
    assert rel_err(st["F"], ref["F"]) < tol
    assert rel_err(st["y"], ref["y"]) < tol * (1 if precision == 0 else 10)
    eng.close()


@pytest.mark.parametrize("counts", list(COUNTS.values())[6:], ids=list(COUNTS)[6:])
@pytest.mark.parametrize("M", [0.0, 15.0])
def test_phase_field_solve(counts, M):
    """The damage solve's sums of two and of four values (the parity tests'
    bounds; M > 0 makes the system diagonally dominant)."""
    s = _scene(counts)
    eng, ora = make_pair(s)
    kw = dict(l0=0.5 * s["dx"], one_over_sigma_c=np.full(len(s["mass"]), 0.02))
    eng.set_phase_field(phase_field_opts(parabolic_M=M, cg_tolerance=0.0), **kw)
    ora.set_phase_field(oracle.pf_opts(parabolic_M=M, cg_tolerance=0.0), **kw)
    eng.sortParticlesAndPolluteGrid()
    eng.particlesToGrid()
    ora.sort_and_pollute()
    ora.update_stress()
    ora.p2g()
    eng.phase_field_solve(1e-4)
    ora.phase_field_solve(1e-4)
    pg, po = eng.get_phase_field(), ora.get_phase_field()
    assert rel_err(pg["c"], po["c"]) < 1e-10
    assert rel_err(pg["H"], po["H"]) < 1e-12
    assert rel_err(pg["pf_Fp"], po["pf_Fp"]) < 1e-12
    eng.close()
