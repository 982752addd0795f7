"""The kernels that a mesh's size chooses, on what the steps of a case may carry:
immersed nodes, ghosts that keep their initial state, empty patches, the power-of-two
time steps.  Below 65,536 cells a stage is one kernel by default; with
PLBFS_BLOCK_CELLS it is the gradient and the flux kernel, as on any larger mesh, whose
flux blocks have 176 to 256 cells.  Every path does the same arithmetic a face, a
cell and a node, so all results agree bit for bit.
"""
import numpy as np
import pytest

from helpers import channel_mesh, oracle_for, perturbed_state, rel_err
from plbfs import case as pc
from plbfs import objects
from plbfs.solver import GpuSolver, HostMesh
from test_gpu_bc_types import empty_case_and_mesh
from test_gpu_parabolic import ghost_start, para_case, para_mesh

import pyoracle

pytestmark = pytest.mark.gpu


def solver(monkeypatch, pm, case, st, env=(), ibm=None, ghost=None):
    for name in ("BLOCK_CELLS", "GRAD_STAGE", "FLUX_STAGE"):
        monkeypatch.delenv("PLBFS_" + name, raising=False)
    for name, value in dict(env).items():
        monkeypatch.setenv("PLBFS_" + name, str(value))
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    s = GpuSolver(hm, case.params, case.patches_for(pm.patch_names))
    s.set_state(*st)
    if ghost:
        s.set_ghost_state(*ghost)
    if ibm:
        s.set_ibm(**ibm)
    return s


def results(s, steps, ibm=None):
    """Return code, then the fields (with nodes, also theirs) and, last, the history."""
    r = s.run(steps)
    out = list(s.state()) + [s.dt_local()]
    if ibm:
        out += list(s.ibm_state()) + [s.body_force()]
        assert np.abs(out[-1]).max() > 0
    s.close()
    return r["rc"], out, r["hist"]


def assert_equal(a, b, hist=True):
    assert a[0] == b[0]
    for x, y in zip(a[1], b[1]):
        assert np.array_equal(x, y, equal_nan=True)
    if hist:
        assert np.array_equal(a[2], b[2], equal_nan=True)


def sphere(case, centre, radius, n, h=1.0, kernel=1):
    # nodes off their anchors, so that the first step has a force already
    X, dA = objects.fibonacci_sphere(n, centre, radius)
    return dict(x_ref=X, x=X + 0.1, stiffness=0.5, node_area=dA, dt=case.time_marching_step, h=h, kernel=kernel)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("tets,h,kernel", [(False, 1.0, 1), (False, 1.0, 0), (True, 1.0, 1)])
def test_stage_kernel_with_immersed_nodes(gpu_available, monkeypatch, precision, tets, h, kernel):
    pm, case = channel_mesh(13, 10, 9, tets=tets), pc.channel_case(re=40.0, length_scale=4.0, fneq_min=0.55)
    case.lsq_exact_det = 1 if tets else 0
    case.precision = precision
    st = perturbed_state(case, oracle_for(pm, case), amp=0.01, seed=4)
    ibm = sphere(case, (5.0, 5.0, 4.5), 2.0, 70, h, kernel)
    one, two, blocks = (results(solver(monkeypatch, pm, case, st, env, ibm), 10, ibm)
                        for env in ({}, {"BLOCK_CELLS": 64}, {"BLOCK_CELLS": 256}))
    assert one[0] == 0
    assert_equal(one, two)
    assert_equal(one, blocks, hist=False)  # its partial sums are other cells'


@pytest.mark.parametrize("block_cells", [64, 192, 256])
@pytest.mark.parametrize("tets", [False, True])
def test_two_kernels_with_immersed_nodes_match_oracle(gpu_available, monkeypatch, tets, block_cells):
    """The bars of test_gpu_ibm.py, which runs this case through the stage kernel."""
    pm, case = channel_mesh(16, 10, 10, tets=tets, jitter=0.12), pc.channel_case(re=40.0, length_scale=4.0)
    case.lsq_exact_det = 1 if tets else 0
    o = oracle_for(pm, case)
    st = perturbed_state(case, o, amp=0.01, seed=4)
    o.set_state(*st)
    ibm = sphere(case, (6.0, 5.0, 5.0), 2.0, 80)
    X = ibm["x_ref"]
    pyoracle.set_ibm(o, X, ibm["x"], **{k: ibm[k] for k in ("stiffness", "node_area", "dt", "h", "kernel")})
    s = solver(monkeypatch, pm, case, st, {"BLOCK_CELLS": block_cells}, ibm)
    assert o.run(20)["rc"] == 0 and s.run(20)["rc"] == 0
    for a, b, at in zip(s.ibm_state(), pyoracle.ibm_state(o), (X, 0, 0)):
        assert rel_err(a - at, b - at) < 1e-9
    assert rel_err(s.body_force(), pyoracle.body_force(o)) < 1e-9
    for a, b in zip(s.state(), o.state()):
        assert rel_err(a, b) < 1e-10


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("dims,tets", [((41, 40, 40), False), ((23, 24, 24), True)])
def test_chosen_block_size_with_immersed_nodes(gpu_available, monkeypatch, dims, tets, precision):
    """Just above 65,536 cells: blocks of a size that is no multiple of a wavefront, some
    of which hold cells that the nodes spread force to, against blocks of 256."""
    pm, case = channel_mesh(*dims, tets=tets), pc.channel_case(re=40.0, length_scale=6.0, fneq_min=0.55)
    case.lsq_exact_det = 1 if tets else 0
    case.precision = precision
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    g = hm.geometry()
    n = pm.n_cells
    rho, u, v, w = case.initial_state(g["cx"][:n], g["cy"][:n], g["cz"][:n])
    st = (rho + 1e-3 * np.sin(g["cx"][:n]), u * (1 + 0.02 * np.cos(g["cy"][:n])), v, w + 1e-4 * np.sin(g["cz"][:n]))
    ibm = sphere(case, tuple(0.5 * d for d in dims), 4.0, 150)
    out = []
    for env in ({}, {"BLOCK_CELLS": 256}):
        s = solver(monkeypatch, pm, case, st, env, ibm)
        b = s.layout_info()["block_cells"]
        assert b == 256 if env else b % 64 != 0
        out.append(results(s, 6, ibm))
    assert out[0][0] == 0
    assert_equal(*out, hist=False)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind", ["parabolic-N", "parabolic-W", "parabolic", "wall", "thin", "slab", "talts"])
@pytest.mark.parametrize("tets", [False, True])
def test_stage_kernel_on_the_other_cases(gpu_available, monkeypatch, kind, tets, precision):
    ghost = None
    if kind in ("thin", "slab"):
        case, pm = empty_case_and_mesh(kind, tets)
    elif kind == "talts":
        pm, case = channel_mesh(10, 6, 6, tets=tets), pc.channel_case(re=40.0, length_scale=4.0)
        case.time_stepping = "talts"
    else:
        pm, case = para_mesh(tets), para_case(kind)
    case.lsq_exact_det = 1 if tets else 0
    case.precision = precision
    o = oracle_for(pm, case)
    if kind in ("thin", "slab", "talts"):
        st = perturbed_state(case, o, amp=0.01, seed=23)
    else:
        st = ghost_start(case, o, pm.n_cells)
        ghost = [x[pm.n_cells:] for x in st]
    one, two = (results(solver(monkeypatch, pm, case, st, env, ghost=ghost), 10) for env in ({}, {"BLOCK_CELLS": 64}))
    assert_equal(one, two)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("flux_stage,grad_stage", [(0, 0), (1, 0), (1, 1)])
def test_staging_changes_nothing_in_the_two_kernels(gpu_available, monkeypatch, precision, flux_stage, grad_stage):
    """Against the default of larger meshes, unstaged fluxes and staged gradients; the
    block size is given, as the stage kernel takes neither switch."""
    pm, case = channel_mesh(12, 6, 6, tets=True), pc.channel_case(re=40.0, length_scale=4.0)
    case.lsq_exact_det = 1
    case.precision = precision
    st = perturbed_state(case, oracle_for(pm, case), amp=0.01, seed=12)
    out = [results(solver(monkeypatch, pm, case, st, dict(BLOCK_CELLS=128, FLUX_STAGE=f, GRAD_STAGE=g)), 10)
           for f, g in ((0, 1), (flux_stage, grad_stage))]
    assert out[0][0] == 0
    assert_equal(*out)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("mode", ["local", "min"])
@pytest.mark.parametrize("env", [{}, {"BLOCK_CELLS": 64}])
def test_timed_run_launches_what_other_runs_launch(gpu_available, monkeypatch, env, mode, precision):
    """Kernel statistics of a run: one launch a stage where the stage kernel serves the
    mesh, counted as the flux's, a gradient and a flux launch elsewhere; same results."""
    pm, case = channel_mesh(10, 6, 6), pc.channel_case(re=40.0, length_scale=4.0)
    case.time_stepping = mode
    case.precision = precision
    st = perturbed_state(case, oracle_for(pm, case), amp=0.01, seed=3)
    plain = results(solver(monkeypatch, pm, case, st, env), 5)
    s = solver(monkeypatch, pm, case, st, env)
    s.enable_timing(True)
    r = s.run(5)
    stats = [s.kernel_stats(k) for k in range(4)]
    assert [n for _, n in stats] == [20 if env else 0, 20, 0, 5]
    assert all((ms > 0) == (n > 0) for ms, n in stats)
    timed = (r["rc"], list(s.state()) + [s.dt_local()], r["hist"])
    s.close()
    assert_equal(plain, timed)


@pytest.mark.parametrize("dims,tets,most", [((48, 48, 48), False, 255), ((62, 62, 62), False, 256),
                                            ((32, 32, 32), True, 256), ((33, 33, 33), True, 256),
                                            ((35, 35, 35), True, 256), ((66, 65, 65), False, 256)])
def test_small_flux_blocks_all_run_at_once(gpu_available, monkeypatch, dims, tets, most):
    """The mesh size chooses fewer than 256 cells a flux block only while all blocks find a
    place, four a CU: 215,622 and 257,250 tets and 278,850 hexes do not."""
    pm, case = channel_mesh(*dims, tets=tets), pc.channel_case(re=40.0, length_scale=6.0, fneq_min=0.55)
    monkeypatch.delenv("PLBFS_BLOCK_CELLS", raising=False)
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    s = GpuSolver(hm, case.params, case.patches_for(pm.patch_names))
    info = s.layout_info()
    s.close()
    assert 176 <= info["block_cells"] <= most
    assert info["block_cells"] == 256 or info["blocks"] <= 1024
