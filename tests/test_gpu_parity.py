"""GPU parity: the HIP solver (through the C-ABI) against the CPU oracle.

Bars: gradients and one-stage residuals to 1e-11 relative (per field, relative
to the field's max magnitude); fields after 100 steps to 1e-10 relative
(the FP64 plain-method requirement); local time steps to 1e-13.
"""
import numpy as np
import pytest

from helpers import (cavity_mesh, channel_mesh, initial_state, oracle_for, periodic_z_case, periodic_z_mesh,
                     perturbed_state, rel_err)
from plbfs import _native as nat
from plbfs import case as pc
from plbfs import meshgen
from plbfs.solver import GpuBatch, GpuSolver, HostMesh

pytestmark = pytest.mark.gpu


def make_pair(pm, case):
    o = oracle_for(pm, case)
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    s = GpuSolver(hm, case.params, case.patches_for(pm.patch_names))
    return o, hm, s


def field_errs(a, b):
    return [rel_err(a[q], b[q]) for q in range(4)]


@pytest.mark.parametrize("tets", [False, True])
def test_residual_and_gradients_match_oracle(gpu_available, tets):
    pm = cavity_mesh(6, tets=tets)
    case = pc.cavity_case()
    o, hm, s = make_pair(pm, case)
    st = perturbed_state(case, o, amp=0.02, seed=3)
    Ro, go = o.eval_residual(*st)
    s.set_state(*st)
    R, g = s.eval_residual()
    N = pm.n_cells
    for q in range(12):
        assert rel_err(g[:, q], go[:N, q]) < 1e-11, ("grad", q)
    for q in range(4):
        assert rel_err(R[:, q], Ro[:, q]) < 1e-11, ("R", q)


@pytest.mark.parametrize("tets", [False, True])
def test_local_dt_matches_oracle(gpu_available, tets):
    pm = cavity_mesh(5, tets=tets)
    case = pc.cavity_case()
    o, hm, s = make_pair(pm, case)
    st = perturbed_state(case, o, amp=0.05, seed=5)
    o.set_state(*st)
    s.set_state(*st)
    assert rel_err(s.dt_local(), o.dt_local()) < 1e-13


@pytest.mark.parametrize("tets", [False, True])
def test_cavity_100_steps(gpu_available, tets):
    pm = cavity_mesh(6, tets=tets)
    case = pc.cavity_case()
    # the reference's LSQ determinant diverges within a few steps on jittered
    # tetrahedra; long tet runs use the true determinant (same on both sides)
    case.lsq_exact_det = 1 if tets else 0
    o, hm, s = make_pair(pm, case)
    st = initial_state(case, o)
    o.set_state(*st)
    s.set_state(*st)
    ro = o.run(100)
    rg = s.run(100)
    assert ro["rc"] == 0 and rg["rc"] == 0
    assert rg["steps"] == 100
    errs = field_errs(s.state(), o.state())
    assert max(errs) < 1e-10, errs
    # residual history tracks the oracle step by step
    assert np.max(np.abs(rg["hist"][:, 1:] - ro["hist"][:, 1:]) / ro["hist"][:, 1:]) < 1e-8


@pytest.mark.parametrize("tets", [False, True])
def test_channel_100_steps(gpu_available, tets):
    pm = channel_mesh(10, 5, 5, tets=tets)
    case = pc.channel_case(re=40.0, length_scale=4.0)
    case.lsq_exact_det = 1 if tets else 0
    o, hm, s = make_pair(pm, case)
    st = perturbed_state(case, o, amp=0.01, seed=9)
    o.set_state(*st)
    s.set_state(*st)
    # the coarse tet channel amplifies 1e-15 input noise ~1000x over 100 steps;
    # 60 steps keep the comparison well conditioned
    n = 60 if tets else 100
    assert o.run(n)["rc"] == 0
    assert s.run(n)["rc"] == 0
    errs = field_errs(s.state(), o.state())
    assert max(errs) < 1e-10, errs


@pytest.mark.parametrize("tets", [False, True])
def test_periodic_z_steps(gpu_available, tets):
    from helpers import periodic_z_case, periodic_z_mesh
    pm = periodic_z_mesh(10, 5, 6, tets=tets)
    case = periodic_z_case(6.0)
    case.lsq_exact_det = 1 if tets else 0
    o, hm, s = make_pair(pm, case)
    st = perturbed_state(case, o, amp=0.01, seed=13)
    o.set_state(*st)
    s.set_state(*st)
    n = 60 if tets else 100
    assert o.run(n)["rc"] == 0
    assert s.run(n)["rc"] == 0
    errs = field_errs(s.state(), o.state())
    assert max(errs) < 1e-10, errs


def test_flux_block_too_large_for_lds_is_a_clean_error(gpu_available, monkeypatch):
    # 1024 FP64 tets staged: ~2300 face slots x 32 B plus 1024 staged cell
    # records x 160 B, over the 159 KiB a flux block may take; refused on the
    # host before any launch
    monkeypatch.setenv("PLBFS_BLOCK_CELLS", "1024")
    monkeypatch.setenv("PLBFS_FLUX_STAGE", "1")
    pm = channel_mesh(16, 8, 8, tets=True)
    case = pc.channel_case(re=40.0, length_scale=6.0)
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    with pytest.raises(nat.PlbfsError) as ei:
        GpuSolver(hm, case.params, case.patches_for(pm.patch_names))
    assert ei.value.rc == -1 and "LDS" in str(ei.value)


@pytest.mark.parametrize("block_cells,stage", [(64, 1), (128, 1), (192, 0), (256, 0), (512, 0), (768, 0)])
def test_flux_block_sizes(gpu_available, monkeypatch, block_cells, stage):
    # the flux block size changes which faces are duplicated on block borders
    # and how many cells one thread updates; staging changes where a block
    # reads its own cells' records (LDS or global memory); none changes the
    # arithmetic
    monkeypatch.setenv("PLBFS_BLOCK_CELLS", str(block_cells))
    monkeypatch.setenv("PLBFS_FLUX_STAGE", str(stage))
    monkeypatch.setenv("PLBFS_GRAD_STAGE", str(stage))
    pm = channel_mesh(16, 8, 8, tets=True)
    case = pc.channel_case(re=40.0, length_scale=6.0)
    case.lsq_exact_det = 1
    o, hm, s = make_pair(pm, case)
    assert s.layout_info()["block_cells"] == block_cells
    st = perturbed_state(case, o, amp=0.01, seed=4)
    o.set_state(*st)
    s.set_state(*st)
    assert o.run(40)["rc"] == 0
    assert s.run(40)["rc"] == 0
    errs = field_errs(s.state(), o.state())
    assert max(errs) < 1e-10, errs


@pytest.mark.parametrize("precision", [0, 1])
def test_border_pass_is_bitwise_neutral(gpu_available, monkeypatch, precision):
    # faces between two flux blocks evaluated once by the border pass or by
    # both blocks: the same arithmetic summed in the same order, so the same bits
    pm = channel_mesh(16, 8, 8, tets=True)
    case = pc.channel_case(re=40.0, length_scale=6.0)
    case.lsq_exact_det = 1
    case.precision = precision
    st = None
    out = []
    for split in ("1", "0"):
        monkeypatch.setenv("PLBFS_SPLIT_BORDER", split)
        monkeypatch.setenv("PLBFS_BLOCK_CELLS", "64")
        o, hm, s = make_pair(pm, case)
        if st is None:
            st = perturbed_state(case, o, amp=0.01, seed=9)
        s.set_state(*st)
        assert s.run(30)["rc"] == 0
        out.append(s.state())
        s.close()
    for q in range(4):
        assert np.array_equal(out[0][q], out[1][q]), q


def test_reference_determinant_on_jittered_tets(gpu_available):
    """The reference's LSQ determinant on jittered tets: both sides follow it
    for the few steps before the reference algorithm itself blows up."""
    pm = cavity_mesh(6, tets=True, jitter=0.15)
    case = pc.cavity_case()
    o, hm, s = make_pair(pm, case)
    st = initial_state(case, o)
    o.set_state(*st)
    s.set_state(*st)
    assert o.run(3)["rc"] == 0
    assert s.run(3)["rc"] == 0
    assert max(field_errs(s.state(), o.state())) < 1e-10
    R, g = s.eval_residual()
    Ro, go = o.eval_residual(*[np.concatenate([x, np.zeros(o.T - o.N)]) for x in o.state()])
    for q in range(4):
        assert rel_err(R[:, q], Ro[:, q]) < 1e-10


@pytest.mark.parametrize("kind", ["cavity", "channel"])
def test_reference_determinant_on_mildly_jittered_tets_100_steps(gpu_available, kind):
    """The reference's LSQ determinant (src/gradients.cpp:282-284) over 100
    steps on tets: with 5 % jitter the reference algorithm stays stable (it
    diverges from 10 % on), so the GPU can be held to the oracle on
    reference semantics for as long as on the other meshes."""
    if kind == "cavity":
        pm = cavity_mesh(6, tets=True, jitter=0.05)
        case = pc.cavity_case()
    else:
        pm = channel_mesh(10, 5, 5, tets=True, jitter=0.05)
        case = pc.channel_case(re=40.0, length_scale=4.0)
    case.lsq_exact_det = 0
    o, hm, s = make_pair(pm, case)
    st = perturbed_state(case, o, amp=0.01, seed=13)
    o.set_state(*st)
    s.set_state(*st)
    print("reference determinant, tets, jitter 0.05,", kind, "cells", pm.n_cells, flush=True)
    assert o.run(100)["rc"] == 0
    assert s.run(100)["rc"] == 0
    errs = field_errs(s.state(), o.state())
    assert max(errs) < 1e-10, errs


def test_time_stepping_modes(gpu_available):
    pm = cavity_mesh(5, tets=False)
    for mode in ("constant", "min", "talts"):
        case = pc.cavity_case()
        case.time_stepping = mode
        case.time_marching_step = 0.5 if mode != "constant" else 0.002
        o, hm, s = make_pair(pm, case)
        st = perturbed_state(case, o, amp=0.01, seed=1)
        o.set_state(*st)
        s.set_state(*st)
        assert o.run(20)["rc"] == 0
        assert s.run(20)["rc"] == 0
        errs = field_errs(s.state(), o.state())
        assert max(errs) < 1e-10, (mode, errs)


def test_gradient_variants(gpu_available):
    pm = cavity_mesh(5, tets=True)
    for gc in ("hybrid", "GG"):
        case = pc.cavity_case()
        case.gradient_calc = gc
        case.lsq_exact_det = 1
        o, hm, s = make_pair(pm, case)
        st = perturbed_state(case, o, amp=0.01, seed=2)
        o.set_state(*st)
        s.set_state(*st)
        assert o.run(10)["rc"] == 0
        assert s.run(10)["rc"] == 0
        assert max(field_errs(s.state(), o.state())) < 1e-10, gc


def test_convergence_stop_matches_oracle(gpu_available):
    pm = cavity_mesh(4, tets=False, jitter=0.1)
    case = pc.cavity_case(re=10.0)
    case.tolerance = 2e-3
    case.check_interval = 7
    o, hm, s = make_pair(pm, case)
    st = initial_state(case, o)
    o.set_state(*st)
    s.set_state(*st)
    ro = o.run(3000)
    rg = s.run(3000)
    assert ro["converged"] and rg["converged"]
    assert rg["steps"] == ro["steps"]
    assert max(field_errs(s.state(), o.state())) < 1e-10


def test_bitwise_deterministic(gpu_available):
    pm = cavity_mesh(6, tets=True)
    case = pc.cavity_case()
    outs = []
    for _ in range(2):
        o, hm, s = make_pair(pm, case)
        s.set_state(*initial_state(case, o))
        s.run(30)
        outs.append(s.state())
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


def test_nan_state_reports_error(gpu_available):
    pm = cavity_mesh(4, tets=False)
    case = pc.cavity_case()
    o, hm, s = make_pair(pm, case)
    rho, u, v, w = initial_state(case, o)
    rho = rho.copy()
    rho[3] = np.nan
    s.set_state(rho, u, v, w)
    r = s.run(5)
    assert r["rc"] == -2, nat.ERR_NAMES.get(r["rc"])
    assert r["steps"] == 1


def test_wall_forces_match_reference_sums(gpu_available):
    """Drag and lift over each wall patch after 50 steps, against the same sums
    (src/post_processing.cpp:96-107) evaluated from the oracle's state and
    ghost-cell gradients."""
    pm = cavity_mesh(6, tets=False)
    case = pc.cavity_case()
    o, hm, s = make_pair(pm, case)
    st = initial_state(case, o)
    o.set_state(*st)
    s.set_state(*st)
    assert o.run(50)["rc"] == 0 and s.run(50)["rc"] == 0
    so = o.state()
    R, go = o.eval_residual(*[np.concatenate([x, np.zeros(o.T - o.N)]) for x in so])
    f = o.faces()
    N, NI = pm.n_cells, pm.n_internal
    bp = hm.bface_patch()
    gam, nuv = case.gamma, case.visc * case.gamma
    checked = 0
    for q, name in enumerate(pm.patch_names):
        drag = lift = 0.0
        for b in np.flatnonzero(bp == q):
            fi, ow = NI + b, pm.owner[NI + b]
            n = (f["ni"][fi], f["nj"][fi], f["nk"][fi])
            A = f["area"][fi]
            p = so[0][ow] / 3.0 * gam
            gu, gv = go[N + b, 3:6], go[N + b, 6:9]
            drag += ((p - nuv * gu[0]) * n[0] - nuv * gu[1] * n[1]) * A
            lift += (nuv * gv[0] * n[0] - (p - nuv * gv[1]) * n[1]) * A
        dl = s.wall_forces(q)
        assert abs(dl[0] - drag) <= 1e-10 * max(1.0, abs(drag)), (name, dl, drag)
        assert abs(dl[1] - lift) <= 1e-10 * max(1.0, abs(lift)), (name, dl, lift)
        checked += 1
    assert checked == len(pm.patch_names)


@pytest.mark.parametrize("dims,tets,sizes", [((40, 40, 40), False, (64, 64)), ((41, 40, 40), False, (176, 256)),
                                             ((23, 22, 22), True, (176, 256)), ((3, 3, 3), False, (64, 64))])
@pytest.mark.parametrize("precision", [0, 1])
def test_chosen_flux_block_size_changes_no_field(gpu_available, monkeypatch, dims, tets, sizes, precision):
    """The block size that a mesh gets on either side of 65,536 cells, against blocks
    of 256 cells: the same fields, bit for bit."""
    pm = channel_mesh(*dims, tets=tets)
    case = pc.channel_case(re=40.0, length_scale=6.0, fneq_min=0.55)
    case.lsq_exact_det = 1 if tets else 0
    case.precision = precision
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    g = hm.geometry()
    n = pm.n_cells
    rho, u, v, w = case.initial_state(g["cx"][:n], g["cy"][:n], g["cz"][:n])
    st = (rho + 1e-3 * np.sin(g["cx"][:n]), u * (1 + 0.02 * np.cos(g["cy"][:n])), v, w + 1e-4 * np.sin(g["cz"][:n]))
    out = []
    for blk in ("", "256"):
        if blk:
            monkeypatch.setenv("PLBFS_BLOCK_CELLS", blk)
        s = GpuSolver(hm, case.params, case.patches_for(pm.patch_names))
        b = s.layout_info()["block_cells"]
        assert b == 256 if blk else sizes[0] <= b <= sizes[1]
        s.set_state(*st)
        assert s.run(6)["rc"] == 0
        out.append(s.state())
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dims,tets", [((2, 2, 2), False), ((4, 4, 4), False), ((5, 13, 2), False), ((7, 6, 5), True),
                                       ((11, 10, 9), False)])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind,stepping", [("periodic", "min"), ("channel", "local"), ("inlet", "constant")])
def test_one_kernel_stage_equals_two_kernels(gpu_available, monkeypatch, dims, tets, precision, kind, stepping):
    """The small meshes' stage kernel against the gradient and flux kernels on the same
    flux blocks (asked for by size): same fields, residuals and time steps, bit for bit.
    A few cells, one whole block, a block of two cells behind two, several blocks."""
    if kind == "periodic":
        if tets:
            pytest.skip("partners are ambiguous on tets")
        pm, case = periodic_z_mesh(*dims), periodic_z_case(float(dims[2]))
    else:
        pm, case = channel_mesh(*dims, tets=tets), pc.channel_case(re=40.0, length_scale=4.0, fneq_min=0.55)
    if kind == "inlet":
        for bc, types in zip(case.bcs.values(), (("inlet", "inlet"), ("dirichlet", "wall"), ("symmetry-x", "symmetry-x"))):
            bc.update(vel_type=types[0], rho_type=types[1])
    case.lsq_exact_det = 1 if tets else 0
    case.precision = precision
    case.time_stepping = stepping
    if stepping == "constant":
        case.cfl = 0.05
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    g = hm.geometry()
    n = pm.n_cells
    rho, u, v, w = case.initial_state(g["cx"][:n], g["cy"][:n], g["cz"][:n])
    st = (rho + 1e-3 * np.sin(g["cx"][:n]), u * (1 + 0.02 * np.cos(g["cy"][:n])), v, w + 1e-4 * np.sin(g["cz"][:n]))
    out = []
    for blk in ("", "64"):
        if blk:
            monkeypatch.setenv("PLBFS_BLOCK_CELLS", blk)
        s = GpuSolver(hm, case.params, case.patches_for(pm.patch_names))
        s.set_state(*st)
        r = s.run(6)
        out.append([r["rc"], r["hist"], s.dt_local()] + list(s.state()))
        s.close()
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("dims", [(16, 16, 1), (17, 16, 1), (41, 40, 40)])
def test_minimum_time_step_over_many_blocks(gpu_available, dims):
    """The global minimum over 1, 2 and 257 blocks of 256 cells: every cell's step in
    the "min" mode is the smallest of the local ones."""
    pm, case = channel_mesh(*dims), pc.channel_case(re=40.0, length_scale=4.0)
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    g = hm.geometry()
    n = pm.n_cells
    rho, u, v, w = case.initial_state(g["cx"][:n], g["cy"][:n], g["cz"][:n])
    dt = []
    for stepping in ("local", "min"):
        case.time_stepping = stepping
        s = GpuSolver(hm, case.params, case.patches_for(pm.patch_names))
        s.set_state(rho, u * (1 + 0.5 * np.cos(g["cx"][:n])), v, w)
        dt.append(s.dt_local())
        s.close()
    assert dt[0].max() > dt[0].min()
    assert np.all(dt[1] == dt[0].min())


@pytest.mark.parametrize("dims", [(4, 4, 4), (8, 8, 9), (13, 12, 11), (41, 40, 41)])
def test_block_order_over_the_xcds_changes_no_field(gpu_available, monkeypatch, dims):
    """Contiguous ranges of blocks per XCD against dispatch order, on 1, 9, 27 and some 300
    blocks (remainders of 8): the same fields, bit for bit."""
    pm, case = channel_mesh(*dims), pc.channel_case(re=40.0, length_scale=4.0, fneq_min=0.55)
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    g = hm.geometry()
    n = pm.n_cells
    rho, u, v, w = case.initial_state(g["cx"][:n], g["cy"][:n], g["cz"][:n])
    out = []
    for order in ("0", "1"):
        monkeypatch.setenv("PLBFS_XCD_REMAP", order)
        monkeypatch.setenv("PLBFS_BLOCK_CELLS", "64" if n < 65536 else "256")
        s = GpuSolver(hm, case.params, case.patches_for(pm.patch_names))
        s.set_state(rho + 1e-3 * np.sin(g["cx"][:n]), u * (1 + 0.02 * np.cos(g["cy"][:n])), v, w)
        assert s.run(4)["rc"] == 0
        out.append(s.state())
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dims", [(5, 4, 3), (21, 20, 20)])
@pytest.mark.parametrize("precision", [0, 1])
def test_state_reads_back_as_set(gpu_available, dims, precision):
    """The state directly behind plbfs_set_state, before and after steps were taken, in
    one copy and (above 8,192 cells) field by field: what was set, bit for bit."""
    pm, case = channel_mesh(*dims), pc.channel_case(re=40.0, length_scale=3.0)
    case.precision = precision
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    s = GpuSolver(hm, case.params, case.patches_for(pm.patch_names))
    rng = np.random.default_rng(5)
    for _ in range(4):
        st = [1.0 + 0.01 * rng.random(pm.n_cells)] + [0.01 * rng.random(pm.n_cells) for _ in range(3)]
        s.set_state(*st)
        for a, b in zip(s.state(), st):
            assert np.array_equal(a, b)
        assert s.run(3)["rc"] == 0
    s.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("dims,lengths", [((6, 5, 4), (9.0, 6.25, 3.0)), ((17, 9, 9), (25.5, 11.25, 6.75))])
def test_rest_stays_at_rest_bit_for_bit(gpu_available, monkeypatch, dims, lengths, precision):
    """A box of uniform density at rest, whose cells' volume is no power of two: the
    pressure fluxes through a cell's opposite faces are equal and cancel exactly in its
    residual, so nothing ever moves; by the stage kernel, the two kernels and a batch."""
    pm = meshgen.box_mesh(*dims, lengths=lengths, permute_seed=3, patch_types=pc.CAVITY_PATCHES)
    case = pc.cavity_case(lid_u=0.0)
    case.precision = precision
    case.tolerance = 0.0
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    n = pm.n_cells
    st = [np.full(n, 1.03)] + [np.zeros(n)] * 3
    patches = case.patches_for(pm.patch_names)
    for blk in ("", "64"):
        if blk:
            monkeypatch.setenv("PLBFS_BLOCK_CELLS", blk)
        s = GpuSolver(hm, case.params, patches)
        s.set_state(*st)
        assert not s.eval_residual()[0].any()
        assert s.run(20)["steps"] == 20
        for a, b in zip(s.state(), st):
            assert np.array_equal(a, b)
        s.close()
    bt = GpuBatch(hm, case.params, patches, [case.visc] * 3)
    bt.set_state(-1, *st)
    assert bt.run(20)[0] == 0
    for k in range(3):
        for a, b in zip(bt.state(k), st):
            assert np.array_equal(a, b)
    bt.close()
