"""Warm-start network on the GPU (BF16 MFMA kernels) against the NumPy reference.

The reference rounds the same GEMM operands to bfloat16 and accumulates in
float64; the GPU accumulates in FP32, so a few operands round to the
neighbouring bfloat16 value downstream.  Bars (relative L2 per tensor):
outputs 1e-2, every parameter gradient 3e-2.  The reference's own backward is
pinned against finite differences on the CPU (test_mpnn_ref.py).
"""
import numpy as np
import pytest

import mpnn_ref as M
from helpers import channel_mesh
from plbfs import case as pc
from plbfs import mpnn
from plbfs.solver import HostMesh

pytestmark = pytest.mark.gpu


def problem(seed=0):
    pm = channel_mesh(8, 4, 4)
    case = pc.channel_case(re=40.0, length_scale=3.0)
    hm = HostMesh.from_polymesh(pm, case.visc, case.gamma, case.fneq_min)
    geo = hm.geometry()
    N = pm.n_cells
    src, dst, ef, _ = mpnn.graph_from_geometry(geo, N)
    x = mpnn.node_inputs(geo, N, (4.0, 2.0, 2.0), 2.0, 80.0)
    rng = np.random.default_rng(seed)
    tgt = np.zeros((N, 16), np.float32)
    tgt[:, :4] = rng.normal(size=(N, 4))
    return N, src, dst, ef, x, tgt


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


def test_forward_matches_reference(gpu_available):
    N, src, dst, ef, x, _ = problem()
    P = M.init_params(1)
    net = mpnn.Mpnn(N, src, dst, ef, train=False)
    net.set_params(mpnn.flatten_params(P, M.mlp_shapes()))
    y = net.forward(x)
    G = M.Graph(src, dst, N)
    yr, _ = M.forward(P, G, x.astype(np.float64), ef[G.order].astype(np.float64), bf16_mode=True)
    assert rel(y[:, :4], yr[:, :4]) < 1e-2


def test_gradients_match_reference(gpu_available):
    N, src, dst, ef, x, tgt = problem()
    P = M.init_params(2)
    net = mpnn.Mpnn(N, src, dst, ef, train=True)
    shapes = M.mlp_shapes()
    net.set_params(mpnn.flatten_params(P, shapes))
    mask = mpnn.output_mask(N)
    loss, g = net.loss_grad(x, tgt, mask)
    G = M.Graph(src, dst, N)
    lr, _, gr = M.loss_and_grads(P, G, x.astype(np.float64), ef[G.order].astype(np.float64),
                                 tgt.astype(np.float64), mask.astype(np.float64), bf16_mode=True)
    assert abs(loss - lr) / lr < 1e-2
    gg = mpnn.unflatten(g, shapes)
    for name, _, _ in shapes:
        for key in ("W1", "b1", "W2", "b2"):
            assert rel(gg[name][key], gr[name][key]) < 3e-2, (name, key)


def test_gradients_are_deterministic(gpu_available):
    N, src, dst, ef, x, tgt = problem(3)
    net = mpnn.Mpnn(N, src, dst, ef, train=True)
    net.set_params(mpnn.flatten_params(M.init_params(4), M.mlp_shapes()))
    mask = mpnn.output_mask(N)
    _, g1 = net.loss_grad(x, tgt, mask)
    _, g2 = net.loss_grad(x, tgt, mask)
    assert np.array_equal(g1, g2)


def test_training_reduces_loss(gpu_available):
    N, src, dst, ef, x, _ = problem()
    net = mpnn.Mpnn(N, src, dst, ef, train=True)
    net.set_params(mpnn.flatten_params(M.init_params(5), M.mlp_shapes()))
    # a smooth target the inputs determine
    tgt = np.zeros((N, 16), np.float32)
    tgt[:, 0] = x[:, 0] * x[:, 1]
    tgt[:, 1] = np.tanh(3 * x[:, 3])
    tgt[:, 2] = x[:, 2]
    X = np.stack([x] * 4)
    T = np.stack([tgt] * 4)
    hist = net.train(X, T, mpnn.output_mask(N), epochs=40, lr=2e-3, seed=3)
    assert np.all(np.isfinite(hist))
    assert hist[-1] < 0.2 * hist[0], hist


@pytest.mark.parametrize("n,degrees", [
    (1, [0]),                      # one node without edges
    (5, [3, 0, 4, 1, 2]),
    (16, [4]),                     # one tile exactly: 16 nodes, 64 edges
    (17, [4]),                     # one node more
    (33, [6]),                     # tiles end at 60 of 64 edges
    (65, [0, 1, 2, 3]),
    (40, [63, 64, 65, 2, 0]),      # nodes that fill a tile, overfill it, or share one
    (12, [200, 1, 129, 64]),       # a node over several chunks of 64 edges
])
def test_edge_tiles_match_reference(gpu_available, n, degrees):
    """Graphs whose in-degrees meet the edges of the kernels' tiles (16 nodes, 64
    edges, one node of more), forward and backward, at the bars of this file."""
    rng = np.random.default_rng(n)
    dst = np.repeat(np.arange(n), [degrees[k % len(degrees)] for k in range(n)]).astype(np.int32)
    src = rng.integers(0, n, size=len(dst)).astype(np.int32)
    order = rng.permutation(len(dst))
    src, dst = src[order], dst[order]
    ef = rng.normal(size=(len(dst), 16)).astype(np.float32)
    x = rng.normal(size=(n, 16)).astype(np.float32)
    tgt = rng.normal(size=(n, 16)).astype(np.float32)
    P, shapes, mask = M.init_params(6), M.mlp_shapes(), mpnn.output_mask(n)
    net = mpnn.Mpnn(n, src, dst, ef, train=True)
    net.set_params(mpnn.flatten_params(P, shapes))
    y = net.forward(x)
    loss, g = net.loss_grad(x, tgt, mask)
    G = M.Graph(src, dst, n)
    lr, _, gr = M.loss_and_grads(P, G, x.astype(np.float64), ef[G.order].astype(np.float64),
                                 tgt.astype(np.float64), mask.astype(np.float64), bf16_mode=True)
    yr, _ = M.forward(P, G, x.astype(np.float64), ef[G.order].astype(np.float64), bf16_mode=True)
    assert rel(y[:, :4], yr[:, :4]) < 1e-2
    assert abs(loss - lr) / lr < 1e-2
    gg = mpnn.unflatten(g, shapes)
    for name, _, _ in shapes:
        for key in ("W1", "b1", "W2", "b2"):
            assert np.linalg.norm(gg[name][key] - gr[name][key]) < 3e-2 * max(np.linalg.norm(gr[name][key]), 1e-6), (
                name, key)
    # inference buffers give the same prediction
    infer = mpnn.Mpnn(n, src, dst, ef, train=False)
    infer.set_params(mpnn.flatten_params(P, shapes))
    assert np.array_equal(infer.forward(x), y)


@pytest.mark.parametrize("scale", [1e3, 1e6, 1e30])
def test_saturated_units_match_reference(gpu_available, scale):
    """Inputs so large that the encoder's units lie far outside +-88 on both sides, at this
    file's bar for outputs (1e30: finite), and one NaN: it reaches its cell's output and
    no cell more than six edges away."""
    N, src, dst, ef, x, _ = problem()
    P = M.init_params(1)
    net = mpnn.Mpnn(N, src, dst, ef, train=False)
    net.set_params(mpnn.flatten_params(P, M.mlp_shapes()))
    xs = (x * scale).astype(np.float32)
    y = net.forward(xs)
    G = M.Graph(src, dst, N)
    with np.errstate(over="ignore"):
        yr, _ = M.forward(P, G, xs.astype(np.float64), ef[G.order].astype(np.float64), bf16_mode=True)
    assert np.isfinite(y).all()
    assert rel(y[:, :4], yr[:, :4]) < 1e-2
    x = x.copy()
    x[0, 0] = np.nan
    y = net.forward(x)
    near = np.zeros(N, bool)
    near[0] = True
    for _ in range(6):
        near[dst[near[src]]] = True
    assert np.isnan(y[0, :4]).all()
    assert np.isfinite(y[~near]).all()


def test_gradients_without_the_loss(gpu_available):
    """plbfs_mpnn_loss_grad with loss NULL: the gradients of this call's inputs, as with
    a loss, though nothing else is read back."""
    N, src, dst, ef, x, tgt = problem(7)
    net = mpnn.Mpnn(N, src, dst, ef, train=True)
    net.set_params(mpnn.flatten_params(M.init_params(8), M.mlp_shapes()))
    mask = mpnn.output_mask(N)
    for scale in (1.0, 0.5, 2.0):
        t = (tgt * scale).astype(np.float32)
        g = np.zeros(net.P, np.float32)
        mpnn.nat.check(mpnn.nat.lib().plbfs_mpnn_loss_grad(net.h, mpnn.fptr(x), mpnn.fptr(t), mpnn.fptr(mask), None,
                                                           mpnn.fptr(g)))
        assert np.array_equal(g, net.loss_grad(x, t, mask)[1])


def test_parameters_set_behind_an_adam_step(gpu_available):
    """plbfs_mpnn_set_params right behind an Adam step, which returns before its kernel
    has run: the parameters that were set, and moments of zero."""
    N, src, dst, ef, x, tgt = problem(9)
    net = mpnn.Mpnn(N, src, dst, ef, train=True)
    first, mask = mpnn.flatten_params(M.init_params(9), M.mlp_shapes()), mpnn.output_mask(N)
    stepped = []
    for _ in range(3):
        net.set_params(first)
        assert np.array_equal(net.params(), first)
        net.loss_grad(x, tgt, mask)
        net.adam_step(1e-3)
        stepped.append(net.params())
        net.adam_step(1e-3)
    assert not np.array_equal(stepped[0], first)
    assert np.array_equal(stepped[0], stepped[1]) and np.array_equal(stepped[0], stepped[2])


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_overflowed_units_show(gpu_available, sign):
    """A cell whose hidden units overflow to inf or -inf, all weights positive: SiLU is
    a / (1 + e^-a), so its output is inf or NaN, as are those of the cells up to six
    edges away, and no other cell's."""
    N, src, dst, ef, x, _ = problem()
    net = mpnn.Mpnn(N, src, dst, ef, train=False)
    net.set_params(np.full(net.P, 0.01, np.float32))
    x = np.abs(x).astype(np.float32)
    x[0] = sign * 3e38  # 16 columns: beyond the largest float in the encoder's sums
    P = mpnn.unflatten(net.params(), M.mlp_shapes())
    P["enc"]["W1"][:] = 1.0
    net.set_params(mpnn.flatten_params(P, M.mlp_shapes()))
    y = net.forward(x)
    near = np.zeros(N, bool)
    near[0] = True
    for _ in range(6):
        near[dst[near[src]]] = True
    assert 1 < near.sum() < N
    if sign > 0:
        assert np.all(y[near] == np.inf)
    else:
        assert np.isnan(y[near]).all()
    assert np.isfinite(y[~near]).all()
