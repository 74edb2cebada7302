"""Kernels chosen by a rule on sizes or parameters, on both sides of the rule and at
its edges, against the oracle (FP64 bar of the parity tests: 1e-13 relative)."""
import subprocess

import numpy as np
import pytest

import oracle_binding as O
from conftest import ROOT, rel

pytestmark = pytest.mark.gpu
_meshes = {}


def molecule(fa, tmp_path_factory, kind, level, radius, *extra):
    key = (kind, level, radius) + extra
    if key not in _meshes:
        base = str(tmp_path_factory.mktemp("mesh") / "m")
        subprocess.check_call([f"{ROOT}/cuda-fabipb_amd/bin/fbmesh", kind, base, "--level", str(level), "--radius",
                               str(radius), *extra], stdout=subprocess.DEVNULL)
        _meshes[key] = fa.Mesh(base)
    return _meshes[key]


GLOBULE = ("--charges", "inside", "--nq", "40", "--sigma", "0.4", "--depth", "1.5", "--seed", "9", "--merge", "0.45")


@pytest.mark.parametrize("kappa,depth", [(0.0, 2), (1e-4, 2), (0.1257, 2), (0.1257, 1), (0.3, 1), (2.5, 2)])
def test_near_exponential_table(fa, tmp_path_factory, kappa, depth):
    """The nearfield's table of e^{-kappa r} (kappa times the near distances up to 4) and
    the general form beyond it; leaves whose row count leaves every remainder of a tile."""
    mesh = molecule(fa, tmp_path_factory, "globule", 3, 8, *GLOBULE)
    tree = fa.Tree(mesh, depth, order=6, height=min(2, depth))
    op = fa.Operator(tree, kappa, 1.0, 80.0, 1)
    x, y = np.random.default_rng(1).uniform(-1, 1, (2, 2 * tree.n))
    ora = O.Oracle(tree.oracle_layout(kappa, 1.0, 80.0, 1))
    ax = op.matvec(x)
    assert rel(ax, ora.matvec(x)) <= 1e-13
    if op.stats()["m2l_pairs"] == 0:   # one level: the adjoint operator needs M2L tensors
        return
    import torch
    yd = torch.tensor(y, device="cuda")
    at = torch.empty_like(yd)
    op.matvec_t_dev(yd, at)
    scale = np.linalg.norm(ax) * np.linalg.norm(y)
    assert abs(float(at.cpu().numpy() @ x) - float(y @ ax)) <= 1e-13 * scale


@pytest.mark.parametrize("order,depth,mac", [(1, 2, 0.8), (3, 3, 0.8), (4, 2, 0.8), (7, 2, 0.8), (8, 3, 0.7), (9, 2, 0.8)])
def test_far_chain_orders(fa, tmp_path_factory, order, depth, mac):
    """Q2M and L2P from the moment matrix alone, for every split of a column over a wave's
    lanes (one or two slots, one to three strides), forward and transposed."""
    import torch
    mesh = molecule(fa, tmp_path_factory, "globule", 3, 8, *GLOBULE)
    tree = fa.Tree(mesh, depth, order=order, sep=mac)
    op = fa.Operator(tree, 0.1257, 1.0, 80.0, 1)
    x, y = np.random.default_rng(2).uniform(-1, 1, (2, 2 * tree.n))
    ora = O.Oracle(tree.oracle_layout(0.1257, 1.0, 80.0, 1))
    ax = op.matvec(x)
    assert rel(ax, ora.matvec(x)) <= 1e-13
    assert rel(op.far_apply(x), ora.apply(x, parts=1)) <= 1e-13   # the stage form
    yd = torch.tensor(y, device="cuda")
    at = torch.empty_like(yd)
    op.matvec_t_dev(yd, at)
    assert abs(float(at.cpu().numpy() @ x) - float(y @ ax)) <= 1e-13 * np.linalg.norm(ax) * np.linalg.norm(y)


@pytest.mark.parametrize("order,mac", [(1, 0.8), (2, 0.8), (5, 0.8), (6, 0.8), (7, 0.8), (8, 0.7), (9, 0.8)])
def test_charge_walks_orders(fa, tmp_path_factory, order, mac):
    """The walks' far term from one table per cluster (value and derivative along the normal
    by one Horner scheme): energy, its weights' kappa derivative and the right-hand side."""
    import torch
    mesh = molecule(fa, tmp_path_factory, "globule", 3, 12, "--charges", "inside", "--nq", "400", "--sigma", "0.4",
                    "--depth", "1.5", "--seed", "5")
    tree = fa.Tree(mesh, 3, order=order, sep=mac)
    ct = tree.charge_tree()
    op = fa.Operator(tree, 0.1257, 1.0, 80.0, 1)
    ora = O.Oracle(tree.oracle_layout(0.1257, 1.0, 80.0, 1))
    op.set_charges(ct, mesh.pos, mesh.chr)
    b = torch.empty(2 * tree.n, dtype=torch.float64, device="cuda")
    op.rhs_tree_res_dev(b)
    assert rel(b.cpu().numpy(), ora.rhs_tree(ct, mesh.pos, mesh.chr)) <= 1e-13
    e = op.energy_res_dev(b)   # a density that does not cancel
    assert abs(e - ora.energy(ct, mesh.pos, mesh.chr, b.cpu().numpy())) <= 1e-12 * abs(e)
    assert abs(op.energy_res_dev(b, precision="fp32") - e) <= 3e-7 * abs(e)   # its tables built after the FP64 walk's
    assert op.energy_res_dev(b) == e


@pytest.mark.parametrize("nchar", [1, 15, 33, 127, 130, 1000])
def test_direct_charge_sums(fa, tmp_path_factory, nchar):
    """The direct right-hand side (its charges split over the waves of a block) and its
    transpose (tiles of 128 charges), for counts around the splits; 1,272 panels, the last
    block of 64 partly empty.  2e-14: 2,000 roundings of 2^-53 against the largest sum."""
    import torch
    mesh = molecule(fa, tmp_path_factory, "globule", 3, 8, *GLOBULE)
    tree = fa.Tree(mesh, 2, order=6)
    rng = np.random.default_rng(nchar)
    pos = rng.uniform(-2, 2, (nchar, 3))
    q = rng.normal(0, 0.4, nchar)
    op = fa.Operator(tree, 0.1257, 1.0, 80.0, 1)
    ora = O.Oracle(tree.oracle_layout(0.1257, 1.0, 80.0, 1))
    b = op.rhs(pos, q)
    ref = ora.rhs(pos, q)
    one = [ora.rhs(pos[k:k + 1], np.abs(q[k:k + 1])) for k in range(min(nchar, 4))]
    scale = np.abs(ref).max() + sum(np.abs(o).max() for o in one)
    assert np.abs(b - ref).max() <= 2e-14 * scale


@pytest.mark.parametrize("nchar", [7, 127, 130, 400])
def test_direct_gradient_sums(fa, tmp_path_factory, nchar):
    """R^T lam by tiles of 128 charges (the transposed direct right-hand side): the gradient
    of a zero density, against the oracle's right-hand sides of unit charges; counts around
    the tile.  1,278 panels: 3e-13 covers the roundings of 2,556 terms of 2^-53 each."""
    import torch
    mesh = molecule(fa, tmp_path_factory, "globule", 3, 12, "--charges", "inside", "--nq", str(nchar), "--sigma", "0.4",
                    "--depth", "1.5", "--seed", "5", "--merge", "0.6")
    tree = fa.Tree(mesh, 2, order=6)
    op = fa.Operator(tree, 0.1257, 1.0, 80.0, 1)
    ora = O.Oracle(tree.oracle_layout(0.1257, 1.0, 80.0, 1))
    lam = torch.tensor(np.random.default_rng(3).uniform(-1, 1, 2 * tree.n), device="cuda")
    dq, _, _ = op.gradient_tree_dev(tree.charge_tree(), mesh.pos, mesh.chr, torch.zeros_like(lam), lam, tol=1e-8)
    u = lam.cpu().numpy()
    cols = [ora.rhs(mesh.pos[k:k + 1], np.ones(1)) for k in range(nchar)]
    want = np.array([u @ c for c in cols])
    tot = np.array([np.abs(u) @ np.abs(c) for c in cols])
    assert (np.abs(dq - want) <= 3e-13 * tot).all()


@pytest.mark.parametrize("depth", [2, 4])
def test_product_in_place(fa, tmp_path_factory, depth):
    """The product whose combine ends the L2P (up to 10M near pairs; depth 2 of 20,480 panels is
    above it, depth 4 below): alpha, beta and y = x, forward and transposed, against the
    oracle and against the two-argument form."""
    import torch
    mesh = molecule(fa, tmp_path_factory, "sphere", 5, 20, "--charges", "ball", "--nq", "20", "--rq", "12", "--seed", "3")
    tree = fa.Tree(mesh, depth, order=6)
    op = fa.Operator(tree, 0.1257, 1.0, 80.0, 1)
    assert (op.stats()["near_interactions"] > 10_000_000) == (depth == 2)
    x, y0 = np.random.default_rng(4).uniform(-1, 1, (2, 2 * tree.n))
    ora = O.Oracle(tree.oracle_layout(0.1257, 1.0, 80.0, 1))
    ax = ora.matvec(x)
    assert rel(op.matvec(x, 0.75, -0.5, y0.copy()), 0.75 * ax - 0.5 * y0) <= 1e-13
    xd = torch.tensor(x, device="cuda")
    for f in (op.matvec_dev, op.matvec_t_dev):
        y, z = torch.tensor(y0, device="cuda"), xd.clone()
        f(xd, y, alpha=0.75, beta=-0.5)
        f(z, z)
        p = torch.empty_like(xd)
        f(xd, p)
        assert torch.equal(z, p)
        assert rel(y.cpu().numpy(), 0.75 * p.cpu().numpy() - 0.5 * y0) <= 1e-14
