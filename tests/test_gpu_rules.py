"""Kernels on both sides of the rules that choose them, with the sizes asserted: streamed
tiles, the launch limits of the fused downward pass, the exponential table's end, and the
direct charge sums where the last block is partly empty."""
import re
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


def globule(fa, tmp_path_factory, radius, seed, merge, nq=40):
    return molecule(fa, tmp_path_factory, "globule", 3, radius, "--charges", "inside", "--nq", str(nq), "--sigma", "0.4",
                    "--depth", "1.5", "--seed", str(seed), "--merge", str(merge))


def streamed_rows(tree, frac):
    """The rows of the tiles (16 rows of a leaf) that stream: a tile does while the streamed share
    of the pairs so far stays within frac."""
    a, rows, stored, seen = tree.a, np.zeros(tree.n, bool), 0, 0
    for leaf in range(tree.nleaf):
        ncol = int(a["leafCount"][a["nearSrc"][a["nearOff"][leaf]:a["nearOff"][leaf + 1]]].sum())
        s, c = int(a["leafStart"][leaf]), int(a["leafCount"][leaf])
        for r0 in range(0, c, 16):
            pairs = min(16, c - r0) * ncol
            if stored + pairs <= frac * (seen + pairs):
                stored += pairs
                rows[s + r0:s + min(r0 + 16, c)] = True
            seen += pairs
    return rows, stored


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("depth", [1, 2, 3])
def test_streamed_tiles_same_bits(fa, tmp_path_factory, monkeypatch, precision, depth):
    """A tile that streams its coefficients gives the same bits in the kernel of streamed tiles
    alone as in the one that computes other tiles beside it."""
    import torch
    mesh = molecule(fa, tmp_path_factory, "globule", 4, 15, "--charges", "inside", "--nq", "40", "--sigma", "0.4",
                    "--depth", "1.5", "--seed", "11", "--merge", "0.4")
    tree = fa.Tree(mesh, depth, order=6, height=min(2, depth))
    x = torch.tensor(np.random.default_rng(1).uniform(-1, 1, 2 * tree.n), device="cuda")
    rows, stored = streamed_rows(tree, 0.6)
    out = []
    for frac in ("1", "0.6"):
        monkeypatch.setenv("FABIPB_NEAR_STREAM", frac)
        op = fa.Operator(tree, 0.1257, 1.0, 80.0, 1)
        st = op.stats()
        assert st["near_stored"] == (st["near_interactions"] if frac == "1" else stored)
        y = torch.empty_like(x)
        if precision == "fp32":
            op.enable_fp32()
            op.matvec32_dev(x, y)
        else:
            op.matvec_dev(x, y)
        out.append(y.cpu().numpy().reshape(2, -1)[:, rows])
    assert rows.sum() >= 0.4 * tree.n
    assert (out[0] == out[1]).all(), (out[0] != out[1]).mean()


@pytest.mark.parametrize("depth", [14, 15, 18, 19])
def test_deep_trees(fa, tmp_path_factory, depth):
    """L2L and L2P of a leaf's whole ancestry in one block at order 9: from 15 levels on the
    dynamic LDS and the kernel's own arrays come to more than 64 KiB; at 19 there are more
    levels than the kernel takes and the passes run level by level."""
    import torch
    mesh = molecule(fa, tmp_path_factory, "sphere", 1, 10, "--charges", "ball", "--nq", "20", "--rq", "6", "--seed", "3")
    tree = fa.Tree(mesh, depth, order=9)
    op = fa.Operator(tree, 0.1257, 1.0, 80.0, 1)
    x, y = np.random.default_rng(2).uniform(-1, 1, (2, 2 * tree.n))
    ax = op.matvec(x)
    assert rel(ax, O.Oracle(tree.oracle_layout(0.1257, 1.0, 80.0, 1)).matvec(x)) <= 1e-13
    yd = torch.tensor(y, device="cuda")
    at = torch.empty_like(yd)
    op.matvec_t_dev(yd, at)
    assert abs(float(at.cpu().numpy() @ x) - float(y @ ax)) <= 1e-13 * np.linalg.norm(ax) * np.linalg.norm(y)


def near_bound(tree):
    """The operator's bound on the near distances: the leaves' spheres about their cube centres
    over the one-point rule's points."""
    a, n = tree.a, tree.n
    v = a["vtx"].reshape(n, 3, 3)
    p = v[:, 0] + 0.5 * ((v[:, 1] - v[:, 0]) + 0.5 * (v[:, 2] - v[:, 1]))
    c = a["cubeX"].reshape(-1, 3)[:tree.nleaf]
    leaf = np.repeat(np.arange(tree.nleaf), a["leafCount"])
    rad = np.zeros(tree.nleaf)
    np.maximum.at(rad, leaf, np.linalg.norm(p - c[leaf], axis=1))
    D = np.repeat(np.arange(tree.nleaf), np.diff(a["nearOff"]))
    S = a["nearSrc"]
    return float((np.linalg.norm(c[D] - c[S], axis=1) + rad[D] + rad[S]).max())


def table_end():
    """kappa r up to which e^{-kappa r} comes from the table of steps 1/256."""
    src = open(f"{ROOT}/cuda-fabipb_amd/csrc/fabipb_hip.hip").read()
    return (int(re.search(r"#define FLY64_TAB (\d+)", src)[1]) - 3) / 256.0


@pytest.mark.parametrize("part", [0.7, 0.95, 1 - 1e-6, 1 + 1e-6, 1.5])
def test_exponential_table_end(fa, tmp_path_factory, monkeypatch, part):
    """kappa such that the largest near distance lies before the table's last entries, at them
    and beyond the table: the product, its transpose, and the kappa derivative against the
    full rules of every pair."""
    import torch
    mesh = globule(fa, tmp_path_factory, 8, 9, 0.55)
    tree = fa.Tree(mesh, 2, order=6)
    kappa = part * table_end() / near_bound(tree)
    op = fa.Operator(tree, kappa, 1.0, 80.0, 1)
    x, y = np.random.default_rng(3).uniform(-1, 1, (2, 2 * tree.n))
    ax = op.matvec(x)
    assert rel(ax, O.Oracle(tree.oracle_layout(kappa, 1.0, 80.0, 1)).matvec(x)) <= 1e-13
    xd, yd = torch.tensor(x, device="cuda"), torch.tensor(y, device="cuda")
    at = torch.empty_like(yd)
    op.matvec_t_dev(yd, at)
    assert abs(float(at.cpu().numpy() @ x) - float(y @ ax)) <= 1e-13 * np.linalg.norm(ax) * np.linalg.norm(y)
    kappa_derivative_matches_rules(fa, monkeypatch, op, mesh, tree, xd, yd)


def kappa_derivative_matches_rules(fa, monkeypatch, op, mesh, tree, x, lam0):
    def dk():
        lam = lam0.clone()
        return op.gradient_tree_dev(tree.charge_tree(), mesh.pos, mesh.chr, x, lam, tol=1e6)[1], lam

    fast, l1 = dk()
    monkeypatch.setenv("FABIPB_DK_RULES", "1")
    rules, l2 = dk()
    monkeypatch.delenv("FABIPB_DK_RULES")
    assert bool((l1 == l2).all())
    # as the one-mesh comparison of the two forms: 1e-11 relative, here of a sum that cancels less
    assert abs(fast - rules) <= 1e-11 * abs(rules)


def test_kappa_derivative_every_tile_streamed(fa, tmp_path_factory, monkeypatch):
    """The kappa derivative's nearfield where the operator computes no tile and so keeps no table."""
    import torch
    monkeypatch.setenv("FABIPB_NEAR", "stream")
    mesh = globule(fa, tmp_path_factory, 8, 9, 0.55)
    tree = fa.Tree(mesh, 2, order=6)
    op = fa.Operator(tree, 0.1257, 1.0, 80.0, 1)
    assert op.stats()["near_fly_tiles"] == 0
    x, y = (torch.tensor(v, device="cuda") for v in np.random.default_rng(3).uniform(-1, 1, (2, 2 * tree.n)))
    kappa_derivative_matches_rules(fa, monkeypatch, op, mesh, tree, x, y)


@pytest.mark.parametrize("merge,n", [(0.5, 1256), (0.55, 1182)])
@pytest.mark.parametrize("nchar", [1, 33, 130])
def test_direct_sums_partial_block(fa, tmp_path_factory, merge, n, nchar):
    """The direct right-hand side where the last block of 64 panels is partly empty.  2e-14:
    2,000 roundings of 2^-53 against the largest sum."""
    mesh = globule(fa, tmp_path_factory, 8, 9, merge)
    tree = fa.Tree(mesh, 2, order=6)
    assert tree.n == n and n % 64 != 0
    rng = np.random.default_rng(nchar)
    pos, q = rng.uniform(-2, 2, (nchar, 3)), rng.normal(0, 0.4, nchar)
    ora = O.Oracle(tree.oracle_layout(0.1257, 1.0, 80.0, 1))
    b, ref = fa.Operator(tree, 0.1257, 1.0, 80.0, 1).rhs(pos, q), ora.rhs(pos, q)
    tot = sum(np.abs(ora.rhs(pos[k:k + 1], q[k:k + 1])) for k in range(nchar))
    assert (np.abs(b - ref) <= 2e-14 * tot.max()).all()


@pytest.mark.parametrize("nchar", [7, 127, 130, 300])
def test_direct_gradient_partial_block(fa, tmp_path_factory, nchar):
    """R^T lam by tiles of 128 charges over a panel count that fills neither the last staged 256
    panels nor a quarter of them: the gradient of a zero density against the oracle's
    right-hand sides of unit charges.  3e-13 covers the roundings of 2,532 terms of 2^-53 each."""
    import torch
    mesh = globule(fa, tmp_path_factory, 12, 5, 1.1, nchar)
    tree = fa.Tree(mesh, 2, order=6)
    assert tree.n == 1266 and tree.n % 256 != 0 and tree.n % 4 != 0
    op = fa.Operator(tree, 0.1257, 1.0, 80.0, 1)
    ora = O.Oracle(tree.oracle_layout(0.1257, 1.0, 80.0, 1))
    lam = torch.tensor(np.random.default_rng(3).uniform(-1, 1, 2 * tree.n), device="cuda")
    dq, _, _ = op.gradient_tree_dev(tree.charge_tree(), mesh.pos, mesh.chr, torch.zeros_like(lam), lam, tol=1e-8)
    u = lam.cpu().numpy()
    cols = [ora.rhs(mesh.pos[k:k + 1], np.ones(1)) for k in range(nchar)]
    want = np.array([u @ c for c in cols])
    tot = np.array([np.abs(u) @ np.abs(c) for c in cols])
    assert (np.abs(dq - want) <= 3e-13 * tot).all()
