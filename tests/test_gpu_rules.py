"""Kernels on both sides of the rules that choose them, with the sizes asserted."""
import subprocess

import numpy as np
import pytest

from conftest import ROOT

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
