"""The table by which the V-cycle gathers corner sums at the vertices: its packing on the CPU, and solves on
a mesh with a vertex of many elements against the FP64 oracle."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import hoc
from hoc import meshes
from pyoracle import Oracle
from conftest import rel_l2

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ho-cxx_amd", "csrc")


def test_packing(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    exe = tmp_path / "gather_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, os.path.join(ROOT, "tests", "cpp", "gather_check.cpp"),
                    os.path.join(CSRC, "hoc_host.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), out.stdout


def fan(m):
    """m kites round one vertex."""
    t = 2 * np.pi * np.arange(m) / m
    a = 0.6 * np.stack([np.cos(t), np.sin(t)], 1)
    b = np.stack([np.cos(t + np.pi / m), np.sin(t + np.pi / m)], 1)
    i, j = np.arange(m), (np.arange(m) + 1) % m
    el = np.stack([np.zeros(m, int), 1 + i, 1 + m + i, 1 + j], 1).astype(np.int32)
    ed = np.concatenate([el[:, 1:3], el[:, 2:4]]).astype(np.int32)
    names = list(meshes.cavity(2, 2).bnames)
    return meshes.QuadMesh(2, np.concatenate([np.zeros((1, 2)), a, b]), el, ed, np.zeros(2 * m, np.int32), names)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [hoc.HOC_FP64, hoc.HOC_MIXED])
# vertices in the fused dense product (5 and 12 kites: one width for all; 120: slices of their own), and in
# the sparse levels, where the fan stands beside a cavity
@pytest.mark.parametrize("m,beside", [(5, 0), (12, 0), (120, 0), (120, 45)])
def test_solve_on_a_fan(gpu_available, m, beside, precision):
    parts = [fan(m)] + ([meshes.cavity(beside, 2)] if beside else [])
    mesh, off = meshes.concat(parts)
    kw = dict(problem_type=1, Re=100.0, dt=1e-4, time_integration_type=4, advection_type=1, tol=1e-13, maxiter=400)
    g = hoc.HO2D(K=3, precision=precision, **kw)
    g.load_mesh(mesh)
    g.setup()
    w = np.random.default_rng(m).standard_normal(g.D)
    # an oracle for each part: its BiCGSTAB stagnates on the two together
    want = np.concatenate([Oracle(p, 3, **kw).poisson(w[9 * i:9 * j]) for p, i, j in zip(parts, off, off[1:])])
    e = rel_l2(g.poisson(w), want)
    print("kites", m, "beside", beside, "its", g.stats()["last_iters"], "rel", e)
    # both sides solve to 1e-13 of a system whose condition number is below 1e5
    assert g.stats()["last_rel_residual"] <= 1e-13 and e < 1e-8
    g.close()
