"""The request loop: every result of a mixed stream of concurrent requests
is bitwise the result of the same request solved alone, admission by the
memory budget still completes every request, and the timestamps order."""
import numpy as np
import pytest

import foamhip as fh
from foamhip.cases import BoxCase
from foamhip.serve import Server

pytestmark = pytest.mark.gpu


def systems():
    out = []
    for i, (n, ctl) in enumerate([
            (8, {"solver": "PCG", "preconditioner": "DIC", "precision": "mixed"}),
            (12, {"solver": "PCG", "preconditioner": "DIC"}),
            (16, {"solver": "PCG", "preconditioner": "DIC", "precision": "mixed"}),
            (20, {"solver": "GAMG", "smoother": "GaussSeidel"}),
            (24, {"solver": "PCG", "preconditioner": "DIC", "precision": "mixed"}),
            (10, {"solver": "PBiCGStab", "preconditioner": "diagonal"})]):
        c = BoxCase(n)
        mesh = fh.lduAddressing(c.N, c.lower, c.upper)
        gamma = c.lognormal(40 + i, 0.8, 4.0)
        diag, upper, source = c.laplacian_system(gamma, c.rhs(70 + i))
        out.append({"mesh": mesh, "diag": diag, "upper": upper, "source": source,
                    "controls": dict(ctl, tolerance=1e-8, relTol=0, maxIter=3000)})
    return out


def alone(s, source):
    m = fh.lduMatrix(s["mesh"], s["diag"], s["upper"])
    psi = np.zeros(s["mesh"].nCells)
    perf = fh.solver_New("p", m, s["controls"]).solve(psi, source)
    return psi, perf


@pytest.mark.parametrize("budget", [32 << 30, 1])
def test_mix_equals_alone(budget):
    S = systems()
    reqs = []
    for k in range(30):
        s = S[(k * 7) % len(S)]
        src = s["source"] * (1.0 + 0.01 * k)
        reqs.append((s, src))
    ref = [alone(s, src) for s, src in reqs]
    srv = Server(maxConcurrent=6, memoryBudget=budget)
    for k, (s, src) in enumerate(reqs):
        srv.submit(k, s["mesh"], s["diag"], s["upper"], src, s["controls"])
    got = {}
    while len(got) < len(reqs):
        r = srv.wait(60.0)
        assert r is not None, "server stalled"
        assert r["status"] == 0, r["message"]
        assert r["submit"] <= r["start"] <= r["end"]
        got[r["id"]] = (srv.fetch(r["id"]), r)
    assert srv.pending() == 0
    srv.close()
    for k, (psi_ref, perf_ref) in enumerate(ref):
        psi, r = got[k]
        np.testing.assert_array_equal(psi, psi_ref)
        assert r["nIterations"] == perf_ref.nIterations


def test_budget_counts_what_a_request_uses():
    """Mixed solves with the tile-local preconditioner take none of the
    marching sweeps' buffers: 4 matrices of 20^3 cells are solved at once
    under the 4.3 MB each that their values and vectors are priced at."""
    c = BoxCase(20)
    mesh = [fh.lduAddressing(c.N, c.lower, c.upper) for _ in range(4)]
    diag, upper, source = c.laplacian_system(c.lognormal(9, 0.8, 4.0), c.rhs(3))
    # (a tolerance that is never met: each solve lasts 4000 iterations)
    ctl = {"solver": "PCG", "preconditioner": "DIC", "precision": "mixed", "tolerance": 0,
           "relTol": 0, "maxIter": 4000}
    srv = Server(maxConcurrent=4, memoryBudget=4 * 4_300_000)
    for k in range(4):
        srv.submit(k, mesh[k], diag, upper, source, ctl)
    got = [srv.wait(60.0) for _ in range(4)]
    srv.close()
    assert all(r is not None and r["status"] == 0 for r in got)
    assert max(r["start"] for r in got) < min(r["end"] for r in got)


@pytest.mark.parametrize("budget", [1, 2 * 4_300_000, 3 * 4_300_000, 32 << 30])
def test_resident_matrix_takes_more_buffers_later(budget):
    """Requests on two meshes whose later controls add the marching sweeps'
    buffers to matrices that are resident: every request is admitted, also
    where the budget holds one matrix or none, and solved as if alone."""
    c = BoxCase(20)
    mesh = [fh.lduAddressing(c.N, c.lower, c.upper) for _ in range(2)]
    diag, upper, source = c.laplacian_system(c.lognormal(9, 0.8, 4.0), c.rhs(3))
    common = {"tolerance": 1e-8, "relTol": 0, "maxIter": 3000}
    controls = [dict(common, solver="PCG", preconditioner="DIC", precision="mixed"),
                dict(common, solver="PCG", preconditioner="DIC"),
                dict(common, solver="smoothSolver", smoother="symGaussSeidel", maxIter=20)]
    ref = [alone({"mesh": mesh[0], "diag": diag, "upper": upper, "controls": ctl}, source)[0]
           for ctl in controls]
    srv = Server(maxConcurrent=3, memoryBudget=budget)
    for k in range(12):
        srv.submit(k, mesh[k % 2], diag, upper, source, controls[k // 2 % 3])
    for _ in range(12):
        r = srv.wait(60.0)
        assert r is not None and r["status"] == 0, "server stalled"
        np.testing.assert_array_equal(srv.fetch(r["id"]), ref[r["id"] // 2 % 3])
    srv.close()
