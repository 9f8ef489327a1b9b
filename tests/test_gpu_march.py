"""The marching sweeps of hex boxes (16 x 16 pencils along k) against the
oracle's sequential loops at the sizes where they can go wrong: one partial
pencil, several with remainders along each side, the fewest planes they
take, planes around the ring's 64, and more pencils than compute units."""
import numpy as np
import pytest

import foamhip as fh
import oracle as O
from foamhip.cases import BoxCase
from meshes import asym_coeffs, spd_coeffs

pytestmark = pytest.mark.gpu

SIZES = [(2, 2, 17), (2, 3, 70), (5, 3, 70), (16, 16, 16), (17, 33, 19), (16, 64, 63), (40, 18, 133),
         (33, 47, 64), (270, 270, 17)]


def systems(size, kind, seed=5):
    c = BoxCase(*size)
    rng = np.random.default_rng(seed)
    a = O.Addr(c.N, c.lower, c.upper)
    mesh = fh.lduAddressing(c.N, c.lower, c.upper)
    assert mesh.info()["tiled"]
    if kind == "spd":
        co = spd_coeffs(c.N, c.lower, c.upper, rng)
    else:
        co = asym_coeffs(c.N, c.lower, c.upper, rng)
    return c, rng, fh.lduMatrix(mesh, *co), O.Matrix(a, *co)


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("kind,precon", [("spd", "DIC"), ("asym", "DILU")])
def test_march_precondition_bitwise(size, kind, precon):
    c, rng, m, om = systems(size, kind)
    for _ in range(3):       # every launch leaves the halos ready for the next
        r = rng.standard_normal(c.N)
        np.testing.assert_array_equal(m.precondition(precon, r), om.precondition(precon, r))


@pytest.mark.parametrize("size", SIZES[:6])
@pytest.mark.parametrize("kind,precon", [("spd", "DIC"), ("asym", "DILU")])
def test_march_f32(size, kind, precon):
    """The FP32 pass: a row is three products and three differences, and its
    error reaches the rows after it with the couplings of a diagonally
    dominant factor (a sum below one), so a few units of 2^-24 of the
    largest value, 64 allowed."""
    c, rng, m, om = systems(size, kind)
    r = rng.standard_normal(c.N)
    w = m.precondition_f32(precon, r).astype(np.float64)
    ow = om.precondition(precon, r.astype(np.float32).astype(np.float64))
    assert np.abs(w - ow).max() <= 64 * 2.0**-24 * np.abs(ow).max()


@pytest.mark.parametrize("size", SIZES[1:6])
@pytest.mark.parametrize("kind", ["spd", "asym"])
def test_march_solves(size, kind):
    """Solves whose sums w.r come from the backward pass: the oracle's
    iteration count and solution; non-finite input is reported."""
    c, rng, m, om = systems(size, kind)
    ctl = {"solver": "PCG" if kind == "spd" else "PBiCGStab",
           "preconditioner": "DIC" if kind == "spd" else "DILU", "tolerance": 1e-9, "relTol": 0}
    b = rng.standard_normal(c.N)
    psi = np.zeros(c.N)
    perf = fh.solver_New("p", m, ctl).solve(psi, b)
    opsi, operf = om.solve(ctl, np.zeros(c.N), b)
    assert abs(perf.nIterations - operf["nIterations"]) <= 1
    assert np.linalg.norm(psi - opsi) <= 1e-8 * np.linalg.norm(opsi)
    b[c.N // 2] = np.nan
    with pytest.raises(fh.FoamHipError):
        fh.solver_New("p", m, ctl).solve(np.zeros(c.N), b)
    # the halos stay in order after it
    r = rng.standard_normal(c.N)
    p = ctl["preconditioner"]
    np.testing.assert_array_equal(m.precondition(p, r), om.precondition(p, r))


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("kind", ["spd", "asym"])
@pytest.mark.parametrize("smoother", ["GaussSeidel", "symGaussSeidel"])
def test_march_gauss_seidel_bitwise(size, kind, smoother):
    """Gauss-Seidel sweeps from a start that is not zero, two of them and one
    more on the same matrix, and again after its coefficients changed."""
    c, rng, m, om = systems(size, kind)
    psi, b = rng.standard_normal(c.N), rng.standard_normal(c.N)
    for n in (2, 1):
        ref = om.smooth(smoother, psi, b, n)
        np.testing.assert_array_equal(m.smooth(smoother, psi, b, n), ref)
    co = (spd_coeffs if kind == "spd" else asym_coeffs)(c.N, c.lower, c.upper, rng)
    m.set(*co)
    om2 = O.Matrix(O.Addr(c.N, c.lower, c.upper), *co)
    np.testing.assert_array_equal(m.smooth(smoother, psi, b, 1), om2.smooth(smoother, psi, b, 1))


@pytest.mark.parametrize("box_sweep", ["wave", "wide"])
@pytest.mark.parametrize("size", [(2, 3, 70), (17, 33, 19), (40, 18, 133), (33, 47, 64)])
@pytest.mark.parametrize("kind", ["spd", "asym"])
def test_tiles_of_many_planes_bitwise(size, kind, box_sweep, monkeypatch):
    """The tile kernels that boxes beyond the marching sweeps' limits take,
    with tiles waiting on tiles along k as well, and the pencils between
    them on the same matrix."""
    c, rng, m, om = systems(size, kind)
    precon = "DIC" if kind == "spd" else "DILU"
    psi, r = rng.standard_normal(c.N), rng.standard_normal(c.N)
    ref = om.precondition(precon, r), om.smooth("symGaussSeidel", psi, r, 2)
    march32 = m.precondition_f32(precon, r)
    for forced in (box_sweep, "", box_sweep):
        monkeypatch.setenv("FOAMHIP_BOX_SWEEP", forced)
        np.testing.assert_array_equal(m.precondition(precon, r), ref[0])
        np.testing.assert_array_equal(m.smooth("symGaussSeidel", psi, r, 2), ref[1])
    # the same operations in FP32
    np.testing.assert_array_equal(m.precondition_f32(precon, r), march32)


@pytest.mark.parametrize("size", [(2, 2, 20000), (2, 2, 40000), (600, 2, 2000)])
def test_thin_boxes(size):
    """Boxes of which a pencil is mostly padding: up to a GiB of packed
    coefficients they march, beyond that they stay on the tiles, whose
    buffers are a few vectors."""
    torch = pytest.importorskip("torch")
    used = lambda: (lambda free, total: total - free)(*torch.cuda.mem_get_info())
    c, rng, m, om = systems(size, "spd")
    psi, r = rng.standard_normal(c.N), rng.standard_normal(c.N)
    np.testing.assert_array_equal(m.precondition("diagonal", r), om.precondition("diagonal", r))
    before = used()
    np.testing.assert_array_equal(m.precondition("DIC", r), om.precondition("DIC", r))
    np.testing.assert_array_equal(m.smooth("symGaussSeidel", psi, r, 1),
                                  om.smooth("symGaussSeidel", psi, r, 1))
    assert used() - before <= max(1 << 30, 4 * 18 * 8 * c.N)
    if size == (2, 2, 40000):
        assert used() - before <= 32 * 8 * c.N
