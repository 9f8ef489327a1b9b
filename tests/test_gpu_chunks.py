"""The value-polling chunk sweeps, in LDS and in memory, on layered graphs:
rows with as many dependencies as their slots (4, 8, 12, 16, 32), one more,
and more than the largest, against the oracle's sequential loops."""
import numpy as np
import pytest

import foamhip as fh
import oracle as O
from meshes import asym_coeffs, spd_coeffs

pytestmark = pytest.mark.gpu


def layered(width, layers, deg, rng, spread):
    """layers of `width` cells; every cell has deg neighbours in the layer
    before (spread: 1 to deg of them), so the layers are the levels."""
    pairs = []
    for l in range(1, layers):
        for c in range(width):
            n = rng.integers(1, deg + 1) if spread else deg
            for p in rng.choice(width, n, replace=False):
                pairs.append(((l - 1) * width + p, l * width + c))
    pairs = np.array(sorted(pairs), dtype=np.int32)
    return width * layers, pairs[:, 0].copy(), pairs[:, 1].copy()


@pytest.mark.parametrize("deg,spread", [(1, False), (4, False), (5, True), (8, False), (9, True),
                                        (12, False), (16, False), (17, True), (32, False),
                                        (45, True)])
@pytest.mark.parametrize("kind", ["spd", "asym"])
@pytest.mark.parametrize("where", ["lds", "memory"])
def test_chunk_sweeps_bitwise(deg, spread, kind, where):
    rng = np.random.default_rng(41 + deg)
    # more than 4 chunks a level go through memory
    width = 300 if where == "memory" else 70 if deg < 32 else 130
    n, lower, upper = layered(width, 7 if where == "lds" else 4, deg, rng, spread)
    co = (spd_coeffs if kind == "spd" else asym_coeffs)(n, lower, upper, rng)
    m = fh.lduMatrix(fh.lduAddressing(n, lower, upper), *co)
    om = O.Matrix(O.Addr(n, lower, upper), *co)
    psi, b = rng.standard_normal(n), rng.standard_normal(n)
    for smoother in ("GaussSeidel", "symGaussSeidel"):
        np.testing.assert_array_equal(m.smooth(smoother, psi, b, 2),
                                      om.smooth(smoother, psi, b, 2))
    precon = "DIC" if kind == "spd" else "DILU"
    np.testing.assert_array_equal(m.precondition(precon, b), om.precondition(precon, b))


@pytest.mark.parametrize("n", [1, 2, 300, 18432, 18433])
@pytest.mark.parametrize("kind", ["spd", "asym"])
def test_chain_and_lds_limit(n, kind):
    """One row per level, up to the most rows the LDS sweep takes (FP64) and
    one more, with a second diagonal so that a level reads two earlier ones."""
    rng = np.random.default_rng(n)
    i = np.arange(n, dtype=np.int32)
    pairs = np.concatenate([np.stack([i[:-1], i[1:]], 1), np.stack([i[:-3], i[3:]], 1)]) \
        if n > 3 else np.stack([i[:-1], i[1:]], 1)
    pairs = pairs[np.lexsort((pairs[:, 1], pairs[:, 0]))]
    lower, upper = pairs[:, 0].copy(), pairs[:, 1].copy()
    co = (spd_coeffs if kind == "spd" else asym_coeffs)(n, lower, upper, rng)
    m = fh.lduMatrix(fh.lduAddressing(n, lower, upper), *co)
    om = O.Matrix(O.Addr(n, lower, upper), *co)
    psi, b = rng.standard_normal(n), rng.standard_normal(n)
    for smoother in ("GaussSeidel", "symGaussSeidel"):
        np.testing.assert_array_equal(m.smooth(smoother, psi, b, 2),
                                      om.smooth(smoother, psi, b, 2))
    precon = "DIC" if kind == "spd" else "DILU"
    np.testing.assert_array_equal(m.precondition(precon, b), om.precondition(precon, b))


@pytest.mark.parametrize("kind", ["spd", "asym"])
@pytest.mark.parametrize("width", [40, 300])
def test_infinite_factor_of_a_cell_without_faces(width, kind):
    """A cell without faces and with a zero diagonal has an infinite factor:
    its result is that factor times the residual, as it has no neighbour
    values to take (in LDS, and in memory with the wider levels)."""
    rng = np.random.default_rng(width)
    n, lower, upper = layered(width, 5, 3, rng, True)
    alone = np.array([0, n + 1], np.int32)          # two more cells, first and last
    lower, upper = lower + 1, upper + 1
    n += 2
    co = list((spd_coeffs if kind == "spd" else asym_coeffs)(n, lower, upper, rng))
    co[0][alone] = 0.0
    m = fh.lduMatrix(fh.lduAddressing(n, lower, upper), *co)
    om = O.Matrix(O.Addr(n, lower, upper), *co)
    r = rng.standard_normal(n)
    precon = "DIC" if kind == "spd" else "DILU"
    ref = om.precondition(precon, r)
    assert np.isinf(ref[alone]).all() and np.isfinite(np.delete(ref, alone)).all()
    np.testing.assert_array_equal(m.precondition(precon, r), ref)
    w = m.precondition_f32(precon, r)
    np.testing.assert_array_equal(w[alone], ref[alone].astype(np.float32))
    assert np.isfinite(np.delete(w, alone)).all()


@pytest.mark.parametrize("width,deg", [(15900, 3), (16100, 3), (8100, 8), (4100, 12), (2100, 30)])
@pytest.mark.parametrize("kind", ["spd", "asym"])
def test_wide_levels_bitwise(width, deg, kind):
    """Levels of many chunks, where the rows wait for a chunk's last
    dependency before they load them all (4, 8, 16 and 32 slots; just under
    the first limit, too)."""
    rng = np.random.default_rng(width)
    c = np.arange(width)
    hop = rng.choice(np.arange(1, width), deg, replace=False)
    pairs = np.concatenate([np.stack([l * width + (c + h) % width, (l + 1) * width + c], 1)
                            for l in range(3) for h in hop]).astype(np.int32)
    pairs = pairs[np.lexsort((pairs[:, 1], pairs[:, 0]))]
    n, lower, upper = 4 * width, pairs[:, 0].copy(), pairs[:, 1].copy()
    co = (spd_coeffs if kind == "spd" else asym_coeffs)(n, lower, upper, rng)
    m = fh.lduMatrix(fh.lduAddressing(n, lower, upper), *co)
    om = O.Matrix(O.Addr(n, lower, upper), *co)
    psi, b = rng.standard_normal(n), rng.standard_normal(n)
    np.testing.assert_array_equal(m.smooth("symGaussSeidel", psi, b, 2),
                                  om.smooth("symGaussSeidel", psi, b, 2))
    precon = "DIC" if kind == "spd" else "DILU"
    np.testing.assert_array_equal(m.precondition(precon, b), om.precondition(precon, b))


@pytest.mark.parametrize("deg", [16, 17, 40])
@pytest.mark.parametrize("kind", ["spd", "asym"])
def test_few_rows_of_many_entries_in_lds(deg, kind):
    """The LDS sweep's rows past its 16 slots: few enough of them that the
    mesh stays in LDS (a chain of 64-cell levels with hubs of deg lower and
    deg upper neighbours)."""
    rng = np.random.default_rng(deg)
    width, layers = 64, 24
    pairs = {((l - 1) * width + c, l * width + c) for l in range(1, layers) for c in range(width)}
    for l in range(1, layers - 1, 3):
        hub = l * width + int(rng.integers(width))
        pairs |= {((l - 1) * width + int(p), hub) for p in rng.choice(width, deg, replace=False)}
        pairs |= {(hub, (l + 1) * width + int(p)) for p in rng.choice(width, deg, replace=False)}
    pairs = np.array(sorted(pairs), dtype=np.int32)
    n, lower, upper = width * layers, pairs[:, 0].copy(), pairs[:, 1].copy()
    co = (spd_coeffs if kind == "spd" else asym_coeffs)(n, lower, upper, rng)
    m = fh.lduMatrix(fh.lduAddressing(n, lower, upper), *co)
    om = O.Matrix(O.Addr(n, lower, upper), *co)
    psi, b = rng.standard_normal(n), rng.standard_normal(n)
    for smoother in ("GaussSeidel", "symGaussSeidel"):
        np.testing.assert_array_equal(m.smooth(smoother, psi, b, 2),
                                      om.smooth(smoother, psi, b, 2))
    precon = "DIC" if kind == "spd" else "DILU"
    np.testing.assert_array_equal(m.precondition(precon, b), om.precondition(precon, b))
