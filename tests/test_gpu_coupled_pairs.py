"""MD-coupled runs in pairs of steps (the two-step kernel and the boxes around the coupled cells) against single
steps, each with its re-collision: the same bits.  Coupled cells on every face, edge and wrap of the box and
next to solids; both modes, with and without densities; lattices that the rule sends to the pairs."""
import numpy as np
import pytest

from madpac_amd import lbm
from test_gpu_pair import BRICKS, ROWS

pytestmark = pytest.mark.gpu


def _cells(size, rng):
    nx, ny, nz = size
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    region = ((abs(x - nx // 2) < 9) & (abs(y - ny // 3) < 7) & (abs(z - nz // 2) < 8)).reshape(-1)
    ids = np.flatnonzero(region)
    corners = [i + nx * (j + ny * k) for i in (0, nx - 1) for j in (0, ny - 1) for k in (0, nz - 1)]
    return rng.permutation(np.union1d(ids, corners + list(rng.choice(nx * ny * nz, 20, replace=False))))


def _run(size, scene, prec, order, mode, with_rho, chunks, graph=False):
    nx, ny, nz = size
    rng = np.random.default_rng(nx * ny + nz)
    n = nx * ny * nz
    solid = rng.random(n) < (0.1 if scene != "open" else 0.0)
    periodic = (True, True, True) if scene == "open" else ((True, False, True) if scene == "porous" else (False,) * 3)
    out = []
    with lbm.Lattice(nx, ny, nz, 0.6, precision=prec, periodic=periodic, cell_order=order) as lat:
        cells = _cells(size, rng)
        lat.set_coupling_cells(cells)
        lat.set_flags(~solid)  # may switch the cell order: the coupled cells follow
        if scene == "cavity":
            lat.set_cavity_lid(0.05)
        lat.init_equilibrium(1 + 0.01 * rng.standard_normal(n), 0.02 * rng.standard_normal((n, 3)))
        for _ in range(2):
            rho = 1 + 0.01 * rng.standard_normal(len(cells)) if with_rho else None
            lat.set_coupling_data(mode, 0.02 * rng.standard_normal((len(cells), 3)), rho, dt=0.9)
            for k in chunks:
                lat.step(k, graph=graph)
            out += list(lat.get_coupling_data())
        lat.set_coupling_data(mode, None)
        for k in chunks:
            lat.step(k)
        out.append(lat.get_populations())
    return out


@pytest.mark.parametrize("size, scene, prec, order, mode, with_rho", [
    ((96, 90, 88), "cavity", lbm.FP64, ROWS, lbm.COUPLE_DIRICHLET, False),
    ((128, 70, 71), "open", lbm.FP64, ROWS, lbm.COUPLE_OVERWRITE, True),
    ((101, 95, 94), "porous", lbm.FP64, BRICKS, lbm.COUPLE_DIRICHLET, True),
    ((128, 128, 126), "cavity", lbm.FP32_SHIFTED, ROWS, lbm.COUPLE_DIRICHLET, False),
    ((192, 130, 128), "open", lbm.FP32_SHIFTED_F32, ROWS, lbm.COUPLE_OVERWRITE, False),
    ((40, 36, 30), "porous", lbm.FP64, lbm.CELL_ORDER_AUTO, lbm.COUPLE_DIRICHLET, True),  # single steps
])
def test_coupled_pairs_equal_single_steps(size, scene, prec, order, mode, with_rho):
    print(f"[gpu] coupled pairs: {size} {scene} precision {prec} order {order} mode {mode}", flush=True)
    a = _run(size, scene, prec, order, mode, with_rho, [5])
    b = _run(size, scene, prec, order, mode, with_rho, [1] * 5)
    assert all(np.array_equal(u, v) for u, v in zip(a, b))


def test_coupled_pairs_in_a_captured_graph():
    args = ((96, 90, 88), "cavity", lbm.FP64, ROWS, lbm.COUPLE_DIRICHLET, False, [33, 64, 1, 32])
    assert all(np.array_equal(u, v) for u, v in zip(_run(*args), _run(*args, graph=True)))
