"""Runs of steps against single steps, on lattices whose plan (lat.step_plan) is checked first: the kernel that each
case is meant for is the one that runs.  lat.step(1) always takes the one-step kernel; the bits must be the same."""
import numpy as np
import pytest

from madpac_amd import lbm
from test_gpu_coupled_pairs import _cells
from test_gpu_pair import BRICKS, ROWS, _lattice

pytestmark = pytest.mark.gpu
AUTO, PLANES = lbm.POPULATIONS_AUTO, lbm.POPULATIONS_PLANES
F64, F32, F32A = lbm.FP64, lbm.FP32_SHIFTED, lbm.FP32_SHIFTED_F32


@pytest.mark.parametrize("size, scene, prec, order, arr, tile", [
    # tiles of 64 x 8 columns
    ((64, 64, 64), "open", F64, ROWS, AUTO, 64),           # interleaved rows, whole tiles, chunks of two planes
    ((127, 127, 125), "cavity", F64, ROWS, AUTO, 64),      # planes, one idle lane and row, last chunk cut
    ((128, 126, 125), "channel", F64, ROWS, AUTO, 64),     # inlet and outlet classes of a parabolic profile
    ((128, 126, 125), "porous", F64, ROWS, AUTO, 64),
    ((128, 126, 125), "brinkman", F64, ROWS, PLANES, 64),  # planes where rows could be interleaved
    ((128, 64, 64), "brinkman", F64, ROWS, AUTO, 64),      # ordinary stores
    ((128, 56, 120), "porous", F64, BRICKS, AUTO, 64),
    ((64, 72, 128), "cavity", F64, BRICKS, PLANES, 64),
    ((128, 128, 128), "cavity", F32, ROWS, AUTO, 64),
    ((190, 97, 90), "cavity", F32, ROWS, AUTO, 64),        # ordinary stores, last tile of one row
    ((127, 140, 125), "porous", F32, BRICKS, AUTO, 64),
    ((128, 160, 150), "porous", F32A, ROWS, AUTO, 64),
    ((192, 130, 128), "open", F32A, ROWS, AUTO, 64),       # FP32 arithmetic on interleaved rows
    # tiles of 32 x 16 columns
    ((128, 126, 64), "cavity", F64, BRICKS, AUTO, 32),     # boundary classes in bricks
    ((126, 118, 60), "porous", F64, BRICKS, AUTO, 32),     # bricks cut by the box
    ((160, 81, 66), "channel", F64, ROWS, AUTO, 32),
    ((130, 120, 118), "brinkman", F32, ROWS, AUTO, 32),
    ((31, 4090, 15), "channel", F32, ROWS, AUTO, 32),      # FP32 inlet and outlet
    # axes that wrap onto the tile, the plane or the cell itself
    ((64, 8, 512), "open", F64, ROWS, AUTO, 64),           # the row above the tile is its own first row
    ((64, 6, 1024), "open", F64, ROWS, AUTO, 64),
    ((2, 400, 400), "open", F64, ROWS, AUTO, 32),          # both x neighbours are the same cell
    ((1, 400, 300), "open", F64, ROWS, AUTO, 32),          # a cell is its own x neighbour
    ((1, 300, 200), "open", F32, ROWS, AUTO, 32),
    ((1000, 800, 2), "open", F64, ROWS, AUTO, 64),         # the planes above and below are the same one
    ((31, 60000, 1), "open", F64, ROWS, AUTO, 32),         # a cell is its own z neighbour
])
def test_pairs_equal_single_steps(size, scene, prec, order, arr, tile):
    print(f"[gpu] planned pairs: {size} {scene} precision {prec} order {order} arrangement {arr}", flush=True)
    out = []
    for chunks in ([5], [1] * 5):
        with _lattice(size, scene, prec, order, arr) as lat:
            assert lat.step_plan() == (2, tile)
            for n in chunks:
                lat.step(n)
            out.append((lat.get_populations(), lat.moments()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("size, scene, prec", [((128, 64, 64), "porous", F64), ((64, 64, 64), "open", F64),
                                                ((128, 128, 128), "cavity", F32)])
def test_pairs_in_a_captured_graph(size, scene, prec):
    print(f"[gpu] planned pairs in a graph: {size} {scene} precision {prec}", flush=True)
    out = []
    for graph in (False, True):
        with _lattice(size, scene, prec, ROWS) as lat:
            assert lat.step_plan()[0] == 2
            for n in (33, 64, 1, 32):  # replays from both buffers, eager steps between
                lat.step(n, graph=graph)
                lat.moments()
            out.append(lat.get_populations())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("size, order, steps", [
    ((12, 12, 12), ROWS, 4), ((1, 1, 1), ROWS, 4), ((13, 12, 14), BRICKS, 3), ((24, 24, 24), BRICKS, 3),
    ((64, 15, 13), ROWS, 3), ((65, 16, 13), ROWS, 1), ((32, 32, 32), ROWS, 1), ((80, 80, 40), ROWS, 1),
])
def test_plans_of_small_lattices(size, order, steps):
    with _lattice(size, "porous", F32, order) as lat:
        assert lat.step_plan() == (steps, 0)


@pytest.mark.parametrize("size, periodic, prec", [
    ((96, 90, 88), False, F64), ((128, 70, 71), True, F64), ((101, 95, 94), True, F64), ((128, 128, 126), False, F32),
    ((192, 130, 128), True, F32A),
])
def test_coupled_lattices_run_pairs(size, periodic, prec):
    # the lattices on which test_gpu_coupled_pairs compares pairs with single steps
    nx, ny, nz = size
    with lbm.Lattice(nx, ny, nz, 0.6, precision=prec, periodic=(periodic,) * 3, cell_order=ROWS) as lat:
        cells = _cells(size, np.random.default_rng(nx * ny + nz))
        lat.set_coupling_cells(cells)
        with pytest.raises(lbm.LbmError, match="flags"):
            lat.step_plan()
        lat.set_flags(np.ones(lat.n))
        lat.set_coupling_data(lbm.COUPLE_OVERWRITE, np.zeros((len(cells), 3)))
        assert lat.step_plan()[0] == 2


def test_in_place_lattices_take_single_steps():
    for n in (10, 64):
        with lbm.Lattice(n, n, n, 0.6, layout=lbm.LAYOUT_AA) as lat:
            lat.set_flags(np.ones(lat.n))
            assert lat.step_plan() == (1, 0)
