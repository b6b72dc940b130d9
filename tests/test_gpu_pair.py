"""Two steps per launch (k_dense_pair) against single steps: the same bits.

lat.step(1) always runs the one-step kernel, lat.step(n) runs pairs on lattices large enough; sizes around
the tiles (64 x 8 and 32 x 16 columns), ragged in every axis, with every kind of cell the step knows."""
import numpy as np
import pytest

from madpac_amd import lbm

pytestmark = pytest.mark.gpu


def _lattice(size, scene, prec, order, arr=lbm.POPULATIONS_AUTO):
    nx, ny, nz = size
    rng = np.random.default_rng(nx + ny + nz)
    solid = rng.random((nz, ny, nx)) < (0.0 if scene == "open" else 0.12)
    periodic = {"open": (True, True, True), "porous": (True, False, True)}.get(scene, (False, False, False))
    force = (1e-5, -2e-5, 3e-5) if scene in ("porous", "brinkman") else (0.0, 0.0, 0.0)
    lat = lbm.Lattice(nx, ny, nz, 0.57, precision=prec, periodic=periodic, force=force, cell_order=order,
                      populations=arr)
    lat.set_flags(~solid)
    if scene == "cavity":
        lat.set_cavity_lid(0.05)
    elif scene == "channel":
        lat.set_channel(0.04, parabolic=True)
    elif scene == "brinkman":
        lat.set_porosity(rng.random(solid.size))
    lat.init_equilibrium(rho=1.0 + 0.01 * rng.standard_normal(solid.size), u=0.02 * rng.standard_normal((solid.size, 3)))
    return lat


ROWS, BRICKS = lbm.CELL_ORDER_ROWS, lbm.CELL_ORDER_BRICKS


@pytest.mark.parametrize("size, scene, prec, order", [
    ((64, 64, 64), "open", lbm.FP64, ROWS),
    ((128, 57, 63), "porous", lbm.FP64, ROWS),        # last tile of one row
    ((131, 70, 53), "channel", lbm.FP64, ROWS),       # planes, ragged tiles, inlet and outlet faces
    ((66, 81, 80), "cavity", lbm.FP64, BRICKS),       # tiles of two columns and one row
    ((97, 63, 65), "porous", lbm.FP64, BRICKS),       # bricks cut by the box
    ((130, 64, 64), "brinkman", lbm.FP64, ROWS),
    ((64, 65, 96), "cavity", lbm.FP32_SHIFTED, ROWS),
    ((127, 72, 48), "channel", lbm.FP32_SHIFTED, ROWS),
    ((192, 49, 47), "porous", lbm.FP32_SHIFTED, ROWS),
    ((73, 71, 71), "porous", lbm.FP32_SHIFTED, BRICKS),
    ((65, 64, 64), "brinkman", lbm.FP32_SHIFTED, ROWS),
    ((128, 64, 33), "open", lbm.FP32_SHIFTED_F32, ROWS),
    ((2, 400, 400), "open", lbm.FP64, ROWS),          # both x neighbours are the same cell
    ((1, 1, 270000), "porous", lbm.FP64, ROWS),       # a cell is its own neighbour in x
    ((600, 500, 1), "open", lbm.FP64, BRICKS),        # ... and in z
])
def test_pairs_equal_single_steps(size, scene, prec, order):
    print(f"[gpu] pairs: {size} {scene} precision {prec} order {order}", flush=True)
    out = []
    for chunks in ([5], [1] * 5):
        with _lattice(size, scene, prec, order) as lat:
            for n in chunks:
                lat.step(n)
            out.append((lat.get_populations(), lat.moments()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


def test_pairs_in_a_captured_graph():
    out = []
    for graph in (False, True):
        with _lattice((64, 72, 60), "porous", lbm.FP64, ROWS) as lat:
            for n in (33, 64, 1, 32):  # replays from both buffers, eager steps between
                lat.step(n, graph=graph)
            out.append(lat.get_populations())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("size, scene, prec, order", [
    ((127, 100, 90), "cavity", lbm.FP32_SHIFTED, ROWS),       # planes, one idle lane, last tile of four rows
    ((191, 97, 90), "open", lbm.FP32_SHIFTED, ROWS),          # last tile of one row
    ((130, 120, 118), "brinkman", lbm.FP32_SHIFTED, ROWS),    # last tile of two columns
    ((127, 125, 121), "porous", lbm.FP32_SHIFTED, BRICKS),    # bricks cut by the box
    ((128, 130, 120), "porous", lbm.FP32_SHIFTED_F32, ROWS),  # interleaved rows
    ((97, 90, 93), "cavity", lbm.FP64, BRICKS),               # boundary classes in bricks
    ((98, 90, 88), "channel", lbm.FP64, ROWS),                # inlet and outlet classes of a parabolic profile
])
def test_pairs_equal_single_steps_where_they_pay(size, scene, prec, order):
    # sizes that the rule of pair_plan sends to the two-step kernel, with each kind of boundary it weighs
    test_pairs_equal_single_steps(size, scene, prec, order)


@pytest.mark.parametrize("size, scene, prec, order", [
    ((95, 97, 83), "porous", lbm.FP64, ROWS),                # one idle lane, last tile of one row
    ((160, 81, 66), "channel", lbm.FP64, ROWS),              # whole tiles along x, inlet and outlet
    ((96, 90, 88), "cavity", lbm.FP64, ROWS),
    ((159, 147, 150), "brinkman", lbm.FP32_SHIFTED, ROWS),   # last tile of three rows
    ((96, 161, 149), "open", lbm.FP32_SHIFTED, ROWS),        # last tile of one row, wrapping axes
    ((160, 158, 150), "cavity", lbm.FP32_SHIFTED, ROWS),
    ((93, 177, 180), "porous", lbm.FP32_SHIFTED, BRICKS),    # bricks cut by the box
    ((130, 120, 118), "porous", lbm.FP32_SHIFTED_F32, ROWS),  # last tile of two columns
])
def test_pairs_in_tall_tiles_equal_single_steps(size, scene, prec, order):
    # sizes that fill tiles of 32 x 16 columns better than those of 64 x 8
    test_pairs_equal_single_steps(size, scene, prec, order)
