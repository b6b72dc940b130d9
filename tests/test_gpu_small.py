"""Several steps per launch on small lattices (k_dense_small) against single steps: the same bits.

lat.step(1) always runs the one-step kernel.  Sizes on both sides of the boxes (8^3 cells, of which 6^3, 4^3 or 2^3 are
stored) and of the rule's lines (256 boxes), axes shorter than a box that wrap onto themselves, both cell
orders and arrangements, every kind of cell."""
import numpy as np
import pytest

from madpac_amd import lbm
from test_gpu_pair import BRICKS, ROWS, _lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size, scene, prec, order", [
    ((1, 1, 1), "open", lbm.FP64, ROWS),
    ((3, 1, 2), "open", lbm.FP64, BRICKS),
    ((12, 12, 12), "cavity", lbm.FP64, ROWS),            # 216 boxes of 2^3
    ((13, 12, 14), "porous", lbm.FP64, BRICKS),          # 294 of 2^3: three steps
    ((7, 9, 11), "brinkman", lbm.FP32_SHIFTED, ROWS),
    ((16, 5, 4), "channel", lbm.FP64, ROWS),
    ((24, 24, 24), "channel", lbm.FP64, BRICKS),         # 216 boxes of 4^3
    ((64, 8, 8), "open", lbm.FP32_SHIFTED, ROWS),        # interleaved rows, 512 / 64 boxes
    ((64, 15, 13), "porous", lbm.FP32_SHIFTED_F32, ROWS),  # 256 boxes of 4^3
    ((65, 16, 13), "cavity", lbm.FP32_SHIFTED, ROWS),    # 272: single steps
    ((25, 23, 21), "brinkman", lbm.FP64, ROWS),
    ((5, 200, 3), "channel", lbm.FP32_SHIFTED, BRICKS),
])
def test_small_lattices_equal_single_steps(size, scene, prec, order):
    print(f"[gpu] small: {size} {scene} precision {prec} order {order}", flush=True)
    out = []
    for chunks in ([7, 4, 2, 5], [1] * 18):  # whole launches of four and three, and each remainder
        with _lattice(size, scene, prec, order) as lat:
            for n in chunks:
                lat.step(n)
            out.append((lat.get_populations(), lat.moments()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("size", [(11, 12, 10), (18, 17, 16)])
def test_small_lattices_in_a_captured_graph(size):
    out = []
    for graph in (False, True):
        with _lattice(size, "porous", lbm.FP64, ROWS) as lat:
            for n in (49, 1, 97, 37, 150):  # replays from both buffers, eager steps between
                lat.step(n, graph=graph)
            out.append(lat.get_populations())
    assert np.array_equal(out[0], out[1])
