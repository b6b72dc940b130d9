"""The one-step kernel's FP32 forms (csrc/lbm_dense.hip): with and without the branch between the two kinds of store
(up to 98,304 cells without), and with or without terms shared between mirrored directions (by the arrangement of
the populations and the force): the same bits in every form."""
import numpy as np
import pytest

from madpac_amd import lbm
from test_gpu_pair import BRICKS, ROWS, _lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [lbm.FP32_SHIFTED, lbm.FP32_SHIFTED_F32])
@pytest.mark.parametrize("scene", ["open", "cavity", "channel", "porous", "brinkman"])
@pytest.mark.parametrize("size", [(64, 24, 64), (64, 32, 49), (64, 21, 19)])  # at the line, above it, below it
def test_forms_agree(size, scene, prec):
    print(f"[gpu] FP32 forms: {size} {scene} precision {prec}", flush=True)
    out = []
    for order, arr in ((ROWS, lbm.POPULATIONS_PLANES), (ROWS, lbm.POPULATIONS_INTERLEAVED),
                       (BRICKS, lbm.POPULATIONS_PLANES), (BRICKS, lbm.POPULATIONS_INTERLEAVED)):
        with _lattice(size, scene, prec, order, arr) as lat:
            for _ in range(4):
                lat.step(1)
            out.append(lat.get_populations())
    assert all(np.array_equal(out[0], f) for f in out[1:])
    with _lattice(size, scene, prec, ROWS) as lat:  # with the loads issued beside the flag word
        lat.tune(variant=1)
        for _ in range(4):
            lat.step(1)
        assert np.array_equal(out[0], lat.get_populations())
