"""States between 20 and 140 MB are stored through the caches (state_cached), others past them: the same values on
either side of the lines, in the one-step, the in-place and the patch kernels (FP64 against the CPU oracle)."""
import numpy as np
import pytest

import oracle as O
from madpac_amd import lbm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size, order", [
    ((50, 51, 51), lbm.CELL_ORDER_ROWS),    # 20.1 MB with the pad of the planes, rows off the 128-byte lines
    ((64, 40, 51), lbm.CELL_ORDER_ROWS),    # 20.2 MB, interleaved
    ((64, 40, 51), lbm.CELL_ORDER_BRICKS),  # planes of z padded to 52, 20.6 MB
    ((48, 50, 52), lbm.CELL_ORDER_ROWS),    # 19.3 MB: streaming
])
def test_fp64_steps_equal_the_oracle(size, order):
    nx, ny, nz = size
    print(f"[gpu] stores of {size}", flush=True)
    rng = np.random.default_rng(nx)
    rho, u = 1 + 0.01 * rng.standard_normal(nx * ny * nz), 0.02 * rng.standard_normal((nx * ny * nz, 3))
    ref = O.Lattice(nx, ny, nz, (True, True, True))
    ref.set_solid(np.zeros(ref.n, np.uint8))
    ref.params.tau = 0.6
    f = ref.step(ref.equilibrium(rho, u), 3)
    for layout in (lbm.LAYOUT_TWO_BUFFER, lbm.LAYOUT_AA):
        with lbm.Lattice(nx, ny, nz, 0.6, periodic=(True,) * 3, layout=layout, cell_order=order) as lat:
            lat.set_flags(np.ones(lat.n))
            lat.init_equilibrium(rho, u)
            for _ in range(3):
                lat.step(1)
            assert np.array_equal(lat.get_populations(), f)


@pytest.mark.parametrize("n", [20, 28, 32, 48])
def test_patches_equal_the_lattice(n):
    # eight patches of n^3 as one torus: 9.7, 26.7, 39.8 and 134 MB of planes (and their ghost records)
    prec = lbm.FP64
    print(f"[gpu] stores of eight patches of {n}^3", flush=True)
    table = []
    for p in range(8):
        i, j, k = p & 1, (p >> 1) & 1, p >> 2
        table.append((n, 0.6, [((i + c[0]) % 2) + 2 * ((j + c[1]) % 2) + 4 * ((k + c[2]) % 2) for c in lbm.C]))
    u = 0.02 * np.random.default_rng(n).standard_normal((2, n, 2, n, 2, n, 3))  # k z j y i x
    with lbm.Lattice(2 * n, 2 * n, 2 * n, 0.6, precision=prec, periodic=(True,) * 3) as lat:
        lat.set_flags(np.ones(lat.n))
        lat.init_equilibrium(None, u.reshape(-1, 3))
        lat.step(3)
        rho_l, u_l = lat.fields()
    with lbm.PatchSet(table, precision=prec) as ps:
        ps.init(u=u.transpose(0, 2, 4, 1, 3, 5, 6).reshape(-1, 3))
        ps.step(3)
        rho_p, u_p = ps.fields()
    rho_l = rho_l.reshape(2, n, 2, n, 2, n).transpose(0, 2, 4, 1, 3, 5).reshape(-1)
    u_l = u_l.reshape(2, n, 2, n, 2, n, 3).transpose(0, 2, 4, 1, 3, 5, 6).reshape(-1, 3)
    assert np.array_equal(rho_p, rho_l)
    assert np.array_equal(u_p, u_l)
