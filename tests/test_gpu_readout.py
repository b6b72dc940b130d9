"""Large readouts go through pinned pieces moved by several threads (csrc/lbm_readout.cpp): the values
must arrive whole at sizes around the switch to it, at ragged last pieces, and from several threads."""
import threading

import numpy as np
import pytest

from madpac_amd import lbm

pytestmark = pytest.mark.gpu

PER = 216 * 23  # values per block: populations, density, velocity


def _roundtrip(nblocks, seed):
    rng = np.random.default_rng(seed)
    want = [rng.standard_normal((nblocks, 216 * k)) for k in (lbm.Q, 1, 3)]
    with lbm.BlockStore(nblocks) as bs:
        bs.set(0, *want)
        for _ in range(2):
            got = bs.get()
            assert all(np.array_equal(g, w) for g, w in zip(got, want))
        a = nblocks // 3
        got = bs.get(a, nblocks - a)
        assert all(np.array_equal(g, w[a:]) for g, w in zip(got, want))


@pytest.mark.parametrize("nblocks", [1, 633, 634, 1000, 1911])
def test_blocks_arrive_whole(nblocks):
    # 633 / 634 blocks lie on either side of 24 MiB
    print(f"[gpu] readout of {nblocks} blocks", flush=True)
    assert 633 * PER * 8 < 24 << 20 < 634 * PER * 8
    _roundtrip(nblocks, nblocks)


def test_concurrent_readouts():
    print("[gpu] four threads reading back at once", flush=True)
    failed = []

    def work(seed):
        try:
            _roundtrip(800 + seed, seed)
        except BaseException as e:  # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed


def test_fields_of_a_large_lattice():
    n = (160, 100, 70)
    rng = np.random.default_rng(5)
    rho = 1 + 0.01 * rng.standard_normal(n[0] * n[1] * n[2])
    with lbm.Lattice(*n, 0.6, periodic=(True,) * 3) as lat:
        lat.set_flags(np.ones(lat.n))
        lat.init_equilibrium(rho)
        f = lat.get_populations().reshape(lbm.Q, -1)
        r, u = lat.fields()
    total = np.zeros_like(rho)
    for q in range(lbm.Q):
        total += f[q]
    assert np.array_equal(r, total)
    assert np.all(np.abs(u) < 1e-15)
