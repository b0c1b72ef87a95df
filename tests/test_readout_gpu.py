"""Read-outs to host memory (flb_readout.hip): the three ways they take give the same values, at the
sizes where one takes over from the next, with a short last chunk, with more chunks than the ring
holds, from several threads, and after the last block gave the buffers back. The pinned memory that
they hold is counted (flb_readout_paths)."""
import gc
import threading

import numpy as np
import pytest

from freelb_amd import Adjoint, AdjointBatch, BlockLattice, Key_TypePair, abi
from freelb_amd.cases import FLUID, VOID
from freelb_amd.lattice import weights

pytestmark = pytest.mark.gpu

DIRECT, RING = 256 << 10, 32 << 20  # pinned bytes of small moments and of the ring


def _block(nx, ny, storage="f32", seed=0):
    """A periodic D2Q9 block and its populations; cells drawn row by row, so that a block of more
    rows begins with the same cells."""
    rng = np.random.default_rng(seed)
    N = nx * ny
    w = weights(9, np.float64)
    p = (w[:, None] * rng.uniform(0.9, 1.1, size=(N, 9)).T).astype(np.float64 if storage == "f64" else np.float32)
    lat = BlockLattice(9, (nx, ny), omega=1.2, storage=storage, periodic=(True, True))
    lat.upload_flags(np.full(N, FLUID, np.uint8))
    lat.set_tasks([Key_TypePair(FLUID, abi.DYN_BGK)])
    lat.upload_pops(p)
    return lat, p


def _took(before):
    now = abi.readout_paths()
    return tuple(now[k] - before[k] for k in ("direct", "ring", "plain"))


# 36 or 72 bytes per cell: just below and above 4 MiB, 17 and 33 chunks, a last chunk of 128 bytes
@pytest.mark.parametrize("nx,ny,storage,way", [(133, 876, "f32", 2), (352, 331, "f32", 1), (1000, 941, "f32", 1),
                                               (176, 331, "f64", 1), (1000, 941, "f64", 1), (7, 5, "f32", 2)])
def test_populations_come_back(nx, ny, storage, way):
    lat, p = _block(nx, ny, storage)
    with lat:
        was = abi.readout_paths()
        assert np.array_equal(lat.pops(), p)
        assert _took(was) == (0, way == 1, way == 2)


@pytest.mark.parametrize("storage", ["f32", "f64"])
def test_moments_of_the_three_ways_agree(storage):
    rows = {0: 128 if storage == "f64" else 257, 2: 258, 1: 4200}  # direct, plain, ring
    got = {}
    for way, ny in rows.items():
        # the same cells in the same place, the flags of the first rows too
        lat, p = _block(85, ny, storage)
        with lat:
            f = np.where(np.arange(85 * ny) % 17 == 3, VOID, FLUID).astype(np.uint8)
            lat.upload_flags(f)
            first = [lat.moments() for _ in range(4)]  # the buffer of small ones is there from the fifth on
            was = abi.readout_paths()
            m = lat.moments()
            assert _took(was) == tuple(int(k == way) for k in range(3))
            assert all(np.array_equal(v, m) for v in first)
            assert np.array_equal(m[:, f == VOID], np.zeros((3, int((f == VOID).sum()))))
            # 8 additions of terms whose magnitudes sum to at most 1.1
            eps = np.finfo(m.dtype).eps / 2
            assert np.max(np.abs(m[0] - p.astype(np.float64).sum(axis=0))[f == FLUID]) <= 8 * 1.1 * eps
            got[way] = m
    n = 85 * rows[0]
    for way in (1, 2):
        assert np.array_equal(got[way][:, :n], got[0])


def test_small_moments_pin_a_small_buffer_of_their_own():
    gc.collect()
    assert abi.readout_paths()["pinned"] == 0  # no block lives
    for _ in range(2):  # a block closed, the buffers given back, a block made again
        lat, p = _block(40, 30)
        with lat:
            was = abi.readout_paths()
            m = lat.moments()
            for _ in range(3):
                assert np.array_equal(lat.moments(), m)
            assert abi.readout_paths()["pinned"] == 0 and _took(was) == (0, 0, 4)
            assert np.array_equal(lat.moments(), m)
            assert abi.readout_paths()["pinned"] == DIRECT and _took(was) == (1, 0, 4)
            big, q = _block(400, 331)
            with big:
                assert np.array_equal(big.pops(), q)
                assert abi.readout_paths()["pinned"] == DIRECT + RING
            assert np.array_equal(lat.pops(), p)
        assert abi.readout_paths()["pinned"] == 0


def test_threads_read_at_once():
    """Two large read-outs at a time share or miss the ring; small moments never take it."""
    (a, pa), (b, pb), (c, _) = _block(1000, 941, seed=1), _block(700, 641, "f64", seed=2), _block(85, 100)
    wrong = []

    def read(lat, want, n):
        for _ in range(n):
            if not np.array_equal(lat.pops(), want):
                wrong.append(lat)
    try:
        was = abi.readout_paths()
        t = [threading.Thread(target=read, args=v) for v in ((a, pa, 6), (b, pb, 6))]
        for x in t:
            x.start()
        for x in t:
            x.join()
        direct, ring, plain = _took(was)
        assert not wrong and direct == 0 and ring >= 1 and ring + plain == 12
        for _ in range(4):
            m = c.moments()
        was = abi.readout_paths()
        t = threading.Thread(target=read, args=(a, pa, 6))
        t.start()
        for _ in range(50):
            assert np.array_equal(c.moments(), m)
        t.join()
        assert not wrong and _took(was) == (50, 6, 0)
    finally:
        for lat in (a, b, c):
            lat.close()


@pytest.mark.parametrize("storage,dims,way", [("f32", [(64, 60, 50), (63, 61, 49), (7, 5, 3)] * 3, 1),
                                              ("f64", [(64, 60, 50), (130, 61, 49), (7, 5, 3)], 1),
                                              ("f32", [(20, 11, 9), (7, 5, 3)], 2)])
def test_gradients_of_a_batch_are_one_read_out(storage, dims, way):
    """Equal to the members' own, with parts of more than a chunk, of less, and of a few bytes."""
    rng = np.random.default_rng(3)
    boxes = []
    try:
        for d in dims:
            boxes.append(Adjoint(d, omega=1.5, periodic=(True, False, False), storage=storage))
            N = boxes[-1].N
            boxes[-1].set_fraction(rng.uniform(0, 1, N))
            boxes[-1].init_equilibrium(np.ones(N), rng.uniform(-0.01, 0.01, (3, N)))
        alone = []
        for a in boxes:
            a.forward(3, 0)
            alone.append(a.backward())
        with AdjointBatch(boxes) as b:
            b.forward(3, 0)
            was = abi.readout_paths()
            got = b.backward()
            assert _took(was) == (0, way == 1, way == 2)
        for g, w in zip(got, alone):
            assert np.array_equal(g, w)
    finally:
        for a in boxes:
            a.close()
