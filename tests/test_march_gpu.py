"""Runs of steps against the same steps one at a time, bit for bit: blocks of
32 MiB of populations and more take two steps per pass in a run (and a single
call steps alone), so the two must agree on every population, for partial and
single tiles along each axis, periodic axes, walls inside the block, moving
walls, each dynamics the passes serve, and run lengths that begin and end at
either parity. The single steps are pinned against the oracle elsewhere; one
cavity here is compared with it directly."""
import numpy as np
import pytest

from freelb_amd import BlockLattice, BlockLatticeManager, HalfwayBB, Key_TypePair, abi
from freelb_amd.cases import FLUID, VOID, cavity_block, cavity_flags
from oracle import oracle as O
from tests.gpu_case import gpu_lattice

pytestmark = pytest.mark.gpu


def _box(dims, periodic, storage, dyn, obstacles, layout_seed=5):
    """A box of dims updated cells, walls on its other faces, 3 % of its cells void (obstacles)."""
    shape = [n if p else n + 2 for n, p in zip(dims, periodic)]
    rng = np.random.default_rng(layout_seed)
    f = np.full(shape[::-1], VOID, dtype=np.uint8)
    f[tuple(slice(None) if p else slice(1, -1) for p in periodic[::-1])] = FLUID
    if obstacles:
        f[(rng.random(f.shape) < 0.03) & (f == FLUID)] = VOID
    f = f.reshape(-1)
    lat = BlockLattice(19, shape, omega=1 / 0.8, storage=storage, periodic=periodic)
    lat.upload_flags(f)
    lat.set_tasks([Key_TypePair(FLUID, dyn, 0.17 if dyn == abi.DYN_SMAG_MRT else 0.0)])
    lat.set_halfway_bc([HalfwayBB(FLUID, VOID)])
    lat.set_force((1e-5, 2e-6, -3e-6))
    lat.init_equilibrium(np.ones(f.size), rng.uniform(-0.02, 0.02, size=(3, f.size)))
    return lat


def _agree(make, runs):
    with make() as a, make() as b:
        for n in runs:
            a.step(n)
            for _ in range(n):
                b.step(1)
            assert a.info().parity == b.info().parity and a.info().step == b.info().step
            assert np.array_equal(a.pops(), b.pops())
        assert np.array_equal(a.moments(), b.moments())


@pytest.mark.parametrize("storage,dims", [("f32", (97, 71, 87)), ("f32", (23, 29, 880)), ("f32", (700, 31, 27)),
                                          ("f32", (258, 19, 119)), ("f32", (260, 560, 4)), ("f32", (64, 78, 117)),
                                          ("f64", (61, 61, 79)), ("f64", (257, 15, 76)), ("f64", (7, 9, 4610))])
@pytest.mark.parametrize("periodic,dyn,obstacles", [((False, False, False), abi.DYN_BGK, True),
                                                    ((True, False, False), abi.DYN_BGK_FORCE, True),
                                                    ((False, True, True), abi.DYN_BGK, True),
                                                    ((True, True, True), abi.DYN_BGK_FORCE, False)])
def test_runs_equal_single_steps(storage, dims, periodic, dyn, obstacles):
    print(f"[march] {storage} {dims} {periodic} dynamics {dyn}", flush=True)
    _agree(lambda: _box(dims, periodic, storage, dyn, obstacles), (5, 4, 9))


@pytest.mark.parametrize("storage,dims,collision", [("f32", (92, 80, 80), "bgk"), ("f32", (90, 70, 73), "mrt_les"),
                                                    ("f64", (70, 65, 64), "bgk"),
                                                    ("f64", (150, 138, 128), "mrt_les"), ("f16s", (130, 90, 80), "bgk"),
                                                    ("f32", (40, 40, 40), "bgk")])
def test_moving_lid_runs_equal_single_steps(storage, dims, collision):
    """Lid and side walls; FP32 MRT-LES, 16-bit storage and the smallest take single steps either way."""
    print(f"[march] lid {storage} {dims} {collision}", flush=True)
    _agree(lambda: cavity_block(dims, storage=storage, collision=collision, tau=0.6, u0_amp=0.03, seed=3), (11, 6, 1, 7))


def test_run_after_changed_set_up():
    """Walls, tasks, flags and populations changed between runs: the next run sees them."""
    def make():
        return cavity_block((92, 83, 77), tau=0.6, u0_amp=0.02, seed=9)
    with make() as a, make() as b:
        N = a.N
        flags = cavity_flags(92, 83, 77)
        for change in ("none", "omega", "flags", "open walls", "pops"):
            for lat in (a, b):
                if change == "omega":
                    lat.set_omega(1.4)
                elif change == "flags":
                    g = flags.copy()
                    g[np.random.default_rng(4).random(N) < 0.02] = VOID
                    lat.upload_flags(g)
                elif change == "open walls":
                    lat.set_halfway_bc([HalfwayBB(4, VOID)])  # the lid's links are no walls any more
                elif change == "pops":
                    lat.set_halfway_bc([HalfwayBB(4 | 8, VOID)])
                    lat.init_equilibrium(np.ones(N), np.random.default_rng(6).uniform(-0.02, 0.02, size=(3, N)))
            a.step(10)
            for _ in range(10):
                b.step(1)
            assert np.array_equal(a.pops(), b.pops()), change


def test_cavity_run_matches_oracle():
    case, p0 = O.cavity_case("hw", 92, 83, 77)
    lat = gpu_lattice(case, pops=p0)
    with lat:
        lat.step(14)
        got = lat.pops()
    ref = case.run(p0.copy(), 14)
    sel = case.flags != O.VOID
    assert np.array_equal(got[:, sel], ref[:, sel])


def test_watchdog_inside_a_run():
    """Checks fall on the same steps as in single stepping; the state is unchanged by them."""
    def make():
        lat = cavity_block((92, 83, 77), tau=0.6, u0_amp=0.02, seed=2)
        lat.set_watchdog(7)
        return lat
    _agree(make, (20, 3))


# large enough together that the batch takes passes of two steps
BATCH_DIMS = [(16, 16, 16), (96, 93, 97), (63, 90, 77), (64, 62, 64), (131, 60, 83), (5, 6, 7), (40, 81, 4),
              (60, 75, 90), (96, 91, 94)]


def _batch_agrees(make, runs, between=lambda k, blocks: None):
    """BlockLatticeManager runs against the blocks stepped one at a time; runs of "replay" replay
    a recorded graph of 10 steps."""
    a, b = make(), make()
    try:
        with BlockLatticeManager(a) as m:
            m.capture(10)
            for k, n in enumerate(runs):
                between(k, a)
                between(k, b)
                if n == "replay":
                    m.replay()
                else:
                    m.step(n)
                m.synchronize()
                for lat in b:
                    for _ in range(10 if n == "replay" else n):
                        lat.step(1)
                for x, y in zip(a, b):
                    assert np.array_equal(x.pops(), y.pops()), (k, n, x.dims)
    finally:
        for lat in a + b:
            lat.close()


@pytest.mark.parametrize("storage,collision", [("f32", "bgk"), ("f64", "bgk"), ("f32", "mrt_les")])
def test_batch_runs_equal_single_steps(storage, collision):
    dims = BATCH_DIMS if collision == "bgk" else BATCH_DIMS * 2

    def make():
        return [cavity_block(d, storage=storage, collision=collision, tau=0.6 + 0.01 * k, u_lid=0.03, u0_amp=0.02,
                             seed=k) for k, d in enumerate(dims)]
    _batch_agrees(make, ("replay", 5, 1, "replay", 12))


def test_batch_of_mixed_periodic_boxes():
    per = [(False, False, False), (True, False, False), (False, True, True), (True, True, True)]

    def make():
        return [_box(d, per[k % 4], "f32", abi.DYN_BGK_FORCE, k % 2 == 0) for k, d in enumerate(BATCH_DIMS)]
    _batch_agrees(make, ("replay", 7, 1, "replay"))


def test_batch_replay_after_changed_walls():
    """A recorded graph replayed after a change that its passes of two steps no longer serve, and
    after the change is taken back."""
    def make():
        return [cavity_block(d, tau=0.7, u_lid=0.03, u0_amp=0.02, seed=k) for k, d in enumerate(BATCH_DIMS)]

    def between(k, blocks):
        if k == 1:
            blocks[3].set_halfway_bc([HalfwayBB(4, VOID)])
        elif k == 2:
            blocks[3].set_halfway_bc([HalfwayBB(4, VOID), HalfwayBB(8, VOID, True)])
            blocks[1].set_omega(1.2)
    _batch_agrees(make, ("replay", "replay", "replay", 6), between)
