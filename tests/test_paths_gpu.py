"""Which kernels served a run (flb_block_paths, flb_adjoint_paths): the boxes of the bit-for-bit
tests of two-step launches do take them, and the ones meant to step singly do not. Moving a
threshold past one of those boxes fails here, where it would otherwise compare single steps with
single steps."""
import numpy as np
import pytest

from freelb_amd import Adjoint, AdjointBatch, BlockLatticeManager, HalfwayBB, abi
from freelb_amd.cases import VOID, cavity_block, heated_cavity
from tests import test_adjoint_gpu as adjoint_tests
from tests import test_march_gpu as march_tests

pytestmark = pytest.mark.gpu


def _params(test, names):
    """The values of a test's parametrize mark over `names`."""
    return next(m.args[1] for m in test.pytestmark if m.name == "parametrize" and m.args[0] == names)


@pytest.mark.parametrize("storage,dims", _params(march_tests.test_runs_equal_single_steps, "storage,dims"))
@pytest.mark.parametrize("periodic,dyn,obstacles",
                         _params(march_tests.test_runs_equal_single_steps, "periodic,dyn,obstacles"))
def test_boxes_of_the_run_tests_take_two_steps(storage, dims, periodic, dyn, obstacles):
    if dyn == abi.DYN_BGK_FORCE and dims in ((23, 29, 880), (700, 31, 27)):
        pytest.skip("steps singly, which is faster; larger boxes of these rows below")
    with march_tests._box(dims, periodic, storage, dyn, obstacles) as lat:
        for n, two in ((4, 0), (5, 2), (9, 4), (1, 0)):  # parities 0, 0, 1, 0
            before = lat.paths()["two_step"]
            lat.step(n)
            assert lat.paths()["two_step"] - before == two, n
        assert lat.paths()["coupled"] == 0


@pytest.mark.parametrize("dims", [(23, 29, 4800), (700, 31, 40)])
@pytest.mark.parametrize("periodic,obstacles", [((True, False, False), True), ((True, True, True), False)])
def test_forced_rows_of_large_boxes_equal_single_steps(dims, periodic, obstacles):
    """Narrow and wide rows, periodic in x and with a force: boxes large enough to march, bit for
    bit against single steps."""
    def make():
        return march_tests._box(dims, periodic, "f32", abi.DYN_BGK_FORCE, obstacles)
    with make() as lat:
        lat.step(9)
        assert lat.paths()["two_step"] == 4
    march_tests._agree(make, (5, 4, 9))


@pytest.mark.parametrize("storage,dims,collision",
                         _params(march_tests.test_moving_lid_runs_equal_single_steps, "storage,dims,collision"))
def test_lid_boxes_take_the_meant_path(storage, dims, collision):
    marches = storage != "f16s" and dims != (40, 40, 40) and (collision == "bgk" or storage == "f64")
    with cavity_block(dims, storage=storage, collision=collision, tau=0.6) as lat:
        lat.step(9)
        assert lat.paths()["two_step"] == (4 if marches else 0)


# around the sizes where one population array fits the memory-side cache and two do not
@pytest.mark.parametrize("storage,dyn,dims,per,marches", [
    ("f32", abi.DYN_BGK, (134, 130, 122), 0, True), ("f32", abi.DYN_BGK, (136, 136, 134), 0, False),
    ("f32", abi.DYN_BGK, (148, 146, 141), 0, True), ("f32", abi.DYN_BGK, (97, 160, 160), 0, True),
    ("f32", abi.DYN_BGK, (256, 97, 100), 0, True), ("f64", abi.DYN_BGK, (104, 100, 95), 0, True),
    ("f64", abi.DYN_BGK, (110, 110, 105), 0, False), ("f64", abi.DYN_BGK, (117, 117, 115), 0, True),
    ("f32", abi.DYN_BGK_FORCE, (97, 140, 120), 1, True), ("f32", abi.DYN_BGK_FORCE, (97, 160, 160), 1, False),
    ("f32", abi.DYN_BGK_FORCE, (136, 150, 152), 1, True), ("f64", abi.DYN_BGK_FORCE, (97, 100, 90), 0, True),
    ("f64", abi.DYN_BGK_FORCE, (110, 110, 105), 1, False), ("f64", abi.DYN_BGK_FORCE, (117, 118, 120), 1, True),
    ("f64", abi.DYN_BGK_FORCE, (256, 70, 70), 1, False), ("f64", abi.DYN_BGK_FORCE, (256, 70, 70), 0, True),
    ("f32", abi.DYN_BGK_FORCE, (256, 97, 100), 0, True), ("f32", abi.DYN_BGK_FORCE, (256, 97, 100), 1, False),
    ("f32", abi.DYN_BGK_FORCE, (400, 64, 100), 1, True), ("f32", abi.DYN_BGK, (20, 200, 600), 0, False),
    ("f32", abi.DYN_BGK, (20, 200, 350), 0, True), ("f32", abi.DYN_BGK_FORCE, (20, 200, 300), 1, False),
    ("f32", abi.DYN_BGK, (97, 160, 170), 0, True), ("f32", abi.DYN_BGK, (97, 160, 170), 1, False),
    ("f64", abi.DYN_BGK, (700, 20, 81), 1, False), ("f64", abi.DYN_BGK_FORCE, (300, 50, 70), 1, False),
    ("f64", abi.DYN_BGK, (60, 90, 180), 0, True), ("f64", abi.DYN_BGK, (60, 90, 240), 0, False)])
def test_band_of_the_memory_side_cache_steps_singly(storage, dyn, dims, per, marches):
    with march_tests._box(dims, (bool(per), False, False), storage, dyn, False) as lat:
        lat.step(5)
        assert lat.paths()["two_step"] == (2 if marches else 0)


def test_open_walls_and_watchdog():
    with cavity_block((92, 83, 77), tau=0.6) as lat:
        lat.set_watchdog(7)
        lat.step(14)  # 7 steps to each check: 1, 4 in two launches, 2; then 4 in two launches, 3
        assert lat.paths()["two_step"] == 4
        lat.set_halfway_bc([HalfwayBB(4, VOID)])
        lat.step(9)
        assert lat.paths()["two_step"] == 4


def test_batches_take_two_steps():
    blocks = [cavity_block(d, tau=0.7, u_lid=0.03, seed=k) for k, d in enumerate(march_tests.BATCH_DIMS)]

    def two():
        counts = {b.paths()["two_step"] for b in blocks}
        assert len(counts) == 1
        return counts.pop()
    try:
        with BlockLatticeManager(blocks) as m:
            m.capture(10)
            assert two() == 0
            m.replay()
            assert two() == 4
            m.step(9)
            assert two() == 8
            m.step(1)
            blocks[3].set_halfway_bc([HalfwayBB(4, VOID)])
            m.replay()
            assert two() == 8
    finally:
        for b in blocks:
            b.close()


ADJ = "storage,dims,per,solids"


@pytest.mark.parametrize(ADJ, _params(adjoint_tests.test_two_steps_per_pass_equal_single_steps, ADJ))
def test_adjoint_boxes_take_two_steps(storage, dims, per, solids):
    with Adjoint(dims, omega=1.6, periodic=per, storage=storage) as adj:
        N = int(np.prod(dims))
        adj.init_equilibrium(np.ones(N), np.zeros((3, N)))
        back = 0 if storage == "f64" else 1
        for T, K, f, b in ((7, 1, 0, 0), (7, 0, 3, 3), (7, 3, 2 + 2, 2), (8, 4, 4 + 4, 4)):
            was = adj.paths()
            adj.forward(T, K)
            adj.backward()
            now = adj.paths()
            assert now["forward_two"] - was["forward_two"] == f, (T, K)
            assert now["backward_two"] - was["backward_two"] == b * back, (T, K)


@pytest.mark.parametrize("dims,recompute", [((56, 55, 76), 0), ((62, 60, 80), 4)])
def test_small_fp64_boxes_recompute_singly(dims, recompute):
    with Adjoint(dims, omega=1.6, periodic=(True, False, False), storage="f64") as adj:
        adj.init_equilibrium(np.ones(adj.N), np.zeros((3, adj.N)))
        adj.forward(8, 4)
        assert adj.paths()["forward_two"] == 4
        adj.backward()
        assert adj.paths()["forward_two"] == 4 + recompute


@pytest.mark.parametrize("storage", ["f32", "f64"])
def test_adjoint_batch_takes_two_steps(storage):
    members = []
    try:
        for dims in ((131, 60, 60), (75, 66, 101), (64, 96, 80), (200, 130, 32), (10, 6, 5), (96, 93, 97), (90, 80, 70)):
            members.append(Adjoint(dims, omega=1.6, periodic=(True, False, False), storage=storage))
            N = int(np.prod(dims))
            members[-1].init_equilibrium(np.ones(N), np.zeros((3, N)))
        with AdjointBatch(members) as b:
            b.forward(9, 0)
            b.backward()
            two = (4, 0 if storage == "f64" else 4)
            assert all((a.paths()["forward_two"], a.paths()["backward_two"]) == two for a in members)
            was = members[0].paths()
            b.forward(9, 1)
            b.backward()
            assert all(a.paths()[k] == was[k] for a in members for k in ("forward_two", "backward_two"))
    finally:
        for a in members:
            a.close()


@pytest.mark.parametrize("storage,dims,T,K,pulls", [("f32", (33, 20, 17), 9, 0, 9), ("f32", (33, 20, 17), 9, 4, 9),
                                                    ("f64", (96, 60, 60), 7, 0, 7), ("f64", (96, 60, 60), 7, 3, 7),
                                                    ("f32", (131, 60, 60), 7, 1, 7), ("f32", (131, 60, 60), 1, 0, 1),
                                                    ("f32", (131, 60, 60), 7, 0, 0), ("f32", (131, 60, 60), 7, 3, 0)])
def test_single_backward_steps_pull(storage, dims, T, K, pulls):
    """Backward runs without launches of two steps read their neighbours (the faster form of a
    single step); odd steps between such launches push. Alone and in a batch of one."""
    with Adjoint(dims, omega=1.6, periodic=(True, False, False), storage=storage) as adj:
        N = int(np.prod(dims))
        rng = np.random.default_rng(5)
        adj.set_fraction(rng.uniform(0, 1, N))
        adj.init_equilibrium(np.ones(N), rng.uniform(-0.01, 0.01, (3, N)))
        J = adj.forward(T, K)
        g = adj.backward()
        assert adj.paths()["backward_pull"] == pulls
        was = adj.paths()
        with AdjointBatch([adj]) as b:
            assert b.forward(T, K)[0] == J
            assert np.array_equal(b.backward()[0], g)
        now = adj.paths()
        # the batch decides on launches of two by its own estimate
        two = now["backward_two"] > was["backward_two"]
        assert now["backward_pull"] - was["backward_pull"] == (0 if two else T)


@pytest.mark.parametrize("n,d,storage", [(5, 3, "f32"), (23, 3, "f64"), (64, 3, "f32"), (40, 2, "f32"), (250, 2, "f64")])
def test_coupled_pairs_take_one_launch(n, d, storage):
    flow, temp, cpl = heated_cavity(n, d, storage)
    try:
        cpl.step(5)
        assert flow.paths() == temp.paths() == dict(two_step=0, coupled=5, plans=0)
        flow.step(1)
        cpl.step(3)
        assert flow.paths()["coupled"] == 5
    finally:
        flow.close()
        temp.close()


@pytest.mark.parametrize("n,d,storage,one", [(124, 3, "f32", True), (144, 3, "f32", False), (148, 3, "f32", True),
                                             (114, 3, "f64", False), (117, 3, "f64", True), (1900, 2, "f32", True),
                                             (1300, 2, "f64", True)])
def test_coupled_pairs_around_the_cache_take_the_faster_way(n, d, storage, one):
    flow, temp, cpl = heated_cavity(n, d, storage)
    try:
        cpl.step(2)
        assert flow.paths()["coupled"] == (2 if one else 0)
    finally:
        flow.close()
        temp.close()


def test_tiles_are_planned_once():
    with cavity_block((300, 60, 40), tau=0.6) as lat:
        for _ in range(3):
            lat.step(9)
        lat.set_omega(1.3)
        lat.set_halfway_bc([HalfwayBB(4, VOID), HalfwayBB(8, VOID, True)])
        lat.step(9)
        assert lat.paths()["two_step"] == 16 and lat.paths()["plans"] == 1
    for storage, plans in (("f32", 2), ("f64", 1)):  # FP64 goes back in single steps
        with Adjoint((131, 60, 60), omega=1.6, storage=storage) as adj:
            adj.init_equilibrium(np.ones(adj.N), np.zeros((3, adj.N)))
            for K in (0, 3, 0):
                adj.forward(7, K)
                adj.backward()
            assert adj.paths()["plans"] == plans


@pytest.mark.parametrize("storage,plans", [("f32", 2), ("f64", 1)])
def test_batches_plan_the_directions_they_take(storage, plans):
    """FP64 goes back in single steps, so only its forward passes are planned."""
    members = []
    try:
        for dims in ((131, 60, 60), (75, 66, 101), (64, 96, 80), (200, 130, 32), (10, 6, 5), (96, 93, 97), (90, 80, 70)):
            members.append(Adjoint(dims, omega=1.6, periodic=(True, False, False), storage=storage))
            members[-1].init_equilibrium(np.ones(members[-1].N), np.zeros((3, members[-1].N)))
        with AdjointBatch(members) as b:
            for K in (0, 3):
                b.forward(5, K)
                b.backward()
        assert all(a.paths()["forward_two"] > 0 and a.paths()["plans"] == plans for a in members)
    finally:
        for a in members:
            a.close()


def test_bad_count_is_refused():
    with cavity_block((8, 8, 8)) as lat:
        with pytest.raises(abi.FLBError):
            abi.paths(abi.lib().flb_block_paths, lat.handle, abi.BLOCK_PATHS + ("x",))
