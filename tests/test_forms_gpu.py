"""Wave mappings of the cell form against each other and the oracle: row
segments (one wavefront per 64 cells of a row) and linear runs (wavefronts
across row ends, taken for short rows), on compact (short-row) and wide row
pitches. Same per-cell arithmetic, so results agree bit for bit."""
import numpy as np
import pytest

from freelb_amd import BlockLattice, BlockLatticeManager, HalfwayBB, Key_TypePair, abi
from freelb_amd.cases import FLUID, LID, VOID, WALL, cavity_flags
from gpu_case import gpu_lattice, interior_mask
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _with_form(monkeypatch, form, make):
    if form is None:
        return make()
    monkeypatch.setenv("FLB_LAUNCH", form)
    try:
        return make()
    finally:
        monkeypatch.delenv("FLB_LAUNCH")


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("mode", ["fw", "hw", "smag"])
@pytest.mark.parametrize("dims", [(8, 7, 6), (100, 9, 7), (257, 3, 3), (33, 33, 3), (230, 4, 3)])
def test_row_and_linear_forms_agree_with_oracle(monkeypatch, storage, mode, dims):
    dt = np.float64 if storage == "f64" else np.float32
    case, p = O.cavity_case(mode, *dims, dtype=dt)
    p0 = p.copy()
    case.run(p, 9)
    # fullway walls: FreeLB's wall cells also hold values streamed in from the
    # void layer, which the kernels do not keep; compare the fluid cells
    inner = interior_mask(case) if mode == "hw" else case.flags == O.AABB
    for form in (None, "-1,4", "-3,4", "-3,1"):
        lat = _with_form(monkeypatch, form, lambda: gpu_lattice(case, storage, p0))
        try:
            lat.step(9)
            got = lat.pops()
        finally:
            lat.close()
        assert np.array_equal(got[:, inner], p[:, inner]), (form, mode, dims)


@pytest.mark.parametrize("mode", ["fw", "hw"])
def test_d2q9_linear_form(monkeypatch, mode):
    case, p = O.cavity_case(mode, 40, 13, 0, dtype=np.float32)
    p0 = p.copy()
    case.run(p, 11)
    inner = interior_mask(case) if mode == "hw" else case.flags == O.AABB
    lat = _with_form(monkeypatch, "-3,2", lambda: gpu_lattice(case, "f32", p0))
    try:
        lat.step(11)
        assert np.array_equal(lat.pops()[:, inner], p[:, inner])
    finally:
        lat.close()


@pytest.mark.parametrize("storage", ["f32", "f64", "f16s", "f16c", "bf16s"])
@pytest.mark.parametrize("dyn", [abi.DYN_BGK, abi.DYN_SMAG_MRT, abi.DYN_BGK_FORCE, abi.DYN_BGK_WRITE])
@pytest.mark.parametrize("dims", [(70, 9, 7), (23, 11, 5), (262, 5, 4)])
def test_kernels_of_one_dynamics_equal_the_general_ones(storage, dyn, dims):
    """A block whose cells share one dynamics steps in a kernel of that dynamics alone; the batched
    step carries every dynamics of the family. Same bits, also in the fields."""
    shape = tuple(n + 2 for n in dims)
    flags = cavity_flags(*dims)
    rng = np.random.default_rng(3)
    u0 = rng.uniform(-0.02, 0.02, size=(3, flags.size))

    def make():
        lat = BlockLattice(19, shape, omega=1 / 0.6, storage=storage)
        lat.upload_flags(flags)
        lat.set_tasks([Key_TypePair(FLUID | WALL | LID, dyn, 0.17 if dyn == abi.DYN_SMAG_MRT else 0.0)])
        lat.set_halfway_bc([HalfwayBB(WALL, VOID), HalfwayBB(LID, VOID, True)])
        lat.set_field_rho(np.ones(flags.size))
        lat.set_field_u(np.where(flags == LID, 0.05, 0.0) * np.array([[1.0], [0.0], [0.0]]))
        lat.set_force((1e-5, 2e-6, -3e-6))
        lat.init_equilibrium(np.ones(flags.size), u0)
        return lat
    a, b = make(), make()
    try:
        with BlockLatticeManager([b]) as m:
            for n in (1, 2, 4):
                for _ in range(n):
                    a.step(1)
                    m.step(1)
                m.synchronize()
                assert np.array_equal(a.pops(), b.pops()), n
                assert np.array_equal(a.download_fields(), b.download_fields()), n
    finally:
        a.close()
        b.close()
