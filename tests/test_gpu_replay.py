"""Fixed-dt replays without a leading eager step: graph mode and batched
ensembles give what eager stepping gives, bit for bit, for even and odd step
counts, every solver, NoDemagSpins and extra field terms (which are prepared
before the capture), and ensembles large enough for several chains."""
import numpy as np
import pytest

from cases import random_unit
from umagnus_amd.params import exchange_lut

pytestmark = pytest.mark.gpu
SOLVERS = {"heun": 2, "rk23": 3, "rk4": 4, "rk45dp": 5}


@pytest.fixture(scope="module")
def gpu():
    import torch
    from umagnus_amd import umhip
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    umhip.init(0)
    return umhip


def _sim(gpu, N, i, solver, graph, extra=None, temp=300.0):
    s = gpu.Sim(N, (2e-9,) * 3, dtype=np.float32)
    s.set_scalar(gpu.P_MSAT, 8e5)
    s.set_scalar(gpu.P_ALPHA, 0.05)
    s.set_scalar(gpu.P_TEMP, temp)
    s.set_exchange_luts(exchange_lut(1.3e-11, dtype=np.float32), None)
    s.set_thermal_seed(11, i)
    shape = (N[2], N[1], N[0])
    if extra == "nodemag":
        s.set_regions((np.arange(np.prod(shape)).reshape(shape) % 3 == 0).astype(np.uint8))
        lut = np.zeros(256, np.float32)
        lut[1] = 1
        s.set_nodemag_lut(lut)
    if extra == "field":
        s.add_field_term(1, 0.01 * random_unit(shape, 50 + i), mul=2.0)
    s.set_solver(SOLVERS[solver])
    s.set_solver_params(dt=5e-15, fixdt=5e-15)
    s.set_m(random_unit(shape, i + 1))
    s.set_graph(graph)
    return s


def _same(a, b, what):
    assert np.array_equal(a.get_m(), b.get_m()), what
    sa, sb = a.state(), b.state()
    assert {k: v for k, v in sa.items()} == {k: v for k, v in sb.items()}, (what, sa, sb)


@pytest.mark.parametrize("temp", [0.0, 300.0])
@pytest.mark.parametrize("solver", list(SOLVERS))
def test_graph_replays_from_the_first_step(gpu, solver, temp):
    print("replay", solver, temp, flush=True)
    for extra in (None, "nodemag", "field"):
        a, b = (_sim(gpu, (48, 20, 2), 0, solver, g, extra, temp) for g in (0, 1))
        for n in (4, 1, 2, 3, 8):
            a.steps(n)
            b.steps(n)
            _same(a, b, (solver, temp, extra, n))


def test_batched_chains(gpu):
    """30 members of ten shapes: more than one chain; special terms among them."""
    sizes = [(32, 32, 1), (48, 20, 2), (64, 32, 3), (35, 24, 1), (96, 16, 4), (40, 30, 1), (32, 48, 6), (64, 64, 1),
             (48, 48, 1), (28, 50, 2)]
    extra = {3: "nodemag", 7: "field", 12: "nodemag", 21: "field"}
    make = lambda i, g: _sim(gpu, sizes[i % 10], i, "heun", g, extra.get(i))
    alone, batch = ([make(i, g) for i in range(30)] for g in (0, 1))
    for n in (2, 5, 6):
        gpu.sims_steps_batched(batch, n)
        for s in alone:
            s.steps(n)
        for i in range(30):
            _same(alone[i], batch[i], (i, n))


def test_batched_skewed_ensemble(gpu):
    """One member with more than half of the work among 48: its share of the
    cost skips whole chains, which must not be kept without members."""
    for big in (0, 24, 47):
        print("skewed ensemble", big, flush=True)
        make = lambda i, g: _sim(gpu, (512, 512, 1) if i == big else ((64, 64, 1), (60, 64, 1))[i % 2], i, "heun", g)
        alone, batch = ([make(i, g) for i in range(48)] for g in (0, 1))
        for n in (4, 5):
            gpu.sims_steps_batched(batch, n)
            for s in alone:
                s.steps(n)
            for i in range(48):
                _same(alone[i], batch[i], (big, i, n))


def test_batched_two_steps_of_changed_members(gpu):
    """Two steps of a few changed members are not worth a new plan; the second
    such call on unchanged members is, and so are two steps of many."""
    def launches(sims, n):
        with gpu.KernelTrace() as tr:
            gpu.sims_steps_batched(sims, n)
        return sum("k_batch" in k for k in tr.names)

    alone, batch = ([_sim(gpu, (nx, 20, 1), i, "heun", g)
                     for i, nx in enumerate((32, 36, 40, 42, 48, 50, 54, 56))] for g in (0, 1))
    for count, builds in ((3, (False, True, False, False)), (8, (True, False, False, True))):
        for call, build in enumerate(builds):
            print("two steps", count, call, flush=True)
            if call in (0, 3):
                for s in alone[:count] + batch[:count]:
                    s.set_vector(gpu.P_BEXT, (0.01 * (call + count), 0.0, 0.0))
            assert (launches(batch[:count], 2) > 0) == build, (count, call)
            for i, s in enumerate(alone[:count]):
                s.steps(2)
                _same(s, batch[i], (count, call, i))
