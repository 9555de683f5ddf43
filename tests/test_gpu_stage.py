"""Solver stages formed inside the X forward pass of the demag convolution
(small grids): every solver's stages (2 to 6 sources, with and without
normalisation), rows of one pair, remainders of a work-group, several z
planes, a geometry, lengths with a compiled X pass and odd rows (which keep
the separate stage kernel), and the largest component array that takes it.

Against the FP64 oracle over 3 fixed steps.  dt gammaLL |B| is about 2e-3, so
the convolution's 2e-6 adds 1e-8 and rounding m (6e-8 a stage, up to 6 stages
a step) dominates FP32: 2e-6.  FP64: 1e-12 likewise."""
import numpy as np
import pytest

from cases import random_unit
from umagnus_amd.params import exchange_lut

pytestmark = pytest.mark.gpu
SOLVERS = (2, 3, 4, 5)   # Heun, RK23, RK4, RK45DP


@pytest.fixture(scope="module")
def gpu():
    import torch
    from umagnus_amd import umhip
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    umhip.init(0)
    return umhip


@pytest.mark.parametrize("dtype,tol", [(np.float32, 2e-6), (np.float64, 1e-12)])
@pytest.mark.parametrize("N,geom", [((2, 8, 1), False), ((30, 7, 1), True), ((10, 6, 5), False), ((64, 9, 2), True),
                                    ((96, 5, 1), False), ((128, 32, 1), False), ((35, 6, 1), True)])
def test_stages_match_oracle(gpu, oracle, N, geom, dtype, tol):
    shape = (N[2], N[1], N[0])
    for solver in SOLVERS:
        print("stages", N, dtype.__name__, solver, flush=True)
        out = []
        for mod, dt in ((oracle, np.float64), (gpu, dtype)):
            s = mod.Sim(N, (4e-9, 3e-9, 2e-9), dtype=dt)
            s.set_scalar(mod.P_MSAT, 8e5)
            s.set_scalar(mod.P_ALPHA, 0.1)
            s.set_exchange_luts(exchange_lut(1.3e-11, dtype=dt), None)
            if geom:
                v = np.ones(shape, dt)
                v.reshape(-1)[::5] = 0
                v.reshape(-1)[1::7] = 0.5
                s.set_geometry(v)
            s.set_m(random_unit(shape, 3).astype(dt))
            s.set_solver(solver)
            s.set_solver_params(dt=1e-14, fixdt=1e-14)
            s.steps(3)
            out.append(np.asarray(s.get_m(), np.float64))
        assert np.abs(out[0] - out[1]).max() <= tol, solver


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_largest_component_array(gpu, dtype):
    """The largest component arrays up to 1 MiB take the path, the next ones do
    not; m stays normalised on both."""
    for rows, want in ((640, 12), (672, 0)) if dtype == np.float32 else ((320, 12), (336, 0)):
        s = gpu.Sim((400, rows, 1), (4e-9, 3e-9, 2e-9), dtype=dtype)
        s.set_scalar(gpu.P_MSAT, 8e5)
        s.set_scalar(gpu.P_ALPHA, 0.1)
        s.set_exchange_luts(exchange_lut(1.3e-11, dtype=dtype), None)
        s.set_m(random_unit((1, rows, 400), 5).astype(dtype))
        s.set_solver(5)
        s.set_solver_params(dt=1e-14, fixdt=1e-14)
        with gpu.KernelTrace() as tr:
            s.steps(2)
        fused = sum("k_rxstage" in k for k in tr.names)
        assert fused == want, tr.names
        m = np.asarray(s.get_m(), np.float64)
        assert np.abs((m * m).sum(0) - 1).max() < 1e-6


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("solver", SOLVERS)
def test_time_functions_see_the_stage(gpu, monkeypatch, solver, dtype):
    """A time function, of a parameter or of a field term, that reads m finds
    every stage's m in it: what it reads, and a trajectory fed back from it, are
    those of a handle whose stages are always kernels of their own."""
    N = (30, 14, 2)
    shape = (N[2], N[1], N[0])
    for term in (False, True):
        print("time function", solver, dtype.__name__, term, flush=True)
        runs = []
        for fused in ("1", "0"):
            monkeypatch.setenv("UMHIP_FUSED_FIELD", fused)
            s = gpu.Sim(N, (4e-9, 3e-9, 2e-9), dtype=dtype)
            s.set_scalar(gpu.P_MSAT, 8e5)
            s.set_scalar(gpu.P_ALPHA, 0.1)
            s.set_exchange_luts(exchange_lut(1.3e-11, dtype=dtype), None)
            s.set_m(random_unit(shape, 9).astype(dtype))
            s.set_solver(solver)
            s.set_solver_params(dt=1e-13, fixdt=1e-13)
            seen = []

            def feedback(t):
                seen.append(np.array(s.get_m()))
                return 0.05 * s.average_m()[0]

            if term:
                s.add_field_term(s.FIELD_TERM_CUSTOM, random_unit(shape, 4).astype(dtype), fn=feedback)
            else:
                s.set_time_function(gpu.P_BEXT, lambda t: (feedback(t), 0.0, 0.0), 3)
            s.steps(3)
            runs.append((seen, np.array(s.get_m())))
        (seen, m), (want, mw) = runs
        assert len(seen) == len(want) >= 6
        # FixDt of 1e-13 turns m by 1e-2 a step: no stage repeats the one before
        for i in range(1, len(want)):
            assert not np.array_equal(want[i], want[i - 1]), i
        for i, (a, b) in enumerate(zip(seen, want)):
            assert np.array_equal(a, b), (i, np.abs(a.astype(float) - b).max())
        assert np.array_equal(m, mw)


# rows of one pair, remainders of a work-group, periodic axes (half and odd
# lengths), several planes, the largest component array that takes the path
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("N,pbc", [((2, 8, 1), (0, 0, 0)), ((30, 7, 1), (0, 0, 0)), ((30, 20, 3), (2, 0, 0)),
                                   ((42, 10, 1), (0, 1, 0)), ((20, 12, 5), (1, 1, 1)), ((250, 50, 1), (0, 0, 0)),
                                   ((160, 16, 10), (0, 0, 0)), ((400, 320, 1), (0, 0, 0))])
def test_same_bits_as_separate_stages(gpu, monkeypatch, N, pbc, dtype):
    """m after fixed and after device-controlled adaptive steps does not depend
    on which kernel forms the stages."""
    shape = (N[2], N[1], N[0])
    for solver, geom in ((2, False), (3, True), (4, False), (5, True), (5, False)):
        print("same bits", N, pbc, dtype.__name__, solver, geom, flush=True)
        out, fused = [], []
        for env in ("1", "0"):
            monkeypatch.setenv("UMHIP_FUSED_FIELD", env)
            s = gpu.Sim(N, (4e-9, 3e-9, 2e-9), pbc=pbc, dtype=dtype)
            s.set_scalar(gpu.P_MSAT, 8e5)
            s.set_scalar(gpu.P_ALPHA, 0.1)
            s.set_exchange_luts(exchange_lut(1.3e-11, dtype=dtype), None)
            if geom:
                v = np.ones(shape, dtype)
                v.reshape(-1)[::5] = 0
                v.reshape(-1)[1::7] = 0.5
                s.set_geometry(v)
            s.set_m(random_unit(shape, 6).astype(dtype))
            s.set_solver(solver)
            s.set_solver_params(dt=1e-13, fixdt=1e-13)
            with gpu.KernelTrace() as tr:
                s.steps(3)
            fused.append(sum("k_rxstage" in k for k in tr.names))
            m = [np.array(s.get_m())]
            if solver == 5:
                s.set_graph(1)
                s.set_solver_params(dt=1e-14)
                s.run(3e-13)
                m.append(np.array(s.get_m()))
            out.append(m)
        assert fused[0] > 0 and fused[1] == 0, fused
        for a, b in zip(*out):
            assert np.array_equal(a, b), np.abs(a.astype(float) - b).max()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_time_function_switches_demag(gpu, monkeypatch, dtype):
    """A time function that switches the demag field off and on between stages:
    every stage is formed all the same."""
    N, shape = (30, 14, 2), (2, 14, 30)
    out = []
    for fused in ("1", "0"):
        monkeypatch.setenv("UMHIP_FUSED_FIELD", fused)
        s = gpu.Sim(N, (4e-9, 3e-9, 2e-9), dtype=dtype)
        s.set_scalar(gpu.P_MSAT, 8e5)
        s.set_scalar(gpu.P_ALPHA, 0.1)
        s.set_exchange_luts(exchange_lut(1.3e-11, dtype=dtype), None)
        s.set_m(random_unit(shape, 2).astype(dtype))
        s.set_solver(5)
        s.set_solver_params(dt=1e-13, fixdt=1e-13)
        calls = [0]

        def switch(t):
            calls[0] += 1
            s.set_flags(int(calls[0] % 3 != 0))
            return (0.01, 0.0, 0.0)

        s.set_time_function(gpu.P_BEXT, switch, 3)
        print("switch", dtype.__name__, fused, flush=True)
        s.steps(4)
        s.set_time_function(gpu.P_BEXT, None, 3)
        s.set_flags(1)
        s.steps(2)
        out.append(np.array(s.get_m()))
    assert np.array_equal(*out)
    assert np.abs((out[0].astype(float) ** 2).sum(0) - 1).max() < 1e-6


def test_profiled_steps_keep_stages_apart(gpu):
    """The demag share of um_sim_kernel_times holds no solver stage; profiled
    steps give the same bits."""
    N, out = (30, 20, 3), []
    for profiling in (0, 1):
        s = gpu.Sim(N, (4e-9, 3e-9, 2e-9), dtype=np.float32)
        s.set_scalar(gpu.P_MSAT, 8e5)
        s.set_scalar(gpu.P_ALPHA, 0.1)
        s.set_exchange_luts(exchange_lut(1.3e-11, dtype=np.float32), None)
        s.set_m(random_unit((3, 20, 30), 8).astype(np.float32))
        s.set_solver(5)
        s.set_solver_params(dt=1e-13, fixdt=1e-13)
        s.set_profiling(profiling)
        with gpu.KernelTrace() as tr:
            s.steps(2)
        assert any("k_rxstage" in k for k in tr.names) == (not profiling), tr.names
        out.append(np.array(s.get_m()))
    assert np.array_equal(*out)
