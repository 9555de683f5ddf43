"""The launch-schedule autotuner on the GPU: every radix schedule of the
generic Stockham engine, forced through a tuning file, gives the demag field of
the oracle; tuned plans (including the ensemble grid sizes with a factor 3,
odd periodic Nx and 2D) stay within the convolution tolerances; results are
kept per shape, written to the tuning file and reused by mode 2.

Tolerances as for the convolution parity tests: FP64 1e-12, FP32 2e-6
normwise against the FP64 oracle."""
import sys

import numpy as np
import pytest

from cases import random_unit

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def gpu():
    import torch
    from umagnus_amd import umhip
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    umhip.init(0)
    yield umhip
    umhip.set_autotune(0)


def _t(a, dtype):
    import torch
    return torch.as_tensor(np.ascontiguousarray(a, dtype)).cuda()


def _check(gpu, oracle, N, pbc, prec, cs=(2e-9, 3e-9, 2.5e-9)):
    rng = np.random.default_rng(sum(N))
    m = random_unit((N[2], N[1], N[0]), sum(N) + 1)
    Ms = rng.uniform(5e5, 1e6, (N[2], N[1], N[0]))
    Bo = oracle.Demag(N, cs, pbc=pbc, dtype=np.float64).exec(m, Ms)
    dt = np.float32 if prec == 0 else np.float64
    conv = gpu.DemagConvolution(N, cs, pbc=pbc, precision=prec)
    B = [_t(np.zeros_like(m[0]), dt) for _ in range(3)]
    conv.Exec(B, [_t(m[k], dt) for k in range(3)], None, _t(Ms, dt))
    Bg = np.stack([b.cpu().numpy() for b in B]).astype(np.float64)
    err = np.abs(Bg - Bo).max() / np.abs(Bo).max()
    assert err < (1e-12 if prec == 1 else 2e-6), (N, pbc, prec, conv.schedule(), err)
    return conv.schedule()


def _key(oracle, N, pbc, prec):
    P = oracle.pad_size(N, pbc)
    return "%s N=%d,%d,%d P=%d,%d,%d" % (("f32", "f64")[prec], *N, *P)


SHAPES = [((96, 48, 2), (0, 0, 0)), ((48, 96, 3), (0, 0, 0)), ((192, 64, 1), (0, 0, 0)),
          ((40, 24, 6), (0, 0, 0)), ((7, 6, 3), (1, 0, 0)), ((24, 20, 4), (0, 0, 2))]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("N,pbc", SHAPES)
def test_every_radix_schedule(gpu, oracle, tmp_path, N, pbc, prec):
    _say("schedules", N, pbc, prec)
    gpu.set_autotune(0)
    base = _check(gpu, oracle, N, pbc, prec)
    for sc in range(4):
        f = tmp_path / ("s%d.txt" % sc)
        v = base[:5] + [sc, sc, sc]
        v[2] = 0     # Stockham X inverse, so its schedule is used too
        f.write_text("%s: %s\n" % (_key(oracle, N, pbc, prec), " ".join(map(str, v))))
        gpu.set_autotune(2, str(f))
        got = _check(gpu, oracle, N, pbc, prec)
        assert got == v, (got, v)
    gpu.set_autotune(0)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("N,pbc", SHAPES + [((256, 256, 1), (0, 0, 0)), ((64, 64, 8), (0, 0, 0)),
                                            ((128, 96, 4), (0, 0, 0))])
def test_tuned_plans(gpu, oracle, tmp_path, N, pbc, prec):
    _say("tuned", N, pbc, prec)
    f = tmp_path / "tune.txt"
    gpu.set_autotune(1, str(f))
    try:
        sched = _check(gpu, oracle, N, pbc, prec)
        lines = f.read_text().splitlines()
        assert len(lines) == 1 and lines[0].startswith(_key(oracle, N, pbc, prec) + ":")
        assert [int(x) for x in lines[0].split(":")[1].split()] == sched
        # known shape: reused without a second entry
        assert _check(gpu, oracle, N, pbc, prec) == sched
        assert len(f.read_text().splitlines()) == 1
    finally:
        gpu.set_autotune(0)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("N", [(100, 100, 2), (250, 250, 1), (64, 64, 8), (90, 80, 15)])
def test_no_choice_among_equals(gpu, oracle, tmp_path, N, prec):
    """A pass that ignores the rows or columns knob (register passes at schedule
    0, four-step X, register Y of 64 and 256) keeps its static value: tuning
    does not pick one of many timings of the same kernel."""
    _say("equals", N, prec)
    gpu.set_autotune(0)
    base = _check(gpu, oracle, N, (0, 0, 0), prec)
    gpu.set_autotune(1, str(tmp_path / "tune.txt"))
    try:
        got = _check(gpu, oracle, N, (0, 0, 0), prec)
    finally:
        gpu.set_autotune(0)
    assert got[2] == base[2] == 1
    if got[5] == 0:
        assert got[:2] == base[:2]
    if got[6] == 0:
        assert got[3] == base[3]
    if got[6 if N[2] == 1 else 7] == 0:
        assert got[4] == base[4]


def test_entries_without_generation(gpu, oracle, tmp_path):
    """An entry without a generation mark, whose schedules meant other kernels:
    tuned again in mode 1 and written with the mark; applied in mode 2."""
    N = (60, 50, 3)
    f = tmp_path / "old.txt"
    old = "%s: 4 4 1 4 4 2 2 2\n" % _key(oracle, N, (0, 0, 0), 0)
    f.write_text(old)
    try:
        gpu.set_autotune(2, str(f))
        assert _check(gpu, oracle, N, (0, 0, 0), 0) == [4, 4, 1, 4, 4, 2, 2, 2]
        assert f.read_text() == old
        gpu.set_autotune(1, str(f))
        sched = _check(gpu, oracle, N, (0, 0, 0), 0)
        lines = f.read_text().splitlines()
        assert len(lines) == 2 and lines[1] == "%s: %s : 2" % (old.split(":")[0], " ".join(map(str, sched)))
        # the marked entry is the one that counts from now on, in both modes
        for mode in (1, 2):
            gpu.set_autotune(mode, str(f))
            assert _check(gpu, oracle, N, (0, 0, 0), 0) == sched
            assert len(f.read_text().splitlines()) == 2
    finally:
        gpu.set_autotune(0)


# lengths without a register split: X rows (FP64 has fewer radices), Y columns,
# the film's and the z axis' convolution
STOCKHAM = [((625, 4, 2), 0, ("k_xfwd", "k_xinv")), ((625, 4, 2), 1, ("k_xfwd", "k_xinv")),
            ((375, 6, 1), 1, ("k_xfwd", "k_xinv")), ((784, 3, 1), 1, ("k_xfwd", "k_xinv")),
            ((4, 625, 2), 0, ("k_colfft",)), ((4, 625, 2), 1, ("k_colfft",)),
            ((6, 625, 1), 0, ("k_conv",)), ((6, 625, 1), 1, ("k_conv",)),
            ((3, 2, 625), 0, ("k_conv",)), ((3, 2, 625), 1, ("k_conv",))]


@pytest.mark.parametrize("N,prec,kernels", STOCKHAM)
def test_lengths_of_the_stockham_engine(gpu, oracle, tmp_path, N, prec, kernels):
    """The run-time Stockham engine at every schedule, where it is the pass of
    the length: the static plan (schedule 0) launches it."""
    gpu.set_autotune(0)
    base = _check(gpu, oracle, N, (0, 0, 0), prec)
    dt = np.float32 if prec == 0 else np.float64
    m = [_t(np.ones((N[2], N[1], N[0])), dt) for _ in range(3)]
    B = [_t(np.zeros((N[2], N[1], N[0])), dt) for _ in range(3)]
    conv = gpu.DemagConvolution(N, (2e-9, 3e-9, 2.5e-9), precision=prec)
    with gpu.KernelTrace() as tr:
        conv.Exec(B, m, None, 8e5)
    assert base[5:] == [0, 0, 0]
    for k in kernels:
        assert any("um::%s<" % k in name for name in tr.names), (k, tr.names)
    for sc in (1, 2, 3):
        _say("stockham", N, prec, sc)
        f = tmp_path / ("s%d.txt" % sc)
        v = base[:5] + [sc, sc, sc]
        f.write_text("%s: %s\n" % (_key(oracle, N, (0, 0, 0), prec), " ".join(map(str, v))))
        gpu.set_autotune(2, str(f))
        try:
            assert _check(gpu, oracle, N, (0, 0, 0), prec) == v
        finally:
            gpu.set_autotune(0)
