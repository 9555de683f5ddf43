"""Register-stage FFT passes of the demag convolution against the FP64 oracle:
every radix they use, one to three stages, remainders of a tile (rows, columns
and work items that do not fill a work-group), odd and periodic lengths, short
z columns in registers, per-cell Ms with a geometry, and component arrays that
are not aligned for pairwise access.

Tolerances as for the convolution parity tests: FP64 1e-12, FP32 2e-6
normwise against the FP64 oracle."""
import numpy as np
import pytest

from cases import random_unit

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    from umagnus_amd import umhip
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    umhip.init(0)
    return umhip


CASES = [
    # X radices: 1 stage up to 16, odd lengths (no pairwise access), 2 and 3 stages
    ((1, 4, 1), (0, 0, 0)), ((2, 3, 1), (0, 0, 0)), ((7, 5, 1), (0, 0, 0)), ((15, 9, 1), (0, 0, 0)),
    ((16, 14, 2), (0, 0, 0)), ((35, 21, 1), (0, 0, 0)), ((45, 50, 3), (0, 0, 0)), ((63, 28, 1), (0, 0, 0)),
    ((98, 12, 1), (0, 0, 0)), ((144, 10, 4), (0, 0, 0)), ((162, 6, 1), (0, 0, 0)), ((225, 7, 1), (0, 0, 0)),
    ((400, 5, 2), (0, 0, 0)), ((720, 3, 1), (0, 0, 0)), ((1008, 2, 1), (0, 0, 0)),
    # Y columns and the film convolution
    ((6, 81, 2), (0, 0, 0)), ((10, 160, 6), (0, 0, 0)), ((6, 245, 3), (0, 0, 0)), ((20, 500, 1), (0, 0, 0)),
    ((6, 640, 1), (0, 0, 0)), ((420, 64, 1), (0, 0, 0)),
    # z columns in registers (Nz 2..7, 9, 10, 12) and in LDS, odd column counts
    ((12, 9, 2), (0, 0, 0)), ((12, 9, 3), (0, 0, 0)), ((70, 6, 4), (0, 0, 0)), ((60, 7, 5), (0, 0, 0)),
    ((30, 10, 6), (0, 0, 0)), ((70, 8, 7), (0, 0, 0)), ((12, 15, 9), (0, 0, 0)), ((14, 6, 10), (0, 0, 0)),
    ((20, 5, 12), (0, 0, 0)), ((10, 6, 15), (0, 0, 0)), ((9, 4, 20), (0, 0, 0)), ((6, 5, 70), (0, 0, 0)),
    # periodic axes: half lengths, odd lengths, no z padding
    ((20, 12, 6), (1, 0, 0)), ((21, 10, 1), (0, 1, 0)), ((18, 15, 5), (0, 1, 1)), ((14, 6, 9), (0, 0, 2)),
]


def _misaligned(a, dtype):
    """A device copy of a that starts one value past the allocator's alignment."""
    import torch
    t = torch.empty(a.size + 1, dtype=dtype, device="cuda")
    v = t[1:].view(*a.shape)
    v.copy_(torch.as_tensor(a))
    return v


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("N,pbc", CASES)
def test_register_passes_vs_oracle(gpu, oracle, N, pbc, prec):
    import torch
    print("register passes", N, pbc, prec, flush=True)
    dt = torch.float32 if prec == 0 else torch.float64
    shape, cs = (N[2], N[1], N[0]), (2e-9, 3e-9, 2.5e-9)
    rng = np.random.default_rng(sum(N))
    m = random_unit(shape, sum(N) + 1)
    Ms = rng.uniform(5e5, 1e6, shape)
    vol = rng.choice([0.0, 0.5, 1.0], shape)
    conv = gpu.DemagConvolution(N, cs, pbc=pbc, precision=prec)
    od = oracle.Demag(N, cs, pbc=pbc, dtype=np.float64)
    up = lambda a: torch.as_tensor(np.ascontiguousarray(a)).to(dt).cuda()
    for place, v, ms in ((up, None, 8e5), (up, vol, Ms), (lambda a: _misaligned(a, dt), vol, Ms)):
        B = [place(np.zeros(shape)) for _ in range(3)]
        conv.Exec(B, [place(m[c]) for c in range(3)], None if v is None else place(v),
                  ms if np.isscalar(ms) else place(ms))
        got = np.stack([b.cpu().numpy() for b in B]).astype(np.float64)
        ref = od.exec(m, np.full(shape, ms) if np.isscalar(ms) else ms, vol=v)
        err = np.abs(got - ref).max() / np.abs(ref).max()
        assert err < (1e-12 if prec == 1 else 2e-6), (N, pbc, prec, err)


# periodic z: dense columns in registers (FP32, 2..8 and 16 points, the latter
# from 24576 columns) and in LDS (9, 16 below that, FP64); odd column counts,
# rows with and without a mirror
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("N,pbc", [((10, 6, 2), (0, 0, 1)), ((35, 7, 3), (0, 0, 2)), ((30, 5, 4), (1, 0, 1)),
                                   ((12, 9, 5), (0, 0, 1)), ((9, 4, 6), (1, 1, 1)), ((70, 6, 7), (0, 0, 1)),
                                   ((20, 7, 8), (0, 1, 1)), ((12, 10, 9), (0, 0, 1)), ((20, 12, 16), (0, 0, 1)),
                                   ((126, 98, 16), (0, 0, 1))])
def test_periodic_z_vs_oracle(gpu, oracle, N, pbc, prec):
    test_register_passes_vs_oracle(gpu, oracle, N, pbc, prec)


def test_periodic_z_kernels(gpu):
    """FP32 dense columns run in registers from 2 to 8 points and, with enough
    columns, of 16."""
    import torch
    for N, short in (((64, 8, 3), True), ((32, 8, 8), True), ((32, 8, 9), False), ((32, 8, 16), False),
                     ((128, 96, 16), True)):
        m = [torch.ones(N[2], N[1], N[0], device="cuda") for _ in range(3)]
        B = [torch.zeros_like(x) for x in m]
        conv = gpu.DemagConvolution(N, (2e-9,) * 3, pbc=(0, 0, 1), precision=0)
        with gpu.KernelTrace() as tr:
            conv.Exec(B, m, None, 8e5)
        assert any("k_rshort" in k for k in tr.names) == short, (N, tr.names)
