"""Demag convolution whose spectrum is taken in parts of its kx columns: FP32
grids above the size that fits the last-level cache, against the FP64 plan of
the same grid (never split)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    from umagnus_amd import umhip
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    umhip.init(0)
    return umhip


# register Z pass with the Nyquist column alone in its tile; general Z pass,
# ragged last part; short Z pass; part widths that leave a narrow rest; deep
# columns: a width rounded down to the budget, and grids that stay whole
# because parts within it would be narrow
@pytest.mark.parametrize("N,parts", [((512, 640, 32), 3), ((400, 400, 40), 2), ((1000, 600, 10), 2),
                                     ((1080, 1024, 8), 3), ((525, 1000, 32), 4), ((320, 1080, 32), 3),
                                     ((70, 1000, 64), 1), ((800, 1000, 40), 1)])
def test_parts_match_fp64(gpu, N, parts):
    import torch
    g = torch.Generator(device="cuda").manual_seed(5)
    m = [torch.randn(N[2], N[1], N[0], device="cuda", generator=g) for _ in range(3)]
    out = []
    for prec, dt in ((0, torch.float32), (1, torch.float64)):
        mv = [x.to(dt) for x in m]
        B = [torch.full_like(x, float("nan")) for x in mv]
        conv = gpu.DemagConvolution(N, (2e-9, 3e-9, 4e-9), precision=prec)
        with gpu.KernelTrace() as tr:
            conv.Exec(B, mv, None, 8e5)
        torch.cuda.synchronize()
        conv.Free()
        # FP64 columns of 2000 have no register split
        cols = sum("k_rcol" in k or "k_colfft" in k for k in tr.names)
        assert cols == 2 * (parts if prec == 0 else 1), tr.names
        out.append(B)
    # as the convolution parity tests: FP32 within 2e-6 of the field's scale of
    # FP64 (whose plan these compare with the oracle at 1e-12)
    scale = max(float(b.abs().max()) for b in out[1])
    for a, b in zip(*out):
        assert float((a.double() - b).abs().max()) <= 2e-6 * scale
