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
# ragged last part; short Z pass; part widths that leave a narrow rest
@pytest.mark.parametrize("N", [(512, 640, 32), (400, 400, 40), (1000, 600, 10), (1080, 1024, 8)])
def test_parts_match_fp64(gpu, N):
    import torch
    g = torch.Generator(device="cuda").manual_seed(5)
    m = [torch.randn(N[2], N[1], N[0], device="cuda", generator=g) for _ in range(3)]
    out = []
    for prec, dt in ((0, torch.float32), (1, torch.float64)):
        mv = [x.to(dt) for x in m]
        B = [torch.full_like(x, float("nan")) for x in mv]
        conv = gpu.DemagConvolution(N, (2e-9, 3e-9, 4e-9), precision=prec)
        conv.Exec(B, mv, None, 8e5)
        torch.cuda.synchronize()
        conv.Free()
        out.append(B)
    # three FP32 transforms each way: some 25 levels of rounding at 6e-8, and
    # the tensor's own rounding, on the scale of the field
    scale = max(float(b.abs().max()) for b in out[1])
    for a, b in zip(*out):
        assert float((a.double() - b).abs().max()) <= 1e-5 * scale
