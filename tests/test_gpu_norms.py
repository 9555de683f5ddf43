"""The RK45DP controller norms (um_rk45dp_error) against numpy in FP64: sizes of
the scalar and the 16-byte kernels around a work-group and a full grid, cells
with |k7| = 0, NaN in Err, infinities, and magnitudes whose squares' products
leave the FP64 range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
E = (0.125, -0.25, 0.5, 0.0625, -0.375, 0.03125)


@pytest.fixture(scope="module")
def gpu():
    import torch
    from umagnus_amd import umhip
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    umhip.init(0)
    return umhip


def _ref(k, h):
    err = np.sqrt((sum(e * v for e, v in zip(E, k)) ** 2).sum(0))
    k7 = np.sqrt((k[-1] ** 2).sum(0))
    with np.errstate(divide="ignore", invalid="ignore"):
        rel = np.where(k7 == 0, 0.0, err / k7)
    return err.max() * h, np.nanmax(rel) if np.isfinite(rel).any() else 0.0, k7.max()


def _run(gpu, k, prec, h):
    import torch
    dt = torch.float32 if prec == 0 else torch.float64
    return gpu.RK45DPError([[torch.as_tensor(np.ascontiguousarray(c)).to(dt).cuda() for c in v] for v in k], E, h)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 4, 255, 1024, 1028, 4099, 262144, 262148, 300001])
def test_norms_sizes(gpu, n, prec):
    print("norms", n, prec, flush=True)
    rng = np.random.default_rng(n)
    k = rng.standard_normal((6, 3, n)).astype(np.float32).astype(np.float64)
    k[5][:, rng.random(n) < 0.3] = 0.0   # no torque: relative error 0 there
    got, want = _run(gpu, k, prec, 0.5), _ref(k, 0.5)
    # Err is a sum of six products in the working precision; the norms are FP64
    tol = 6 * (2.0 ** -23 if prec == 0 else 2.0 ** -52)
    for g, w in zip(got, want):
        assert abs(g - w) <= tol * 8 * abs(w), (n, prec, got, want)


@pytest.mark.parametrize("scale", [1e-150, 1e-120, 1e-80, 1e80, 1e140])
def test_norms_range_f64(gpu, scale):
    """Err and k7 both `scale` in magnitude: the quotient stays what it is."""
    rng = np.random.default_rng(3)
    k = rng.standard_normal((6, 3, 5000)) * scale
    got, want = _run(gpu, k, 1, 1.0), _ref(k / scale, 1.0)
    assert abs(got[1] - want[1]) <= 1e-13 * want[1], (got, want)


def test_norms_nan_and_infinity(gpu):
    rng = np.random.default_rng(4)
    k = rng.standard_normal((6, 3, 1000))
    k[2, 1, 77] = np.nan
    got = _run(gpu, k, 1, 1.0)
    assert np.isnan(got[0]) and np.isfinite(got[1]) and np.isfinite(got[2])
    k = rng.standard_normal((6, 3, 1000))
    k[2, 1, 77] = np.inf   # Err infinite, k7 finite there
    got = _run(gpu, k, 1, 1.0)
    assert got[0] == np.inf and got[1] == np.inf and np.isfinite(got[2])
