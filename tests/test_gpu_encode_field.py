"""GPU parity of the MATLAB encodings (oph_encode_field) against the FP64
restatement of OpenHolo_Encoding/fn_encoding.m, on the same complex64 input."""
import numpy as np
import pytest

from conftest import rel_l2
from oracle import encoding_ref as E

pytestmark = pytest.mark.gpu

METHODS = {"ssb": E.SSB, "ni": E.NI, "p2a": E.P2A, "real": E.REAL, "burckhardt": E.BURCKHARDT,
           "two_phase": E.TWO_PHASE}


def _field(ny, nx, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((ny, nx)) + 1j * rng.standard_normal((ny, nx))).astype(np.complex64)


def _away_from_cuts(u, cuts, eps=1e-5):
    """Pixels whose phase angle + pi is not within eps of a branch boundary
    (float rounding may put those in the neighbouring branch)."""
    ph = np.angle(u.astype(np.complex128)) + np.pi
    return np.all([np.abs(ph - c) > eps for c in cuts], axis=0)


@pytest.mark.parametrize("method", list(METHODS))
def test_encode_field_vs_oracle(ctx, method):
    print(f"case: encode_field {method} 128x64", flush=True)
    u = _field(64, 128, 11)
    out = ctx.encode_field(u, method)
    ref = E.encode(u.astype(np.complex128), METHODS[method])
    assert out.shape == ref.shape
    if method in ("burckhardt", "two_phase", "p2a"):
        k = ref.shape[1] // u.shape[1]
        ok = _away_from_cuts(u, [0.0, 2 * np.pi / 3, 4 * np.pi / 3, 2 * np.pi])
        ok = np.repeat(ok, k, axis=1)
        assert ok.mean() > 0.99
        err = rel_l2(out[ok], ref[ok])
    else:
        err = rel_l2(out, ref)
    print(method, "rel-L2", err)
    assert err < 1e-5


@pytest.mark.parametrize("passband", ["left", "right", "top", "bottom"])
def test_encode_ssb_passbands(ctx, passband):
    u = _field(32, 256, 12)
    out = ctx.encode_field(u, "ssb", passband=passband)
    ref = E.ssb(u.astype(np.complex128), {"left": E.LEFT, "right": E.RIGHT, "top": E.TOP,
                                          "bottom": E.BOTTOM}[passband])
    assert rel_l2(out, ref) < 1e-5


def test_encode_field_device_and_errors(ctx):
    from openhologram_amd import OphError
    u = _field(16, 16, 13)
    d = ctx.to_device(u)
    out = ctx.empty((16, 32), np.float32)
    ctx.encode_field(d, "two_phase", device=True, out=out)
    assert np.allclose(out.numpy(), ctx.encode_field(u, "two_phase"))
    with pytest.raises(OphError):
        ctx.encode_field(_field(16, 24, 1), "ssb")   # SSB needs power-of-two sides
    with pytest.raises(OphError):
        ctx.encode_field(u, "ssb", asynchronous=True)  # async needs device pointers


@pytest.mark.parametrize("passband", ["left", "right", "top", "bottom"])
@pytest.mark.parametrize("ny,nx", [(16, 32), (64, 16), (128, 1024), (512, 256), (2048, 64), (32, 4096), (8192, 16),
                                   (16, 8192)])
def test_encode_ssb_line_lengths(ctx, ny, nx, passband):
    """One-dimensional sideband filter at every transform length, whole and
    partial groups of lines.  Bound: a forward and an inverse FP32 transform of
    at most four stages, about 1e-7 a stage: 2e-6 with the scaling."""
    print(f"case: ssb {nx}x{ny} {passband}", flush=True)
    u = _field(ny, nx, ny + nx)
    ref = E.ssb(u.astype(np.complex128), {"left": E.LEFT, "right": E.RIGHT, "top": E.TOP,
                                          "bottom": E.BOTTOM}[passband])
    assert rel_l2(ctx.encode_field(u, "ssb", passband=passband), ref) < 2e-6


def test_encode_ssb_aliased_and_not_finite(ctx):
    """The output may overlap the field; a field with a NaN gives NaN everywhere
    (as a two-dimensional transform of it does)."""
    u = _field(64, 128, 5)
    ref = ctx.encode_field(u, "ssb", passband="top")
    d = ctx.to_device(u)
    ctx.encode_field(d, "ssb", passband="top", device=True, out=d.ptr)
    assert np.array_equal(d.numpy().view(np.float32).ravel()[:64 * 128], ref.ravel())
    u[3, 5] = np.nan
    assert np.isnan(ctx.encode_field(u, "ssb")).all()


@pytest.mark.parametrize("mean", [3.0, -3.0])
@pytest.mark.parametrize("passband", ["right", "bottom"])
@pytest.mark.parametrize("n", [16, 32, 64])
def test_encode_ssb_one_sided(ctx, n, passband, mean):
    """A carrier in the passband: the filtered field lies on one side of zero,
    so a zero that enters the minimum or the maximum shows.  Lines of 16 and 32
    columns are workgroups of less than a wave.  Bound: the transforms' 2e-6 of
    the mean, against a spread of at least a thirtieth of it: 6e-5 of outputs
    that are about half of one: 1.2e-4."""
    print(f"case: ssb one-sided {n} {passband} mean {mean}", flush=True)
    u = (mean + 0.1 * _field(*((n, 64) if passband == "bottom" else (64, n)), n)).astype(np.complex64)
    ref = E.ssb(u.astype(np.complex128), {"right": E.RIGHT, "bottom": E.BOTTOM}[passband])
    assert rel_l2(ctx.encode_field(u, "ssb", passband=passband), ref) < 1.2e-4
