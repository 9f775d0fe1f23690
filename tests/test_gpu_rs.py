"""GPU parity of the exact RS point-cloud field (oph_pc_rs) against the FP64
oracle (tolerance rel-L2 1e-5 on the complex field) and the reference's
FP32 fringe fixtures."""
import numpy as np
import pytest

from conftest import rel_l2
from oracle import oracle as O
import openhologram_amd as oph
from openhologram_amd import scenes

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _s64(spec):
    return dict(nx=spec["nx"], ny=spec["ny"], pitch=spec["pitch"], lambda_=spec["lambda_"],
                scale=spec.get("scale", (1, 1, 1)), offset_z=spec.get("offset_z", 0.0),
                tilt_deg=spec.get("tilt_deg", (0, 0)))


def test_rs_1000pts_1024sq_full_size(ctx):
    """1000 seeded points, 1024^2 at 8 um, 532 nm, complex128 out."""
    print("case: rs 1024x1024 P=1000", flush=True)
    x, y, z, a, ph = scenes.rs_points(1000, seed=1)
    spec = dict(scenes.RS_SPEC)
    U = ctx.pc_rs(spec, x, y, z, a, ph)
    ref = O.rs(_s64(spec), x, y, z, a, ph)
    err = rel_l2(U, ref)
    print("rel-L2", err)
    assert err < TOL


@pytest.mark.parametrize("nx,ny,tilt", [(100, 37, (0, 0)), (64, 64, (22.5, 22.5)), (130, 70, (3, -7))])
def test_rs_ragged_and_tilt(ctx, nx, ny, tilt):
    print(f"case: rs ragged {nx}x{ny} tilt {tilt}", flush=True)
    x, y, z, a, ph = scenes.rs_points(300, seed=7)
    spec = dict(nx=nx, ny=ny, pitch=(8e-6, 6e-6), lambda_=633e-9, tilt_deg=tilt)
    U = ctx.pc_rs(spec, x, y, z, a, ph)
    assert rel_l2(U, O.rs(_s64(spec), x, y, z, a, ph)) < TOL


def test_rs_near_field_exact_path(ctx):
    """Points 0.5-2 mm from the plane with wide lateral spread take the FP64
    per-pixel path (second-order expansion out of range)."""
    print("case: rs near field", flush=True)
    g = scenes.SplitMix64(11)
    n = 200
    x, y = g.uniform(n, -2e-3, 2e-3), g.uniform(n, -2e-3, 2e-3)
    z = g.uniform(n, 0.5e-3, 2e-3)
    a = g.uniform(n)
    spec = dict(nx=256, ny=192, pitch=8e-6, lambda_=532e-9)
    U = ctx.pc_rs(spec, x, y, z, a)
    assert rel_l2(U, O.rs(_s64(spec), x, y, z, a)) < TOL


def test_rs_keti_fringe_fixtures(ctx, golden_keti):
    """Float fringe mode vs the reference fixtures (the reference's own FP32
    noise bounds the match) and vs the FP64 oracle (tight)."""
    pts = golden_keti["points"]
    for name in golden_keti["case_names"]:
        print("case: keti fixture", name, flush=True)
        s = golden_keti[f"spec_{name}"]
        spec = dict(nx=int(s[6]), ny=int(s[7]), pitch=(float(s[4]), float(s[5])),
                    lambda_=float(s[8]), scale=tuple(float(v) for v in s[0:3]),
                    offset_z=float(s[3]), tilt_deg=(float(s[9]), float(s[10])))
        fr = ctx.pc_rs(spec, pts[:, 0], pts[:, 1], pts[:, 2], pts[:, 3], fmt=oph.OUT_FRINGE)
        assert fr.dtype == np.float32
        ref64 = O.rs(_s64(spec), pts[:, 0], pts[:, 1], pts[:, 2], pts[:, 3]).real
        assert rel_l2(fr, ref64) < 1e-5
        assert rel_l2(fr, golden_keti[f"fringe_{name}"]) < 0.1


def test_rs_accumulate_device_and_c64(ctx):
    print("case: rs accumulate / device / c64", flush=True)
    x, y, z, a, ph = scenes.rs_points(500, seed=3)
    spec = dict(nx=128, ny=96, pitch=8e-6, lambda_=532e-9)
    ref = O.rs(_s64(spec), x, y, z, a, ph)
    out = ctx.pc_rs(spec, x, y, z, a, ph)
    ctx.pc_rs(spec, x, y, z, a, ph, out=out, accumulate=True)
    assert rel_l2(out, 2 * ref) < TOL
    d = [ctx.to_device(v) for v in (x, y, z, a, ph)]
    dout = ctx.pc_rs(spec, *d, fmt=oph.OUT_C64, device=True)
    U = dout.numpy()
    assert U.dtype == np.complex64 and rel_l2(U, ref) < 2e-5


def test_rs_empty_point_set(ctx):
    spec = dict(nx=64, ny=64, pitch=8e-6, lambda_=532e-9)
    e = np.zeros(0)
    U = ctx.pc_rs(spec, e, e, e, e)
    assert np.all(U == 0)


def test_rs_invalid_args(ctx):
    with pytest.raises(oph.OphError):
        ctx.pc_rs(dict(nx=0, ny=64, pitch=8e-6, lambda_=532e-9), [0.0], [0.0], [0.1], [1.0])
    with pytest.raises(oph.OphError):
        ctx.pc_rs(dict(nx=64, ny=64, pitch=8e-6, lambda_=-1.0), [0.0], [0.0], [0.1], [1.0])


@pytest.mark.parametrize("nx,ny,z", [(256, 192, 0.1), (130, 70, 0.02)])
def test_huygens_vs_oracle(ctx, nx, ny, z):
    """cwoPLS::Huygens (1/r amplitude, CWO grid) against the FP64 oracle,
    including points close enough for the per-pixel FP64 path."""
    print(f"case: huygens {nx}x{ny} z {z}", flush=True)
    rng = np.random.default_rng(nx)
    n = 700
    x, y = rng.uniform(-5e-4, 5e-4, (2, n))
    zz = rng.uniform(-0.005, 0.005, n)
    a, ph = rng.uniform(0, 1, n), rng.uniform(0, 2 * np.pi, n)
    U = ctx.huygens(nx, ny, 8e-6, 532e-9, z, x, y, zz, a, ph, ph=0.25)
    ref = O.huygens(nx, ny, 8e-6, 532e-9, z, x, y, zz, a, ph, ph=0.25)
    err = rel_l2(U, ref)
    print("rel-L2", err)
    assert err < 1e-5
    V = ctx.huygens(nx, ny, 8e-6, 532e-9, z, x, y, zz, a, ph, ph=0.25, fmt=oph.OUT_C64, out=U.astype(np.complex64),
                    accumulate=True)
    assert rel_l2(V, 2 * ref) < 1e-5


@pytest.mark.parametrize("nx,ny,n,zlo,zhi,near", [
    (70, 45, 1, 0.1, 0.1, 0),        # one point, partial blocks
    (33, 97, 63, 0.09, 0.11, 0),     # one short batch of the contraction
    (128, 64, 65, 0.2, 0.3, 0),      # one point past a batch, whole tiles
    (200, 130, 1100, 0.04, 0.06, 0),  # two to five terms, split over chunks
    (96, 100, 130, 0.1, 0.12, 7),    # some points out of the expansion's range
    (100, 70, 300, 2e-3, 4e-3, 0),   # tiles too close: a sin and cos per pixel
])
@pytest.mark.parametrize("huygens", [False, True])
def test_rs_contraction_edges(ctx, nx, ny, n, zlo, zhi, near, huygens):
    """Separable contraction at its edges (partial blocks, batches of 64
    points, one to five terms, points out of range summed per pixel) and the
    direct form.  Bound per term: reduced phases 2 x 2^-25 turns and the centre
    phase 2^-25 (5e-7 rad), dropped terms 3e-7 rad, FP32 products and sums of
    at most 64 terms (under 5e-7): 2e-6 in the 2-norm."""
    print(f"case: rs contraction {nx}x{ny} P={n} z {zlo}..{zhi} near {near} huygens {huygens}", flush=True)
    g = scenes.SplitMix64(100 + n)
    x, y, z = g.uniform(n, -5e-3, 5e-3), g.uniform(n, -5e-3, 5e-3), g.uniform(n, zlo, zhi)
    z[:near] = 3e-3
    a, ph = g.uniform(n, 0.1, 1.0), g.uniform(n, 0.0, 2 * np.pi)
    if huygens:
        U = ctx.huygens(nx, ny, 8e-6, 532e-9, 0.0, x, y, z, a, ph)
        ref = O.huygens(nx, ny, 8e-6, 532e-9, 0.0, x, y, z, a, ph)
    else:
        spec = dict(nx=nx, ny=ny, pitch=(8e-6, 6e-6), lambda_=532e-9)
        U = ctx.pc_rs(spec, x, y, z, a, ph)
        ref = O.rs(_s64(spec), x, y, z, a, ph)
    err = rel_l2(U, ref)
    print("rel-L2", err)
    assert err < 2e-6


@pytest.mark.parametrize("huygens", [False, True])
@pytest.mark.parametrize("z0", [0.3, 0.5, 1.0])
def test_rs_error_at_long_distances(ctx, z0, huygens):
    """Beyond 0.3 m a sum per pixel of 100 points has 2.0e-7 to 2.2e-7 from
    FP64 (one rounded phase, FP32 sums of 100); the contraction, which rounds
    two phases but sums 16 products at a time, stays within 2.5e-7."""
    print(f"case: rs z {z0} huygens {huygens}", flush=True)
    n = 100
    g = scenes.SplitMix64(n)
    x, y, z = g.uniform(n, -5e-3, 5e-3), g.uniform(n, -5e-3, 5e-3), g.uniform(n, z0, 1.02 * z0)
    a, ph = g.uniform(n), g.uniform(n, 0.0, 2 * np.pi)
    if huygens:
        U = ctx.huygens(300, 200, 8e-6, 532e-9, 0.0, x, y, z, a, ph)
        ref = O.huygens(300, 200, 8e-6, 532e-9, 0.0, x, y, z, a, ph)
    else:
        spec = dict(nx=300, ny=200, pitch=8e-6, lambda_=532e-9)
        U, ref = ctx.pc_rs(spec, x, y, z, a, ph), O.rs(_s64(spec), x, y, z, a, ph)
    err = rel_l2(U, ref)
    print("rel-L2", err)
    assert err < 2.5e-7


@pytest.mark.parametrize("huygens", [False, True])
@pytest.mark.parametrize("amp", [np.inf, -np.inf, 3e38])
@pytest.mark.parametrize("n,at", [(1, 0), (100, 37), (600, 599)])
def test_rs_huge_amplitudes(ctx, n, at, amp, huygens):
    """A point of infinite amplitude adds +-inf to both parts of every pixel,
    one near the largest float its finite value: no NaN from the contraction's
    intermediate sums.  Signs are compared where the cosine or sine is above
    1e-3 (phases agree to 1e-6)."""
    print(f"case: rs amplitude {amp} at {at} of {n} huygens {huygens}", flush=True)
    g = scenes.SplitMix64(n)
    x, y, z = g.uniform(n, -5e-4, 5e-4), g.uniform(n, -5e-4, 5e-4), g.uniform(n, 1.05, 1.1)
    a, ph = g.uniform(n, 0.1, 1.0), g.uniform(n, 0.0, 2 * np.pi)
    one = [v[at:at + 1] for v in (x, y, z)] + [np.ones(1), ph[at:at + 1]]
    a[at] = amp
    if huygens:
        U = ctx.huygens(150, 70, 8e-6, 532e-9, 0.0, x, y, z, a, ph, fmt=oph.OUT_C64)
        one = O.huygens(150, 70, 8e-6, 532e-9, 0.0, *one)
    else:
        spec = dict(nx=150, ny=70, pitch=8e-6, lambda_=532e-9)
        U, one = ctx.pc_rs(spec, x, y, z, a, ph, fmt=oph.OUT_C64), O.rs(_s64(spec), *one)
    if np.isinf(amp):
        for got, unit in ((U.real, one.real), (U.imag, one.imag)):
            ok = np.abs(unit) > 1e-3
            assert np.all(np.isinf(got[ok])) and np.all(np.sign(got[ok]) == np.sign(unit[ok] * amp))
    else:
        assert rel_l2(U / np.float32(amp), one) < 2e-6
