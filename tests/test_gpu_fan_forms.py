"""2D operators.  Forward: the line walk over the geometries it accepts (both walks and the
tiles that take the two, two to four pixels per cell, both staging pitches, odd sizes, both
detectors, every storage type) and the candidate form for one it does not, against the FP64
oracle.  Backprojection: the same geometries (footprints of one to eight cells, partly or
wholly off the detector, an odd number of views) in every storage type.

Tolerances: relative L2 <= 1e-5, the repository's FP32 gate, and no cell farther than 1e-4 of
the largest one (a pixel dropped or counted twice on one ray is about 1e-2 of it), each widened
to three times the FP32 oracle's own distance where that is larger, as the other parity tests
do: the DD footprint jumps between a pixel's x and y edges where |cos| = |sin|, which the
central ray of the diagonal views meets exactly.  FP16 / BF16 storage: the rounding of the type, 2^-11 and 2^-8, on input and output."""
import numpy as np
import pytest

from conftest import rel_l2
from helpers import geometry_from_g2

pytestmark = pytest.mark.gpu

DIAG = np.arange(16) * np.pi / 8  # the axes and the exact diagonals among them
CASES = {
    # n, d, o, nu, du, ou, sad, sdd, detector
    "odd": ((33, 70), (0.8, 0.8), (0.0, 0.0), 130, 1.0, 0.25, 1000.0, 1500.0, 1),
    "oblong_pixels": ((61, 47), (0.5, 0.9), (1.3, -2.2), 101, 0.9, -1.5, 1000.0, 1500.0, 1),
    "fine_pixels": ((150, 140), (0.6, 0.6), (0.0, 0.0), 75, 2.0, 0.0, 1000.0, 1500.0, 1),
    "coarse_pixels": ((40, 41), (1.5, 1.5), (0.0, 0.0), 300, 0.4, 0.0, 1000.0, 1500.0, 1),
    "wide_strips": ((210, 190), (0.6, 0.6), (0.0, 0.0), 170, 1.5, 0.0, 1000.0, 1500.0, 1),
    "arc": ((64, 57), (0.8, 0.8), (0.5, 0.0), 129, 1.0, 0.25, 600.0, 1100.0, 0),
    "one_cell": ((9, 1), (0.8, 0.8), (0.0, 0.0), 1, 1.0, 0.0, 1000.0, 1500.0, 1),
    "source_near": ((48, 48), (1.0, 1.0), (0.0, 0.0), 96, 1.5, 0.0, 45.0, 90.0, 1),  # candidate form
}


@pytest.mark.parametrize("kind", ["dd", "tf"])
@pytest.mark.parametrize("name", list(CASES))
def test_fan_forward_vs_fp64_oracle(name, kind):
    from oracle import oracle as O
    from ctsim_amd.device import DeviceArray
    from ctsim_amd.projector import Projector
    n, d, o, nu, du, ou, sad, sdd, det = CASES[name]
    rng = np.random.default_rng(len(name))
    betas = np.concatenate([DIAG, rng.uniform(0, 2 * np.pi, 9)])
    g = O.G2(n[0], n[1], d[0], d[1], o[0], o[1], nu, du, ou, sad, 0.0, sdd, betas, det)
    img = (0.2 + rng.uniform(0, 1, n)).astype(np.float32)
    want = O.fbct(f"proj,{kind}", g, img, prec=64)
    P = Projector(geometry_from_g2(g))
    out = DeviceArray(P.n_sino(), "f32")
    P.proj(P.upload_volume(img), out, f"proj,{kind}")
    got = P.download_sino(out)
    o32 = O.fbct(f"proj,{kind}", g, img)
    assert rel_l2(got, want) <= max(1e-5, 3 * rel_l2(o32, want)), rel_l2(got, want)
    assert np.abs(got - want).max() <= max(1e-4 * np.abs(want).max(), 3 * np.abs(o32 - want).max())
    ex = DeviceArray(P.n_sino(), "f32")
    P.proj(P.upload_volume(img), ex, f"proj,{kind}", exhaustive=True)
    np.testing.assert_array_equal(P.download_sino(ex), got)
    for dt, tol in (("f16", 2.0 ** -11), ("bf16", 2.0 ** -8)):
        half = DeviceArray(P.n_sino(), dt)
        P.proj(P.upload_volume(img, dt), half, f"proj,{kind}")
        assert rel_l2(P.download_sino(half), want) <= max(2 * tol, 3 * rel_l2(o32, want)), dt


@pytest.mark.parametrize("kind", ["dd", "tf"])
@pytest.mark.parametrize("name", list(CASES))
def test_fan_back_vs_fp64_oracle(name, kind):
    from oracle import oracle as O
    from ctsim_amd.device import DeviceArray
    from ctsim_amd.projector import Projector
    n, d, o, nu, du, ou, sad, sdd, det = CASES[name]
    rng = np.random.default_rng(len(name) + 50)
    betas = np.concatenate([DIAG, rng.uniform(0, 2 * np.pi, 9)])
    g = O.G2(n[0], n[1], d[0], d[1], o[0], o[1], nu, du, ou, sad, 0.0, sdd, betas, det)
    sino = (0.2 + rng.uniform(0, 1, (nu, betas.size))).astype(np.float32)
    want = O.fbct(f"back,{kind}", g, sino, prec=64)
    o32 = O.fbct(f"back,{kind}", g, sino)
    P = Projector(geometry_from_g2(g))
    out = DeviceArray(P.n_img, "f32")
    P.back(P.upload_sino(sino), out, f"back,{kind}")
    got = P.download_volume(out)
    assert rel_l2(got, want) <= max(1e-5, 3 * rel_l2(o32, want)), rel_l2(got, want)
    assert np.abs(got - want).max() <= max(1e-4 * np.abs(want).max(), 3 * np.abs(o32 - want).max())
    for dt, tol in (("f16", 2.0 ** -11), ("bf16", 2.0 ** -8)):
        P.back(P.upload_sino(sino, dt), out, f"back,{kind}")
        assert rel_l2(P.download_volume(out), want) <= max(2 * tol, 3 * rel_l2(o32, want)), dt
