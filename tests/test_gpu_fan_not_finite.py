"""2D operators: a value that is not finite (a dead detector cell, an overflow of FP16 storage)
stays with the pixels or cells that it weighs on, and a pixel that no view sees is zero.

Which those are comes from the oracle.  A footprint edge that meets a cell edge to within the
rounding may fall on either side of it, so the value `must` reach what it weighs on by more than
1e-6 of its largest weight and `may` reach what it weighs on at all on any of three detectors
shifted by 1e-3 cells against each other (the FP32 edges are within 1e-4 cells)."""
import numpy as np
import pytest

from helpers import geometry_from_g2

pytestmark = pytest.mark.gpu

SHIFTS = (-1e-3, 0.0, 1e-3)
# image sizes, pixel, detector cells, cell, detector offset, SAD, SDD, detector type
FANS = {
    # the image overhangs the detector on both sides, by most of it on the low side
    "overhang": ((60, 50), (1.2, 1.2), 40, 1.0, 14.0, 1000.0, 1500.0, 1),
    "overhang_arc": ((60, 50), (1.2, 1.2), 40, 1.0, 14.0, 600.0, 1100.0, 0),
    # the same so far that views are passed over (images of 256^2 pixels and more)
    "far_overhang": ((260, 256), (1.2, 1.2), 40, 1.0, 14.0, 1000.0, 1500.0, 1),
    # pixels of two to four cells, inside the detector; oblong pixels
    "fine_cells": ((31, 44), (1.5, 1.1), 200, 0.7, 0.25, 1000.0, 1500.0, 1),
}
# cells of one value each, and their views: the ends of the detector that the image overhangs
CELLS = {"overhang": ((0, 1), (2, 0), (20, 2), (39, 4)), "overhang_arc": ((0, 1), (2, 0), (20, 2), (39, 4)),
         "far_overhang": ((0, 1), (39, 4)), "fine_cells": ((70, 0), (101, 2), (130, 4))}
BETAS = np.array([0.05, 0.2, np.pi / 4, 0.9, 1.1])  # a short arc, so that pixels stay unseen


def _fan(name, shift=0.0):
    from oracle import oracle as O
    n, d, nu, du, ou, sad, sdd, det = FANS[name]
    return O.G2(n[0], n[1], d[0], d[1], 0.0, 0.0, nu, du, ou + shift, sad, 0.0, sdd, BETAS, det)


def _back(name, kind, sino, dt, batch):
    from ctsim_amd.batch2 import Batch2
    from ctsim_amd.device import DeviceArray
    from ctsim_amd.projector import Projector
    geom = geometry_from_g2(_fan(name))
    if not batch:
        P = Projector(geom)
        out = DeviceArray(P.n_img, "f32")
        P.back(P.upload_sino(sino, dt), out, f"back,{kind}")
        return P.download_volume(out)
    B = Batch2([geom, geom])
    out = DeviceArray(B.img_elems, "f32")
    B.back(DeviceArray.from_numpy(np.tile(sino.ravel(order="F"), 2), dt), out, f"back,{kind}")
    a, b = B.unpack_images(out.to_numpy())
    np.testing.assert_array_equal(a, b)
    return a


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("kind", ["dd", "tf"])
@pytest.mark.parametrize("name", list(FANS))
def test_back_keeps_values_that_are_not_finite_in_their_pixels(name, kind, dt, batch):
    from oracle import oracle as O
    rng = np.random.default_rng(3)
    nu = FANS[name][2]
    clean = (0.2 + rng.uniform(0, 1, (nu, BETAS.size))).astype(np.float32)
    want = _back(name, kind, clean, dt, batch)
    assert np.isfinite(want).all()
    unseen = ~sum(O.fbct(f"back,{kind}", _fan(name, s), np.ones_like(clean), prec=64) != 0 for s in SHIFTS).astype(bool)
    assert unseen.any() == (name != "fine_cells")
    assert not want[unseen].any()
    for value in (np.nan, np.inf):
        for cell, view in CELLS[name]:
            only = np.zeros_like(clean)
            only[cell, view] = 1
            low, weight, high = (O.fbct(f"back,{kind}", _fan(name, s), only, prec=64) for s in SHIFTS)
            must = weight > 1e-6 * weight.max()
            may = (low != 0) | (weight != 0) | (high != 0)
            assert must.any()
            sino = clean.copy()
            sino[cell, view] = value
            got = _back(name, kind, sino, dt, batch)
            bad = ~np.isfinite(got)
            assert not (must & ~bad).any(), (value, cell, view)
            assert not (bad & ~may).any(), (value, cell, view, int((bad & ~may).sum()))
            np.testing.assert_array_equal(got[~may], want[~may])


@pytest.mark.parametrize("det", [1, 0])
@pytest.mark.parametrize("kind", ["dd", "tf"])
def test_back_of_images_far_beyond_the_detector_vs_fp64_oracle(kind, det):
    """The form that passes over views, an odd number of them, alone and in a batch with a slice
    that would not take it: relative L2 <= 1e-5, the repository's FP32 gate, or three times the
    FP32 oracle's own distance where that is larger, as in the other parity tests."""
    from conftest import rel_l2
    from oracle import oracle as O
    from ctsim_amd.batch2 import Batch2
    from ctsim_amd.device import DeviceArray
    from ctsim_amd.projector import Projector
    rng = np.random.default_rng(5)
    betas = rng.uniform(0, 2 * np.pi, 27)
    far = O.G2(259, 257, 1.1, 1.0, 2.0, -1.0, 41, 1.3, 3.0, 1000.0, 0.0, 1500.0, betas, det)
    near = O.G2(70, 61, 0.8, 0.8, 0.0, 0.0, 130, 1.0, 0.25, 1000.0, 0.0, 1500.0, betas[:6], det)
    sinos = [(0.2 + rng.uniform(0, 1, (g.nu, g.nviews))).astype(np.float32) for g in (far, near)]
    wants = [O.fbct(f"back,{kind}", g, s, prec=64) for g, s in zip((far, near), sinos)]
    tols = [max(1e-5, 3 * rel_l2(O.fbct(f"back,{kind}", g, s), w)) for g, s, w in zip((far, near), sinos, wants)]
    P = Projector(geometry_from_g2(far))
    out = DeviceArray(P.n_img, "f32")
    P.back(P.upload_sino(sinos[0]), out, f"back,{kind}")
    assert rel_l2(P.download_volume(out), wants[0]) <= tols[0]
    B = Batch2([geometry_from_g2(near), geometry_from_g2(far)])
    img = DeviceArray(B.img_elems, "f32")
    flat = np.concatenate([s.ravel(order="F") for s in sinos[::-1]])
    for split in (1, 2, 4):
        B.set_schedule(1, split)
        B.back(DeviceArray.from_numpy(flat, "f32"), img, f"back,{kind}")
        for got, want, tol in zip(B.unpack_images(img.to_numpy()), wants[::-1], tols[::-1]):
            assert rel_l2(got, want) <= tol, (split, rel_l2(got, want))


def _proj(name, kind, img, dt, batch):
    from ctsim_amd.batch2 import Batch2
    from ctsim_amd.device import DeviceArray
    from ctsim_amd.projector import Projector
    geom = geometry_from_g2(_fan(name))
    if not batch:
        P = Projector(geom)
        out = DeviceArray(P.n_sino(), "f32")
        P.proj(P.upload_volume(img, dt), out, f"proj,{kind}")
        return P.download_sino(out)
    B = Batch2([geom, geom])
    out = DeviceArray(B.sino_elems, "f32")
    B.proj(DeviceArray.from_numpy(B.pack_images([img, img]), dt), out, f"proj,{kind}")
    a, b = B.unpack_sinos(out.to_numpy())
    np.testing.assert_array_equal(a, b)
    return a


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("kind", ["dd", "tf"])
@pytest.mark.parametrize("name", [n for n in FANS if n != "far_overhang"])
def test_proj_keeps_values_that_are_not_finite_in_their_cells(name, kind, dt, batch):
    """the other cells keep their values to the repository's FP32 gate, 1e-5 of the largest (the
    same products may be added in another order)"""
    from oracle import oracle as O
    rng = np.random.default_rng(4)
    nx, ny = FANS[name][0]
    clean = (0.2 + rng.uniform(0, 1, (nx, ny))).astype(np.float32)
    want = _proj(name, kind, clean, dt, batch)
    assert np.isfinite(want).all()
    for value in (np.nan, np.inf):
        for ix, iy in ((nx // 2 - 4, ny // 2), (nx // 2, 0), (nx // 2 - 2, ny - 1)):
            only = np.zeros_like(clean)
            only[ix, iy] = 1
            low, weight, high = (O.fbct(f"proj,{kind}", _fan(name, s), only, prec=64) for s in SHIFTS)
            must = weight > 1e-6 * weight.max()
            may = (low != 0) | (weight != 0) | (high != 0)
            assert must.any()
            img = clean.copy()
            img[ix, iy] = value
            got = _proj(name, kind, img, dt, batch)
            bad = ~np.isfinite(got)
            assert not (must & ~bad).any(), (value, ix, iy)
            assert not (bad & ~may).any(), (value, ix, iy, int((bad & ~may).sum()))
            np.testing.assert_allclose(got[~may], want[~may], rtol=0, atol=1e-5 * want.max())
