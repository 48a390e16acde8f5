"""The 3D backprojector's four-column form: 4 to 32 voxels per lane and z-slabs, each gather
class (voxels of less than one to three rows), one to several 64-row chunks and odd row counts,
each storage type, footprints of more than four cells, a detector that the image overhangs,
both detector types, couch, map and odd image sizes, against the FP64 oracle; the same bits from
both column orders.

Tolerance: relative L2 <= 1e-5, widened to three times the FP32 oracle's own distance where that
is larger, as in the other parity tests."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_parity import TOL, _cone_case, geometry_from_g3

pytestmark = pytest.mark.gpu

CASES = {
    # nx * ny columns enough for the form: 16384 of up to 64 slices, 6400 of more
    "lanes4": (dict(seed=60, n=(129, 128, 61), nuv=(256, 57), nviews=18, dz=0.6, dv=1.1), "f32"),
    "few_rows": (dict(seed=61, n=(131, 127, 5), nuv=(250, 4), nviews=5, dz=0.6, dv=1.1), "bf16"),
    "lanes8": (dict(seed=62, n=(81, 80, 65), nuv=(180, 66), nviews=17, dz=1.0, dv=1.0, dettype=0, couch=True), "f16"),
    "odd_rows": (dict(seed=63, n=(80, 83, 100), nuv=(180, 65), nviews=7, dz=1.0, dv=1.2, dettype=0), "f32"),
    "odd_rows_16": (dict(seed=63, n=(80, 83, 100), nuv=(180, 65), nviews=7, dz=1.0, dv=1.2), "f16"),  # one column
    "lanes16": (dict(seed=64, n=(81, 80, 129), nuv=(180, 202), nviews=16, dz=0.7, dv=0.6, offsets=True), "bf16"),
    "rows3": (dict(seed=65, n=(81, 80, 70), nuv=(180, 300), nviews=5, dz=0.9, dv=0.5, couch=True), "f32"),
    "lanes32": (dict(seed=66, n=(80, 81, 300), nuv=(170, 205), nviews=4, dz=0.3, dv=0.6), "f32"),
    "slabs": (dict(seed=67, n=(80, 80, 525), nuv=(170, 768), nviews=3, dz=0.3, dv=0.3, map_=False), "f32"),
    "too_many_rows": (dict(seed=68, n=(80, 80, 70), nuv=(170, 769), nviews=3, dz=0.9, dv=0.4), "f32"),
    # detector shorter and narrower than the image's shadow: columns and views without cells
    "overhang": (dict(seed=69, n=(90, 81, 130), nuv=(61, 131), nviews=19, dz=0.9, dv=0.55, couch=True), "f32"),
    "overhang_16": (dict(seed=70, n=(90, 81, 130), nuv=(62, 130), nviews=19, dz=0.9, dv=0.55), "bf16"),
}


def _check(g, sino, mp, kind, dt):
    from oracle import oracle as O
    from ctsim_amd.device import DeviceArray
    from ctsim_amd.projector import Projector
    P = Projector(geometry_from_g3(g, mp))
    d_sino = P.upload_sino(sino, dtype=dt)
    seen = np.asarray(P.download_sino(d_sino), np.float32)
    want = O.cbct(f"back,{kind}", g, seen, mp, prec=64, nthreads=8)
    tol = max(TOL, 3 * rel_l2(O.cbct(f"back,{kind}", g, seen, mp, nthreads=8), want))
    img = DeviceArray(P.n_img, "f32")
    P.back(d_sino, img, f"back,{kind}")
    got = P.download_volume(img)
    assert rel_l2(got, want) <= tol, (rel_l2(got, want), tol)
    if mp is not None:
        assert not got[~mp].any()
    P.set_schedule(back_sched=0)
    P.back(d_sino, img, f"back,{kind}")
    np.testing.assert_array_equal(P.download_volume(img), got)
    # onto what the volume holds, scaled
    P.set_schedule(back_sched=1)
    P.back(d_sino, img, f"back,{kind}", scale=0.5, accumulate=True)
    assert rel_l2(P.download_volume(img), 1.5 * want) <= tol


@pytest.mark.parametrize("kind", ["dd", "tf"])
@pytest.mark.parametrize("name", list(CASES))
def test_four_column_form_vs_fp64_oracle(name, kind):
    case, dt = CASES[name]
    g, _, sino, mp = _cone_case(**case)
    print(name, kind, g.n.tolist(), flush=True)
    _check(g, sino, mp, kind, dt)


@pytest.mark.parametrize("dt", ["f32", "f16"])
@pytest.mark.parametrize("kind,du", [("dd", 0.36), ("tf", 0.36), ("tf", 0.2)])
def test_four_column_form_wide_footprints(kind, du, dt):
    """pixels of up to seven cells, and (du = 0.2) more than the form takes"""
    from oracle import oracle as O
    rng = np.random.default_rng(71)
    g = O.G3((81, 82, 66), (0.9, 0.9, 1.0), (0, 0, 0), (330, 70), (du, 1.4), (0.5, 0), 1000.0, 0.0, 1500.0,
             np.sort(rng.uniform(0, 2 * np.pi, 6)))
    _check(g, rng.uniform(0, 1, (70, 330, 6)).astype(np.float32), None, kind, dt)


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_four_column_form_keeps_values_that_are_not_finite_in_their_columns(value):
    """one such cell reaches every voxel that weighs it (by more than the rounding of its edges,
    1e-6 of its largest weight) and no other column; columns without it keep their bits"""
    from oracle import oracle as O
    from ctsim_amd.device import DeviceArray
    from ctsim_amd.projector import Projector
    g, _, sino, _ = _cone_case(seed=72, n=(81, 80, 130), nuv=(180, 131), nviews=18, dz=0.7, dv=0.9, couch=True)
    P = Projector(geometry_from_g3(g, None))
    img = DeviceArray(P.n_img, "f32")
    P.back(P.upload_sino(sino), img, "back,tf")
    clean = P.download_volume(img)
    only = np.zeros_like(sino)
    only[66, 90, 3] = 1
    weight = O.cbct("back,tf", g, only, None, prec=64, nthreads=8)
    sino[66, 90, 3] = value
    P.back(P.upload_sino(sino), img, "back,tf")
    got = P.download_volume(img)
    bad = ~np.isfinite(got)
    assert not (~bad & (weight > 1e-6 * weight.max())).any()
    may = ~np.isfinite(O.cbct("back,tf", g, sino, None, nthreads=8)).any(axis=2) | weight.any(axis=2)
    assert not bad[~may].any()
    np.testing.assert_array_equal(got[~may], clean[~may])
