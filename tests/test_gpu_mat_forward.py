"""The 3D forward's matrix form: every gather class (voxels of 1/4 to 14 rows), one and two row
chunks per item, both staging sizes, split and whole items, detectors of few and of odd rows,
footprints of more than four tile cells, both detector types, couch and map, against the FP64
oracle; the same bits from exhaustive candidate lists; values that are not finite.

Tolerance: relative L2 <= 1e-5, widened to three times the FP32 oracle's own distance where
that is larger, as in the other parity tests."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_parity import TOL, _cone_case, geometry_from_g3

pytestmark = pytest.mark.gpu

CASES = {
    "class5": dict(seed=40, n=(30, 26, 120), nuv=(60, 33), nviews=5, dz=0.3, dv=1.55),   # 0.29 rows per voxel
    "class4": dict(seed=41, n=(34, 30, 128), nuv=(75, 64), nviews=6, dz=0.4, dv=1.5),    # 0.4
    "class3": dict(seed=42, n=(34, 30, 61), nuv=(75, 17), nviews=6, dz=0.7, dv=1.5),     # 0.7
    "class2": dict(seed=43, n=(29, 37, 77), nuv=(75, 93), nviews=7, dz=1.0, dv=0.9, dettype=0, couch=True),
    "thick": dict(seed=44, n=(28, 28, 9), nuv=(64, 130), nviews=6, dz=4.0, dv=0.5),      # 12 rows per voxel
    "one_row": dict(seed=45, n=(30, 30, 20), nuv=(70, 1), nviews=6, dz=0.5, dv=0.75),
    "one_slice": dict(seed=46, n=(30, 30, 1), nuv=(70, 40), nviews=6, dz=1.0, dv=1.0, map_=False),
}


def _run(P, d_vol, kind, sched, exhaustive=False):
    from ctsim_amd.device import DeviceArray
    out = DeviceArray(P.n_sino(), "f32")
    P.set_schedule(proj_sched=sched)
    P.proj(d_vol, out, f"proj,{kind}", exhaustive=exhaustive)
    return P.download_sino(out)


@pytest.mark.parametrize("kind", ["dd", "tf"])
@pytest.mark.parametrize("name", list(CASES))
def test_matrix_form_vs_fp64_oracle(name, kind):
    from oracle import oracle as O
    from ctsim_amd.projector import Projector
    g, vol, _, mp = _cone_case(**CASES[name])
    print(name, kind, g.n.tolist(), flush=True)
    want = O.cbct(f"proj,{kind}", g, vol, mp, prec=64)
    tol = max(TOL, 3 * rel_l2(O.cbct(f"proj,{kind}", g, vol, mp), want))
    P = Projector(geometry_from_g3(g, mp))
    d_vol = P.upload_volume(vol)
    for sched in (1 | 1 << 2, 1 | 2 << 2, 3 | 1 << 2):  # whole items, shared items, two row chunks
        got = _run(P, d_vol, kind, sched)
        assert rel_l2(got, want) <= tol, (sched, rel_l2(got, want))
        np.testing.assert_array_equal(_run(P, d_vol, kind, sched, exhaustive=True), got)


@pytest.mark.parametrize("kind", ["dd", "tf"])
def test_matrix_form_wide_footprints(kind):
    """pixels of four to seven detector cells: several records per column"""
    from oracle import oracle as O
    from ctsim_amd.projector import Projector
    rng = np.random.default_rng(50)
    g = O.G3((31, 27, 20), (1.2, 1.2, 1.0), (0, 0, 0), (300, 40), (0.35, 1.0), (0.5, 0), 1000.0, 0.0, 1500.0,
             np.sort(rng.uniform(0, 2 * np.pi, 6)))
    vol = rng.uniform(0, 1, (31, 27, 20)).astype(np.float32)
    want = O.cbct(f"proj,{kind}", g, vol, None, prec=64)
    tol = max(TOL, 3 * rel_l2(O.cbct(f"proj,{kind}", g, vol, None), want))
    P = Projector(geometry_from_g3(g, None))
    d_vol = P.upload_volume(vol)
    for sched in (1 | 1 << 2, 1 | 2 << 2, 3 | 1 << 2):
        got = _run(P, d_vol, kind, sched)
        assert rel_l2(got, want) <= tol, (sched, rel_l2(got, want))
        np.testing.assert_array_equal(_run(P, d_vol, kind, sched, exhaustive=True), got)


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_matrix_form_keeps_values_that_are_not_finite_in_their_rays(value):
    """one such voxel reaches every cell that it weighs on (by more than the rounding of its
    edges, 1e-6 of its largest weight) and no cell outside its footprint and the rows beside
    it; every other cell of the tile keeps its value"""
    from oracle import oracle as O
    from ctsim_amd.projector import Projector
    g, vol, _, _ = _cone_case(seed=51, n=(24, 24, 30), nuv=(70, 40), nviews=5, dz=0.7, dv=1.0)
    P = Projector(geometry_from_g3(g, None))
    clean = _run(P, P.upload_volume(vol), "tf", 1 | 2 << 2)
    only = np.zeros_like(vol)
    only[11, 13, 14] = 1
    weight = O.cbct("proj,tf", g, only, None, prec=64)
    must = weight > 1e-6 * weight.max()
    vol[11, 13, 14] = value
    may = ~np.isfinite(O.cbct("proj,tf", g, vol, None)) | must
    may[1:] |= may[:-1]
    may[:-1] |= may[1:]
    for sched in (1 | 1 << 2, 1 | 2 << 2, 3 | 1 << 2):
        got = _run(P, P.upload_volume(vol), "tf", sched)
        bad = ~np.isfinite(got)
        assert not (must & ~bad).any() and not (bad & ~may).any(), sched
        np.testing.assert_allclose(got[~may], clean[~may], rtol=1e-5)
