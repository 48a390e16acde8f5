"""The 3D backprojector's four-column form where the image's shadow is several times the
detector: views that miss all four columns of a wave, views that miss some of them, a number of
views that is no multiple of its batch, against the FP64 oracle with the tolerance of
test_gpu_quad_back.py (relative L2 <= 1e-5, or three times the FP32 oracle's own distance where
that is larger); the same bits from both column orders."""
import pytest

from test_gpu_parity import _cone_case
from test_gpu_quad_back import _check

pytestmark = pytest.mark.gpu

CASES = {
    "couch_f32": (dict(seed=80, n=(150, 140, 66), nuv=(50, 70), nviews=19, dz=0.9, dv=1.0, couch=True), "f32"),
    "offsets_bf16": (dict(seed=81, n=(150, 140, 66), nuv=(60, 70), nviews=33, dz=0.9, dv=1.0, offsets=True), "bf16"),
    "short_arc": (dict(seed=82, n=(200, 190, 40), nuv=(140, 60), nviews=18, dz=0.9, dv=1.0, dettype=0), "f32"),
    "narrow_16": (dict(seed=83, n=(260, 256, 70), nuv=(30, 40), nviews=5, dz=0.9, dv=2.0, map_=False), "f16"),
    # narrower still: one column
    "refused": (dict(seed=84, n=(130, 128, 40), nuv=(30, 40), nviews=7, dz=0.9, dv=1.0), "f32"),
}


@pytest.mark.parametrize("kind", ["dd", "tf"])
@pytest.mark.parametrize("name", list(CASES))
def test_four_column_form_on_narrow_detectors(name, kind):
    case, dt = CASES[name]
    g, _, sino, mp = _cone_case(**case)
    print(name, kind, g.n.tolist(), flush=True)
    _check(g, sino, mp, kind, dt)
