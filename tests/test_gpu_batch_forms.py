"""The batched 2D forward's one form for all slices: line walk (flat, arc), and the candidate form
where one slice lies outside the walk's range or the detectors are of both types, against the FP64
oracle: relative L2 <= 1e-5, the repository's FP32 gate, or three times the FP32 oracle's own
distance where that is larger, as in the other parity tests."""
import numpy as np
import pytest

from conftest import rel_l2
from helpers import geometry_from_g2

pytestmark = pytest.mark.gpu

# image, pixel, cells, cell, SAD, SDD, detector type
SLICES = {
    "flat": ((33, 70), 0.8, 130, 1.0, 1000.0, 1500.0, 1),
    "flat_large": ((97, 64), 0.6, 75, 2.0, 1000.0, 1500.0, 1),
    "arc": ((64, 57), 0.8, 129, 1.0, 600.0, 1100.0, 0),
    "arc_small": ((20, 31), 1.0, 64, 0.9, 600.0, 1100.0, 0),
    "source_near": ((48, 48), 1.0, 96, 1.5, 45.0, 90.0, 1),
}
BATCHES = {"flat": ("flat", "flat_large"), "arc": ("arc", "arc_small"), "mixed": ("flat", "arc", "flat_large"),
           "refused": ("flat_large", "source_near", "flat")}


@pytest.mark.parametrize("kind", ["dd", "tf"])
@pytest.mark.parametrize("name", list(BATCHES))
def test_batched_forward_form_vs_fp64_oracle(name, kind):
    from oracle import oracle as O
    from ctsim_amd.batch2 import Batch2
    from ctsim_amd.device import DeviceArray
    rng = np.random.default_rng(6)
    gs, imgs = [], []
    for n, d, nu, du, sad, sdd, det in (SLICES[s] for s in BATCHES[name]):
        betas = np.concatenate([np.arange(4) * np.pi / 4, rng.uniform(0, 2 * np.pi, 5)])
        gs.append(O.G2(n[0], n[1], d, d, 0.0, 0.0, nu, du, 0.25, sad, 0.0, sdd, betas, det))
        imgs.append((0.2 + rng.uniform(0, 1, n)).astype(np.float32))
    B = Batch2([geometry_from_g2(g) for g in gs])
    out = DeviceArray(B.sino_elems, "f32")
    for split in (1, 2, 4):
        B.set_schedule(split, 4)
        B.proj(DeviceArray.from_numpy(B.pack_images(imgs), "f32"), out, f"proj,{kind}")
        for g, img, got in zip(gs, imgs, B.unpack_sinos(out.to_numpy())):
            want = O.fbct(f"proj,{kind}", g, img, prec=64)
            tol = max(1e-5, 3 * rel_l2(O.fbct(f"proj,{kind}", g, img), want))
            assert rel_l2(got, want) <= tol, (split, rel_l2(got, want), tol)
