"""The schedule cache's key: an entry that another build of the kernels measured is not reused."""
import json
from types import SimpleNamespace

import numpy as np

from ctsim_amd import _lib, autotune
from ctsim_amd.geometry import Geometry


def _plan():
    geom = Geometry(reconSize=(16, 16, 8), reconSpacing=(1, 1, 1), reconOffset=(0, 0, 0), detSize=(24, 10),
                    detSpacing=(1, 1), detOffset=(0, 0), SAD=1000.0, ADD=500.0, SDD=1500.0,
                    betas=np.arange(4) * np.pi / 2)
    set_to, timed = [], []

    def measure(*args, **kw):
        timed.append(1)
        return {"best": 1 | 2 << 2, "candidates": [(1 | 2 << 2, 0.5)]}

    return SimpleNamespace(geom=geom, compute=0, autotune=measure,
                           set_schedule=lambda **kw: set_to.append(kw)), set_to, timed


def test_a_schedule_is_measured_again_with_other_kernels(tmp_path, monkeypatch):
    monkeypatch.setenv("CTSIM_SCHEDULE_CACHE", str(tmp_path / "s.json"))
    arr = SimpleNamespace(dtype=_lib.F32)
    builds = []
    for i in range(2):
        lib = tmp_path / f"lib{i}.so"
        lib.write_bytes(b"kernels of build %d" % i)
        builds.append(str(lib))
    P, set_to, timed = _plan()
    for lib, n in ((builds[0], 1), (builds[0], 1), (builds[1], 2), (builds[0], 2)):
        monkeypatch.setattr(_lib, "LIB_PATH", lib)
        autotune.tuned(P, arr, arr, "proj,tf")
        assert len(timed) == n
        assert set_to[-1] == {"proj_sched": 1 | 2 << 2}
    assert len(json.loads((tmp_path / "s.json").read_text())) == 2
