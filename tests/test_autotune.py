"""The autotuner's candidates: every setting that changes something, once."""
from __future__ import annotations

import pytest

from srs_amd.autotune import autotune

LIVE = ("tile", "plane_pad", "compact", "nt_state", "occupancy")


class _Ctx:
    """Steps take 1 ms, and 0.5 with tiles of 256."""

    def __init__(self, layout):
        self.layout = layout

    def tune(self, **kw):
        pass

    def explicit_step(self, n, flags=0):
        pass

    def prepare(self, n, flags=0):
        pass

    def last_timing(self):
        return (20 * (0.5 if self.layout["tile"] == 256 else 1.0), 0.0)

    def close(self):
        pass


@pytest.mark.parametrize("kw", [{}, dict(groups=(1, 2, 4)), dict(nt_geometry=(0, 1), lds=(0, 1)),
                                dict(groups=(4,), lds=(1,))])
def test_candidates_differ_in_more_than_ignored_keys(kw):
    best, trials = autotune(_Ctx, **kw)
    seen = [tuple(cfg[k] for k in LIVE) for cfg, _ in trials]
    assert len(seen) == len(set(seen)) == 3 * 2 * 2 * 2
    assert best["tile"] == 256
    for k, default in (("nt_geometry", (0,)), ("lds", (1,))):
        assert best[k] == kw.get(k, default)[0]
    assert best.get("group", 1) == kw.get("groups", (1,))[0]
