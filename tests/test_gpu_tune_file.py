"""Recorded autotuner picks (CUBE_AUTOTUNE_FILE) are those of the present kernels: a
pick that an earlier form of a kernel was timed with is not taken, whatever its
number, and the trials run and are recorded again.
"""
import pytest

from cube_nu_amd import P3M
from inputs import buffered_set

pytestmark = pytest.mark.gpu


def _timed(p, seed=3):
    """The choices whose candidates were timed in two kicks."""
    xp, vp, _, rhoc = buffered_set(p.geo, seed=seed, mean=4.0)
    for _ in range(2):
        p.kick(xp, vp.copy(), rhoc, a_mid=0.5, dt=0.1)
    return {k.split(":")[1] for k, v in p.timing_report().items() if k.startswith("autotune:") and v["ms"] > 0}


def test_picks_of_earlier_kernels_are_not_taken(tmp_path, monkeypatch):
    f = tmp_path / "picks"
    monkeypatch.setenv("CUBE_AUTOTUNE_FILE", str(f))
    first = P3M(64)
    made = _timed(first)
    first.close()
    assert any(k.startswith("pp_depth") for k in made) and any(k.startswith("interp_shape") for k in made)
    recorded = {line.split()[0] for line in f.read_text().splitlines()}
    assert made <= recorded
    # this build's own picks save the trials
    again = P3M(64)
    assert not _timed(again)
    again.close()
    # the same levels under the names that earlier kernels were recorded with
    old = [k.replace(k.split("_l")[0], name, 1) for k in made for name in ("pp_depth", "interp_shape")
           if k.startswith(name)]
    f.write_text("".join(f"{k} {6 if k.startswith('pp') else 2}\n" for k in old))
    p = P3M(64)
    assert _timed(p) >= {k for k in made if k.startswith(("pp_depth", "interp_shape"))}
    p.close()
