"""The autotuner's saved measurements: those of the same kernels are used, older ones are measured again (on the CPU: a
stand-in for the solver says that a measurement has begun)."""
import json

import pytest

from peps_mg_amd import autotune, geometry, multigrid


class Measuring(Exception):
    pass


@pytest.fixture
def cache(tmp_path, monkeypatch):
    def solver(*args, **kw):
        raise Measuring
    path = tmp_path / "tune.json"
    monkeypatch.setenv("PEPSMG_TUNE_CACHE", str(path))
    monkeypatch.setattr(multigrid, "Multigrid", solver)
    return path


def sdm():
    return geometry.geometry_subdomain_create(geometry.geometry_domain_create(32, 32, 32, 0.0, 0.0, 0.0, 1.0, 1.0, 1.0))


TILE = {"tile_x": 128, "tile_y": 16, "fused_smoother": 1, "smoother_ms": 1.0, "timings": {}}


@pytest.mark.parametrize("key", ["tile:32x32x32:p1", "tile:32x32x32:p1:v2"])
def test_older_tile_measured_again(cache, key):
    cache.write_text(json.dumps({key: TILE}))
    with pytest.raises(Measuring):
        autotune.tune_tiles(sdm(), 3, 1)


@pytest.mark.parametrize("key", ["solve:32x32x32:p1:nl3:nu2:v2"])
def test_older_schedule_measured_again(cache, key):
    cache.write_text(json.dumps({key: dict(TILE, inner_nu=1)}))
    with pytest.raises(Measuring):
        autotune.tune_solver(sdm(), 3, None, None)


def test_saved_measurement_used(cache):
    cache.write_text(json.dumps({autotune._key("tile", sdm(), 1): TILE}))
    assert autotune.tune_tiles(sdm(), 3, 1) == TILE
