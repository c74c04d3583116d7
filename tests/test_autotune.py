"""CPU checks of the tile autotuner's cache: a choice made among other kernels is
not applied, the same kernels' is, and TaylorF2 without time marginalisation,
whose kernel takes no tile, is neither timed nor cached."""
import json
import types

import pytest

from bilby_amd import autotune as at


@pytest.fixture
def stub(monkeypatch, tmp_path):
    monkeypatch.setattr(at.torch.cuda, "get_device_name", lambda device=None: "card")
    monkeypatch.setattr(at, "CACHE_PATH", str(tmp_path / "cache.json"))
    log = types.SimpleNamespace(set=[], timed=[])
    monkeypatch.setattr(at, "set_tile", lambda lk, *tile: log.set.append(tile))
    monkeypatch.setattr(at, "time_tile",
                        lambda lk, rows, tile, *a: log.timed.append(tile) or 1.0 + sum(tile))
    log.path = at.CACHE_PATH
    return log


class _Detectors(list):
    frequency_array = range(16385)


def _likelihood(time, approximant):
    return types.SimpleNamespace(
        interferometers=_Detectors("abc"), device=0, precision="fp64", _flags=lambda: 7,
        waveform_generator=types.SimpleNamespace(approximant=approximant),
        time_marginalization=time)


ROWS = types.SimpleNamespace(shape=(4096, 16))


def test_choices_among_other_kernels_are_not_applied(stub):
    lk = _likelihood(True, at.TAYLORF2)
    key = at.bucket_key(lk, 4096)
    former = "|".join(key.split("|")[1:])       # the key without the generation
    with open(stub.path, "w") as fh:
        json.dump({former: {"tile": [8, 4]}}, fh)
    tile, sweep = at.autotune(lk, ROWS)
    assert tile[0] == 0 and len(stub.timed) == len(at.DEFAULT_CANDIDATES_TIME)
    del stub.timed[:]
    assert at.autotune(lk, ROWS)[0] == tile and not stub.timed and stub.set[-1] == tile


def test_nothing_to_tune_without_time_marginalisation(stub):
    assert at.autotune(_likelihood(False, at.TAYLORF2), ROWS) == ((0, 0), {})
    assert not stub.timed and stub.set == [(0, 0)]
    at.autotune(_likelihood(False, 1), ROWS)    # sine-Gaussian tiles are tuned
    assert stub.timed == at.DEFAULT_CANDIDATES_PLAIN
