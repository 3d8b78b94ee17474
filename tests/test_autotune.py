"""Autotuner logic without a device - CPU only.

Coordinate descent picks the fastest option of the first space with the
default of the second, then the fastest of the second with that choice;
choices persist in the JSON cache (atomic rewrite, unreadable or unwritable
files tolerated); workload keys depend on the shapes, not their order.
"""

import json

import numpy as np
import pytest

from stencil_benchmarks_amd import autotune


def test_descend_is_coordinate_descent():
    space_a = ({"by": 8}, {"by": 16}, {"by": 32})
    space_b = ({"variant": 4}, {"variant": 3})
    cost = {(8, 4): 5.0, (16, 4): 3.0, (32, 4): 4.0, (8, 3): 0.5, (16, 3): 2.0, (32, 3): 9.0}
    calls = []

    def measure(a, b):
        calls.append((a["by"], b["variant"]))
        return cost[(a["by"], b["variant"])]

    a, b, t, trials = autotune.descend(space_a, space_b, measure, space_b[0])
    # (8, 3) would be the global optimum, but descent fixes a = 16 first
    assert (a, b, t) == ({"by": 16}, {"variant": 3}, 2.0)
    assert calls == [(8, 4), (16, 4), (32, 4), (16, 3)] and len(trials) == 4


def test_cache_roundtrip_and_tolerance(tmp_path):
    path = tmp_path / "sub" / "tune.json"
    cache = autotune.TuneCache(path)
    assert cache.get("k") is None
    cache.put("k", {"hdiff": {"by": 16}, "vadv": {}, "seconds": 1.0})
    assert json.loads(path.read_text())["k"]["hdiff"] == {"by": 16}
    assert autotune.TuneCache(path).get("k")["seconds"] == 1.0
    path.write_text("not json")
    assert autotune.TuneCache(path).entries == {}
    blocked = tmp_path / "file"
    blocked.write_text("")
    autotune.TuneCache(blocked / "tune.json").put("k", {})  # parent is a file: no error


def test_workload_key_ignores_order_and_names_types():
    a = autotune.workload_key("batch", [(32, 40, 50), (64, 64, 80)], np.float32, np.float64)
    b = autotune.workload_key("batch", [(64, 64, 80), (32, 40, 50)], "float32", "float64")
    c = autotune.workload_key("batch", [(64, 64, 80), (32, 40, 51)], "float32", "float64")
    assert a == b != c and "float32|float64" in a


def test_spaces_hold_only_built_combinations():
    built = {(16, 2, 2), (16, 2, 0), (16, 8, 2), (16, 8, 0), (8, 1, 2), (32, 2, 2), (16, 4, 2),
             (16, 1, 2)}  # (tile rows, planes, cache flags) of the batched hdiff kernel
    for h in autotune.BATCH_HDIFF_SPACE:
        flags = (h.get("unroll", 0) & 3) if h.get("unroll") else 2
        assert (h["by"], h["bz"], flags) in built
    assert len(autotune.PLAIN_HDIFF_SPACE) == 3 * 5 * 4
    for v in autotune.BATCH_VADV_SPACE:  # levels per step 4 / 8, prefetch depth 4 / 8
        assert v["variant"] in (3, 4) and v.get("unroll", 0) in (0, 4, 8)
        assert v.get("bx", 0) in (0, 4, 5) and (v["variant"] == 4 or "bx" not in v)


def test_launch_from_sets_fields():
    launch = autotune.launch_from({"variant": 4, "by": 16})
    assert (launch.variant, launch.by, launch.bz) == (4, 16, 0)


class _NoDevice:
    base = span = 8

    def pointer(self):
        return self.base

    def free(self):
        pass


def _tune_without_device(monkeypatch, tmp_path, name, fastest):
    """The tuner over calls that take 1 s with the options `fastest` accepts, else 2 s."""
    from stencil_benchmarks_amd import device, native

    def call(function, *arguments):
        if function == "sb_" + name and arguments[-1] is not None:
            arguments[-1]._obj.value = 1.0 if fastest(arguments[-2]) else 2.0

    monkeypatch.setattr(autotune, "device_key", lambda: "device")
    monkeypatch.setattr(native, "call", call)
    monkeypatch.setattr(device.DeviceField, "group",
                        lambda shape, dtype, strides, count, halo: [_NoDevice()] * count)
    tune = {"hdiff": autotune.tune_hdiff, "vadv": autotune.tune_vadv}[name]
    return lambda: tune((20, 10, 8), "float32", repeats=1,
                        cache=autotune.TuneCache(tmp_path / "tune.json"))


@pytest.mark.parametrize("name", ["hdiff", "vadv"])
def test_plain_tuners_return_no_options_where_those_are_fastest(monkeypatch, tmp_path, name):
    def fields(options):
        return [getattr(options, f) for f in ("variant", "bx", "by", "bz", "unroll")]

    tune = _tune_without_device(monkeypatch, tmp_path, name,
                                lambda options: not any(fields(options)))
    for from_cache in (False, True):
        tuned = tune()
        assert tuned.defaults and tuned.seconds == 1.0 and tuned.from_cache == from_cache
        assert not any(fields(getattr(tuned, name + "_options")))


@pytest.mark.parametrize("name", ["hdiff", "vadv"])
def test_plain_tuners_return_the_fastest_options(monkeypatch, tmp_path, name):
    tune = _tune_without_device(monkeypatch, tmp_path, name,
                                lambda options: options.variant > 0 and options.unroll == 4)
    for from_cache in (False, True):
        tuned = tune()
        assert not tuned.defaults and tuned.seconds == 1.0 and tuned.from_cache == from_cache
        assert getattr(tuned, name + "_options").unroll == 4


@pytest.mark.parametrize("name", ["hdiff", "vadv"])
def test_choices_between_older_kernels_are_made_anew(monkeypatch, tmp_path, name):
    tune = _tune_without_device(monkeypatch, tmp_path, name, lambda options: options.variant == 1)
    # the key of an entry written before keys named a revision
    key = autotune.workload_key(name, [(20, 10, 8)], "float32", "float32", (3, 3, 3))
    old = "device|" + key[key.index(name):]
    autotune.TuneCache(tmp_path / "tune.json").put(
        old, {"hdiff": {"variant": 3}, "vadv": {"variant": 3}, "seconds": 0.1, "trials": 60})
    assert not tune().from_cache and tune().from_cache
    monkeypatch.setattr(autotune, "REVISION", autotune.REVISION + 1)
    assert not tune().from_cache
