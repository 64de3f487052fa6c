"""The launch-shape tuner on a stand-in target with a clock of its own: what it
measures, what it tries and which cached entries it applies."""
import ctypes as C
import json
import types

import pytest

from mutracer_amd import abi, autotune


class Target:
    """Renders whose time depends on the tuning; render_timed is another
    launch sequence, for which other tunings are best."""

    def __init__(self, clock):
        self.clock, self.probed = clock, []
        self.settings = types.SimpleNamespace(width=96, height=64, bounces=6, direct_light_candidates=2)
        self.scene = types.SimpleNamespace(info=lambda: dict(triangles=1_000_000))
        self.current = dict(max_paths_in_flight=1 << 25, trace_kernel=0, lds_stack=16, trace_oversubscription=1,
                            shade_oversubscription=1, shade_waves_per_simd=2, use_graphs=1, graph_replays=0,
                            graph_captures=0, tail_paths=0, queue_sort=0, lds_stack_closest=0)

    def tuning(self):
        return dict(self.current)

    def set_tuning(self, **kw):
        self.current.update(kw)
        self.probed.append(dict(self.current))

    def restart_samples(self):
        pass

    def synchronize(self):
        pass

    def render(self, samples):
        t = self.current
        self.clock.now += samples * (1.0 + (0.1 if t["tail_paths"] else 0.0) - (0.2 if t["lds_stack"] == 24 else 0.0))

    def render_timed(self, samples):
        t = dict.fromkeys(("generate_accumulate", "trace", "shade", "shadow", "tail"), 0.0)
        return dict(t, trace=1.0 if self.current["tail_paths"] == 65536 else 2.0)


@pytest.fixture
def target(monkeypatch):
    clock = types.SimpleNamespace(now=0.0)
    monkeypatch.setattr("time.perf_counter", lambda: clock.now)
    return Target(clock)


def test_measures_the_launches_of_a_render(target, tmp_path):
    best = autotune.tune(target, cache_path=str(tmp_path / "tune.json"))
    assert best["tail_paths"] == 0 and best["lds_stack"] == 24
    assert autotune.tune(target, cache_path=str(tmp_path / "tune.json")) == best


def test_tries_no_two_tunings_with_the_same_kernels(target, tmp_path):
    target.current["lds_stack_closest"] = 32
    autotune.tune(target, cache_path=str(tmp_path / "tune.json"))
    assert {t["lds_stack_closest"] for t in target.probed} == {0}
    assert target.probed[0]["lds_stack"] == 32


def test_entries_of_earlier_launch_forms_are_not_applied(target, tmp_path):
    name, cus = C.create_string_buffer(256), C.c_int32(0)
    abi.lib().mtx_device_info(name, 256, C.byref(cus))
    old = f"{name.value.decode()}|{cus.value}|tris~{1 << 19}|96x64|b6|c2"
    path = tmp_path / "tune.json"
    path.write_text(json.dumps({old: dict(tuning=dict(target.current, tail_paths=65536))}))
    assert autotune.tune(target, cache_path=str(path))["tail_paths"] == 0
    assert set(json.loads(path.read_text())) == {old, autotune._key(target)}
