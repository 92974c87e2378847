"""The traversal autotuner's search and cache, with a synthetic timer (no
GPU): coordinate descent finds the fastest shape of a separable cost, every
shape it tries is a valid one, and the cache round-trips."""
import json

from cavalry_amd import tune


def test_descent_finds_separable_minimum(monkeypatch):
    tried, cur = [], {}

    def setter(ctx, which, shape):
        tried.append(dict(shape))
        cur.update(shape)

    monkeypatch.setattr(tune, "set_launch", setter)
    cost = lambda s: ((s["workgroups_per_cu"] - 3) ** 2 + abs(s["ray_chunk"] - 512) / 128
                      + (0 if s["lds_stack"] == 48 else 0.5) + 10)
    best, timings = tune._descend(None, tune.STANDALONE, lambda: cost(cur),
                                  {"workgroups_per_cu": 5, "ray_chunk": 256, "lds_stack": 32}, reps=2)
    assert best == {"workgroups_per_cu": 3, "ray_chunk": 512, "lds_stack": 48, "workgroup_size": 256,
                    "shade_workgroup_size": 256, "handoff_steps": 1024, "any_hit_step": 0,
                    "any_hit_whole_line": 0}
    assert tried[-1] == best  # the winner is left set
    for s in tried:
        assert s["workgroups_per_cu"] in tune.PER_CU and s["ray_chunk"] in tune.CHUNKS and s["lds_stack"] in tune.LDS
        assert s["workgroup_size"] in tune.SIZES and s["shade_workgroup_size"] in tune.SIZES
        assert s["handoff_steps"] in tune.HANDOFFS
        assert s["any_hit_step"] in (0,) + tune.ANY_STEPS
    assert min(timings.values()) == cost(best)


def test_descent_over_workgroup_sizes(monkeypatch):
    """The workgroup size is tried at the same waves per CU, then the
    workgroups per CU at the chosen size, and (render loops) the shading
    workgroup size."""
    tried, cur = [], {}

    def setter(ctx, which, shape):
        tried.append(dict(shape))
        cur.update(shape)

    monkeypatch.setattr(tune, "set_launch", setter)

    def cost(s):
        waves = s["workgroups_per_cu"] * s["workgroup_size"] // 64
        return ((0 if s["workgroup_size"] == 128 else 1) + abs(waves - 16) / 4
                + (0 if s["shade_workgroup_size"] == 64 else 0.25) + 5)

    start = {"workgroups_per_cu": 3, "ray_chunk": 256, "lds_stack": 32, "workgroup_size": 256,
             "shade_workgroup_size": 256}
    best, timings = tune._descend(None, tune.WAVEFRONT, lambda: cost(cur), start, reps=1, shade=True)
    assert best["workgroup_size"] == 128 and best["workgroups_per_cu"] == 8
    assert best["shade_workgroup_size"] == 64
    # the size step keeps the start's 12 waves per CU
    sized = [s for s in tried if s["ray_chunk"] == 256 and s["lds_stack"] == 32 and s["shade_workgroup_size"] == 256]
    assert {(s["workgroup_size"], s["workgroups_per_cu"]) for s in sized[:4]} >= {(64, 12), (128, 6), (256, 3)}
    assert tried[-1] == best
    assert min(timings.values()) == cost(best)
    # without shade, the shading size is never changed
    tried.clear()
    tune._descend(None, tune.STANDALONE, lambda: cost(cur), start, reps=1)
    assert all(s["shade_workgroup_size"] == 256 for s in tried)


def test_cache_round_trip(tmp_path):
    p = str(tmp_path / "t.json")
    tune._store(p, "k1", {"shape": {"workgroups_per_cu": 2, "ray_chunk": 128, "lds_stack": 48}, "ms": 1.5})
    tune._store(p, "k2", {"shape": {"workgroups_per_cu": 4, "ray_chunk": 256, "lds_stack": 32}, "ms": 2.5})
    data = json.load(open(p))
    assert set(data["entries"]) == {"k1", "k2"}
    assert tune._load(p)["entries"]["k1"]["shape"]["lds_stack"] == 48
    assert tune._load(str(tmp_path / "missing.json")) == {}


def test_descent_over_the_wide_tree(monkeypatch):
    """Where the traces walk the wide tree, workgroups per CU and LDS depth do
    nothing: they keep their values, whatever noise the timer adds, unless the
    search ends at a shape that walks the reference's tree."""
    cur, tried = {}, []

    def setter(ctx, which, shape):
        cur.clear()
        cur.update(shape)

    monkeypatch.setattr(tune, "set_launch", setter)
    start = {"workgroups_per_cu": 5, "ray_chunk": 256, "lds_stack": 32}
    wide = lambda: cur["handoff_steps"] < 1 << 30 and cur["any_hit_step"] != 2

    def timer(ref):  # the reference's tree takes `ref` times as long; per_cu and lds lure
        tried.append(dict(cur))
        return (1.0 if wide() else ref) + 0.01 * cur["workgroups_per_cu"] + (0.1 if cur["lds_stack"] == 32 else 0)

    best, _ = tune._descend(None, tune.STANDALONE, lambda: timer(100.0), start, reps=1, wide=wide)
    assert (best["workgroups_per_cu"], best["lds_stack"]) == (5, 32) and best["handoff_steps"] < 1 << 30
    assert {(s["workgroups_per_cu"], s["lds_stack"]) for s in tried} == {(5, 32)}
    best, _ = tune._descend(None, tune.STANDALONE, lambda: timer(0.1), start, reps=1, wide=wide)
    assert not wide() and best["lds_stack"] == 48 and best["workgroups_per_cu"] == min(tune._per_cu_for(best["workgroup_size"]))


def test_cached_shapes_of_other_traversals_are_not_reused(monkeypatch, tmp_path):
    """An entry stored when traces walked the reference's tree (its key named no
    traversal) is not applied: its sibling pairs would switch the wide tree off."""
    p = str(tmp_path / "t.json")
    shape = {"workgroups_per_cu": 2, "ray_chunk": 128, "lds_stack": 48, "any_hit_step": 2}
    for old in ("standalone|tris=2^20|rays=2^20", "rounds|tris=2^20|rays=2^20|traces=1|any=False|cands=0,1"):
        tune._store(p, f"{tune._device_name()}|{old}", {"shape": shape, "ms": 1.0, "rounds": 1})
    applied = []
    monkeypatch.setattr(tune, "set_launch", lambda ctx, which, s: applied.append(s))

    class Bvh:
        n = 1 << 20

    class Timed(Exception):
        pass

    def timed(*a, **k):
        raise Timed

    import torch
    monkeypatch.setattr(torch, "empty", timed)  # (the first thing it does when it has to time)
    try:
        tune.tune_trace(None, Bvh, None, 1 << 20, cache_path=p)
        assert False
    except Timed:
        assert not applied
