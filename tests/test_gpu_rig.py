"""GPU tests of the multi-camera rig: one launch chain (phase A over every camera's segments, one
heavy-first order of the joint pixel space, one walk launch, captured into a hipGraph) must give
every camera exactly what advancing it alone gives: the same events bit for bit, the same saved state
and the same work counters. Cameras of mixed resolutions, ragged runs with heavy-tailed sample counts,
cameras at different model times, event-buffer overflow, graph on and off, both photoreceptor kinds,
the autotuner (it changes no camera) and the refusals (before any camera changes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WORK = ("substeps", "substep_attempts", "settled_substeps", "leaf_intervals", "fallbacks", "quarantines", "pieces",
        "events", "input_clamps")


def _params(kind, **over):
    import ballasim_amd as bsx
    if kind == "instant":
        p = bsx.preset("prophesee_gen3")
        p.photoreceptor = "instantaneous"
        p.noise = False
        p.leak_rate_hz = 0.5
        p.refractory_s = 5e-5
    elif kind == "noise":
        p = bsx.preset("prophesee_gen3")
    else:
        p = bsx.preset("samsung_gen3")
        p.noise = False
    for k, v in over.items():
        setattr(p, k, v)
    return p


def heavy_runs(rng, P, t0, t1, G=1, mu=np.log(6.0), sigma=1.5, cap=300, frac=0.85):
    """Ragged runs with log-normal sample counts (clipped to [1, cap]) for a random subset of pixels in
    random order: strictly increasing times in (t0, t1], log-normal irradiance drifting per pixel."""
    ids = np.nonzero(rng.random(P) < frac)[0].astype(np.uint32)
    rng.shuffle(ids)
    counts = np.clip(np.round(np.exp(rng.normal(mu, sigma, size=len(ids)))), 1, cap).astype(np.int64)
    counts = np.minimum(counts, t1 - t0)
    ts, irs = [], []
    for n in counts:
        tt = np.sort(rng.choice(np.arange(t0 + 1, t1 + 1, max(1, (t1 - t0) // 4096)), size=int(n), replace=False))
        ts.append(tt.astype(np.int64))
        walk = np.cumsum(rng.normal(0.0, 0.35, size=(int(n), G)), axis=0) + rng.normal(3.0, 1.0)
        irs.append(np.exp(walk).astype(np.float32))
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    t = np.concatenate(ts) if ts else np.zeros(0, np.int64)
    irr = np.concatenate(irs).reshape(-1, G) if irs else np.zeros((0, G), np.float32)
    return ids, t, irr, offs


def to_device(ids, t, irr, offs):
    import torch
    dev = torch.device("cuda:0")
    return (torch.from_numpy(ids.astype(np.int32)).to(dev), torch.from_numpy(offs[:-1].copy()).to(dev),
            torch.from_numpy(np.diff(offs).astype(np.int32)).to(dev), torch.from_numpy(t).to(dev),
            torch.from_numpy(np.ascontiguousarray(irr.reshape(-1))).to(dev))


SHAPES = [(40, 24), (23, 17), (64, 9), (31, 31)]


def make_cameras(kind, shapes, seed=5, G=1, **over):
    import ballasim_amd as bsx
    cams = []
    for c, (W, H) in enumerate(shapes):
        extra = dict(over)
        if kind == "instant" and c == 1:
            extra.setdefault("shot_rate_hz", 40.0)  # one camera with the shot process
        cams.append(bsx.SensorModel(_params(kind, **extra), W, H, seed + c, ["constant"] * G, c, device="cuda"))
    return cams


def run_pair(kind, shapes, calls=3, graph=True, G=1, t0s=None, caps=None, tuning=None, seed=11):
    """Advances a rig and an identical set of cameras advanced one by one on the same device runs;
    asserts equality after every call."""
    import torch

    import ballasim_amd as bsx
    rng = np.random.default_rng(seed)
    rig_cams = make_cameras(kind, shapes, G=G)
    solo = make_cameras(kind, shapes, G=G)
    t0s = t0s or [0] * len(shapes)
    for c, (W, H) in enumerate(shapes):
        irr0 = np.exp(rng.normal(3, 1, (W * H, G))).astype(np.float32)
        rig_cams[c].init(t0s[c], irr0)
        solo[c].init(t0s[c], irr0)
        if caps is not None and caps[c]:
            rig_cams[c].set_launch_policy(event_capacity=caps[c])
            solo[c].set_launch_policy(event_capacity=caps[c])
    rig = bsx.Rig(rig_cams)
    rig.set_graph(graph)
    if tuning:
        rig.set_tuning(**tuning)
    t_end = max(t0s)
    for call in range(calls):
        t_end += int(rng.integers(2 ** 21, 2 * 2 ** 23))
        runs, keep = [], []
        for c, (W, H) in enumerate(shapes):
            t_from = rig_cams[c].time_ns
            r = heavy_runs(rng, W * H, t_from, t_end, G=G)
            d = to_device(*r)
            keep.append(d)
            runs.append(d)
        torch.cuda.synchronize()
        got = rig.advance_device(runs, t_end)
        for c in range(len(shapes)):
            ptr, count = solo[c].advance_device(*runs[c], t_end)
            want = solo[c].download_events(ptr, count)
            have = rig_cams[c].download_events(*got[c])
            assert got[c][1] == count, f"call {call} camera {c}: {got[c][1]} events, alone {count}"
            for k in want:
                assert np.array_equal(have[k], want[k]), f"call {call} camera {c}: {k}"
            assert rig_cams[c].save_state() == solo[c].save_state(), f"call {call} camera {c}: state"
    for c in range(len(shapes)):
        a, b = rig_cams[c].stats(), solo[c].stats()
        for k in WORK:
            assert a[k] == b[k], (c, k, a[k], b[k])
    return rig, rig_cams


def test_rig_instant_equals_cameras_alone_graph():
    rig, cams = run_pair("instant", SHAPES)
    st = rig.stats()
    assert st["launches"] == 3 and st["graph_launches"] == 3 and st["captures"] >= 1
    assert sum(c.stats()["events"] for c in cams) > 500


def test_rig_instant_without_graph_and_persistent_queue():
    rig, _ = run_pair("instant", SHAPES, graph=False, tuning=dict(queue_chunk=2, block_size=128, walk_budget=16,
                                                                  search_batch=4))
    assert rig.stats()["graph_launches"] == 0


# Head groups and the queue of 64-pixel groups, which the walk with in-path noise takes: groups that divide the head,
# leave a remainder, cover the whole order or more groups than a grab.
@pytest.mark.parametrize("graph,tuning", [
    (True, dict(head_lanes=16, head_per_mille=250)),
    (False, dict(head_lanes=8, head_per_mille=500, queue_chunk=2, block_size=128)),
    (True, dict(head_lanes=7, head_per_mille=333, queue_chunk=1)),
    (True, dict(head_lanes=1, head_per_mille=1000, queue_chunk=64)),
    (False, dict(queue_chunk=1, block_size=64)),
    (True, dict(queue_chunk=3)),
])
def test_rig_noise_head_groups_and_queue(graph, tuning):
    """The heaviest pixels of the order walked in groups of fewer than 64 (idle lanes in those waves), and groups taken
    from the queue, give every camera the events, state and counters of advancing it alone in 64-pixel groups."""
    rig, _ = run_pair("noise", [(24, 16), (17, 9)], calls=2, graph=graph, tuning=tuning)
    got = rig.tuning()
    for f, v in tuning.items():
        assert got[f] == v
    rig.set_tuning(head_per_mille=-1)
    assert rig.tuning()["head_per_mille"] == 0


# The heads of the other walks: lanes of a wave dealt pixels before the queue (instantaneous: one, a few, with refills
# at 48 idle lanes or a whole wave), and none (cascade).
@pytest.mark.parametrize("kind,graph,tuning", [
    ("instant", True, dict(head_lanes=16, head_per_mille=250)),
    ("instant", False, dict(head_lanes=8, head_per_mille=500, queue_chunk=2, block_size=128)),
    ("instant", True, dict(head_lanes=1, head_per_mille=8, queue_chunk=64)),
    ("instant", True, dict(head_lanes=2, head_per_mille=8, queue_chunk=64, block_size=64)),
    ("cascade", True, dict(head_lanes=32, head_per_mille=300)),
])
def test_rig_heads_without_noise(kind, graph, tuning):
    rig, _ = run_pair(kind, SHAPES if kind == "instant" else [(24, 16), (17, 9)], calls=2, graph=graph, tuning=tuning)
    got = rig.tuning()
    assert got["head_lanes"] == tuning["head_lanes"] and got["head_per_mille"] == tuning["head_per_mille"]
    rig.set_tuning(head_per_mille=-1)
    assert rig.tuning()["head_per_mille"] == 0


@pytest.mark.parametrize("head", [1, 2, 63])
def test_lanes_dealt_and_from_the_queue(head):
    """More pixels than the walk's resident waves, so that lanes that are dealt none take theirs from the queue."""
    import torch

    import ballasim_amd as bsx
    rng = np.random.default_rng(head)
    shapes = [(331, 97), (64, 9)]
    cams, solo = make_cameras("instant", shapes), make_cameras("instant", shapes)
    for c, (W, H) in enumerate(shapes):
        irr0 = np.exp(rng.normal(3, 1, (W * H, 1))).astype(np.float32)
        cams[c].init(0, irr0)
        solo[c].init(0, irr0)
    rig = bsx.Rig(cams)
    rig.set_tuning(head_lanes=head, head_per_mille=8, queue_chunk=64)
    t_end = 2 ** 21
    runs = [to_device(*heavy_runs(rng, W * H, 0, t_end, mu=np.log(2.0), cap=40)) for (W, H) in shapes]
    torch.cuda.synchronize()
    got = rig.advance_device(runs, t_end)
    for c in range(len(shapes)):
        ptr, count = solo[c].advance_device(*runs[c], t_end)
        want, have = solo[c].download_events(ptr, count), cams[c].download_events(*got[c])
        for k in want:
            assert np.array_equal(have[k], want[k]), (c, k)
        assert cams[c].save_state() == solo[c].save_state()
        for k in WORK:
            assert cams[c].stats()[k] == solo[c].stats()[k], (c, k)


def test_rig_cameras_at_different_times_and_overflow():
    rig, _ = run_pair("instant", SHAPES[:3], t0s=[0, 2 ** 23 + 777, 3 * 2 ** 22 - 5], caps=[32, 0, 16],
                      tuning=dict(queue_chunk=1))
    assert rig.stats()["walk_reruns"] >= 1


def test_rig_two_light_groups():
    run_pair("instant", SHAPES[:2], G=2, calls=2)


def test_rig_cascade_equals_cameras_alone():
    rig, cams = run_pair("cascade", [(24, 16), (17, 9)], calls=2)
    assert sum(c.stats()["events"] for c in cams) > 50


def test_rig_autotune_changes_no_camera():
    import torch

    import ballasim_amd as bsx
    rng = np.random.default_rng(3)
    cams = make_cameras("instant", SHAPES)
    for c, (W, H) in enumerate(SHAPES):
        cams[c].init(0, np.exp(rng.normal(3, 1, (W * H, 1))).astype(np.float32))
    rig = bsx.Rig(cams)
    runs = [to_device(*heavy_runs(rng, W * H, 0, 2 ** 23)) for (W, H) in SHAPES]
    torch.cuda.synchronize()
    before = [c.save_state() for c in cams]
    trials = rig.autotune(runs, 2 ** 23, reps=1)
    assert len(trials) >= 10
    best = min(ms for _, ms in trials)
    tu = rig.tuning()
    assert any(t == tu and ms == best for t, ms in trials)
    assert [c.save_state() for c in cams] == before
    assert all(c.time_ns == 0 for c in cams)
    # the tuned rig still equals the cameras alone
    solo = make_cameras("instant", SHAPES)
    rng = np.random.default_rng(3)
    for c, (W, H) in enumerate(SHAPES):
        solo[c].init(0, np.exp(rng.normal(3, 1, (W * H, 1))).astype(np.float32))
    got = rig.advance_device(runs, 2 ** 23)
    for c in range(len(SHAPES)):
        ptr, count = solo[c].advance_device(*runs[c], 2 ** 23)
        want = solo[c].download_events(ptr, count)
        have = cams[c].download_events(*got[c])
        for k in want:
            assert np.array_equal(have[k], want[k]), (c, k)
        assert cams[c].save_state() == solo[c].save_state()


# The fields each kind of walk reads, and values of them that must be among the candidates.
@pytest.mark.parametrize("kind,live", [
    ("instant", dict(block_size={64, 128, 256}, walk_budget={4, 8}, search_batch={1, 2, 4}, queue_chunk={0, 1},
                     head_lanes={64, 8, 2}, head_per_mille={0, 8})),
    ("cascade", dict(block_size={64, 128, 256})),
    ("noise", dict(block_size={64, 128, 256}, queue_chunk={0, 1, 16}, head_lanes={64, 16, 32}, head_per_mille={0, 8, 32})),
])
def test_rig_autotune_tries_what_the_walk_reads(kind, live):
    import torch

    import ballasim_amd as bsx
    rng = np.random.default_rng(7)
    shapes = [(24, 16), (17, 9)]
    cams = make_cameras(kind, shapes)
    for c, (W, H) in enumerate(shapes):
        cams[c].init(0, np.exp(rng.normal(3, 1, (W * H, 1))).astype(np.float32))
    rig = bsx.Rig(cams)
    runs = [to_device(*heavy_runs(rng, W * H, 0, 2 ** 21)) for (W, H) in shapes]
    torch.cuda.synchronize()
    base = rig.tuning()
    trials = [t for t, _ in rig.autotune(runs, 2 ** 21, reps=1)]
    assert len({tuple(sorted(t.items())) for t in trials}) == len(trials)  # no shape twice
    for f in base:
        seen = {t[f] for t in trials}
        assert seen >= live[f] if f in live else seen == {base[f]}, (f, seen)


def test_rig_refusals_change_no_camera():
    import torch

    import ballasim_amd as bsx
    rng = np.random.default_rng(4)
    cams = make_cameras("instant", SHAPES[:3])
    for c, (W, H) in enumerate(SHAPES[:3]):
        cams[c].init(0, np.exp(rng.normal(3, 1, (W * H, 1))).astype(np.float32))
    rig = bsx.Rig(cams)
    runs = [heavy_runs(rng, W * H, 0, 2 ** 23) for (W, H) in SHAPES[:3]]
    bad = list(runs[1])
    bad[0] = bad[0].copy()
    bad[0][0] = SHAPES[1][0] * SHAPES[1][1] + 5  # pixel id out of range in camera 1
    dev = [to_device(*runs[0]), to_device(*bad), to_device(*runs[2])]
    torch.cuda.synchronize()
    before = [c.save_state() for c in cams]
    with pytest.raises(ValueError, match="camera 1"):
        rig.advance_device(dev, 2 ** 23)
    assert [c.save_state() for c in cams] == before
    nan = list(runs[2])
    nan[2] = nan[2].copy()
    nan[2][len(nan[2]) // 2] = np.nan  # a non-finite sample in camera 2: found by phase A, after the launch
    dev = [to_device(*runs[0]), to_device(*runs[1]), to_device(*nan)]
    torch.cuda.synchronize()
    with pytest.raises(ValueError, match="camera 2.*non-finite"):
        rig.advance_device(dev, 2 ** 23)
    assert [c.save_state() for c in cams] == before and all(c.initialized for c in cams)
    dev = [to_device(*r) for r in runs]
    rig.advance_device(dev, 2 ** 23)
    assert all(c.time_ns == 2 ** 23 for c in cams)
    with pytest.raises(ValueError):
        bsx.Rig([cams[0], cams[0]])
    other = bsx.SensorModel(_params("cascade"), 8, 8, 1, device="cuda")
    with pytest.raises(ValueError):
        bsx.Rig([cams[0], other])
    with pytest.raises(ValueError):
        rig.set_tuning(block_size=96)
