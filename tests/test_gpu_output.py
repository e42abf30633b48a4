"""GPU parity of the output stage with its oracle (oracle/output_oracle.py, pinned against the
reference's output_order / readout / label_s1): per window the released events, their order and
every C4 column are identical, and the held count matches; with a crop and a readout with delay,
quantum and clock offset and drift; then flush. Also the C4 file written from the released columns
(t monotone, ms_to_idx)."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from oracle import output_oracle as Q
from tests.helpers import random_runs

pytestmark = pytest.mark.gpu

W = 1 << 23


@pytest.mark.parametrize("crop,readout", [
    (None, {}),
    ((3, 2, 31, 19), dict(readout_delay_s=7e-4, readout_quantum_s=1e-6, clock_offset_ns=-12345, clock_drift_ppm=35.0)),
])
def test_output_stage_matches_oracle(crop, readout, tmp_path):
    import ballasim_amd as bsx
    from ballasim_amd.output import EventFile, OutputStage
    p = bsx.preset("prophesee_gen3")
    p.photoreceptor = "instantaneous"
    p.noise = False
    p.leak_rate_hz = 5.0
    p.refractory_s = 1e-5
    for k, v in readout.items():
        setattr(p, k, v)
    Wd, Hd = 40, 24
    m = bsx.SensorModel(p, Wd, Hd, 3, ["constant"], 0, device="cuda")
    ref = O.OracleModel(p.c, Wd, Hd, 3, 1, 0)
    rng = np.random.default_rng(5)
    irr0 = np.exp(rng.normal(3, 1, (Wd * Hd, 1))).astype(np.float32)
    m.init(0, irr0)
    ref.init(0, irr0)
    info = m._info()
    rd = dict(quantum=round(p.readout_quantum_s * 1e9), delay=round(p.readout_delay_s * 1e9),
              phase=int(info.readout_phase_ns), offset=int(p.clock_offset_ns), drift_ppm=float(p.clock_drift_ppm))
    stage = OutputStage(m, crop=crop, t_offset_us=1000)
    oracle = Q.OutputOracle(Wd, Hd, rd, crop=crop, t_offset_us=1000)
    f = EventFile(tmp_path / "cam.npz", "cam0", Wd, Hd, t_offset_us=1000)
    released = 0
    for w in range(5):
        ids, ts, ir, offs = random_runs(rng, Wd * Hd, w * W, (w + 1) * W, max_n=24, log_sigma=2.0)
        import torch
        dev = torch.device("cuda:0")
        runs = (torch.from_numpy(ids.astype(np.int32)).to(dev), torch.from_numpy(offs[:-1].copy()).to(dev),
                torch.from_numpy(np.diff(offs).astype(np.int32)).to(dev), torch.from_numpy(ts).to(dev),
                torch.from_numpy(np.ascontiguousarray(ir.reshape(-1))).to(dev))
        torch.cuda.synchronize()
        events = m.advance_device(*runs, (w + 1) * W)
        raw, _ = ref.advance_runs(ids, ts, ir, offs, (w + 1) * W)
        assert events[1] == len(raw)
        got = stage.window(events, w * W)
        want = oracle.window(raw, w * W)
        assert len(got["t"]) == len(want["t"]), w
        for k_got, k_want in (("x", "x"), ("y", "y"), ("p", "p"), ("t", "t"), ("t_ns_rem", "t_ns_rem"),
                              ("t_reported_ns", "t_reported"), ("t_cross_ns", "t_cross"), ("label", "label"),
                              ("flags", "flags")):
            assert np.array_equal(got[k_got], want[k_want]), (w, k_got)
        assert stage.held == len(oracle.held["t_cross"])
        f.append({"x": got["x"], "y": got["y"], "p": got["p"], "t": got["t"], "t_ns_rem": got["t_ns_rem"],
                  "label": got["label"], "t_cross_ns": got["t_cross_ns"], "flags": got["flags"]})
        released += len(got["t"])
    got = stage.flush()
    want = oracle.flush()
    assert np.array_equal(got["t_reported_ns"], want["t_reported"]) and np.array_equal(got["x"], want["x"])
    assert stage.held == 0
    f.append({"x": got["x"], "y": got["y"], "p": got["p"], "t": got["t"], "t_ns_rem": got["t_ns_rem"],
              "label": got["label"], "t_cross_ns": got["t_cross_ns"], "flags": got["flags"]})
    released += len(got["t"])
    assert released > 300
    f.close()
    d = np.load(tmp_path / "cam.npz")
    t = d["events/t"]
    assert len(t) == released and np.all(np.diff(t) >= 0)
    ms = d["ms_to_idx"].astype(np.int64)
    k = np.arange(len(ms))
    assert len(ms) == t[-1] // 1000 + 1
    # entry k is the FIRST event with t >= 1000 k
    assert np.all((ms == len(t)) | (t[np.minimum(ms, len(t) - 1)] >= 1000 * k))
    assert np.all((ms == 0) | (t[np.maximum(ms - 1, 0)] < 1000 * k))


def test_output_order_of_millions_of_events():
    """The stage's stable radix passes at scale: about 2.5 M synthetic raw events per window over a
    1280x720 camera (several hundred sort tiles per pass), their crossing times on a coarse grid and a
    1-us readout quantum, so that the reported time, x and y each tie among many events and the order rests
    on every pass being stable. Two windows and the flush, against the oracle's lexsort."""
    import torch

    import ballasim_amd as bsx
    from ballasim_amd.output import OutputStage
    p = bsx.preset("prophesee_gen3")
    p.photoreceptor = "instantaneous"
    p.noise = False
    p.readout_delay_s = 3e-4
    p.readout_quantum_s = 1e-6
    Wd, Hd = 1280, 720
    m = bsx.SensorModel(p, Wd, Hd, 3, ["constant"], 0, device="cuda")
    m.init(0, np.full((Wd * Hd, 1), 50.0, np.float32))
    info = m._info()
    rd = dict(quantum=round(p.readout_quantum_s * 1e9), delay=round(p.readout_delay_s * 1e9),
              phase=int(info.readout_phase_ns), offset=int(p.clock_offset_ns), drift_ppm=float(p.clock_drift_ppm))
    stage = OutputStage(m, t_offset_us=0)
    oracle = Q.OutputOracle(Wd, Hd, rd, t_offset_us=0)
    rng = np.random.default_rng(11)
    for w in range(2):
        n = 2_600_000
        pix = rng.integers(0, Wd * Hd, n).astype(np.uint32)
        tc = (w * W + rng.integers(0, W // 4096, n) * 4096 + rng.integers(0, 3, n)).astype(np.int64)
        key = pix.astype(np.int64) * (1 << 24) + (tc - w * W)
        _, first = np.unique(key, return_index=True)  # one event per (pixel, t_cross): a total order
        first = rng.permutation(first)
        raw = np.zeros(len(first), O.EVENT_DTYPE)
        raw["pixel"] = pix[first]
        raw["t_cross"] = tc[first]
        raw["polarity"] = rng.integers(0, 2, len(first))
        raw["label"] = rng.integers(0, 8, len(first))  # the class is the label's two low bits
        raw["flags"] = rng.integers(0, 4, len(first))
        dev = torch.from_numpy(raw.view(np.uint8).copy()).cuda()
        torch.cuda.synchronize()
        got = stage.window((dev.data_ptr(), len(raw)), w * W)
        want = oracle.window(raw, w * W)
        assert len(got["t"]) == len(want["t"]) > 10 ** 6, w
        for k_got, k_want in (("x", "x"), ("y", "y"), ("p", "p"), ("t_reported_ns", "t_reported"),
                              ("t_cross_ns", "t_cross"), ("label", "label"), ("flags", "flags")):
            assert np.array_equal(got[k_got], want[k_want]), (w, k_got)
        assert stage.held == len(oracle.held["t_cross"]) > 0
        del dev
    got = stage.flush()
    want = oracle.flush()
    for k_got, k_want in (("x", "x"), ("y", "y"), ("t_reported_ns", "t_reported"), ("t_cross_ns", "t_cross")):
        assert np.array_equal(got[k_got], want[k_want]), k_got


RAW_EVENT = np.dtype([("pixel", np.uint32), ("polarity", np.uint8), ("label", np.uint8), ("flags", np.uint16),
                      ("t_cross", np.int64), ("ds", np.float32), ("dn", np.float32), ("dl", np.float32),
                      ("l_first", np.float32)])


# One block's sort and its edges, the first sizes that are bucketed, quanta that the key divides out (up to two reports
# a window), a drift that gives neighbouring times one report, keys of more than 64 bits (the digit sort), and a column
# copy of several chunks.
@pytest.mark.parametrize("n,size,readout,span", [
    (1, (3, 2), {}, W), (2, (3, 2), {}, 3), (63, (40, 24), {}, W), (65, (40, 24), dict(readout_quantum_s=1e-6), W),
    (2048, (640, 480), dict(readout_quantum_s=2e-5), W), (2049, (640, 480), {}, W),
    (30000, (2048, 1536), dict(readout_quantum_s=5e-3), W), (30000, (64, 48), dict(readout_quantum_s=0.0,
     clock_drift_ppm=-4000.0), 60000), (5000, (65535, 3), dict(readout_quantum_s=1.0), 1 << 40),
    (300001, (1280, 720), dict(readout_quantum_s=1e-6, clock_drift_ppm=35.0), W),
    (5000, (65535, 3), dict(readout_quantum_s=0.0, clock_drift_ppm=-4000.0), 1 << 40),
    (200000, (1280, 720), dict(readout_quantum_s=2e-5), W),
    (200000, (1280, 720), dict(readout_quantum_s=1e-3, clock_drift_ppm=35.0), W)])
def test_output_order_of_any_size(n, size, readout, span):
    import torch

    import ballasim_amd as bsx
    from ballasim_amd.output import OutputStage
    p = bsx.preset("prophesee_gen3")
    p.photoreceptor = "instantaneous"
    p.noise = False
    for k, v in readout.items():
        setattr(p, k, v)
    p.readout_delay_s = max(p.readout_delay_s, p.readout_quantum_s)
    w, h = size
    m = bsx.SensorModel(p, w, h, 3, ["constant"], 0, device="cuda")
    rd = dict(quantum=round(p.readout_quantum_s * 1e9), delay=round(p.readout_delay_s * 1e9),
              phase=int(m._info().readout_phase_ns), offset=int(p.clock_offset_ns), drift_ppm=float(p.clock_drift_ppm))
    rng = np.random.default_rng(n)
    ev = np.zeros(n, RAW_EVENT)
    ev["pixel"] = rng.integers(0, w * h, n)
    ev["polarity"] = rng.integers(0, 2, n)
    ev["label"] = rng.integers(0, 4, n)
    ev["flags"] = rng.integers(0, 1 << 14, n)
    ev["t_cross"] = 1 + rng.permutation(np.arange(n) * (span - 1) // n)  # (distinct, or distinct per pixel below)
    keep = np.unique(ev[["pixel", "t_cross"]], return_index=True)[1]
    ev = ev[np.sort(keep)]
    stage = OutputStage(m)
    oracle = Q.OutputOracle(w, h, rd)
    dev = torch.from_numpy(ev.view(np.uint8).reshape(len(ev), 32)).cuda()
    torch.cuda.synchronize()
    raw = np.zeros(len(ev), O.EVENT_DTYPE)
    for f in ("pixel", "polarity", "label", "flags", "t_cross"):
        raw[f] = ev[f]
    for got, want in ((stage.window((dev.data_ptr(), len(ev)), 0), oracle.window(raw, 0)),
                      (stage.flush(), oracle.flush())):
        for a, b in (("x", "x"), ("y", "y"), ("p", "p"), ("t", "t"), ("t_ns_rem", "t_ns_rem"),
                     ("t_reported_ns", "t_reported"), ("t_cross_ns", "t_cross"), ("label", "label"), ("flags", "flags")):
            assert np.array_equal(got[a], want[b]), a
    assert stage.held == 0


# A column copy by several threads (more than two 1 MiB chunks) behind the columns' kernel, whatever stream the caller
# names: the null stream, one of its own, and the handle that names another stream in each thread. The second window
# differs from the first, whose columns the stage's buffers still hold.
@pytest.mark.parametrize("kind", ["null", "own", "per_thread"])
def test_columns_on_any_stream(kind):
    import torch

    import ballasim_amd as bsx
    from ballasim_amd.output import OutputStage
    p = bsx.preset("prophesee_gen3")
    p.photoreceptor = "instantaneous"
    p.noise = False
    Wd, Hd, n = 640, 480, 200000
    m = bsx.SensorModel(p, Wd, Hd, 3, ["constant"], 0, device="cuda")
    rd = dict(quantum=round(p.readout_quantum_s * 1e9), delay=round(p.readout_delay_s * 1e9),
              phase=int(m._info().readout_phase_ns), offset=int(p.clock_offset_ns), drift_ppm=float(p.clock_drift_ppm))
    own = torch.cuda.Stream()
    stream = {"null": 0, "own": own, "per_thread": 2}[kind]  # 2: hipStreamPerThread
    stage, oracle = OutputStage(m), Q.OutputOracle(Wd, Hd, rd)
    rng = np.random.default_rng(3)
    for w in range(2):
        ev = np.zeros(n, RAW_EVENT)
        ev["pixel"] = rng.integers(0, Wd * Hd, n)
        ev["polarity"] = rng.integers(0, 2, n)
        ev["label"] = rng.integers(0, 4, n)
        ev["t_cross"] = w * W + 1 + rng.permutation(n) * (W // n)
        raw = np.zeros(n, O.EVENT_DTYPE)
        for f in ("pixel", "polarity", "label", "flags", "t_cross"):
            raw[f] = ev[f]
        dev = torch.from_numpy(ev.view(np.uint8).reshape(n, 32)).cuda()
        torch.cuda.synchronize()
        got, want = stage.window((dev.data_ptr(), n), w * W, stream=stream), oracle.window(raw, w * W)
        assert len(got["t"]) == len(want["t"]) > 100000
        for a, b in (("x", "x"), ("y", "y"), ("p", "p"), ("t", "t"), ("t_ns_rem", "t_ns_rem"),
                     ("t_reported_ns", "t_reported"), ("t_cross_ns", "t_cross"), ("label", "label"), ("flags", "flags")):
            assert np.array_equal(got[a], want[b]), (w, a)


@pytest.mark.parametrize("missing", ["x", "t", "flags"])
def test_fetch_refuses_a_null_column(missing):
    import torch

    import ballasim_amd as bsx
    from ballasim_amd import _abi
    from ballasim_amd.output import _COLUMNS, OutputColumns, OutputStage
    p = bsx.preset("prophesee_gen3")
    p.photoreceptor = "instantaneous"
    p.noise = False
    m = bsx.SensorModel(p, 40, 24, 3, ["constant"], 0, device="cuda")
    stage = OutputStage(m)
    ev = np.zeros(100, RAW_EVENT)
    ev["pixel"] = np.arange(100)
    ev["t_cross"] = 1 + 10000 * np.arange(100)  # (each with a report of its own)
    dev = torch.from_numpy(ev.view(np.uint8).reshape(100, 32)).cuda()
    torch.cuda.synchronize()
    n, held = C.c_size_t(), C.c_size_t()
    lib = _abi.load_library()
    _abi.check(lib.bsx_output_window_count(stage._h, C.byref(_abi.DeviceEvents(dev.data_ptr(), 100)), 0, None,
                                           C.byref(n), C.byref(held)))
    assert n.value == 100
    cols = {name: np.zeros(100, dt) for name, dt in _COLUMNS}
    ptr = [None if name == missing else a.ctypes.data for name, a in cols.items()]
    with pytest.raises(ValueError, match="null column"):
        _abi.check(lib.bsx_output_fetch(stage._h, None, C.byref(OutputColumns(*ptr))))
    # refused before anything is written, and the events are still there to fetch
    assert all(not a.any() for a in cols.values())
    _abi.check(lib.bsx_output_fetch(stage._h, None, C.byref(OutputColumns(*[a.ctypes.data for a in cols.values()]))))
    assert np.array_equal(cols["x"], np.arange(100) % 40) and np.array_equal(cols["t_cross_ns"], ev["t_cross"])


# Bursts: buckets past what a block sorts leave the events to the digit sort, with a window's other events around them
# or not; the largest that still fits, and one event more.
@pytest.mark.parametrize("burst,spread", [(2048, 700), (2049, 700), (60000, 700), (60000, 0), (300000, 50000)])
def test_bursts(burst, spread):
    import torch

    import ballasim_amd as bsx
    from ballasim_amd.output import OutputStage
    p = bsx.preset("prophesee_gen3")
    p.photoreceptor = "instantaneous"
    p.noise = False
    p.readout_quantum_s = 0.0
    Wd, Hd = 1280, 720
    m = bsx.SensorModel(p, Wd, Hd, 3, ["constant"], 0, device="cuda")
    rd = dict(quantum=0, delay=round(p.readout_delay_s * 1e9), phase=0, offset=int(p.clock_offset_ns),
              drift_ppm=float(p.clock_drift_ppm))
    rng = np.random.default_rng(burst)
    n = burst + spread
    ev = np.zeros(n, RAW_EVENT)
    ev["pixel"] = rng.permutation(Wd * Hd)[:n]
    ev["polarity"] = rng.integers(0, 2, n)
    ev["t_cross"] = np.where(rng.permutation(n) < burst, 3000000 + rng.integers(0, 2, n), 1 + rng.integers(0, W - 1, n))
    stage, oracle = OutputStage(m), Q.OutputOracle(Wd, Hd, rd)
    dev = torch.from_numpy(ev.view(np.uint8).reshape(n, 32)).cuda()
    torch.cuda.synchronize()
    raw = np.zeros(n, O.EVENT_DTYPE)
    for f in ("pixel", "polarity", "label", "flags", "t_cross"):
        raw[f] = ev[f]
    for got, want in ((stage.window((dev.data_ptr(), n), 0), oracle.window(raw, 0)), (stage.flush(), oracle.flush())):
        for a, b in (("x", "x"), ("y", "y"), ("p", "p"), ("t_reported_ns", "t_reported"), ("t_cross_ns", "t_cross")):
            assert np.array_equal(got[a], want[b]), a
    assert stage.held == 0


class OutputEvents(C.Structure):
    """bsx_output_events: host columns owned by the stage."""
    _fields_ = [("count", C.c_size_t), ("x", C.c_void_p), ("y", C.c_void_p), ("p", C.c_void_p), ("t", C.c_void_p),
                ("t_ns_rem", C.c_void_p), ("t_reported_ns", C.c_void_p), ("t_cross_ns", C.c_void_p),
                ("label", C.c_void_p), ("flags", C.c_void_p), ("held", C.c_size_t)]


# bsx_output_window and bsx_output_flush, whose columns the stage itself holds, against the calls that fetch them: no
# events, one staging chunk (of 1 MiB: 30,840 events), two, and several.
@pytest.mark.parametrize("n", [0, 1, 30000, 50000, 150000])
def test_columns_held_by_the_stage_equal_the_fetched(n):
    import torch

    import ballasim_amd as bsx
    from ballasim_amd import _abi
    from ballasim_amd.output import _COLUMNS, OutputStage
    p = bsx.preset("prophesee_gen3")
    p.photoreceptor = "instantaneous"
    p.noise = False
    p.readout_delay_s = 2e-3  # a quarter of the events is held for the flush
    Wd, Hd = 640, 480
    m = bsx.SensorModel(p, Wd, Hd, 3, ["constant"], 0, device="cuda")
    rng = np.random.default_rng(n)
    ev = np.zeros(n, RAW_EVENT)
    ev["pixel"] = rng.integers(0, Wd * Hd, n)
    ev["polarity"] = rng.integers(0, 2, n)
    ev["label"] = rng.integers(0, 4, n)
    ev["flags"] = rng.integers(0, 1 << 14, n)
    ev["t_cross"] = 1 + rng.permutation(n) * (W // max(n, 1))
    dev = torch.from_numpy(ev.view(np.uint8).reshape(n, 32)).cuda()
    torch.cuda.synchronize()
    fetched, own = OutputStage(m, t_offset_us=17), OutputStage(m, t_offset_us=17)
    lib = _abi.load_library()
    events = _abi.DeviceEvents(dev.data_ptr() if n else None, n)
    for call in ("window", "flush"):
        out = OutputEvents()
        if call == "window":
            want = fetched.window((dev.data_ptr() if n else 0, n), 0)
            _abi.check(lib.bsx_output_window(own._h, C.byref(events), 0, None, C.byref(out)))
        else:
            want = fetched.flush()
            _abi.check(lib.bsx_output_flush(own._h, None, C.byref(out)))
        assert out.count == len(want["t"]) and out.held == fetched.held
        assert n < 100 or out.count > n // 8  # both calls release events
        for name, dt in _COLUMNS:
            got = np.zeros(0, dt)
            if out.count:
                got = np.frombuffer(C.string_at(getattr(out, name), out.count * np.dtype(dt).itemsize), dt)
            assert np.array_equal(got, want[name]), (call, name)
