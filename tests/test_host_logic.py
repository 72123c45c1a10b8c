"""Host-side logic that needs no GPU: sweep draws, tile tables, table layouts,
checkpoint files."""

import ctypes

import numpy as np
import pytest
import torch


def test_sweep_draws_are_reproducible():
    from latticeboltzmann_amd.batch import SIZES, shear_wave_sweep
    a, b = shear_wave_sweep(512, 0), shear_wave_sweep(512, 0)
    assert a == b and len(a) == 512
    assert {p["nx"] for p in a} <= set(SIZES) and {p["ny"] for p in a} <= set(SIZES)
    assert all(0.3 <= p["omega"] <= 1.9 and 0.01 <= p["amplitude"] <= 0.1 for p in a)
    assert {p["direction"] for p in a} == {"x", "y"}
    # the draws of numpy.random.default_rng(0), in the documented order
    rng = np.random.default_rng(0)
    nx = rng.choice(SIZES, 512)
    assert [p["nx"] for p in a] == nx.tolist()
    assert shear_wave_sweep(512, 1) != a


def test_instance_and_tile_records_match_the_c_structs():
    from latticeboltzmann_amd.batch import INST_DTYPE, TILE_DTYPE

    class Inst(ctypes.Structure):
        _fields_ = [("offset", ctypes.c_int64), ("nx", ctypes.c_int32), ("ny", ctypes.c_int32),
                    ("omega", ctypes.c_double), ("u0", ctypes.c_double), ("bc", ctypes.c_int32),
                    ("dir", ctypes.c_int32)]

    class Tile(ctypes.Structure):
        _fields_ = [("inst", ctypes.c_int32), ("first", ctypes.c_int32)]

    assert INST_DTYPE.itemsize == ctypes.sizeof(Inst) == 40
    assert TILE_DTYPE.itemsize == ctypes.sizeof(Tile) == 8
    for name, _ in Inst._fields_:
        assert INST_DTYPE.fields[name][1] == getattr(Inst, name).offset


def test_tiles_cover_every_node_once():
    from latticeboltzmann_amd.batch import _tiles
    sizes = [64 * 64, 64 * 1024, 128 * 192]
    for tile in (64, 256, 1024):
        t = _tiles(range(3), sizes, tile)
        for i, n in enumerate(sizes):
            firsts = np.sort(t["first"][t["inst"] == i])
            assert firsts[0] == 0 and np.all(np.diff(firsts) == tile)
            assert firsts[-1] < n <= firsts[-1] + tile


def test_size_class_rounds_up_to_powers_of_two():
    from latticeboltzmann_amd.autotune import size_class
    assert size_class(1000, 1000) == "1024x1024"
    assert size_class(64, 65) == "64x128"
    assert size_class(1, 1) == "1x1"


def _bare(cls, **attrs):
    # the host arithmetic of a lattice without touching a device
    obj = cls.__new__(cls)
    obj.__dict__.update(attrs)
    return obj


def test_lattice_launch_count():
    from latticeboltzmann_amd.lattice import Lattice, StepGraph
    lat = _bare(Lattice, multi_variant=10, multi_k=3)
    assert [lat.launches(n) for n in (0, 1, 2, 3, 4, 1000, 1001)] == [0, 1, 2, 1, 2, 334, 335]
    single = _bare(Lattice, multi_variant=None, multi_k=1)
    assert single.launches(1000) == 1000
    # a graph is captured only when the state ends in the buffer it started in
    assert StepGraph(lat, 1000).enabled and not StepGraph(lat, 999).enabled
    assert not StepGraph(_bare(Lattice, multi_variant=12, multi_k=4), 1001).enabled
    assert StepGraph(single, 2).enabled and not StepGraph(single, 3).enabled


def test_deviation_lattice_launch_count():
    from latticeboltzmann_amd.precision import DeviationLattice
    lat = _bare(DeviationLattice, multi_variant=2, multi_k=3)
    assert [lat.launches(n) for n in (1, 3, 7, 9)] == [1, 1, 3, 3]
    assert _bare(DeviationLattice, multi_variant=None, multi_k=1).launches(7) == 7


class _FakeLattice:
    """Host stand-in with a Lattice's checkpointed attributes (CPU tensors)."""

    def __init__(self, nx=4, ny=6, omega=1.2, dtype=torch.float64):
        self.nx, self.ny, self.omega, self.bc, self.u0, self.layout = nx, ny, omega, "cavity", 0.1, 1
        self.f = torch.zeros((nx, 9, ny), dtype=dtype)
        self.time = 0


class _FakeDeviationLattice(_FakeLattice):
    def __init__(self, fmt=2, **kw):
        super().__init__(**kw)
        del self.f
        self.fmt, self.scale, self.rounding, self.seed, self.compute, self.store_every = \
            fmt, 1024.0, 1, 7, 0, 4
        raw = torch.float32 if fmt == 0 else torch.int16
        self.d = torch.zeros((self.nx, 9, self.ny), dtype=raw)


def test_checkpoint_round_trip_and_parameter_checks(tmp_path):
    from latticeboltzmann_amd import checkpoint
    rng = np.random.default_rng(5)
    a = _FakeLattice()
    a.f.copy_(torch.from_numpy(rng.standard_normal(a.f.shape)))
    a.f[0, 0, 0] = float("nan")  # every bit, NaN payloads included
    a.time = 1234
    p = str(tmp_path / "lat.npz")
    checkpoint.save(a, p)
    b = _FakeLattice()
    checkpoint.restore(b, p)
    assert b.time == 1234
    assert np.array_equal(b.f.numpy().view(np.uint64), a.f.numpy().view(np.uint64))
    for attr, val in (("omega", 1.3), ("bc", "periodic"), ("layout", 0)):
        c = _FakeLattice()
        setattr(c, attr, val)
        with pytest.raises(ValueError):
            checkpoint.restore(c, p)
    with pytest.raises(ValueError):  # grid shape
        checkpoint.restore(_FakeLattice(nx=5), p)
    with pytest.raises(ValueError):  # storage type
        checkpoint.restore(_FakeLattice(dtype=torch.float32), p)
    with pytest.raises(ValueError):  # kind
        checkpoint.restore(_FakeDeviationLattice(), p)


def test_checkpoint_deviation_words(tmp_path):
    from latticeboltzmann_amd import checkpoint
    a = _FakeDeviationLattice()
    a.d.copy_(torch.arange(a.d.numel(), dtype=torch.int16).view(a.d.shape))
    a.time = 48
    p = str(tmp_path / "dev.npz")
    checkpoint.save(a, p)
    b = _FakeDeviationLattice()
    checkpoint.restore(b, p)
    assert b.time == 48 and torch.equal(a.d, b.d)
    c = _FakeDeviationLattice()
    c.seed = 8  # another dither stream: not the same run
    with pytest.raises(ValueError):
        checkpoint.restore(c, p)
    d = _FakeDeviationLattice()
    d.store_every = 1
    with pytest.raises(ValueError):
        checkpoint.restore(d, p)


@pytest.mark.parametrize("dtype,nx,ny,periodic,walls", [
    (torch.float64, 64, 64, False, False), (torch.float64, 2048, 2048, True, True),
    (torch.float32, 2048, 2048, True, True), (torch.float32, 512, 512, False, False),
    (torch.float64, 700, 1500, True, True), (torch.float64, 6000, 100, True, False),
    (torch.float32, 100000, 160, True, False),
    # values of one or two bytes, short rows, a few long rows
    (torch.uint8, 3000, 2000, False, False), (torch.float16, 2048, 2048, False, False),
    (torch.float64, 100000, 10, False, False), (torch.float32, 1000000, 8, False, False),
    (torch.float64, 3, 500000, False, False), (torch.float32, 64, 20000, False, False),
    (torch.float32, 256, 100000, True, True)])
def test_streaming_route(dtype, nx, ny, periodic, walls):
    # in place exactly where that was measured to be no slower than a second array
    from latticeboltzmann_amd.PyLB import Streaming
    f = torch.empty((9, nx, ny), dtype=dtype, device="meta")
    assert Streaming._in_place(f, False) == periodic
    assert Streaming._in_place(f, True) == walls


def test_streaming_route_beyond_one_launch():
    # grids that take more than 2^32 threads in place go through a second array,
    # which takes fewer; the in-place calls say so before any launch
    from latticeboltzmann_amd import _native as nat
    from latticeboltzmann_amd.PyLB import Streaming
    lib = nat.load()
    for nx, fits in ((5 << 20, True), (8 << 20, False)):
        f = torch.empty((9, nx, 128), dtype=torch.float32, device="meta")
        assert Streaming._in_place(f, False) == fits
        assert (lib.lbm_stream_inplace_scratch(nx, 128, 0) > 0) == fits
        assert (lib.lbm_stream_inplace_scratch(nx, 128, 1) > 0) == fits
    assert lib.lbm_stream_inplace_scratch(8 << 20, 128, 0) == -2
    # every grid that the route takes fits
    for nx in (1, 255, 256, 5000, 1 << 20, 5592405, 1 << 23, 1 << 24):
        for ny in (128, 255, 256, 1000, 6144, 6145, 1 << 20, 1 << 26):
            f = torch.empty((9, nx, ny), dtype=torch.float64, device="meta")
            for walls in (False, True):
                assert not Streaming._in_place(f, walls) or lib.lbm_stream_inplace_scratch(nx, ny, walls) > 0


class _FailingRun:
    """Stands for the native library: its run makes an odd number of launches,
    then fails."""

    def call(self, name, *args):
        assert "_run_" in name
        args[-2]._obj.value = 1
        raise RuntimeError("HIP error")


def test_failed_lattice_run_leaves_the_state_of_its_launches(monkeypatch):
    from latticeboltzmann_amd import _native as nat
    from latticeboltzmann_amd import kernels
    from latticeboltzmann_amd.lattice import Lattice
    monkeypatch.setattr(nat, "call", _FailingRun().call)
    monkeypatch.setattr(nat, "stream_ptr", lambda: 0)
    monkeypatch.setattr(kernels, "_require_device", lambda *t: None)
    a, b = (torch.zeros((64, 9, 64), dtype=torch.float64) for _ in range(2))
    lat = _bare(Lattice, f=a, _g=b, omega=1.2, bc="cavity", u0=0.1, layout=nat.LAYOUT_ROWS, variant=-1,
                multi_variant=None, multi_k=1, time=0)
    with pytest.raises(RuntimeError):
        lat.step(3)
    assert lat.f is b and lat._g is a and lat.time == 0


def test_failed_ghost_run_leaves_the_state_of_its_launches(monkeypatch):
    from latticeboltzmann_amd import _native as nat
    from latticeboltzmann_amd.ghost import GhostLattice
    monkeypatch.setattr(nat, "call", _FailingRun().call)
    monkeypatch.setattr(nat, "stream_ptr", lambda: 0)
    a, b = (torch.zeros((30, 9, 40), dtype=torch.float64) for _ in range(2))
    lat = _bare(GhostLattice, f=a, _g=b, nx=30, ny=40, omega=1.2, layout=nat.LAYOUT_ROWS, rules=[],
                _rules=(nat.GhostRule * 1)(), _pbc=None, dtype=torch.float64, time=0)
    with pytest.raises(RuntimeError):
        lat.step(3)
    assert lat.f is b and lat._g is a and lat.time == 0


def test_native_ghost_run_says_where_the_state_is():
    # *in_b is 0 when a run is refused before its first launch, whatever it held
    from latticeboltzmann_amd import _native as nat
    lib = nat.load()
    for nx, steps, status in ((2, 3, -2), (30, -1, -2)):
        in_b = ctypes.c_int(7)
        assert lib.lbm_ghost_run_f64(1 << 20, 1 << 30, nx, 40, 0, 1.2, None, 0, None, steps, None, None, None,
                                     ctypes.byref(in_b), None) == status
        assert in_b.value == 0


@pytest.mark.parametrize("cin,cout,transposed", [(16384, 8192, 0), (8192, 16384, 1), (65536, 2048, 0)])
def test_packing_leaves_out_layers_beyond_the_packed_kernels(cin, cout, transposed):
    # weights past 2^31 packed bytes run unpacked: no packed place, and packing a
    # network that has such a layer is no error
    from latticeboltzmann_amd import _native as nat
    lib = nat.load()
    assert lib.lbm_nn_packed_size(cin, cout) == 0
    assert lib.lbm_nn_packed_fits(1, 2, 2, cin, cout) == 0
    frm, to = (ctypes.c_int64 * 1)(0), (ctypes.c_int64 * 1)(0)
    ci, co = (ctypes.c_int * 1)(cin), (ctypes.c_int * 1)(cout)
    # nothing is launched, so no pointer is read
    assert lib.lbm_nn_pack_weights(1 << 20, ctypes.addressof(frm), ctypes.addressof(ci), ctypes.addressof(co), 1,
                                   transposed, 1 << 20, ctypes.addressof(to), None) == 0
    assert lib.lbm_nn_packed_size(8192, 8192) == 9 * 8192 * 8192
    # a network of such layers has a workspace without room for their packed weights
    widths = (ctypes.c_int * 1)(32)
    small = lib.lbm_nn_unet_workspace(1, 2, 2, 32, ctypes.addressof(widths), 1, 32, 3)
    large = lib.lbm_nn_unet_workspace(1, 2, 2, 32, ctypes.addressof(widths), 1, 16384, 3)
    assert 0 < small < large < small + (1 << 25)


def test_small_tiles_are_tuned_on_small_grids_only():
    from latticeboltzmann_amd import _native as nat
    from latticeboltzmann_amd import kernels
    from latticeboltzmann_amd.autotune import multi_candidates
    info = {v: kernels.step_multi_info(v) for v in range(nat.load().lbm_step_multi_variant_count())}
    small = {v for v, (k, mnx, mny) in info.items() if 0 < mny - 2 * k <= 16}
    assert len(small) == 3
    assert small <= set(multi_candidates(256, 256, info, 256))
    for nx, ny in ((933, 933), (2048, 2048), (100, 6000)):
        got = set(multi_candidates(nx, ny, info, 256))
        assert not got & small
        # the others are those that fit
        assert got == {v for v, (k, mnx, mny) in info.items() if nx >= mnx and ny >= mny} - small
    assert multi_candidates(15, 15, info, 256) == []


def test_tuner_times_close_variants_again(monkeypatch, tmp_path):
    from latticeboltzmann_amd import _native as nat
    from latticeboltzmann_amd import autotune
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda d: "none")
    monkeypatch.setattr(nat, "build_id", lambda: "0")
    monkeypatch.setenv("LBM_TUNE_CACHE", str(tmp_path / "tune.json"))
    monkeypatch.setattr(autotune, "_MEMO", {})
    true = {1: 4.0, 2: 4.4, 3: 9.0, 4: 8.0}  # per launch; variant 4 makes two steps
    rounds = []

    def timed(launch, variants, reps=10, warmup=2):
        rounds.append(list(variants))
        slow = 1.25 if len(rounds) == 1 else 1.0  # the first timing of variant 1 was disturbed
        return {v: true[v] * (slow if v == 1 else 1.0) for v in variants}

    monkeypatch.setattr(autotune, "time_variants", timed)
    best = autotune.best_variant("k", 64, 64, "f64", 0, 0, lambda nx, ny: None, [1, 2, 3])
    assert best == 1 and rounds == [[1, 2, 3], [1, 2], [1, 2]]
    del rounds[:]
    best = autotune.best_variant("m", 64, 64, "f64", 0, 0, lambda nx, ny: None, [2, 3, 4],
                                 normalize=lambda t: {v: x / (2 if v == 4 else 1) for v, x in t.items()})
    assert best == 4 and rounds == [[2, 3, 4], [2, 4], [2, 4]]
    assert autotune.best_variant("k", 64, 64, "f64", 0, 0, None, [1, 2, 3]) == 1  # kept
