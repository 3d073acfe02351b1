"""Two timesteps per launch (k_pair) against the oracle and against the two
half steps, bit for bit: tiles whose rims and last, partly filled tiles fall
anywhere, chunks down to one plane, sources (voltage and current) on rims and
chunk ends, UPML in both layouts with slab faces inside tiles and hook-only
cells from random fields, both coefficient layouts, odd step counts, samples
that force single steps between pairs, and graph replays of either parity."""
import time

import numpy as np
import pytest

from oracle.operator_ref import RefOperator
from oracle.oracle import RefEngine
from openems_amd import scenes
from openems_amd._native import NativeError
from openems_amd.engine import EngineHIP
from openems_amd.operator import Operator
from openems_amd.simulation import Simulation

pytestmark = pytest.mark.gpu


def _cavity(nx, ny, nz, curr=False):
    s = scenes.pec_cavity(8, 100)
    s["lines"] = [np.arange(n, dtype=np.float64) for n in (nx, ny, nz)]
    a = (nx // 2, ny // 2, nz // 2)
    s["excitations"] = [{"type": 0, "val": (0.5, 0.0, 1.0), "start": a, "stop": (a[0] + 1, a[1], a[2] + 1)}]
    if curr:
        s["excitations"].append({"type": 2, "val": (0.0, 1.0, 0.3), "start": (2.5, 1.5, 1.5), "stop": (2.5, 2.5, 2.5)})
    s["probes"] = []
    return s


def _graded(n, pml):
    return scenes.upml_bricks(n, 100, nbricks=6, pml=pml, dump=False)


def _sheet(nx, ny, nz):
    """a source in every column of a plane, mesh edges included"""
    s = _cavity(nx, ny, nz)
    s["excitations"] = [{"type": 0, "val": (1.0, 0.5, 0.0), "start": (0, 0, nz // 2), "stop": (nx - 1, ny - 1, nz // 2)}]
    return s


def _columns(nx, ny, nz):
    """columns with one entry a plane, with a gap, with several entries on some planes, and of currents"""
    s = _cavity(nx, ny, nz)
    s["excitations"] = [
        {"type": 0, "val": (0.0, 0.0, 1.0), "start": (12, 0, 0), "stop": (12, ny - 1, nz - 1)},
        {"type": 0, "val": (0.0, 0.5, 0.0), "start": (20, 3, 2), "stop": (20, 14, 6)},
        {"type": 0, "val": (0.0, 0.5, 0.0), "start": (20, 3, 12), "stop": (20, 14, nz - 1)},
        {"type": 0, "val": (0.3, 0.0, 0.7), "start": (4, 8, 5), "stop": (9, 8, 16)},
        {"type": 2, "val": (0.0, 0.2, 0.0), "start": (14.5, 2.5, 1.5), "stop": (14.5, 20.5, nz - 2.5)},
    ]
    return s


def _upml_sheet(axis, thick=0):
    """all components on a sheet (or slab) normal to `axis`, along z over all chunks, UPML cells included"""
    s = _graded(40, 8)
    L = s["lines"]
    lo, hi = [l[3] for l in L], [l[-4] for l in L]
    lo[axis], hi[axis] = L[axis][17], L[axis][17 + thick]
    s["excitations"] = [{"type": 0, "val": (1.0, -0.5, 0.25), "start": tuple(lo), "stop": tuple(hi)},
                        {"type": 2, "val": (0.0, 0.3, 0.1), "start": tuple(lo), "stop": tuple(hi)}]
    return s


CASES = [
    # scene, tile (columns x, y, planes; None: the automatic one), layout, steps
    ("cavity_5x4x3", lambda: _cavity(5, 4, 3), None, "auto", 9),
    ("cavity_23x17x9_current_source", lambda: _cavity(23, 17, 9, True), "7,6,1", "auto", 21),
    ("cavity_23x17x9_plain", lambda: _cavity(23, 17, 9, True), "10,6,4", "plain", 20),
    ("cavity_66x34x12", lambda: _cavity(66, 34, 12), "64,16,5", "auto", 20),
    ("cavity_64", lambda: _cavity(64, 64, 64), None, "auto", 41),
    ("sheet_40x26x18", lambda: _sheet(40, 26, 18), "13,8,3", "auto", 30),
    ("upml_40", lambda: _graded(40, 8), "16,12,7", "compressed", 60),
    ("upml_40_plain", lambda: _graded(40, 8), "16,12,7", "plain", 61),
    ("upml_45_pml6", lambda: _graded(45, 6), None, "compressed", 60),
    ("upml_40_pml6_one_plane", lambda: _graded(40, 6), "40,9,1", "compressed", 40),
    ("columns_30x24x22", lambda: _columns(30, 24, 22), "11,9,6", "plain", 31),
    ("columns_30x24x22_tables", lambda: _columns(30, 24, 22), "11,9,6", "compressed", 30),
    ("upml_40_x_sheet", lambda: _upml_sheet(0), "16,12,7", "compressed", 41),
    ("upml_40_y_slab", lambda: _upml_sheet(1, 2), "13,11,9", "plain", 40),
    ("wires_36", lambda: scenes.wire_antenna(36, 100), "11,36,36", "auto", 80),
]


@pytest.mark.parametrize("name,make,tile,layout,steps", CASES, ids=[c[0] for c in CASES])
def test_pairs_match_oracle_and_halves(gpu, monkeypatch, name, make, tile, layout, steps):
    monkeypatch.setenv("EMS_PAIR", "1")
    if tile:
        monkeypatch.setenv("EMS_PAIR_TILE", tile)
    scene = make()
    print("case pairs", name, tile, layout, "steps", steps, flush=True)
    op = Operator(scene)
    eng = EngineHIP(op, layout=layout)
    assert eng.pair()[0] == 1
    eng.IterateTS(steps)
    assert eng.pair()[2] == steps // 2
    ref = RefEngine(RefOperator(scene).build(), "basic")
    ref.iterate(steps)
    rv, rc = ref.raw_views()
    assert np.max(np.abs(rv)) > 0
    assert np.array_equal(eng.get_volt(), rv)
    assert np.array_equal(eng.get_curr(), rc)
    ref.close()
    # from random fields in every cell, the last lines included
    rng = np.random.default_rng(5)
    v = rng.standard_normal((3,) + tuple(op.N)).astype(np.float32)
    c = rng.standard_normal((3,) + tuple(op.N)).astype(np.float32)
    half = EngineHIP(op, layout=layout, fused=False)
    assert half.pair()[0] == 0
    half.IterateTS(steps)
    for e in (eng, half):
        e.set_volt(v)
        e.set_curr(c)
        e.IterateTS(steps)
    assert np.array_equal(eng.get_volt(), half.get_volt())
    assert np.array_equal(eng.get_curr(), half.get_curr())
    eng.close()
    half.close()


@pytest.mark.parametrize("n,graph", [(40, 0), (40, 24), (64, 7)])
def test_pairs_with_samples_and_graphs(gpu, monkeypatch, n, graph):
    """Probes and dumps fall on odd and even steps: their steps run singly
    where needed; replayed chunks equal direct launches and the half steps."""
    monkeypatch.setenv("EMS_PAIR", "1")
    scene = scenes.upml_bricks(n, 700, nbricks=4) if n == 40 else scenes.pec_cavity(n, 700)
    print("case pairs with samples", n, "graph", graph, flush=True)
    out = []
    for fused in (None, False):
        sim = Simulation(scene, fused=fused, graph=graph)
        sim.run(301)
        sim.run(3)
        sim.run(396)
        assert (sim.eng.pair()[2] > 100) == (fused is None)
        out.append((sim.results(), sim.eng.get_volt(), sim.eng.get_curr(), sim.eng.energy()))
        sim.close()
    (ra, va, ca, ea), (rb, vb, cb, eb) = out
    for k in rb["probes"]:
        assert np.array_equal(ra["probes"][k]["td"], rb["probes"][k]["td"])
    for k in rb["dumps"]:
        assert np.array_equal(ra["dumps"][k]["fd"], rb["dumps"][k]["fd"])
    assert np.array_equal(va, vb) and np.array_equal(ca, cb) and ea == eb


def test_pair_policy(gpu, monkeypatch):
    """Automatic engines without hooks between the half steps take pairs, UPML
    meshes from a million cells on; asked-for step forms and lane widths do not."""
    monkeypatch.delenv("EMS_PAIR", raising=False)
    small, pml = Operator(_cavity(24, 20, 16)), Operator(_graded(40, 6))
    for op, kw, want in ((small, {}, 1), (small, {"fused": False}, 0), (small, {"quad": True}, 0), (small, {"quad": False}, 0),
                         (small, {"fused": "lds"}, 0), (pml, {}, 0),
                         (Operator(scenes.mur_layers(24, 20, 16, 10)), {}, 0), (Operator(scenes.dispersive_rlc(40, 10)), {}, 0),
                         (Operator(_cavity(260, 12, 10)), {}, 1)):
        eng = EngineHIP(op, **kw)
        assert eng.pair()[0] == want, (op.N, kw)
        eng.close()
    # UPML above a million cells: a sheet, a block of voltages, of currents half as many
    for lo, hi, typ, want in ((50, 50, 0, 1), (34, 69, 0, 0), (38, 65, 0, 1), (38, 65, 2, 0)):
        s = scenes.upml_bricks(104, 100, nbricks=4, dump=False)
        x, y, z = s["lines"]
        a, b = (x[lo], y[34], z[34]), (x[hi], y[69], z[69])
        s["excitations"] = [{"type": typ, "val": (0.0, 0.0, 1.0), "start": a, "stop": b}]
        op = Operator(s)
        entries = len(op.excitation(bool(typ))["dir"]) * (2 if typ else 1)
        eng = EngineHIP(op)
        assert eng.pair()[0] == want == (25 * entries <= 104 ** 3), (lo, hi, typ, entries)
        eng.close()


def test_sheet_source_over_many_tiles(gpu, monkeypatch):
    """A source in every column of 600 x 600 and 14400 tiles: set-up does not
    test every column against every tile (12.9 s; as it is 0.08 s)."""
    monkeypatch.setenv("EMS_PAIR", "1")
    op = Operator(_sheet(600, 600, 4))
    half = EngineHIP(op, fused=False)
    half.IterateTS(7)
    monkeypatch.setenv("EMS_PAIR_TILE", "8,8,4")
    print("case pairs sheet source set-up", flush=True)
    t = time.perf_counter()
    eng = EngineHIP(op)
    t = time.perf_counter() - t
    print("set-up %.2f s" % t, flush=True)
    assert eng.pair()[0] == 1
    assert t < 3.0
    eng.IterateTS(7)
    assert np.max(np.abs(half.get_volt())) > 0
    assert np.array_equal(eng.get_volt(), half.get_volt()) and np.array_equal(eng.get_curr(), half.get_curr())
    eng.close()
    half.close()


@pytest.mark.parametrize("pml,few,most,samples", [(False, 8, 12, 2), (True, 15, 26, 3)])
def test_pairs_make_room(gpu, monkeypatch, pml, few, most, samples):
    """Device memory asked for after set-up is taken from the buffers that only
    pairs need, in the middle of a run; an engine short of it from the start
    has no pairs.  Limits in MB: fields 4.6 (with UPML 9.9 and fluxes), as much
    again for pairs, dump samples of 2.3 (3.1)."""
    monkeypatch.setenv("EMS_PAIR", "1")
    op = Operator(_graded(64, 8) if pml else _cavity(64, 60, 50))
    last = [n - 1 for n in op.N]
    print("case pairs make room, UPML", pml, flush=True)

    def dump(e, capacity):
        return e.add_td_dump((0, 0, 0), last, 4, capacity=capacity)

    half = EngineHIP(op, fused=False)
    half.IterateTS(2)
    hid, box = dump(half, samples)
    half.IterateTS(11)
    want = half.get_volt(), half.get_curr(), half.td_dump_results(hid, box)
    monkeypatch.setenv("EMS_DEVICE_BYTES", str(few * 1000000))
    eng = EngineHIP(op)
    assert eng.pair()[0] == 0
    eng.IterateTS(13)
    assert np.array_equal(eng.get_volt(), want[0]) and np.array_equal(eng.get_curr(), want[1])
    eng.close()
    monkeypatch.setenv("EMS_DEVICE_BYTES", str(most * 1000000))
    eng = EngineHIP(op)
    eng.set_graph(2)
    eng.IterateTS(2)
    assert eng.pair()[0] == 1 and eng.pair()[2] == 1
    did, box = dump(eng, samples)
    assert eng.pair()[0] == 0
    with pytest.raises(NativeError, match="hipMalloc"):
        dump(eng, 5)
    eng.IterateTS(11)
    assert np.max(np.abs(want[0])) > 0
    assert np.array_equal(eng.get_volt(), want[0]) and np.array_equal(eng.get_curr(), want[1])
    for a, b in zip(eng.td_dump_results(did, box), want[2]):
        assert np.array_equal(a, b)
    eng.close()
    half.close()


def test_engines_of_different_tiles_in_turn(gpu, monkeypatch):
    """An engine whose tiles take 72 KB of LDS goes on beside one made later
    whose tiles take 5 KB, direct launches and replayed chunks."""
    monkeypatch.setenv("EMS_PAIR", "1")
    op = Operator(_cavity(70, 40, 20, True))
    half = EngineHIP(op, fused=False)
    half.IterateTS(40)
    engs = []
    for tile in ("64,16,5", "64,16,20", "8,8,4"):
        monkeypatch.setenv("EMS_PAIR_TILE", tile)
        engs.append(EngineHIP(op))
        assert engs[-1].pair()[1] == tuple(int(k) for k in tile.split(","))
    print("case pairs of three tiles in turn", flush=True)
    for e in engs:
        e.set_graph(6)
    for n in (4, 1, 15, 20):
        for e in engs:
            e.IterateTS(n)
    for e in engs:
        assert np.array_equal(e.get_volt(), half.get_volt()) and np.array_equal(e.get_curr(), half.get_curr())
        e.close()
    assert np.max(np.abs(half.get_volt())) > 0
    half.close()


@pytest.mark.parametrize("graph", [0, 6, 9])
@pytest.mark.parametrize("shape,interval,curr", [((260, 12, 10), 0, False), ((256, 17, 9), 3, True), ((264, 10, 21), 5, False)])
def test_pairs_beside_quad_sweeps(gpu, monkeypatch, shape, interval, curr, graph):
    """On rows of 64 quads the single steps between pairs are the quad sweep's,
    which swaps the field buffers and not the counters and writes no last
    line: from random fields, against the half steps and the oracle."""
    monkeypatch.delenv("EMS_PAIR", raising=False)
    scene = _cavity(*shape, curr)
    print("case pairs beside quad sweeps", shape, interval, graph, flush=True)
    op = Operator(scene)
    ref = RefEngine(RefOperator(scene).build(), "basic")
    ref.iterate(41)
    rv, rc = ref.raw_views()
    rng = np.random.default_rng(9)
    v = rng.standard_normal((3,) + tuple(op.N)).astype(np.float32)
    c = rng.standard_normal((3,) + tuple(op.N)).astype(np.float32)
    out = []
    for fused in (None, False):
        eng = EngineHIP(op, fused=fused)
        assert eng.pair()[0] == (fused is None) and (eng.fused()[0] == 3) == (fused is None)
        eng.set_graph(graph)
        if interval:
            pos = np.repeat(np.array([[k // 2] for k in shape], np.uint32), 3, 1)
            pid = eng.add_probe(2, [0, 1, 2], pos, None, [1.0] * 3, interval, 0, 0, 10 ** 6, 400)
        eng.IterateTS(5)
        eng.IterateTS(36)
        assert np.array_equal(eng.get_volt(), rv) and np.array_equal(eng.get_curr(), rc)
        for n in (41, 7, 30, 90):
            eng.set_volt(v)
            eng.set_curr(c)
            eng.IterateTS(n)
            out.append((eng.get_volt(), eng.get_curr()))
        if interval:
            out.append(eng.probe_results(pid))
        if fused is None:
            assert eng.pair()[2] > 0
            if graph:
                assert eng.graph()[2] > 0
        eng.close()
    ref.close()
    half = len(out) // 2
    for a, b in zip(out[:half], out[half:]):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def test_setting_a_field_does_not_wait_for_other_engines(gpu, monkeypatch):
    """Fields of a small engine are set while a large one advances."""
    monkeypatch.delenv("EMS_PAIR", raising=False)
    small, large = EngineHIP(Operator(_cavity(20, 18, 16))), EngineHIP(Operator(_cavity(250, 240, 250)))
    assert small.pair()[0] == 1
    rng = np.random.default_rng(2)
    v = rng.standard_normal((3,) + tuple(small.N)).astype(np.float32)
    large.IterateTS(64)                    # its chunk is captured
    small.set_volt(v)
    print("case set a field beside a running engine", flush=True)
    large.set_async(True)
    t = time.perf_counter()
    large.IterateTS(6400)
    small.set_volt(2 * v)
    small.write_field(True, (1, 2, 3), (2, 3, 4), v[:, :2, :2, :2])
    t_set = time.perf_counter() - t
    large.sync()
    t_all = time.perf_counter() - t
    print("set after %.3f s, all done after %.3f s" % (t_set, t_all), flush=True)
    assert t_set < 0.5 * t_all
    assert np.array_equal(small.get_volt(), 2 * v)
    assert np.array_equal(small.read_field(True, (1, 2, 3), (2, 3, 4)), v[:, :2, :2, :2])
    small.close()
    large.close()


def test_creating_an_engine_does_not_wait_for_others(gpu, monkeypatch):
    """An engine with pairs is set up while a large one advances."""
    monkeypatch.setenv("EMS_PAIR", "1")
    large, op = EngineHIP(Operator(_cavity(250, 240, 250))), Operator(_graded(40, 8))
    EngineHIP(op).close()
    large.IterateTS(64)
    print("case engine set up beside a running one", flush=True)
    large.set_async(True)
    t = time.perf_counter()
    large.IterateTS(6400)
    eng = EngineHIP(op)
    t_made = time.perf_counter() - t
    large.sync()
    t_all = time.perf_counter() - t
    print("made after %.3f s, all done after %.3f s" % (t_made, t_all), flush=True)
    assert eng.pair()[0] == 1 and t_made < 0.5 * t_all
    eng.close()
    large.close()
