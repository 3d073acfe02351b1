"""Extension hooks sharing a launch: every combination in which one hook reads
or sets an element that another sets (Mur faces that meet at edges, a single
axis of Mur faces, sources and ADE cells on face and neighbour lines, lumped
elements in dispersive cells, steady-state probes on a face) against the
oracle, bit for bit."""
import numpy as np
import pytest

from oracle.operator_ref import RefOperator
from oracle.oracle import RefEngine
from openems_amd import scenes
from openems_amd.engine import EngineHIP
from openems_amd.operator import Operator
from openems_amd.simulation import steady_state_probes
from tests.test_engine_gpu import _oracle_ade

pytestmark = pytest.mark.gpu


def _layers(bc, at=None):
    """Mur layers, the sheet source across every face line, or one on line `at` of x"""
    s = dict(scenes.mur_layers(30, 26, 22, 120), bc=bc)
    if at is not None:
        lx, ly, lz = s["lines"]
        s["excitations"] = [{"type": 0, "val": (0.0, 1.0, 0.5), "start": (lx[at], ly[8], lz[6]), "stop": (lx[at], ly[9], lz[7])}]
    return s


def _dispersive(bc):
    """ADE cells and lumped elements beside and on Mur lines: the Drude box reaches to the x = 0 face"""
    s = scenes.dispersive_rlc(36, 120)
    L = s["lines"]
    s["bc"] = bc
    s["materials"][0]["start"] = (L[0][0], L[1][0], L[2][10])
    s["lumped"][1]["start"] = (L[0][12], L[1][15], L[2][16])      # inside the Drude box: both set its elements
    s["lumped"][1]["stop"] = (L[0][12], L[1][15], L[2][20])
    s["materials"][0]["stop"] = (L[0][14], L[1][24], L[2][24])
    return s


CASES = [
    ("mur_all", lambda: _layers([2] * 6), True),
    ("mur_x_pair", lambda: _layers([2, 2, 0, 0, 0, 0], 15), False),
    ("mur_x_pair_source_on_neighbour", lambda: _layers([2, 2, 0, 0, 0, 0], 1), True),
    ("mur_x_low_source_on_face", lambda: _layers([2, 0, 1, 0, 0, 1], 0), False),
    ("dispersive_pml", lambda: _dispersive([3] * 6), False),
    ("dispersive_mur_all", lambda: _dispersive([2] * 6), False),
    ("dispersive_mur_x", lambda: _dispersive([2, 2, 0, 0, 0, 0]), False),
]


@pytest.mark.parametrize("name,make,steady", CASES, ids=[c[0] for c in CASES])
def test_hooks_match_oracle(gpu, name, make, steady):
    scene = make()
    print("case hooks", name, flush=True)
    op = Operator(scene)
    ss = steady_state_probes(op) if steady else None
    eng = EngineHIP(op, fused=False, steady_state=ss)
    eng.IterateTS(120)
    ref = RefOperator(scene).build()
    lor, rlc = _oracle_ade(ref) if scene.get("lumped") else ([], None)
    e = RefEngine(ref, "basic", lorentz=lor, rlc=rlc) if lor else RefEngine(ref, "basic")
    e.iterate(120)
    rv, rc = e.raw_views()
    assert np.max(np.abs(rv)) > 0
    assert np.array_equal(eng.get_volt(), rv)
    assert np.array_equal(eng.get_curr(), rc)
    eng.close()
    e.close()


@pytest.mark.parametrize("mur", [False, True])
def test_long_unordered_ade_lists(gpu, mur):
    """Three orders over most cells of the mesh (faces included), in random
    order and overlapping, with lumped elements among them: lists long enough
    for the counting sort, against the oracle."""
    scene = dict(scenes.mur_layers(40, 36, 30, 60), bc=[2] * 6) if mur else scenes.upml_bricks(40, 60, nbricks=6, dump=False)
    print("case hooks long ADE lists, Mur", mur, flush=True)
    op = Operator(scene)
    rng = np.random.default_rng(8)
    cells = int(np.prod(op.N))
    lor = []
    for share, lorentz, curr in ((0.7, True, True), (0.5, False, True), (0.02, False, False)):
        at = rng.permutation(cells)[:int(share * cells)]
        k = len(at)
        o = {"pos": np.stack(np.unravel_index(at, tuple(op.N))).astype(np.uint32), "volt": True, "curr": curr}
        for s in "vi":
            o[s + "_int"] = rng.uniform(0.8, 0.95, (3, k)).astype(np.float32)
            o[s + "_ext"] = rng.uniform(1e-3, 5e-3, (3, k)).astype(np.float32)
            o[s + "_lor"] = rng.uniform(1e-3, 5e-3, (3, k)).astype(np.float32) if lorentz else None
        lor.append(o)
    assert lor[0]["pos"].shape[1] > 16384 and lor[2]["pos"].shape[1] < 16384
    rlc = {"pos": np.stack([rng.choice(np.arange(3, n - 3), 6, replace=False) for n in op.N]).astype(np.uint32),
           "dir": rng.integers(0, 3, 6).astype(np.int32)}
    for name in ("i2v", "ilv", "vvd", "vv2", "vj1", "vj2", "ib0", "b1", "b2"):
        rlc[name] = rng.uniform(0.5, 0.9, 6).astype(np.float32) if name == "vvd" else rng.uniform(-0.05, 0.05, 6).astype(np.float32)
    eng = EngineHIP(op, fused=False, lorentz=lor, rlc=rlc)
    eng.IterateTS(60)
    ref = RefEngine(RefOperator(scene).build(), "basic", lorentz=lor, rlc=rlc)
    ref.iterate(60)
    rv, rc = ref.raw_views()
    assert np.max(np.abs(rv)) > 0
    assert np.array_equal(eng.get_volt(), rv)
    assert np.array_equal(eng.get_curr(), rc)
    eng.close()
    ref.close()


def _sweep_mur(nx, faces=(2, 2, 2, 2, 2, 2)):
    return lambda: dict(scenes.mur_layers(nx, 26, 22, 120), bc=list(faces))


@pytest.mark.parametrize("graph", [0, 8])
@pytest.mark.parametrize("make,kw", [
    (lambda: _layers([2] * 6), dict(fused=False)),
    (lambda: _dispersive([3] * 6), dict(fused=False, quad=False)),
    (lambda: _dispersive([3] * 6), dict(fused=False, quad=True)),
    (lambda: _dispersive([2, 2, 0, 0, 0, 0]), dict(fused=False)),
    (_sweep_mur(32, (2, 3, 3, 3, 3, 3)), dict(fused=False, quad=True)),
    (_sweep_mur(32), dict(fused="quads")),
    (_sweep_mur(264), dict(fused="quads")),                              # the x faces inside the sweep
    (_sweep_mur(264, (2, 2, 0, 0, 0, 0)), dict(fused="quads")),          # no face left around it
    (_sweep_mur(264, (0, 0, 0, 0, 0, 2)), dict(fused="quads")),
], ids=["layers", "ade_pml", "ade_pml_quads", "ade_mur", "mur_pml", "sweep", "sweep_fold", "sweep_fold_only", "sweep_z"])
def test_calls_of_any_length_agree(gpu, make, kw, graph):
    """The next step's hooks run beside the currents only within a call: calls
    of one step (which never do that), calls of every length, replayed chunks,
    and fields set between calls give the same bits."""
    scene = make()
    print("case hooks calls", scene["bc"], kw, graph, flush=True)
    op = Operator(scene)
    got = []
    for lengths in ([1] * 45, [1, 2, 37, 3, 2], [40, 5]):
        eng = EngineHIP(op, **kw)
        eng.set_graph(graph)
        n = 0
        for k in lengths:
            if n == 40:                # a field set between two calls
                eng.set_volt(np.ascontiguousarray(eng.get_volt() * np.float32(0.5)))
            eng.IterateTS(k)
            n += k
        got.append((eng.get_volt(), eng.get_curr()))
        eng.close()
    assert np.max(np.abs(got[0][0])) > 0
    for v, c in got[1:]:
        assert np.array_equal(v, got[0][0])
        assert np.array_equal(c, got[0][1])


@pytest.mark.parametrize("nprobe", [1, 191, 400])
def test_steady_state_of_many_probes(gpu, nprobe):
    """More probes than the evaluation has threads, and one."""
    scene = _layers([2] * 6)
    op = Operator(scene)
    period, _, _ = steady_state_probes(op)
    rng = np.random.default_rng(nprobe)
    dirs = rng.integers(0, 3, nprobe).tolist()
    pos = [[int(rng.integers(0, k)) for k in op.N] for _ in range(nprobe)]
    print("case steady state,", nprobe, "probes", flush=True)
    eng = EngineHIP(op, fused=False, steady_state=(period, dirs, pos))
    eng.IterateTS(6 * period + 3)
    ref = RefEngine(RefOperator(scene).build(), "basic", steady_state=(period, dirs, pos))
    ref.iterate(6 * period + 3)
    last, hist = eng.steady_state()
    want = ref.steady_history()
    assert len(hist) == len(want) and len(want) > 3 and last == hist[-1][1]
    for (t1, d1), (t2, d2) in zip(hist, want):
        assert t1 == t2
        # the energy is summed in another order than the oracle's
        assert d1 == pytest.approx(d2, rel=1e-9, abs=1e-300)
    eng.close()
    ref.close()
