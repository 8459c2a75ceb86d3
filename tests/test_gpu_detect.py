"""Particle-pair drivers on the GPU against the oracle: every contact field
bit for bit, the emission order, and the statistics."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as ol
import scenes
from delta_amd import _lib, contact, shapes
from delta_amd.device import DeviceArray

pytestmark = pytest.mark.gpu

METHODS = {
    "bf": (contact.bf, _lib.DH_BF),
    "penalty": (contact.penalty, _lib.DH_PENALTY),
    "hybrid_batch": (contact.hybridWithPerBatchFallBack, _lib.DH_HYBRID_BATCH),
    "hybrid_triangle": (contact.hybridWithPerTriangleFallBack, _lib.DH_HYBRID_TRIANGLE),
    "penalty_stat": (contact.penaltyStat, _lib.DH_PENALTY_STAT),
    "hybrid_batch_stat": (contact.hybridBatchStat, _lib.DH_HYBRID_BATCH_STAT),
    "hybrid_triangle_stat": (contact.hybridTriangleStat, _lib.DH_HYBRID_TRIANGLE_STAT),
    "gjk": (lambda xA, yA, zA, nA, eA, fA, iA, xB, yB, zB, nB, eB, fB, iB:
            contact.gjk(nA, xA, yA, zA, eA, fA, iA, nB, xB, yB, zB, eB, fB, iB), _lib.DH_GJK),
}
FIELDS = ["x", "normal", "depth", "P", "Q", "eps_total", "master", "slave", "penetration",
          "friction", "triA", "triB"]
EPS = 1e-4


def same_contacts(a, b):
    assert len(a) == len(b), (len(a), len(b))
    for f in FIELDS:
        va, vb = np.ascontiguousarray(a[f]), np.ascontiguousarray(b[f])
        if va.dtype == np.float64:
            assert np.array_equal(va.view(np.uint64), vb.view(np.uint64)), f
        else:
            assert np.array_equal(va, vb), f


@pytest.mark.parametrize("method", list(METHODS))
@pytest.mark.parametrize("case", range(len(scenes.pair_cases())))
def test_pair_driver_matches_oracle(method, case):
    name, A, B = scenes.pair_cases()[case]
    fn, code = METHODS[method]
    if code == _lib.DH_HYBRID_TRIANGLE and len(B) > len(A):
        A, B = B, A
    xa, xb = shapes.to_soa(A), shapes.to_soa(B)
    contact.reset_all_statistics()
    got = fn(*xa, len(A), EPS, True, 7, *xb, len(B), EPS, True, 9)
    st = contact._stats
    rc, want, ost = ol.or_detect(code, A, B, EPS, EPS, 1, 1, 7, 9)
    assert rc == 0
    same_contacts(got, want)
    assert list(st.newton_histogram) == list(ost.newton_histogram)
    for f in ("penalty_fails", "batch_fails", "batch_size", "triangle_checks",
              "pairs_evaluated", "fallback_rows"):
        assert getattr(st, f) == getattr(ost, f), f
    assert st.batch_error == ost.batch_error


def soup(n, seed, shift=0.0):
    """n triangles of 0.3 across in a unit cube: crossing, close and apart."""
    rng = np.random.default_rng(seed)
    t = rng.uniform(0.0, 1.0, (n, 1, 3)) + rng.uniform(-0.15, 0.15, (n, 3, 3))
    t[:, :, 0] += shift
    return t


TILE_SIZES = [(1, 1, 0.2), (16, 16, 0.1), (17, 15, 0.1), (321, 79, 1e-3), (321, 79, 1e-5)]
NOTED_SIZES = [(1100, 1000, 1e-3), (1100, 1000, 1e-5)]  # the notes are the hybrids'


@pytest.mark.parametrize("method,na,nb,eps", [
    (m, *size) for m in ("bf", "penalty", "hybrid_batch", "hybrid_triangle", "hybrid_batch_stat")
    for size in TILE_SIZES + (NOTED_SIZES if m in ("hybrid_batch", "hybrid_triangle") else [])])
def test_tiles_of_one_pair_match_oracle(method, na, nb, eps):
    """Partial tiles, rows over several workgroups, and (1,100 x 1,000) tiles
    of more pairs than a hybrid tile notes; at 1e-5 most rows fall back, at
    the larger margins none."""
    A, B = soup(na, 3), soup(nb, 4, 0.4)
    fn, code = METHODS[method]
    contact.reset_all_statistics()
    got = fn(*shapes.to_soa(A), na, eps, True, 7, *shapes.to_soa(B), nb, eps, True, 9)
    st = contact._stats
    rc, want, ost = ol.or_detect(code, A, B, eps, eps, 1, 1, 7, 9)
    assert rc == 0
    same_contacts(got, want)
    for f in ("penalty_fails", "batch_fails", "batch_size", "triangle_checks",
              "pairs_evaluated", "fallback_rows"):
        assert getattr(st, f) == getattr(ost, f), f


def test_hybrid_triangle_rejects_reference_out_of_bounds():
    A = scenes.particle(0, 0.5e-3, 1, [0, 0, 0])
    B = scenes.particle(1, 0.5e-3, 2, [1e-3, 0, 0])
    with pytest.raises(_lib.DhError) as e:
        contact.hybridWithPerTriangleFallBack(*shapes.to_soa(A), len(A), EPS, 0, 0,
                                              *shapes.to_soa(B), len(B), EPS, 0, 1)
    assert e.value.code == 4


@pytest.mark.parametrize("method", ["bf", "penalty", "hybrid_batch", "hybrid_batch_stat", "gjk"])
def test_batched_pairs_match_per_pair_oracle(method):
    """dh_detect_pairs over several particle pairs: contacts grouped by pair
    in pair order, each group in reference order."""
    _batched_pairs(method)


@pytest.mark.parametrize("screen", [0, 1])
@pytest.mark.parametrize("max_tiles", [1, 16])
def test_batched_bf_through_the_survivor_queue(max_tiles, screen):
    """The same with the survivor queue forced on (every item's survivors
    solved from one queue, one per lane), with and without the binary32
    screen: bit-exact and in order."""
    from delta_amd import tuning
    tuning.set(detect_queue_min_items=0, detect_max_tiles=max_tiles, detect_fp32_screen=screen)
    try:
        _batched_pairs("bf")
    finally:
        tuning.set(**tuning.default())


@pytest.mark.parametrize("max_tiles", [1, 7])
@pytest.mark.parametrize("eps", [1e-3, 5e-3, 2e-2, 1e-1])
def test_survivor_queue_at_its_limits(eps, max_tiles):
    """Segments below and above the 256 entries that one wave takes, items that
    go on in the pool's blocks, of more than the 2,048 entries that may queue
    and of more than 160 kept boxes, uneven ones, empty ones and one triangle:
    the contacts, their order and the counters are the oracle's."""
    from delta_amd import tuning
    parts = [soup(80, 1), soup(80, 2, 0.1), soup(320, 3, 0.5), soup(100, 4, 0.7), soup(8, 5, 0.2),
             soup(1, 6), soup(700, 7, 5.0), soup(64, 8, 4.2)]
    pairs = [(0, 1), (0, 2), (0, 4), (1, 2), (1, 3), (2, 3), (2, 4), (4, 2), (5, 0), (0, 6), (6, 7)]
    tuning.set(detect_queue_min_items=0, detect_max_tiles=max_tiles)
    try:
        _batched_pairs("bf", parts, pairs, eps)
    finally:
        tuning.set(**tuning.default())


def _batched_pairs(method, parts=None, pairs=None, eps=EPS):
    if parts is None:
        parts = [scenes.particle(1 + (i % 2), 0.5e-3, 50 + i, [0.98e-3 * i, 0.05e-3 * (i % 3), 0])
                 for i in range(6)]
        parts.append(scenes.floor(-0.45e-3))
        pairs = [(i, i + 1) for i in range(5)] + [(i, 6) for i in range(6)] + [(0, 2)]
    offs = np.cumsum([0] + [len(p) for p in parts]).astype(np.int32)
    allm = np.concatenate(parts)
    x, y, z = (DeviceArray.from_host(v) for v in shapes.to_soa(allm))
    d_off = DeviceArray.from_host(offs)
    n = len(parts)
    d_eps = DeviceArray.from_host(np.full(n, eps))
    d_fr = DeviceArray.from_host(np.ones(n, np.int32))
    d_id = DeviceArray.from_host(np.arange(n, dtype=np.int32) * 10)
    d_pairs = DeviceArray.from_host(np.array(pairs, np.int32).reshape(-1))
    g = _lib.DhGeometry(x.ptr, y.ptr, z.ptr, d_off.ptr, d_eps.ptr, d_fr.ptr, d_id.ptr, n,
                        int(offs[-1]))
    code = METHODS[method][1]
    cap = 200000
    out = DeviceArray((cap * 144,), np.uint8)
    cnt = DeviceArray((len(pairs),), np.int32)
    nout = C.c_int(0)
    st = _lib.DhStats()
    L = _lib.lib()
    L.dh_detect_pairs.argtypes = [C.c_int, C.POINTER(_lib.DhGeometry), C.c_void_p, C.c_int,
                                  C.c_void_p, C.c_int, C.POINTER(C.c_int), C.c_void_p,
                                  C.POINTER(_lib.DhStats), C.c_void_p]
    _lib.check(L.dh_detect_pairs(code, C.byref(g), d_pairs.ptr, len(pairs), out.ptr, cap,
                                 C.byref(nout), cnt.ptr, C.byref(st), None), "detect_pairs")
    got = np.frombuffer(out.download().tobytes()[:144 * nout.value], dtype=contact.CONTACT_DTYPE)
    counts = cnt.download()
    want = []
    ost_total = ol.DhStats()
    for k, (a, b) in enumerate(pairs):
        rc, w, ost = ol.or_detect(code, parts[a], parts[b], eps, eps, 1, 1, 10 * a, 10 * b)
        assert rc == 0
        assert counts[k] == len(w)
        w = w.copy()
        w["pair"] = k
        want.append(w)
        for f in ("penalty_fails", "batch_fails", "batch_size", "triangle_checks",
                  "pairs_evaluated", "fallback_rows"):
            setattr(ost_total, f, getattr(ost_total, f) + getattr(ost, f))
    want = np.concatenate(want)
    same_contacts(got, want)
    assert np.array_equal(got["pair"], want["pair"])
    for f in ("penalty_fails", "batch_fails", "batch_size", "triangle_checks",
              "pairs_evaluated", "fallback_rows"):
        assert getattr(st, f) == getattr(ost_total, f), f


def _wall_touching_particle():
    """The 2,048-triangle funnel and an 80-triangle sphere pressed 0.05 mm
    into its wall at mid height."""
    from delta_amd import workloads
    funnel = shapes.cone_funnel(2e-3, 20e-3, 30.0)
    t = np.tan(np.radians(30.0))
    y = 15e-3
    inward = -np.array([1.0, -t, 0.0]) / np.hypot(1.0, t)
    c = np.array([2e-3 + y * t, y, 0.0]) + inward * 0.45e-3
    return funnel, scenes.particle(1, 0.5e-3, 61, c)


@pytest.mark.parametrize("queue", [0, 1])
@pytest.mark.parametrize("max_tiles", [1, 16])
@pytest.mark.parametrize("swap", [False, True])
def test_bf_large_particle_matches_oracle(max_tiles, swap, queue):
    """A particle with more rows than one LDS block holds (the funnel as A:
    2,048 rows, staged in blocks of 320 when one workgroup takes them all)
    and as B (2,048 columns: the unstaged pass): contacts bit-exact and in
    the reference's order."""
    from delta_amd import tuning
    A, B = _wall_touching_particle()
    if swap:
        A, B = B, A
    tuning.set(detect_max_tiles=max_tiles, detect_queue_min_items=0 if queue else 1 << 30)
    try:
        got = contact.bf(*shapes.to_soa(A), len(A), EPS, True, 7, *shapes.to_soa(B), len(B),
                         EPS, True, 9)
    finally:
        tuning.set(**tuning.default())
    rc, want, _ = ol.or_detect(_lib.DH_BF, A, B, EPS, EPS, 1, 1, 7, 9)
    assert rc == 0 and len(want) > 0
    same_contacts(got, want)


def _facing_lines(n):
    """n triangles on a line, 1 cm apart, and n beside them: every 4,001st within
    the margin, the others 1 m away."""
    rng = np.random.default_rng(9)
    tri = rng.uniform(-1e-3, 1e-3, (3, 3))
    at = 1e-2 * np.arange(n)[:, None, None] * np.array([1.0, 0.0, 0.0])
    A, B = tri + at, tri + at + np.array([0.0, 1.0, 0.0])
    B[::4001, :, 1] -= 1.0 - 5e-5
    return A, B


@pytest.mark.parametrize("n", [46341, 65537])
def test_penalty_over_more_pairs_than_32_bits_number(n):
    """n x n triangles are more than 2^31 (2^32) pairs: the contacts are those
    of A called part by part, in order, and come from every tile."""
    A, B = _facing_lines(n)
    contact.reset_all_statistics()
    got = contact.penalty(*shapes.to_soa(A), n, EPS, True, 7, *shapes.to_soa(B), n, EPS, True, 9)
    assert contact._stats.pairs_evaluated == n * n
    want = []
    for lo in range(0, n, 16384):
        a = A[lo:lo + 16384]
        w = contact.penalty(*shapes.to_soa(a), len(a), EPS, True, 7, *shapes.to_soa(B), n, EPS,
                            True, 9).copy()
        w["triA"] += lo
        want.append(w)
    same_contacts(got, np.concatenate(want))
    assert set(range(0, n, 4001)) <= set(got["triB"].tolist())


@pytest.mark.parametrize("n", [233015, 233016])
def test_largest_particles_through_pinned_memory(n):
    """The last pair of particles that is staged in pinned memory (16 MiB with
    its header) and the first that is copied: the oracle's contacts, and a
    small call after them."""
    A, _ = _facing_lines(n)
    B = A[n // 2:n // 2 + 1] + np.array([0.0, 5e-5, 0.0])
    for a in (A, A[n // 2 - 3:n // 2 + 3]):
        got = contact.bf(*shapes.to_soa(a), len(a), EPS, True, 7, *shapes.to_soa(B), 1, EPS, True, 9)
        rc, want, _ = ol.or_detect(_lib.DH_BF, a, B, EPS, EPS, 1, 1, 7, 9)
        assert rc == 0 and len(want) > 0
        same_contacts(got, want)
