"""The DEM step with its survivor queue solved by the learned narrow phase
(DH_BF_LEARNED) against the brute-force step (DH_BF) and the oracle: the
learned decision returns bfSolver's points bit for bit, so contacts, forces
and every state array must be identical, eager and captured."""
import numpy as np
import pytest

import oracle_lib as ol
from delta_amd import _lib, engine, learn
from delta_amd.device import DeviceArray
from test_gpu_engine import STATE, compare, sincos_branch_used

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def network():
    """A network trained briefly on the lattice's own triangle pairs (the
    results do not depend on its quality, only the share it finishes)."""
    soa = learn.c1_pairs(1 << 18, seed=6)
    ds = learn.Dataset(DeviceArray.from_host(soa), soa.shape[1])
    tr = learn.Trainer(seed=0)
    tr.fit(ds, epochs=3, batch=8192, lr=3e-3)
    tr.install()
    return tr


def _scene(name):
    if name == "c1":
        return engine.c1_scene()
    if name.startswith("drum-"):
        # the rotating box's meshes on a lattice tighter than the largest
        # particles, so that some pairs are in contact from the first step
        from delta_amd import workloads
        return workloads.drum_scene(n=int(name.split("-")[1]), pitch=1.3e-3)
    from delta_amd import scene_io
    return scene_io.hopper_scene(num=int(name.split("-")[1]), sphere_level=1)


def _params(hs, method, name):
    if name.startswith("hopper"):
        return engine.step_params(method=method, dt=1e-6, gravity=(0.0, 0.0, -10.0), spring=1e6,
                                  damper=0.1, friction=0.0, cell=hs.cell_size())
    dt = 5e-7 if name.startswith("drum") else 1e-6
    return engine.step_params(method=method, dt=dt, spring=1e5, damper=0.1, friction=0.0,
                              cell=hs.cell_size())


@pytest.mark.parametrize("name", ["c1", "hopper-6", "drum-3000"])
def test_learned_step_equals_brute_force_step(network, name):
    """Eager steps with DH_BF_LEARNED and with DH_BF on two copies: the same
    counts and every state array bit for bit after each step."""
    hs = _scene(name)
    a = engine.DeviceScene(hs)
    b = engine.DeviceScene(hs)
    pl = _params(hs, _lib.DH_BF_LEARNED, name)
    pb = _params(hs, _lib.DH_BF, name)
    total = 0
    for s in range(4):
        ia = engine.step(a, pl)
        ib = engine.step(b, pb)
        assert (ia.candidate_pairs, ia.contacts, ia.triangle_checks) == \
            (ib.candidate_pairs, ib.contacts, ib.triangle_checks), (name, s)
        total += ia.contacts
        for f in STATE:
            assert np.array_equal(a.download(f).view(np.uint64), b.download(f).view(np.uint64)), \
                (name, s, f)
    assert total > 0, name


def test_learned_step_matches_oracle(network):
    """The C1 lattice's first steps (where its contacts are) against the
    oracle's brute-force step: counts exact, states bitwise while expmap stays
    in its series branch, else to 1e-10 (device vs host libm)."""
    hs = engine.c1_scene()
    ds = engine.DeviceScene(hs)
    p = _params(hs, _lib.DH_BF_LEARNED, "c1")
    for s in range(3):
        info = engine.step(ds, p)
        nc, checks, npairs = ol.or_step(hs, _lib.DH_BF, 1e5, 0.1, 0.0, 1e-6, (0.0, -9.81, 0.0))
        assert (info.contacts, info.candidate_pairs, info.triangle_checks) == (nc, npairs, checks)
        compare(ds, hs, s, exact=not sincos_branch_used(hs, 1e-6), rtol=1e-10)


@pytest.mark.parametrize("name", ["c1", "drum-2000"])
def test_learned_step_graph_equals_eager(network, name):
    """The captured learned step replayed against eager learned steps: the
    lattice (a full queue) and a rotating box of 2,000 particles (its wall
    pairs culled before the queue, which stays short against its capacity:
    the network and brute-force passes stop at the live entries)."""
    hs = _scene(name)
    de = engine.DeviceScene(hs)
    dg = engine.DeviceScene(hs)
    p = _params(hs, _lib.DH_BF_LEARNED, name)
    info0 = engine.step(engine.DeviceScene(hs), p)
    _lib.check(_lib.lib().dh_synchronize(), "sync")
    # the box's contacts grow over the steps: room for all of them
    g = engine.StepGraph(dg, p, pair_cap=max(4096, 2 * info0.candidate_pairs + 1024),
                         contact_cap=1 << 16 if name == "c1" else 1 << 20)
    try:
        for s in range(5):
            info = engine.step(de, p)
            _lib.check(_lib.lib().dh_synchronize(), "sync")
            g.launch()
            ginfo, overflow = g.status()
            assert overflow == 0
            assert (ginfo.candidate_pairs, ginfo.contacts) == (info.candidate_pairs, info.contacts)
            for f in STATE:
                assert np.array_equal(de.download(f).view(np.uint64),
                                      dg.download(f).view(np.uint64)), (s, f)
    finally:
        g.close()


@pytest.mark.parametrize("method", [_lib.DH_BF, _lib.DH_BF_LEARNED])
@pytest.mark.parametrize("captured", [False, True])
def test_step_with_more_survivors_than_the_queue(network, method, captured):
    """125 icospheres pushed into one another with hardly a margin: several
    survivors per contact, more than the queue's segments and pool hold and,
    for some pairs, than an item may queue.  The states are those of the brute
    force without the queue, bit for bit."""
    from delta_amd import shapes, tuning
    rs, rr = shapes.Rng(21), shapes.Rng(22)
    at = np.stack(np.meshgrid(*[np.arange(5)] * 3, indexing="ij"), -1).reshape(-1, 3)
    meshes = [shapes.jittered_icosphere(1, 0.5e-3, 0.1, rs) @ shapes.random_rotation(rr).T
              + 0.35e-3 * c for c in at]
    hs = engine.HostScene(meshes, 1e-9, 0, np.arange(len(meshes)), 2500.0, 0)
    prm = lambda m: engine.step_params(method=m, dt=1e-8, spring=1.0, damper=0.1, friction=0.0,
                                       cell=hs.cell_size())
    want, got = engine.DeviceScene(hs), engine.DeviceScene(hs)
    try:
        tuning.set(detect_queue_min_items=1 << 30)
        infos = [engine.step(want, prm(_lib.DH_BF)) for _ in range(3)]
        tuning.set(detect_queue_min_items=0, detect_max_tiles=1)
        info = infos[0]
        held = max(16 * 2 * info.candidate_pairs + 65536, 5 * (info.contacts + 1024) // 2)
        assert info.triangle_checks - info.pairs_culled > held
        if captured:
            g = engine.StepGraph(got, prm(method), pair_cap=info.candidate_pairs + 64,
                                 contact_cap=info.contacts + 1024)
            try:
                for i in infos:
                    g.launch()
                    s, overflow = g.status()
                    assert overflow == 0
                    assert (s.candidate_pairs, s.contacts) == (i.candidate_pairs, i.contacts)
            finally:
                g.close()
        else:
            for i in infos:
                s = engine.step(got, prm(method))
                assert (s.candidate_pairs, s.contacts) == (i.candidate_pairs, i.contacts)
    finally:
        tuning.set(**tuning.default())
    for f in STATE:
        assert np.array_equal(want.download(f).view(np.uint64), got.download(f).view(np.uint64)), f
