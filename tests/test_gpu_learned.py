"""The learned narrow phase on the GPU: network forward and gradient against
the numpy restatement, training, and its results against the oracle's
bfSolver: P, Q and d bit for bit on every pair (generated, ragged and
degenerate), whatever the network predicts."""
import ctypes as C

import numpy as np
import pytest

import mlp_ref
import oracle_lib as ol
from delta_amd import _lib, learn, narrow
from delta_amd.device import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def train_set():
    b = narrow.PairBatch(1 << 20, seed=11)
    return b, learn.Dataset(b.soa, b.n)


def test_forward_matches_numpy(train_set):
    _, ds = train_set
    tr = learn.Trainer(seed=4)
    out = tr.forward(ds, 4096)
    X = ds.X.download()[:4096]
    ref = mlp_ref.forward(learn.init_params(4), X)[4]
    assert np.allclose(out[:, :20], ref[:, :20], rtol=2e-2, atol=2e-2)
    assert np.median(np.abs(out[:, :20] - ref[:, :20])) < 1e-4


def test_gradient_matches_numpy(train_set):
    _, ds = train_set
    tr = learn.Trainer(seed=5)
    g, loss = tr.grad_at(ds, 128, 1024)
    X = ds.X.download()[128:1152]
    feat = ds.feat.download()[128:1152].astype(np.int64)
    bary = ds.bary.download()[128:1152]
    flag = ds.flag.download()[128:1152]
    lref, gref = mlp_ref.loss_and_grad(learn.init_params(5), X, feat, bary, flag)
    assert loss == pytest.approx(lref, rel=1e-3)
    rel = np.linalg.norm(g - gref) / np.linalg.norm(gref)
    assert rel < 1e-2, rel
    for lo, hi in ((learn.W1, learn.B1), (learn.W2, learn.B2), (learn.W3, learn.B3),
                   (learn.B3, learn.N_PARAMS)):
        seg = np.linalg.norm(g[lo:hi] - gref[lo:hi]) / (np.linalg.norm(gref[lo:hi]) + 1e-30)
        assert seg < 3e-2, (lo, seg)


@pytest.mark.parametrize("batch", [1, 15, 16, 17, 127, 128, 129, 1000, 256 * 128 + 77])
def test_gradient_across_batch_sizes(batch, train_set):
    """Partial 16-pair tiles and 128-pair chunks, several workgroups, and more
    chunks than workgroups, from an odd first pair.  bf16 operands (2^-8 each,
    rounded at other sums) bound the relative difference as above."""
    _, ds = train_set
    tr = learn.Trainer(seed=5)
    first = 61
    assert ds.n >= first + batch
    g, loss = tr.grad_at(ds, first, batch)
    rows = slice(first, first + batch)
    lref, gref = mlp_ref.loss_and_grad(learn.init_params(5), ds.X.download()[rows],
                                       ds.feat.download()[rows].astype(np.int64),
                                       ds.bary.download()[rows], ds.flag.download()[rows])
    assert loss == pytest.approx(lref, rel=1e-3)
    assert np.linalg.norm(g - gref) < 1e-2 * np.linalg.norm(gref)


def run_learned(batch, method="learned"):
    batch.run(method)
    L = _lib.lib()
    cnt = _lib.DhPairCounters()
    _lib.check(L.dh_tri_pairs_counters(C.byref(cnt)), "counters")
    return batch.results(), cnt


def oracle_bf(batch):
    """The oracle's bfSolver (CPU restatement of bf.cpp:217-1178, no
    threads) on the batch's own pairs: P, Q, d."""
    soa = np.ascontiguousarray(batch.soa.download())
    n = soa.shape[1]
    P = np.zeros((3, n)); Q = np.zeros((3, n)); d = np.zeros(n)
    rc = ol.oracle().or_tri_pairs(0, ol.dptr(soa), C.c_int64(n), C.c_double(2e-4), ol.dptr(P),
                                  ol.dptr(Q), ol.dptr(d), None)
    assert rc == 0
    return P, Q, d


def assert_bits(a, b, what):
    eq = np.ascontiguousarray(a).view(np.uint64) == np.ascontiguousarray(b).view(np.uint64)
    if not eq.all():
        bad = np.argwhere(~eq)[:5]
        raise AssertionError(f"{what}: {int((~eq).sum())} of {eq.size} differ, e.g. {bad.tolist()}")


def fp64_features_per_pair(cnt, n):
    """FP64 feature evaluations per pair: the learned path's own (2 per
    pair, plus ties) and the brute force's 15 for every queued pair."""
    return (cnt.features_fp64 + 15 * cnt.rechecked) / n


def test_trained_network_matches_oracle_bit_for_bit(train_set):
    """Every pair's P, Q and d equal the oracle's bfSolver bit for bit,
    certified or not (so the contact points, normals and the contact set are
    the reference's); the trained network finishes most pairs itself."""
    _, ds = train_set
    tr = learn.Trainer(seed=0)
    l0 = tr.grad_at(ds, 0, 8192)[1]
    tr.fit(ds, epochs=6, batch=4096, lr=3e-3)
    l1 = tr.grad_at(ds, 0, 8192)[1]
    assert l1 < 0.5 * l0
    test = narrow.PairBatch(1 << 16, seed=3)
    P0, Q0, d0 = oracle_bf(test)
    tr.install()
    (P, Q, d, flags), cnt = run_learned(test)
    assert_bits(P, P0, "P")
    assert_bits(Q, Q0, "Q")
    assert_bits(d, d0, "d")
    cert = (flags & 8) != 0
    assert cnt.certified == cert.sum() and cnt.rechecked == (~cert).sum()
    # measured 0.82 after these 6 epochs (the certificate requires the
    # network's feature to be bfSolver's own choice)
    assert cert.mean() > 0.7, cert.mean()


def test_network_gain_over_brute_force(train_set):
    """What the trained network buys: FP64 feature evaluations per pair
    against the brute force's 15, and against the same path with an
    untrained network (whose wrong predictions fall back to the brute
    force).  Results are bfSolver's in all three."""
    _, ds = train_set
    test = narrow.PairBatch(1 << 16, seed=5)
    P0, Q0, d0 = oracle_bf(test)
    tr = learn.Trainer(seed=0)
    tr.fit(ds, epochs=6, batch=4096, lr=3e-3)
    tr.install()
    (P, Q, d, _), cnt = run_learned(test)
    assert_bits(d, d0, "d trained")
    trained = fp64_features_per_pair(cnt, test.n)
    un = learn.Trainer(seed=0)
    un.install()
    (Pu, Qu, du, _), cnt_u = run_learned(test)
    assert_bits(Pu, P0, "P untrained")
    assert_bits(du, d0, "d untrained")
    untrained = fp64_features_per_pair(cnt_u, test.n)
    tr.install()
    # measured: about 6.4 for the trained network (the near-parallel 5% go
    # to the brute force's 15), 12-15 untrained
    assert trained < 8.0, (trained, untrained)
    assert trained < 0.6 * untrained, (trained, untrained)


@pytest.mark.parametrize("n", [1, 63, 65, 5000, 100003])
def test_learned_ragged_sizes(train_set, n):
    """Sizes that leave partial chunks, partial workgroups and a single pair:
    every result equal to the oracle's bit for bit, and the per-workgroup
    tallies add up to n."""
    _, ds = train_set
    tr = learn.Trainer(seed=0)
    tr.fit(ds, epochs=1, batch=8192, lr=3e-3)
    tr.install()
    test = narrow.PairBatch(n, seed=29)
    P0, Q0, d0 = oracle_bf(test)
    (P, Q, d, flags), cnt = run_learned(test)
    assert ((flags & 8) != 0).sum() + ((flags & 2) != 0).sum() == n
    assert cnt.certified + cnt.rechecked == n
    assert_bits(P, P0, "P")
    assert_bits(Q, Q0, "Q")
    assert_bits(d, d0, "d")


def test_learned_degenerate_pairs(train_set):
    """Ties and degenerate pairs built by hand: a vertex against a vertex, a
    vertex against an edge, parallel edges, parallel faces (a segment or an
    area of closest points), touching and intersecting triangles: bit for bit
    equal to the oracle."""
    import scenes
    tr = learn.Trainer(seed=0)
    tr.fit(train_set[1], epochs=1, batch=8192, lr=3e-3)
    tr.install()
    soa = scenes.degenerate_pairs()
    test = narrow.PairBatch.from_host(soa)
    P0, Q0, d0 = oracle_bf(test)
    (P, Q, d, _), _ = run_learned(test)
    assert_bits(P, P0, "P")
    assert_bits(Q, Q0, "Q")
    assert_bits(d, d0, "d")


def test_network_warm_start_of_the_penalty_newton(train_set):
    """DH_PAIR_LEARNED_PENALTY starts the penalty Newton iteration from the
    network's barycentric outputs; DH_PAIR_PENALTY_CERT from the reference's
    0.33.  Both certify or fall back, so both are correct.  The network's
    start is far closer to the solution's barycentric parameters than 0.33
    (held-out pairs, against the brute force's labels); the Newton step
    count barely follows, because the penalty schedule (three steps at the
    first regularisation, then x1e5 per step until the relative step is
    below 1e-20) sets it: the trained start needs slightly fewer steps and
    certifies at least as many pairs."""
    _, ds = train_set
    tr = learn.Trainer(seed=0)
    tr.fit(ds, epochs=6, batch=4096, lr=3e-3)
    tr.install()
    test = narrow.PairBatch(1 << 16, seed=3)
    held = learn.Dataset(test.soa, test.n)
    guess = tr.forward(held)[:, 16:20]
    truth = held.bary.download()
    err_net = np.abs(guess - truth).mean()
    err_033 = np.abs(0.33 - truth).mean()
    # measured: mean absolute error 0.19 from the network against 0.32 from 0.33
    assert err_net < 0.75 * err_033, (err_net, err_033)
    test.run("bf64")
    _, _, d0, _ = test.results()
    stats = {}
    for m in ("learned_penalty", "penalty_cert"):
        test.run(m)
        L = _lib.lib()
        cnt = _lib.DhPairCounters()
        _lib.check(L.dh_tri_pairs_counters(C.byref(cnt)), "counters")
        _, _, d, fl = test.results()
        cert = (fl & 8) != 0
        assert (np.abs(d - d0) / d0).max() <= 1e-6
        assert np.array_equal(d[~cert].view(np.uint64), d0[~cert].view(np.uint64))
        assert cnt.certified == cert.sum() and cnt.rechecked == (~cert).sum()
        stats[m] = (cnt.features_fp64 / test.n, cert.mean())
    (its_w, cert_w), (its_c, cert_c) = stats["learned_penalty"], stats["penalty_cert"]
    assert its_w < its_c, stats
    assert cert_w >= cert_c, stats
