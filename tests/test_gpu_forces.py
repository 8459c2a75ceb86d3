"""dh_contacts_forces over lists whose pairs carry very different numbers of
contacts, bit for bit against the oracle's per-pair sums added in ascending
partner order.  The lists cross the sizes where the device code changes its
split: pairs with none, one, a wave's worth and several waves of contacts,
short and long pair lists, few and many particles.  (What a captured step adds
up after it ran out of contact capacity is not defined, only that it stays
within its buffers: tests of the step graph.)"""
import ctypes as C
import types

import numpy as np
import pytest

import oracle_lib as ol
from delta_amd import _lib, contact
from delta_amd.device import DeviceArray

pytestmark = pytest.mark.gpu


def scene(n, rng):
    hs = types.SimpleNamespace(n=n)
    hs.pos = rng.normal(0, 1, (n, 3))
    hs.linvel = rng.normal(0, 1, (n, 3))
    hs.angvel = rng.normal(0, 1, (n, 3))
    hs.mass = rng.uniform(1, 2, n)
    hs.mass[0] = np.inf
    hs.obstacle = np.zeros(n, np.int32)
    hs.obstacle[0] = 1
    return hs


def contacts(counts, rng):
    c = np.zeros(int(counts.sum()), contact.CONTACT_DTYPE)
    c["x"] = rng.normal(0, 1, (len(c), 3))
    v = rng.normal(0, 1, (len(c), 3))
    c["normal"] = v / np.linalg.norm(v, axis=1)[:, None]
    c["depth"] = rng.uniform(-1e-3, 1e-3, len(c))
    c["friction"] = rng.integers(0, 2, len(c))
    c["normal"][::17, 1] = -0.0
    return c


@pytest.mark.parametrize("n,npairs,many", [(40, 1, False), (40, 301, True), (1500, 301, True),
                                           (1500, 131072, False), (1500, 131073, True),
                                           (1025, 131130, False)])
def test_pair_sums(n, npairs, many):
    rng = np.random.default_rng(n + npairs)
    hs = scene(n, rng)
    i, j = np.triu_indices(n, 1)
    sel = np.sort(rng.permutation(len(i))[:npairs])
    pairs = np.stack([i[sel], j[sel]], 1).astype(np.int32)
    assert len(pairs) == npairs
    counts = rng.choice([0, 0, 1, 2, 5], npairs)
    counts[rng.permutation(npairs)[3000:]] = 0
    if many:
        at = rng.permutation(npairs)[:6]
        counts[at] = [63, 64, 65, 127, 200, 1]
        counts[0], counts[-1] = 70, 64
    cs = contacts(counts, rng)
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    by_pair = [cs[offs[k]:offs[k + 1]] for k in range(npairs)]
    up = DeviceArray.from_host
    d = {f: up(getattr(hs, f)) for f in ("pos", "linvel", "angvel", "mass", "obstacle")}
    z9 = up(np.zeros((n, 9)))
    bodies = _lib.DhBodies(d["pos"].ptr, d["pos"].ptr, d["linvel"].ptr, d["angvel"].ptr,
                           d["angvel"].ptr, z9.ptr, z9.ptr, z9.ptr, d["mass"].ptr,
                           d["obstacle"].ptr, d["obstacle"].ptr, n)
    dc = up(cs.view(np.uint8)) if len(cs) else DeviceArray((144,), np.uint8)
    dp, do = up(pairs), up(offs)
    F, T = DeviceArray((n, 3), np.float64), DeviceArray((n, 3), np.float64)
    t = DeviceArray((n,), np.int32)
    fp = _lib.DhForceParams(1e4, 0.3, 0.5, 0)
    L = _lib.lib()
    L.dh_contacts_forces.argtypes = [C.POINTER(_lib.DhBodies), C.c_void_p, C.c_int, C.c_void_p,
                                     C.c_void_p, C.POINTER(_lib.DhForceParams), C.c_void_p,
                                     C.c_void_p, C.c_void_p, C.c_void_p]
    for _ in range(2):  # the second call on the buffers of the first
        _lib.check(L.dh_contacts_forces(C.byref(bodies), dp.ptr, npairs, dc.ptr, do.ptr,
                                        C.byref(fp), F.ptr, T.ptr, t.ptr, None), "forces")
    fo, to, tch = ol.or_forces_scene(hs, [tuple(p) for p in pairs], by_pair, 1e4, 0.3, 0.5)
    assert np.array_equal(t.download(), tch)
    assert np.array_equal(F.download().view(np.uint64), np.ascontiguousarray(fo).view(np.uint64))
    assert np.array_equal(T.download().view(np.uint64), np.ascontiguousarray(to).view(np.uint64))
