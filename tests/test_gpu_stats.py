"""sph_stats_noalloc of two contexts from two threads at once: each gets its own
maxima, bit for bit those of sph_stats, at sizes of one workgroup and many."""
import threading

import numpy as np
import pytest

import cases
import urbansph

pytestmark = pytest.mark.gpu


def _stepped(nf, sigma_u):
    P, _ = cases.box(nf=nf, walls=3, sigma_u=sigma_u)
    c = urbansph.Case(cases.box_params(urbansph.default_params(), tol=1e-6), len(P))
    c.upload(P)
    c.step(0, 1e-4)
    c.sync()
    return c


def test_contexts_do_not_share_the_working_memory():
    cs = [_stepped(20, 0.3), _stepped(12, 0.01)]
    ref = [np.array(c.stats(), np.float32).view(np.uint32) for c in cs]
    assert (ref[0] != ref[1]).any()
    print("[stats] two threads", flush=True)
    bad = []

    def loop(k):
        for _ in range(300):
            got = np.array(cs[k].stats_noalloc(), np.float32).view(np.uint32)
            if not np.array_equal(got, ref[k]):
                bad.append((k, got))
                return

    ts = [threading.Thread(target=loop, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not any(t.is_alive() for t in ts) and not bad, bad


def test_one_workgroup_and_a_remainder():
    for n in (1, 255, 256, 257):
        P, _ = cases.box(nf=6, walls=3)
        prm = cases.box_params(urbansph.default_params())
        prm.update(ppe_solver=0)
        c = urbansph.Case(prm, n + 300)   # room for more than the case has
        c.upload(P[-n:].copy())
        c.step(0, 1e-6)
        np.testing.assert_array_equal(np.array(c.stats_noalloc(), np.float32), np.array(c.stats(), np.float32))
        c.close()
