"""Renders from several threads at once: each the image that it makes alone."""
import threading

import numpy as np
import pytest

from flam3_amd import genome as G
from flam3_amd.serve import Server

pytestmark = pytest.mark.gpu


def _jobs():
    """Calls of every kind and of different sizes."""
    out = []
    for s in range(12):
        if s % 4 == 0:
            out.append((G.synthetic_preview(s, size=64 + 16 * s, quality=20.0), {}))
        elif s % 4 == 1:
            out.append((G.synthetic_animation(seed=s, width=100 + s, height=60, quality=20.0, supersample=1,
                                              temporal_samples=20), {"time": 3.0}))
        elif s % 4 == 2:
            out.append((G.synthetic_8k(seed=s, width=90, height=60 + s, quality=20.0, supersample=1), {"bits": 64}))
        else:
            out.append((G.synthetic_small(seed=s, width=200, height=100 + s, quality=60.0), {"bits": 32}))
    return out


def _same(a, b):
    return np.array_equal(a, b) or (a.shape == b.shape and np.abs(a.astype(int) - b).max() <= 1)


def test_renders_of_several_threads(prod):
    """Threads with a render call each, one with render_many and one with a
    server, over the same genomes.  (Sums of doubles round by the order of the
    deposits: a count of one at bits 64.)"""
    jobs = _jobs()
    want = [prod.render(g, seed=str(i), **kw) for i, (g, kw) in enumerate(jobs)]
    bad = []

    def check(i, img, st):
        ok = _same(img, want[i][0]) if jobs[i][1].get("bits") == 64 else np.array_equal(img, want[i][0])
        if not ok or st["badvals"] != want[i][1]["badvals"]:
            bad.append(i)

    def single(t):
        try:
            for r in range(3):
                for i in range(t, len(jobs), 3):
                    k = (i + r) % len(jobs)
                    check(k, *prod.render(jobs[k][0], seed=str(k), **jobs[k][1]))
        except Exception as e:
            bad.append(e)

    def many():
        try:
            for _ in range(3):
                r = prod.render_many([dict(kw, genomes=g, seed=str(i)) for i, (g, kw) in enumerate(jobs)])
                for i, x in enumerate(r):
                    check(i, *x)
        except Exception as e:
            bad.append(e)

    def served():
        try:
            s = Server()
            for _ in range(3):
                ts = [s.submit(g, seed=str(i), **kw) for i, (g, kw) in enumerate(jobs)]
                for i, t in enumerate(ts):
                    check(i, *s.wait(t)[:2])
            s.close()
        except Exception as e:
            bad.append(e)

    threads = [threading.Thread(target=single, args=(t,)) for t in range(3)]
    threads += [threading.Thread(target=many), threading.Thread(target=served)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_servers_beside_each_other(prod):
    """Three servers at once, whose groups pass through the same download slots."""
    items = [{"genomes": G.synthetic_preview(s, size=64 + 32 * (s % 5), quality=10.0), "seed": str(s)} for s in range(30)]
    want = [prod.render(it["genomes"], seed=it["seed"])[0] for it in items]
    bad = []

    def served(order):
        try:
            s = Server(max_batch=3)
            for _ in range(3):
                ts = [(i, s.submit(**items[i])) for i in order]
                for i, t in ts:
                    if not np.array_equal(s.wait(t)[0], want[i]):
                        bad.append(i)
            s.close()
        except Exception as e:
            bad.append(e)

    n = range(len(items))
    threads = [threading.Thread(target=served, args=(o,)) for o in (list(n), list(n)[::-1], list(n)[15:] + list(n)[:15])]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
