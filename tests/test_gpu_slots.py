"""Operator slots laid out again and again in kept memory: the product after slots of other
sizes came and went, and after single tensors were replaced, is the one of a new context."""
import threading

import numpy as np
import pytest

import chemps2_amd
from chemps2_amd.problems import mx_table, random_abinitio

pytestmark = pytest.mark.gpu

IRR, T, V = random_abinitio(8, 3, group=0)
MX = mx_table(T, V, 8)
LEFT = [(2, 0), (2, 2), (3, 1), (3, 3), (4, 0), (4, 2)]
RIGHT = [(4, 0), (4, 2), (5, 1), (5, 3), (6, 0), (6, 2)]


def problem(c):
    c.set_problem(8, 0, IRR, 8, 0, 0, MX)


def product(c, d, replaced=False):
    c.set_sectors(3, [(n, s, 0, d + q) for q, (n, s) in enumerate(LEFT)])
    c.set_sectors(4, [(4, 0, 0, 1)])
    c.set_sectors(5, [(n, s, 0, d + q) for q, (n, s) in enumerate(RIGHT)])
    c.fill_synthetic(2, 1, 5)
    c.fill_synthetic(4, 0, 6)
    if replaced:  # a tensor of its own memory in the place of one of the slot's
        n = sum((d + a) * (d + b) for a, (na, sa) in enumerate(LEFT) for b, (nb, sb) in enumerate(LEFT)
                if nb == na + 1 and abs(sb - sa) == 1)
        c.upload(2, 1, "L", 0, 0, 1, 1, int(IRR[2]), np.linspace(-1, 1, n))
    n = c.prepare(3)
    return c.apply(np.random.default_rng(d).normal(size=n))


def test_relaid_slots(tmp_path):
    sizes = [3, 20, 4, 33, 3, 20, 2, 21, 60, 5]
    ref = {}
    for d in sorted(set(sizes)):
        for r in (False, True):
            c = chemps2_amd.Context(0)
            problem(c)
            ref[d, r] = product(c, d, r)
            c.close()
    bad = []

    def run(shift):
        c = chemps2_amd.Context(0)
        problem(c)
        for q, d in enumerate(sizes[shift:] + sizes[:shift]):
            r = q % 3 == 1
            if not np.array_equal(product(c, d, r), ref[d, r]):
                bad.append((shift, d, r))
            if q == 5:
                problem(c)
        c.close()

    print("one context, then two threads", flush=True)
    run(0)
    threads = [threading.Thread(target=run, args=(s,)) for s in (2, 5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
