"""The explicit sector matrix against chained products, at sub-block sizes on both sides of the
assembly's choices (one, two or eight elements a thread) with ragged rests."""
import os

import numpy as np
import pytest

import chemps2_amd
from chemps2_amd.problems import mx_table, random_abinitio

pytestmark = pytest.mark.gpu

LEFT = [(2, 0), (2, 2), (3, 1), (3, 3), (4, 0), (4, 2)]   # (N, 2S) at the left boundary
RIGHT = [(4, 0), (4, 2), (5, 1), (5, 3), (6, 0), (6, 2)]


def product(dims, explicit, mixed=False):
    old = os.environ.get("CHM_EXPLICIT_MAX")
    os.environ["CHM_EXPLICIT_MAX"] = explicit
    try:
        c = chemps2_amd.Context(0)
    finally:
        if old is None:
            del os.environ["CHM_EXPLICIT_MAX"]
        else:
            os.environ["CHM_EXPLICIT_MAX"] = old
    try:
        irr, T, V = random_abinitio(8, 3, group=0)
        c.set_problem(8, 0, irr, 8, 0, 0, mx_table(T, V, 8))
        c.set_sectors(3, [(n, s, 0, dims[0] + q % 2) for q, (n, s) in enumerate(LEFT)])
        c.set_sectors(4, [(4, 0, 0, 1)])
        c.set_sectors(5, [(n, s, 0, dims[1] + q % 3) for q, (n, s) in enumerate(RIGHT)])
        c.fill_synthetic(2, 1, 5)
        c.fill_synthetic(4, 0, 6)
        if mixed:
            c.set_heff_form(chemps2_amd.FORM_MIXED)
        n = c.prepare(3)
        return c.apply(np.random.default_rng(1).normal(size=n)), c.plan_stats()
    finally:
        c.close()


@pytest.mark.parametrize("dims", [(1, 1), (1, 7), (7, 1), (3, 5), (4, 6), (5, 9), (8, 6), (13, 2), (2, 17), (15, 4)])
def test_explicit_equals_chained(dims):
    print(f"case dims {dims}", flush=True)
    y0, s0 = product(dims, "0")
    y1, s1 = product(dims, "100000000")
    y2, _ = product(dims, "100000000", mixed=True)
    assert s1["explicit_pairs"] > 0 and s1["chain_terms"] < max(s0["chain_terms"], 1)
    # FP64 sums of the same products in another order; hi + lo is each element to 2^-48
    assert np.abs(y1 - y0).max() <= 1e-12 * np.abs(y0).max()
    assert np.abs(y2 - y0).max() <= 1e-12 * np.abs(y0).max()
