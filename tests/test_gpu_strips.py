"""Long lists of chained terms (shared intermediates, the cheaper association, the input block
in LDS) against one intermediate per term in the reference's order, at block dimensions
around the tile edges and the limit of the inner dimension, and in several batches of
intermediates."""
import os

import numpy as np
import pytest

import chemps2_amd
from chemps2_amd.problems import mx_table, random_abinitio

pytestmark = pytest.mark.gpu

LEFT = [(2, 0), (2, 2), (3, 1), (3, 3), (4, 0), (4, 2)]   # (N, 2S) at the left boundary
RIGHT = [(4, 0), (4, 2), (5, 1), (5, 3), (6, 0), (6, 2)]


def product(dims, x, share, w_cap=None, **more):
    env = {"CHM_TILE_SHARE_MIN": str(share), "CHM_EXPLICIT_MAX": "1", **more}
    if w_cap:
        env["CHM_TILE_W_CAP"] = str(w_cap)
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        ctx = chemps2_amd.Context(0)
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v
    try:
        irr, T, V = random_abinitio(8, 3, group=0)
        ctx.set_problem(8, 0, irr, 8, 0, 0, mx_table(T, V, 8))
        ctx.set_sectors(3, [(n, s, 0, dims[q % len(dims)]) for q, (n, s) in enumerate(LEFT)])
        ctx.set_sectors(4, [(4, 0, 0, 1)])
        ctx.set_sectors(5, [(n, s, 0, dims[(q + 2) % len(dims)]) for q, (n, s) in enumerate(RIGHT)])
        ctx.fill_synthetic(2, 1, 5)
        ctx.fill_synthetic(4, 0, 6)
        n = ctx.prepare(3)
        x = np.random.default_rng(1).normal(size=n) if x is None else x
        return x, ctx.apply(x), ctx.plan_stats()
    finally:
        ctx.close()


@pytest.mark.parametrize("dims", [(1, 2, 3), (15, 16, 17), (31, 5, 33), (48, 64, 49), (65, 80, 63), (97, 112, 9),
                                  (127, 128, 129), (140, 20, 128)])
def test_long_lists_equal_short_lists(dims):
    print(f"case dims {dims}", flush=True)
    x, y0, s0 = product(dims, None, 10 ** 9)
    _, y1, s1 = product(dims, x, 1)
    _, y2, _ = product(dims, x, 1, w_cap=s1["W_doubles"] // 3 + 1)
    assert s0["chain_terms"] == s1["chain_terms"] > 0 and s1["tiles1"] > 0
    assert s1["W_doubles"] < s0["W_doubles"]
    # the same products of inner dimension up to 140 summed in other orders over up to some
    # thousand terms per element: errors of 2^-53 each, as a random walk
    assert np.abs(y1 - y0).max() <= 64 * 2.0 ** -53 * np.sqrt(s0["chain_terms"]) * np.abs(y0).max()
    assert np.abs(y2 - y0).max() <= 64 * 2.0 ** -53 * np.sqrt(s0["chain_terms"]) * np.abs(y0).max()


@pytest.mark.parametrize("share", [1, 10 ** 9])
@pytest.mark.parametrize("dims", [(1, 2, 3), (31, 5, 33), (65, 80, 63)])
def test_tiles_for_blocks_of_any_size(dims, share):
    # with 64-bit offsets, as for blocks of 2^28 elements and more
    print(f"case dims {dims} share {share}", flush=True)
    x, y0, s0 = product(dims, None, 10 ** 9)
    _, y1, s1 = product(dims, x, share, CHM_TILE_WIDE_MIN="0")
    assert s1["chain_terms"] == s0["chain_terms"] > 0
    assert np.abs(y1 - y0).max() <= 64 * 2.0 ** -53 * np.sqrt(s0["chain_terms"]) * np.abs(y0).max()
