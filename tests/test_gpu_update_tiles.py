"""Operator updates at block dimensions around the edges of the 16 x 16, 32 x 32 and 64 x 64
tiles. Every block is a scalar times u v^T with a unit vector for each sector, so an update of
any dimensions is the update of the scalars (all dimensions 1), times the same u v^T."""
import re

import numpy as np
import pytest

import chemps2_amd
from chemps2_amd.problems import mx_table, random_abinitio
from plancheck import oracle_tensors

pytestmark = pytest.mark.gpu

L, G = 8, 0
LEFT = [(2, 0), (2, 2), (3, 1), (3, 3), (4, 0), (4, 2)]   # (N, 2S) at boundary 3
RIGHT = [(3, 1), (4, 0), (4, 2), (5, 1), (5, 3), (6, 2)]  # and at boundary 4


def op_blocks(sec, two_j, n_elec):
    for n, s in sec:
        for sd in range(s - two_j, s + two_j + 1, 2):
            if (n + n_elec, sd) in sec:
                yield (n, s), (n + n_elec, sd)


def mps_blocks():
    for n, s in LEFT:
        for nr in range(n, n + 3):
            tj = 1 if nr == n + 1 else 0
            for sr in range(s - tj, s + tj + 1, 2):
                if (nr, sr) in RIGHT:
                    yield (n, s), (nr, sr)


def spread(scalars, blocks, uv):
    """The packed tensor (column-major blocks) of the scalars."""
    return np.concatenate([np.outer(uv[a], uv[b]).ravel("F") * x for (a, b), x in zip(blocks, scalars)] or [np.zeros(0)])


@pytest.fixture(scope="module")
def shapes(oracle_lib):
    irr, T, V = random_abinitio(L, 4, group=G)
    o = oracle_lib.OracleDMRG(L, G, irr, 8, 0, 0, T, V)
    o.init(14, 4)
    right = {i: [(kd, k, m, int(t[1]), int(t[2]), int(t[3])) for kd, k, m, t, _ in oracle_tensors(o, i)] for i in (2, 3)}
    o.sweep_left_to(1, 14, rtol=1e-4)  # slots 2 and 3 now hold right operators
    left = {i: [(kd, k, m, int(t[1]), int(t[2]), int(t[3])) for kd, k, m, t, _ in oracle_tensors(o, i)] for i in (2, 3)}
    return o.irreps(), o.mx(), {True: right, False: left}


def update(shapes, mr, dims, uv, scalars):
    irr, mx, sh = shapes
    prev, new = (2, 3) if mr else (3, 2)
    sec = {2: LEFT, 3: RIGHT}  # slot i lies at boundary i + 1
    c = chemps2_amd.Context(0)
    try:
        c.set_problem(L, G, irr, 8, 0, 0, mx)
        c.set_sectors(3, [(n, s, 0, dims["l", n, s]) for n, s in LEFT])
        c.set_sectors(4, [(n, s, 0, dims["r", n, s]) for n, s in RIGHT])
        side = {2: {q: uv["l", q[0], q[1]] for q in LEFT}, 3: {q: uv["r", q[0], q[1]] for q in RIGHT}}
        for q, (kd, k, m, tj, ne, ni) in enumerate(sh[mr][prev]):
            bl = list(op_blocks(sec[prev], tj, ne))
            c.upload(prev, mr, kd, k, m, tj, ne, ni, spread(scalars["op"][q], bl, side[prev]))
        bl = list(mps_blocks())
        out = [np.outer(side[2][a], side[3][b]).ravel("F") * x for (a, b), x in zip(bl, scalars["mps"])]
        c.mps_upload(3, np.concatenate(out))
        c.update_operators(new, mr)
        got = []
        for kd, k, m, tj, ne, ni in sh[mr][new]:
            bl = list(op_blocks(sec[new], tj, ne))
            n = sum(side[new][a].size * side[new][b].size for a, b in bl)
            got.append((bl, c.tensor_download(new, kd, k, m, n) if n else np.zeros(0)))
        return got, side[new]
    finally:
        c.close()


@pytest.mark.parametrize("env", [None, ("CHM_TILE_WIDE_MIN", "0"), ("CHM_TILES_MFMA", "1"), ("CHM_TILES_MFMA", "0")])
@pytest.mark.parametrize("sizes", [(3, 17, 5), (33, 48, 16), (65, 5, 97)])
def test_update_in_workgroup_tiles(monkeypatch, capfd, shapes, sizes, env):
    # the tiles for blocks of any number of elements, and the older kernels on request, take all of
    # the output; by default the blocks of at most 32 x 32 are on wavefronts
    monkeypatch.setenv("CHM_VERBOSE", "1")
    if env:
        monkeypatch.setenv(*env)
    test_update_of_rank_one_blocks(shapes, sizes, True)
    waves = [int(n) for n in re.findall(r"(\d+) of the output's on wavefronts", capfd.readouterr().err)]
    assert waves and (not any(waves) if env else all(waves))


@pytest.mark.parametrize("mr", [True, False])
@pytest.mark.parametrize("sizes", [(1, 2, 17), (15, 16, 33), (31, 32, 9), (33, 48, 16), (63, 64, 31), (65, 5, 97), (128, 64, 129)])
def test_update_of_rank_one_blocks(shapes, sizes, mr):
    print(f"case sizes {sizes} moving_right {mr}", flush=True)
    rng = np.random.default_rng(2)
    keys = [("l", n, s) for n, s in LEFT] + [("r", n, s) for n, s in RIGHT]
    prev = 2 if mr else 3
    scalars = {"op": [rng.normal(size=len(list(op_blocks(LEFT if mr else RIGHT, t[3], t[4])))) for t in shapes[2][mr][prev]],
               "mps": rng.normal(size=len(list(mps_blocks())))}
    ref, _ = update(shapes, mr, {k: 1 for k in keys}, {k: np.ones(1) for k in keys}, scalars)
    dims = {k: sizes[(q + q // 3) % 3] for q, k in enumerate(keys)}
    uv = {k: rng.normal(size=d) for k, d in dims.items()}
    uv = {k: v / np.linalg.norm(v) for k, v in uv.items()}
    got, side = update(shapes, mr, dims, uv, scalars)
    scale = max(np.abs(s).max(initial=0) for _, s in ref)
    seen = 0
    for (bl, s), (_, g) in zip(ref, got):
        # two inner products of up to 129 elements each: an error below 2 * 129 * 2^-53 of every
        # term (2.9e-14), of some ten terms no larger than the largest sum
        assert g.shape == spread(s, bl, side).shape
        assert np.abs(g - spread(s, bl, side)).max(initial=0) <= 3e-13 * scale
        seen += g.size > 0
    assert seen > 30


@pytest.mark.parametrize("rows,cols", [(128, 40), (80, 24)])
def test_blocks_of_more_than_four_gigabytes(rows, cols):
    # Join of a left block of more than 2^29 elements, whose last columns alone are not zero: byte
    # offsets beyond 32 bits, in tiles of 64 x 40, 64 x 24 and 16 x 24
    mid = 2 ** 29 // rows + 48
    print(f"case {rows} x {mid} x {cols}", flush=True)
    c = chemps2_amd.Context(0)
    try:
        irr, T, V = random_abinitio(L, 4, group=G)
        c.set_problem(L, G, irr, 8, 0, 0, mx_table(T, V, 8))
        c.set_sectors(3, [(2, 0, 0, rows)])
        c.set_sectors(4, [(3, 1, 0, mid)])
        c.set_sectors(5, [(4, 0, 0, cols)])
        rng = np.random.default_rng(rows)
        a, b = rng.normal(size=(rows, 48)), rng.normal(size=(48, cols))
        assert c.mps_layout_size(3) == rows * mid and c.mps_layout_size(4) == mid * cols
        left = np.zeros(rows * mid)
        left[-rows * 48:] = a.ravel("F")
        c.mps_upload(3, left)
        del left
        right = np.zeros((cols, mid))
        right[:, -48:] = b.T
        c.mps_upload(4, right.ravel())
        del right
        c.join(3)
        got = c.s_get()
        ref = a @ b
        blocks = [g.reshape(cols, rows).T for g in got.reshape(-1, rows * cols) if np.abs(g).max() > 0]
        assert blocks
        for g in blocks:  # each a recoupling factor times the product; 48 terms a sum
            f = np.vdot(g, ref) / np.vdot(ref, ref)
            assert abs(f) > 0.1
            assert np.abs(g - f * ref).max() <= 48 * 2.0 ** -52 * abs(f) * np.abs(ref).max()
    finally:
        c.close()
