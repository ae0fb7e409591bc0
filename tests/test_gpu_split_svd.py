"""Split's decompositions at the sizes where its kernels change: panels of 16 columns, the
Jacobi sweeps of one launch up to 32 columns and rounds of pairs of 16-column blocks above,
wide and tall sectors, rank deficiency, and the sectors longer than a panel in LDS. That
the own kernels did it, and not the rocSOLVER call that repeats a sector without convergence,
is read from the context's counters. One left and one right sector, so that all three
centre sectors are a x b matrices of the test's choosing."""
import numpy as np
import pytest
import torch

import chemps2_amd
from chemps2_amd.problems import hubbard, mx_table

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 40), (15, 16), (16, 15), (17, 33), (40, 40), (64, 64), (64, 70), (65, 64), (65, 65), (80, 66),
         (97, 130), (200, 190), (257, 130), (600, 610), (1024, 24), (700, 1024), (1030, 5)]
TALL = [(1025, 1), (17, 1025), (1030, 50), (1537, 250), (256, 2049), (4096, 31)]


def own(a, b):
    """The sector is within the limits of the own kernels."""
    return max(a, b) <= 1024 or (max(a, b) <= 4096 and min(a, b) <= 256)


@pytest.mark.parametrize("rank", [None, 0.4])
@pytest.mark.parametrize("a,b", SIZES + TALL)
def test_split_decompositions(a, b, rank):
    L, N, st = 8, 6, 3
    T, V = hubbard(L, U=3.0)
    ctx = chemps2_amd.Context(0)
    try:
        ctx.set_problem(L, 0, np.zeros(L, dtype=np.int32), N, 0, 0, mx_table(T, V, N))
        ctx.set_sectors_auto(10 ** 6)
        ctx.set_sectors(st, [(2, 0, 0, a)])
        ctx.set_sectors(st + 2, [(4, 0, 0, b)])
        ctx.set_sectors(st + 1, [(2, 0, 0, 1), (3, 1, 0, 1), (4, 0, 0, 1)])
        for q in (st, st + 1):
            ctx.mps_upload(q, np.ones(ctx.mps_layout_size(q)))
        # blocks (n1, n2, 2J): (0, 2, 0), (1, 1, 0), (1, 1, 2) (uncoupled: zero), (2, 0, 0)
        assert ctx.join(st) == 4 * a * b
        rng = np.random.default_rng(a * 1000 + b)
        n = min(a, b)
        parts = []
        for _ in range(3):  # rows and columns falling over seven decades in all
            m = rng.normal(size=(a, b)) * np.outer(10.0 ** (-3.5 * np.arange(a) / a), 10.0 ** (-3.5 * np.arange(b) / b))
            if rank is not None:
                r = max(1, int(rank * n))
                m = m[:, :r] @ rng.normal(size=(r, b))
            parts.append(m.T.ravel())
        x = np.concatenate(parts[:2] + [np.zeros(a * b)] + parts[2:])
        x /= np.linalg.norm(x)
        print(f"case {a} x {b} rank {rank}", flush=True)
        ctx.s_set(x)
        assert ctx.split(st, 10 ** 6, moving_right=True) == 0.0
        left, right = ctx.mps_download(st), ctx.mps_download(st + 1)
        ctx.join(st)
        # backward error and loss of orthogonality: n rotations per column and sweep, each
        # of relative error eps, and as many reflections
        tol = 10 * max(n, 4) * 2.0 ** -53
        assert np.linalg.norm(ctx.s_get() - x) <= tol
        for q in range(3):
            u = left[q * a * n:(q + 1) * a * n].reshape(n, a)
            assert np.abs(u @ u.T - np.eye(n)).max() <= tol
            w = right[q * n * b:(q + 1) * n * b].reshape(b, n)  # rows of W: sigma v
            sigma = np.linalg.norm(w, axis=0)
            ref = np.linalg.svd(parts[q].reshape(b, a), compute_uv=False)
            ref *= np.linalg.norm(sigma) / np.linalg.norm(ref)
            assert np.abs(sigma - ref).max() <= tol * ref[0]
            assert np.abs(w.T @ w - np.diag(sigma ** 2)).max() <= tol * ref[0] ** 2
        # the other side: sigma on the left tensor, the right one orthonormal by rows
        ctx.s_set(x)
        ctx.split(st, 10 ** 6, moving_right=False)
        right = ctx.mps_download(st + 1)
        for q, two_sm in enumerate((0, 1, 0)):
            v = right[q * n * b:(q + 1) * n * b].reshape(b, n) / np.sqrt(two_sm + 1.0)
            assert np.abs(v.T @ v - np.eye(n)).max() <= tol
    finally:
        ctx.close()


def boundaries(ctx, a, b):
    """The three centre sectors of site 3 as a x b matrices."""
    T, V = hubbard(8, U=3.0)
    ctx.set_problem(8, 0, np.zeros(8, dtype=np.int32), 6, 0, 0, mx_table(T, V, 6))
    ctx.set_sectors_auto(10 ** 6)
    ctx.set_sectors(3, [(2, 0, 0, a)])
    ctx.set_sectors(5, [(4, 0, 0, b)])
    ctx.set_sectors(4, [(2, 0, 0, 1), (3, 1, 0, 1), (4, 0, 0, 1)])
    for q in (3, 4):
        ctx.mps_upload(q, np.ones(ctx.mps_layout_size(q)))
    ctx.join(3)


def graded(a, b, seed, rank=None):
    """Centre matrices whose rows and columns fall over seven decades, and the object."""
    rng = np.random.default_rng(seed)
    parts = [rng.normal(size=(a, b)) * np.outer(10.0 ** (-3.5 * np.arange(a) / a), 10.0 ** (-3.5 * np.arange(b) / b))
             for _ in range(3)]
    if rank is not None:
        r = max(1, int(rank * min(a, b)))
        parts = [m[:, :r] @ rng.normal(size=(r, b)) for m in parts]
    x = np.concatenate([parts[0].ravel("F"), parts[1].ravel("F"), np.zeros(a * b), parts[2].ravel("F")])
    return parts, x / np.linalg.norm(x)


def sides(ctx, a, b):
    """(U, W = sigma V^T) of the three sectors after a Split to the right."""
    n = min(a, b)
    left, right = ctx.mps_download(3), ctx.mps_download(4)
    return [(left[q * a * n:(q + 1) * a * n].reshape(n, a).T, right[q * n * b:(q + 1) * n * b].reshape(b, n).T)
            for q in range(3)]


@pytest.mark.parametrize("scale", ["flat", "graded"])
@pytest.mark.parametrize("a,b", SIZES + TALL)
def test_singular_vectors_orthonormal(a, b, scale):
    # A column goes through n reflectors and some 10 n rotations, each of which rounds it by half
    # a unit in the last place of its elements: a random walk of sqrt(11 n) such steps, of 0.5 x
    # 2^-53 of its norm, twice in U^T U, for each of the n columns: 3.3 n 2^-53 in all where no
    # rounding is systematic. The re-joined object, whose parts have their share of the norm:
    # sqrt(11 n) of them.
    print(f"case {a} x {b} {scale}", flush=True)
    n = min(a, b)
    parts, x = graded(a, b, 5 * a + b)
    if scale == "flat":
        rng = np.random.default_rng(5 * a + b)
        x = np.concatenate([rng.normal(size=2 * a * b), np.zeros(a * b), rng.normal(size=a * b)])
        x /= np.linalg.norm(x)
    ctx = chemps2_amd.Context(0)
    try:
        boundaries(ctx, a, b)
        ctx.s_set(x)
        ctx.split(3, 10 ** 6, moving_right=True)
        us = [u for u, _ in sides(ctx, a, b)]
        ctx.join(3)
        error = np.linalg.norm(ctx.s_get() - x)
        ctx.s_set(x)
        ctx.split(3, 10 ** 6, moving_right=False)
        vs = [w.T / np.sqrt(q % 2 + 1.0) for q, (_, w) in enumerate(sides(ctx, a, b))]
        loss = max(np.linalg.norm(m.T @ m - np.eye(n)) for m in us + vs) * 2.0 ** 53
        print(f"  {loss / n:.2f} n, {error * 2.0 ** 53 / np.sqrt(n):.2f} sqrt(n) units", flush=True)
        assert loss <= 6 * max(n, 2)
        assert error * 2.0 ** 53 <= 2 * np.sqrt(11 * max(n, 2))
    finally:
        ctx.close()


@pytest.mark.parametrize("n", [2, 3, 5, 8])
def test_small_sectors_stop_at_the_rounding_floor(n):
    # the sweeps end with no pair of columns above sqrt(n) 2^-53; normalising them adds a rounding
    # of half a unit to each element
    print(f"case {n} x {n}", flush=True)
    worst = 0.0
    ctx = chemps2_amd.Context(0)
    try:
        boundaries(ctx, n, n)
        for seed in range(60):
            if seed > 0:
                ctx.join(3)
            x = np.random.default_rng(seed).normal(size=4 * n * n)
            x[2 * n * n:3 * n * n] = 0.0
            ctx.s_set(x)
            ctx.split(3, 10 ** 6, moving_right=False)
            for q, (_, w) in enumerate(sides(ctx, n, n)):
                v = (w / np.sqrt(q % 2 + 1.0)).astype(np.longdouble)
                worst = max(worst, float(np.abs(np.triu(v @ v.T, 1)).max()) * 2.0 ** 53)
        print(f"  {worst:.2f} units", flush=True)
        assert worst <= np.sqrt(n) + 1.5
    finally:
        ctx.close()


@pytest.mark.parametrize("scale", [1e-90, 1e-159, 1e-290, 1e90, 1e160])
@pytest.mark.parametrize("a,b", [(6, 6), (24, 40), (70, 50)])
def test_sectors_of_any_magnitude(a, b, scale):
    # a sector far from order one, whose norms to the second or fourth power leave the range of
    # doubles, beside two of order one
    print(f"case {a} x {b} scale {scale}", flush=True)
    n = min(a, b)
    _, x = graded(a, b, a + b)
    x[:a * b] *= scale
    ctx = chemps2_amd.Context(0)
    try:
        boundaries(ctx, a, b)
        ctx.s_set(x)
        ctx.split(3, 10 ** 6, moving_right=True)
        assert ctx.split_stats() == (3, 0, 0)
        tol = 10 * n * 2.0 ** -53
        for u, _ in sides(ctx, a, b):
            assert np.abs(u.T @ u - np.eye(n)).max() <= tol
        ctx.join(3)
        for got, ref in zip(ctx.s_get().reshape(4, -1), x.reshape(4, -1)):
            big = np.abs(ref).max() or 1.0
            assert np.linalg.norm(got / big - ref / big) <= tol * np.linalg.norm(ref / big)
    finally:
        ctx.close()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("a,b", [(6, 6), (24, 40), (70, 50)])
def test_sector_without_finite_values(a, b, bad):
    # such a sector counts as zero: sigma = 0 and orthonormal vectors; the others are untouched
    print(f"case {a} x {b} {bad}", flush=True)
    n = min(a, b)
    _, x = graded(a, b, a + b)
    y = x.copy()
    y[a * b // 2] = bad
    ctx = chemps2_amd.Context(0)
    try:
        boundaries(ctx, a, b)
        ctx.s_set(y)
        ctx.split(3, 10 ** 6, moving_right=True)
        assert ctx.split_stats() == (3, 0, 0)
        tol = 10 * n * 2.0 ** -53
        for u, _ in sides(ctx, a, b):
            assert np.abs(u.T @ u - np.eye(n)).max() <= tol
        assert not sides(ctx, a, b)[0][1].any()
        ctx.join(3)
        assert np.linalg.norm(ctx.s_get()[a * b:] - x[a * b:]) <= tol
    finally:
        ctx.close()


@pytest.mark.parametrize("rank", [None, 0.4])
@pytest.mark.parametrize("a,b", SIZES + TALL + [(1025, 257), (4097, 3)])
def test_own_kernels_converge(a, b, rank):
    print(f"case {a} x {b} rank {rank}", flush=True)
    ctx = chemps2_amd.Context(0)
    try:
        boundaries(ctx, a, b)
        ctx.s_set(graded(a, b, 1000 * a + b, rank)[1])
        ctx.split(3, 10 ** 6, moving_right=True)
        assert ctx.split_stats() == ((3, 0, 0) if own(a, b) else (0, 3, 0))
    finally:
        ctx.close()


@pytest.mark.parametrize("a,b", [(20, 30), (33, 40), (97, 130)])
def test_sectors_without_convergence(monkeypatch, a, b):
    # one sweep: up to 32 columns the kernel's own flag, above them the counters of the rounds
    # say that the last sweep still rotated
    print(f"case {a} x {b}, one sweep", flush=True)
    monkeypatch.setenv("CHM_SVD_MAX_SWEEPS", "1")
    ctx = chemps2_amd.Context(0)
    try:
        boundaries(ctx, a, b)
        x = graded(a, b, a + b)[1]
        ctx.s_set(x)
        ctx.split(3, 10 ** 6, moving_right=True)
        assert ctx.split_stats() == (3, 0, 3)
        n = min(a, b)
        tol = 10 * n * 2.0 ** -53
        for u, _ in sides(ctx, a, b):
            assert np.abs(u.T @ u - np.eye(n)).max() <= tol
        ctx.join(3)
        assert np.linalg.norm(ctx.s_get() - x) <= tol
    finally:
        ctx.close()


def test_large_workspaces_are_given_back():
    # the matrices of a dozen sectors of up to some 1000 x 1000 take more than the 128 MB that
    # stay with the context
    left = [(1, 1), (2, 0), (2, 2), (3, 1), (3, 3), (4, 0), (4, 2), (5, 1)]
    right = [(3, 1), (4, 0), (4, 2), (5, 1), (5, 3), (6, 0), (6, 2), (7, 1)]
    d = 250
    T, V = hubbard(8, U=3.0)
    ctx = chemps2_amd.Context(0)
    try:
        ctx.set_problem(8, 0, np.zeros(8, dtype=np.int32), 8, 0, 0, mx_table(T, V, 8))
        ctx.set_sectors_auto(10 ** 6)
        ctx.set_sectors(3, [(n, s, 0, d) for n, s in left])
        ctx.set_sectors(5, [(n, s, 0, d) for n, s in right])
        ctx.set_sectors(4, [(n, s, 0, 1) for n in range(1, 8) for s in range(n % 2, 5, 2)])
        for q in (3, 4):
            ctx.mps_upload(q, np.ones(ctx.mps_layout_size(q)))
        ctx.join(3)
        # the first Split allocates the tensors of its dimensions and drops what its sectors lack
        ctx.s_set(np.random.default_rng(3).normal(size=ctx.s_get().size))
        ctx.split(3, 10 ** 6, moving_right=True)
        ctx.join(3)
        x = ctx.s_get() / np.linalg.norm(ctx.s_get())
        ctx.s_set(x)
        ctx.split(3, 10 ** 6, moving_right=True)
        free = torch.cuda.mem_get_info(0)[0]
        ctx.join(3)
        assert np.linalg.norm(ctx.s_get() - x) <= 1e-13
        n = sum(min(sum(d for a, t in left if 0 <= m - a <= 2 and abs(t - s) == (m - a) % 2),
                    sum(d for a, t in right if 0 <= a - m <= 2 and abs(t - s) == (a - m) % 2)) ** 2
                for m in range(1, 8) for s in range(m % 2, 5, 2))
        print(f"sectors of {n} elements in all", flush=True)
        assert 6 * 8 * n > 128 << 20
        tensors = 8 * sum(ctx.mps_layout_size(q) for q in (3, 4))
        ctx.close()
        held = torch.cuda.mem_get_info(0)[0] - free
        print(f"held {held >> 20} MiB, tensors {tensors >> 20} MiB, object {x.nbytes >> 20} MiB", flush=True)
        # the tensors, the object and the join's lists besides, and the math library's own
        assert held <= tensors + 4 * x.nbytes + (128 << 20)
    finally:
        ctx.close()
