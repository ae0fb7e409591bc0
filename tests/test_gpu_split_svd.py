"""Split's decompositions at the sizes where its kernels change: panels of 16 columns, the
one-workgroup Jacobi up to 64 columns, blocked rounds above it (block width 16, then
narrower as the columns get longer), wide and tall sectors, rank deficiency, and the
sectors longer than the in-house limit. One left and one right sector, so that all three
centre sectors are a x b matrices of the test's choosing."""
import numpy as np
import pytest

import chemps2_amd
from chemps2_amd.problems import hubbard, mx_table

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 40), (15, 16), (16, 15), (17, 33), (40, 40), (64, 64), (64, 70), (65, 64), (65, 65), (80, 66),
         (97, 130), (200, 190), (257, 130), (600, 610), (1024, 24), (700, 1024), (1030, 5)]


@pytest.mark.parametrize("rank", [None, 0.4])
@pytest.mark.parametrize("a,b", SIZES)
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
