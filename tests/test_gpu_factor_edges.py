"""The batched inverse factor at the edges of its tiles, panels and workgroup pairs (GPU)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _recurrence(V, lo, up):
    """inverse diagonal blocks of the elimination from both ends towards the middle block, in FP64 (NumPy)"""
    n = len(V)
    m = (n - 1) // 2
    inv = [None] * n
    for i in list(range(m)) + list(range(n - 1, m, -1)) + [m]:
        M = V[i].copy()
        if 0 < i <= m:
            M -= lo[i - 1][:, None] * inv[i - 1] * up[i - 1][None, :]
        if m <= i < n - 1:
            M -= up[i][:, None] * inv[i + 1] * lo[i][None, :]
        inv[i] = np.linalg.inv(M)
    return inv


def _factor(sizes, bs, values, precision):
    import torch
    from spitfire_amd import _native
    dev = torch.device('cuda:0')
    nb = np.asarray(sizes)
    voff = np.cumsum([0] + [v.size for v in values])[:-1].astype(np.int64)
    doff = np.cumsum(np.r_[0, nb * bs * bs])[:-1].astype(np.int64)
    V = torch.tensor(np.concatenate(values), device=dev)
    D = torch.zeros(int((nb * bs * bs).sum()), device=dev,
                    dtype=torch.float64 if precision == 64 else torch.float32)
    t = [torch.tensor(a, device=dev) for a in (nb.astype(np.int32), voff, doff)]
    _native.check(_native.lib().gf_batch_btddod_inverse_factorize(
        len(sizes), t[0].data_ptr(), bs, V.data_ptr(), t[1].data_ptr(), D.data_ptr(), t[2].data_ptr(), precision,
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    d = D.cpu().numpy().astype(np.float64)
    return [d[doff[s]:doff[s] + nb[s] * bs * bs].reshape(nb[s], bs, bs).transpose(0, 2, 1) for s in range(len(sizes))]


@pytest.mark.parametrize('precision', [64, 32])
@pytest.mark.parametrize('bs', [7, 8, 9, 15, 16, 17, 32, 33, 47, 48, 49, 56, 57, 63, 64])
def test_inverse_factor_tile_edges(bs, precision):
    """Block sizes around the panels of 8 and tiles of 16; 515 systems, so that one-block systems share workgroups
    (two that are 256 apart), some with a longer system in the partner's place and the last ones without a
    partner. Rows are scaled and permuted so that every pivot exchanges rows. Tolerance: growth of at most 4 (diagonal
    weights) times N eps cond, cond <= 100 for these blocks after row scaling."""
    rng = np.random.default_rng(bs)
    sizes = [1] * 515
    sizes[3], sizes[260], sizes[270], sizes[514] = 2, 3, 4, 5
    values, parts = [], []
    for n in sizes:
        V = rng.standard_normal((n, bs, bs)) + (4. + 2. * np.sqrt(bs)) * np.eye(bs)
        V = V[:, rng.permutation(bs)] * 10. ** rng.uniform(-1., 1., (n, bs, 1))
        lo, up = 0.1 * rng.standard_normal((n - 1, bs)), 0.1 * rng.standard_normal((n - 1, bs))
        parts.append((V, lo, up))
        values.append(np.concatenate([V.transpose(0, 2, 1).ravel(), lo.ravel(), up.ravel()]))
    got = _factor(sizes, bs, values, precision)
    tol = 4. * bs * 100. * (2.2e-16 if precision == 64 else 6.0e-8)
    for s in list(range(0, 515, 37)) + [3, 4, 259, 260, 14, 270, 256, 513, 514]:
        for a, b in zip(got[s], _recurrence(*parts[s])):
            assert np.max(np.abs(a - b)) <= tol * np.max(np.abs(b))


@pytest.mark.parametrize('bs', [10, 53])
def test_inverse_factor_of_singular_and_nonfinite_blocks(bs):
    """A zero block and a block with a NaN give no finite inverse, and leave the other systems alone."""
    rng = np.random.default_rng(1)
    blocks = [rng.standard_normal((1, bs, bs)) + 20. * np.eye(bs) for _ in range(4)]
    blocks[1] = np.zeros((1, bs, bs))
    blocks[2][0, bs // 2, 1] = np.nan
    got = _factor([1] * 4, bs, [b.transpose(0, 2, 1).ravel() for b in blocks], 64)
    assert not np.isfinite(got[1]).any() and not np.isfinite(got[2]).all()
    for s in (0, 3):
        assert np.max(np.abs(got[s][0] @ blocks[s][0] - np.eye(bs))) <= 1e-12


@pytest.mark.parametrize('precision', [64, 32])
@pytest.mark.parametrize('bs', [1, 2, 7, 8, 9, 11])
def test_inverse_factor_routes_are_bitwise_the_same(bs, precision):
    """Few systems go to the panel kernel, many small ones to the one-wave kernel: the same elimination, entry by entry,
    also where pivots tie, over chains long enough to permute rows and columns of a permuted block. Tolerance: none."""
    rng = np.random.default_rng(bs)
    sizes = [1, 2, 3, 6, 7, 1, 4]
    values = []
    for s, n in enumerate(sizes):
        V = rng.standard_normal(n * bs * bs) if s % 2 else rng.integers(-2, 3, n * bs * bs).astype(float)
        values.append(np.concatenate([V, rng.standard_normal(2 * (n - 1) * bs)]))
    few = _factor(sizes, bs, values, precision)
    many = _factor(sizes * 230, bs, values * 230, precision)  # 1,610 systems
    for s in range(len(sizes)):
        for k in (0, 229):
            a, b = few[s], many[s + k * len(sizes)]
            assert np.array_equal(np.isfinite(a), np.isfinite(b)) and np.array_equal(a[np.isfinite(a)], b[np.isfinite(b)])


@pytest.mark.parametrize('precision', [64, 32])
@pytest.mark.parametrize('bs', [1, 3, 4, 5, 13, 52, 53, 63, 64])
def test_inverse_solve_edges(bs, precision):
    """Block sizes around the four columns of a group and chains from one block to some more than the loads in flight, the
    right-hand side apart from and in place of the solution, against the dense system. Tolerance: the residual of a solve with
    diagonally dominant blocks, 100 N eps of the inverses' precision (FP64) times the norm, 10 times that for the chain."""
    import torch
    from spitfire_amd import _native
    rng = np.random.default_rng(bs)
    sizes = [1, 2, 3, 4, 5, 6, 9, 12] + [1] * 3
    values, dense, rhs = [], [], []
    for n in sizes:
        V = rng.standard_normal((n, bs, bs)) + (4. + 2. * np.sqrt(bs)) * np.eye(bs)
        lo, up = 0.1 * rng.standard_normal((n - 1, bs)), 0.1 * rng.standard_normal((n - 1, bs))
        values.append(np.concatenate([V.transpose(0, 2, 1).ravel(), lo.ravel(), up.ravel()]))
        A = np.zeros((n * bs, n * bs))
        for k in range(n):
            A[k * bs:(k + 1) * bs, k * bs:(k + 1) * bs] = V[k]
        for k in range(n - 1):
            A[(k + 1) * bs:(k + 2) * bs, k * bs:(k + 1) * bs] = np.diag(lo[k])
            A[k * bs:(k + 1) * bs, (k + 1) * bs:(k + 2) * bs] = np.diag(up[k])
        dense.append(A)
        rhs.append(rng.standard_normal(n * bs))
    dev = torch.device('cuda:0')
    nb = np.asarray(sizes)
    offsets = [np.cumsum(np.r_[0, a])[:-1].astype(np.int64) for a in ([v.size for v in values], nb * bs * bs, nb * bs)]
    V, b = (torch.tensor(np.concatenate(a), device=dev) for a in (values, rhs))
    D = torch.zeros(int((nb * bs * bs).sum()), device=dev, dtype=torch.float64 if precision == 64 else torch.float32)
    n, vo, do, xo = (torch.tensor(a, device=dev) for a in (nb.astype(np.int32), *offsets))
    x = torch.zeros_like(b)
    st = torch.cuda.current_stream().cuda_stream
    lib = _native.lib()
    _native.check(lib.gf_batch_btddod_inverse_factorize(len(sizes), n.data_ptr(), bs, V.data_ptr(), vo.data_ptr(),
                                                        D.data_ptr(), do.data_ptr(), precision, st))
    in_place = b.clone()
    for r, out in ((b, x), (in_place, in_place)):
        _native.check(lib.gf_batch_btddod_inverse_solve(len(sizes), n.data_ptr(), bs, V.data_ptr(), vo.data_ptr(),
                                                        D.data_ptr(), do.data_ptr(), precision, r.data_ptr(),
                                                        out.data_ptr(), xo.data_ptr(), st))
    assert torch.equal(x, in_place)
    got = x.cpu().numpy()
    tol = 1e3 * bs * (2.2e-16 if precision == 64 else 6.0e-8)
    for s in range(len(sizes)):
        g = got[offsets[2][s]:offsets[2][s] + nb[s] * bs]
        assert np.max(np.abs(dense[s] @ g - rhs[s])) <= tol * np.max(np.abs(rhs[s]))


@pytest.mark.parametrize('bs', [1, 2, 7, 8, 9, 53, 56, 57, 64])
def test_lapack_factor_and_solve_edges(bs):
    """Block sizes around the eight waves' columns, chains of one to five blocks, rows permuted so that pivots interchange and
    with exact ties (integer blocks): pivots equal to LAPACK's, factors, L blocks and solutions against NumPy. Tolerance: 100 N
    eps times the condition (at most 1e4 here) of the blocks, 10 times that for the chain."""
    import torch
    from scipy.linalg import lu_factor
    from spitfire_amd import _native
    rng = np.random.default_rng(bs)
    sizes = [1, 2, 5, 1, 3]
    parts, values, rhs = [], [], []
    for s, n in enumerate(sizes):
        V = rng.standard_normal((n, bs, bs)) if s % 2 else rng.integers(-1, 2, (n, bs, bs)).astype(float)
        V = (V + (2. + 2. * bs) * np.eye(bs))[:, rng.permutation(bs)]
        lo, up = 0.1 * rng.standard_normal((n - 1, bs)), 0.1 * rng.standard_normal((n - 1, bs))
        parts.append((V, lo, up))
        values.append(np.concatenate([V.transpose(0, 2, 1).ravel(), lo.ravel(), up.ravel()]))
        rhs.append(rng.standard_normal(n * bs))
    dev = torch.device('cuda:0')
    nb = np.asarray(sizes)
    offsets = [np.cumsum(np.r_[0, a])[:-1].astype(np.int64) for a in ([v.size for v in values], nb * bs * bs, nb * bs)]
    V, b = (torch.tensor(np.concatenate(a), device=dev) for a in (values, rhs))
    n, vo, lo, xo = (torch.tensor(a, device=dev) for a in (nb.astype(np.int32), *offsets))
    L = torch.zeros(int((nb * bs * bs).sum()), device=dev, dtype=torch.float64)
    P = torch.zeros(int((nb * bs).sum()), device=dev, dtype=torch.int32)
    x = torch.zeros_like(b)
    st = torch.cuda.current_stream().cuda_stream
    lib = _native.lib()
    _native.check(lib.gf_batch_btddod_full_factorize(len(sizes), n.data_ptr(), bs, V.data_ptr(), vo.data_ptr(), L.data_ptr(),
                                                     lo.data_ptr(), P.data_ptr(), xo.data_ptr(), st))
    _native.check(lib.gf_batch_btddod_full_solve(len(sizes), n.data_ptr(), bs, V.data_ptr(), vo.data_ptr(), L.data_ptr(),
                                                 lo.data_ptr(), P.data_ptr(), xo.data_ptr(), b.data_ptr(), x.data_ptr(),
                                                 xo.data_ptr(), st))
    v, l, p, g = (t.cpu().numpy() for t in (V, L, P, x))
    tol = 1e3 * bs * 2.2e-16 * 1e4
    for s, (B, sub, sup) in enumerate(parts):
        y, inv, A = None, None, None
        for i in range(sizes[s]):
            at = offsets[1][s] + i * bs * bs
            blk = lambda a, o: a[o:o + bs * bs].reshape(bs, bs).T
            D = B[i]
            if i > 0:
                Li = sub[i - 1][:, None] * inv
                assert np.max(np.abs(blk(l, at) - Li)) <= tol * np.max(np.abs(Li))
                D = D - Li * sup[i - 1][None, :]
            lu, piv = lu_factor(D)
            assert np.array_equal(p[offsets[2][s] + i * bs:offsets[2][s] + (i + 1) * bs], piv + 1)
            assert np.max(np.abs(blk(v, offsets[0][s] + i * bs * bs) - lu)) <= tol * np.max(np.abs(lu))
            inv = np.linalg.inv(D)
        xs = g[offsets[2][s]:offsets[2][s] + sizes[s] * bs].reshape(sizes[s], bs)
        r = np.einsum('nij,nj->ni', B, xs)
        if sizes[s] > 1:
            r[1:] += sub * xs[:-1]
            r[:-1] += sup * xs[1:]
        assert np.max(np.abs(r.ravel() - rhs[s])) <= tol * np.max(np.abs(rhs[s]))


@pytest.mark.parametrize('sizes', [[1], [3, 1], [1, 2, 1]])
@pytest.mark.parametrize('bs', [1, 8, 53, 64])
def test_lapack_solve_ends_on_a_one_block_system(bs, sizes):
    """A one-block system has no couplings, and as the last of its batch nothing behind its block. Tolerance: 1,000 N eps of the
    diagonally dominant systems' right-hand sides."""
    import torch
    from spitfire_amd import _native
    rng = np.random.default_rng(bs)
    values, dense, rhs = [], [], []
    for n in sizes:
        V = rng.standard_normal((n, bs, bs)) + (4. + 2. * bs) * np.eye(bs)
        lo, up = 0.1 * rng.standard_normal((n - 1, bs)), 0.1 * rng.standard_normal((n - 1, bs))
        values.append(np.concatenate([V.transpose(0, 2, 1).ravel(), lo.ravel(), up.ravel()]))
        A = np.zeros((n * bs, n * bs))
        for k in range(n):
            A[k * bs:(k + 1) * bs, k * bs:(k + 1) * bs] = V[k]
        for k in range(n - 1):
            A[(k + 1) * bs:(k + 2) * bs, k * bs:(k + 1) * bs] = np.diag(lo[k])
            A[k * bs:(k + 1) * bs, (k + 1) * bs:(k + 2) * bs] = np.diag(up[k])
        dense.append(A)
        rhs.append(rng.standard_normal(n * bs))
    dev = torch.device('cuda:0')
    nb = np.asarray(sizes)
    offsets = [np.cumsum(np.r_[0, a])[:-1].astype(np.int64) for a in ([v.size for v in values], nb * bs * bs, nb * bs)]
    V, b = (torch.tensor(np.concatenate(a), device=dev) for a in (values, rhs))
    n, vo, lo, xo = (torch.tensor(a, device=dev) for a in (nb.astype(np.int32), *offsets))
    L = torch.zeros(int((nb * bs * bs).sum()), device=dev, dtype=torch.float64)
    P = torch.zeros(int((nb * bs).sum()), device=dev, dtype=torch.int32)
    x = torch.zeros_like(b)
    st = torch.cuda.current_stream().cuda_stream
    lib = _native.lib()
    _native.check(lib.gf_batch_btddod_full_factorize(len(sizes), n.data_ptr(), bs, V.data_ptr(), vo.data_ptr(), L.data_ptr(),
                                                     lo.data_ptr(), P.data_ptr(), xo.data_ptr(), st))
    _native.check(lib.gf_batch_btddod_full_solve(len(sizes), n.data_ptr(), bs, V.data_ptr(), vo.data_ptr(), L.data_ptr(),
                                                 lo.data_ptr(), P.data_ptr(), xo.data_ptr(), b.data_ptr(), x.data_ptr(),
                                                 xo.data_ptr(), st))
    got = x.cpu().numpy()
    for s in range(len(sizes)):
        g = got[offsets[2][s]:offsets[2][s] + nb[s] * bs]
        assert np.max(np.abs(dense[s] @ g - rhs[s])) <= 1e3 * bs * 2.2e-16 * np.max(np.abs(rhs[s]))


def _plain_lu(A):
    """LAPACK's unblocked factors in place and the interchanges (0-based): only what lies beyond a pivot is touched"""
    n, piv = len(A), []
    for j in range(n):
        a = np.where(np.isnan(A[j:, j]), -1., np.abs(A[j:, j]))
        p = j + int(np.argmax(a))
        piv.append(p)
        A[[j, p]] = A[[p, j]]
        if A[j, j] != 0.:
            A[j + 1:, j] *= 1. / A[j, j]
        A[j + 1:, j + 1:] -= A[j + 1:, j, None] * A[None, j, j + 1:]
    return piv


def _plain_solve(A, piv, X):
    """X <- A^{-1} X in place with these factors, one division an entry"""
    for j, p in enumerate(piv):
        X[[j, p]] = X[[p, j]]
    for j in range(len(A)):
        X[j + 1:] -= A[j + 1:, j, None] * X[None, j]
    for j in reversed(range(len(A))):
        X[j] /= A[j, j]
        X[:j] -= A[:j, j, None] * X[None, j]


def _plain_system(V, lo, up, b):
    """factors, L blocks, pivots and solution of one system by the two above"""
    D, L, P, n = [], [None], [], len(V)
    for i in range(n):
        A = V[i].copy()
        if i > 0:
            X = np.eye(len(A))
            _plain_solve(D[-1], P[-1], X)
            L.append(lo[i - 1][:, None] * X)
            A -= L[-1] * up[i - 1][None, :]
        P.append(_plain_lu(A))
        D.append(A)
    y = [b[0].copy()]
    for i in range(1, n):
        t = b[i].copy()
        for c in range(len(t)):
            t -= L[i][:, c] * y[-1][c]
        y.append(t)
    x = [None] * n
    for i in reversed(range(n)):
        r = (y[i] - up[i] * x[i + 1] if i + 1 < n else y[i].copy())[:, None]
        _plain_solve(D[i], P[i], r)
        x[i] = r[:, 0]
    return D, L, P, x


def _alike(a, b, tol):
    """the same infinities and NaN, and finite entries within tol of the largest finite one"""
    a, b = np.asarray(a), np.asarray(b)
    f = np.isfinite(b)
    ok = np.array_equal(a[~f], b[~f], equal_nan=True) and np.isfinite(a[f]).all()
    return bool(ok and (not f.any() or np.max(np.abs(a[f] - b[f])) <= tol * np.max(np.abs(b[f]))))


@pytest.mark.parametrize('kind', ['zero column', 'infinity', 'two infinities', 'tiny pivot', 'huge pivot', 'infinite rhs'])
@pytest.mark.parametrize('bs', [2, 9, 53, 64])
def test_lapack_format_of_singular_and_extreme_blocks(bs, kind):
    """Singular blocks, infinities and pivots at the ends of the range, as the first, a middle, the last and the only block of a
    system, give what LAPACK's order of operations gives: the same infinities and NaN, and all else to rounding; ordinary systems
    beside them are what they are. Tolerance: 1,000 N eps, the blocks' growth and condition being below 10 except in the odd entry,
    times 100 for the chain."""
    import torch
    from spitfire_amd import _native
    rng = np.random.default_rng(bs)
    parts = []
    for n, at in ((1, 0), (4, 0), (4, 1), (3, 2), (2, -1), (1, -1)):
        V = rng.uniform(0.5, 1., (n, bs, bs)) * rng.choice([-1., 1.], (n, bs, bs)) + (4. + 2. * bs) * np.eye(bs)
        lo, up = rng.uniform(0.05, 0.1, (2, n - 1, bs))
        b = rng.uniform(0.5, 1., (n, bs))
        k = bs - 1 if kind == 'tiny pivot' else bs // 2  # (zeros below it times its reciprocal would be NaN)
        if at >= 0:
            if kind == 'zero column':
                V[at][:, k] = 0.
                if at > 0:
                    lo[at - 1][:] = 0.
            elif kind == 'infinity':
                V[at][k, bs - 1] = np.inf
            elif kind == 'two infinities':
                V[at][0, bs - 1], V[at][bs - 1, k] = np.inf, -np.inf
            elif kind == 'infinite rhs':
                b[at][k] = np.inf
            else:
                V[at][k], V[at][:, k] = 0., 0.
                V[at][k, k] = 1e-310 if kind == 'tiny pivot' else 1.7e308
                b[at][k] = 1e-310 if kind == 'tiny pivot' else 1e300
                if at > 0:
                    lo[at - 1][k] = up[at - 1][k] = 0.
                if at + 1 < n:
                    lo[at][k] = up[at][k] = 0.
        parts.append((V, lo, up, b))
    sizes = np.array([len(q[0]) for q in parts])
    values = [np.concatenate([V.transpose(0, 2, 1).ravel(), lo.ravel(), up.ravel()]) for V, lo, up, _ in parts]
    dev = torch.device('cuda:0')
    vo, do, xo = [np.cumsum(np.r_[0, a])[:-1].astype(np.int64) for a in ([v.size for v in values], sizes * bs * bs, sizes * bs)]
    V, b = torch.tensor(np.concatenate(values), device=dev), torch.tensor(np.concatenate([q[3].ravel() for q in parts]), device=dev)
    n, vt, dt, xt = (torch.tensor(a, device=dev) for a in (sizes.astype(np.int32), vo, do, xo))
    L = torch.zeros(int((sizes * bs * bs).sum()), device=dev, dtype=torch.float64)
    P = torch.zeros(int((sizes * bs).sum()), device=dev, dtype=torch.int32)
    x = torch.zeros_like(b)
    st = torch.cuda.current_stream().cuda_stream
    lib = _native.lib()
    _native.check(lib.gf_batch_btddod_full_factorize(len(sizes), n.data_ptr(), bs, V.data_ptr(), vt.data_ptr(), L.data_ptr(),
                                                     dt.data_ptr(), P.data_ptr(), xt.data_ptr(), st))
    _native.check(lib.gf_batch_btddod_full_solve(len(sizes), n.data_ptr(), bs, V.data_ptr(), vt.data_ptr(), L.data_ptr(),
                                                 dt.data_ptr(), P.data_ptr(), xt.data_ptr(), b.data_ptr(), x.data_ptr(),
                                                 xt.data_ptr(), st))
    v, l, p, g = (t.cpu().numpy() for t in (V, L, P, x))
    tol = 1e5 * bs * 2.2e-16
    with np.errstate(all='ignore'):
        for s, part in enumerate(parts):
            D, Lb, piv, xs = _plain_system(*part)
            for i in range(sizes[s]):
                at = do[s] + i * bs * bs
                assert _alike(v[vo[s] + i * bs * bs:vo[s] + (i + 1) * bs * bs].reshape(bs, bs).T, D[i], tol), (s, i)
                assert np.array_equal(p[xo[s] + i * bs:xo[s] + (i + 1) * bs] - 1, piv[i]), (s, i)
                if i > 0:
                    assert _alike(l[at:at + bs * bs].reshape(bs, bs).T, Lb[i], tol), (s, i)
                assert _alike(g[xo[s] + i * bs:xo[s] + (i + 1) * bs], xs[i], tol), (s, i)


@pytest.mark.parametrize('precision', [64, 32])
@pytest.mark.parametrize('bs', [16, 17, 20, 22, 23, 28, 29, 33, 48, 53, 64])
def test_one_block_systems_of_a_large_batch_are_bitwise_the_same(bs, precision):
    """In a large batch the one-block systems of these sizes have a kernel of their own; the inverses are those of a small batch,
    where they have not, entry by entry, and so are the longer systems' beside them. Tolerance: none."""
    rng = np.random.default_rng(bs)
    sizes = [1, 1, 3, 1, 2, 1, 1]
    values = []
    for s, n in enumerate(sizes):
        V = rng.standard_normal(n * bs * bs) if s % 2 else rng.integers(-2, 3, n * bs * bs).astype(float)
        values.append(np.concatenate([V, rng.standard_normal(2 * (n - 1) * bs)]))
    few = _factor(sizes, bs, values, precision)
    many = _factor(sizes * 600 + [1], bs, values * 600 + values[:1], precision)  # 4,201 systems: not whole workgroups
    for s in range(len(sizes)):
        for k in (0, 1, 599):
            assert np.array_equal(few[s], many[s + k * len(sizes)], equal_nan=True)
    assert np.array_equal(few[0], many[-1], equal_nan=True)


@pytest.fixture(scope='module')
def host_factor(tmp_path_factory):
    """inverse factors of one system, eliminated pivot by pivot on the host (tests/native/gauss_jordan_host.cpp)"""
    so = str(tmp_path_factory.mktemp('gauss_jordan') / 'libgj.so')
    subprocess.run(['g++', '-O2', '-std=c++17', '-ffp-contract=off', '-mfma', '-shared', '-fPIC', '-o', so,
                    os.path.join(os.path.dirname(os.path.abspath(__file__)), 'native', 'gauss_jordan_host.cpp')], check=True)
    lib = ctypes.CDLL(so)

    def factor(n, bs, values, precision):
        out = np.empty((n, bs, bs), dtype=np.float64 if precision == 64 else np.float32)
        v = np.ascontiguousarray(values)
        getattr(lib, 'inverse_factor_f%d' % precision)(n, bs, v.ctypes.data_as(ctypes.c_void_p),
                                                       out.ctypes.data_as(ctypes.c_void_p))
        return out.transpose(0, 2, 1).astype(np.float64)
    return factor


@pytest.mark.parametrize('precision', [64, 32])
@pytest.mark.parametrize('bs', [1, 4, 5, 8, 12, 16, 17, 31, 32, 33, 48, 49, 53, 57, 64])
def test_inverse_factor_is_bitwise_the_elimination_pivot_by_pivot(bs, precision, host_factor):
    """Whatever the panels and tiles: blocks of one to four tiles, random ones and integers whose pivots tie, alone, in chains that
    permute a permuted block's rows and columns, and one-block systems that share a workgroup (the batch of 300, where 256
    further on there is another one) against an independent elimination on the host. Tolerance: none."""
    rng = np.random.default_rng(100 + bs)
    for sizes in ([1, 2, 3, 4, 7, 1, 2], [1] * 300):
        values = []
        for s, n in enumerate(sizes):
            V = rng.standard_normal(n * bs * bs) if s % 2 else rng.integers(-3, 4, n * bs * bs).astype(float)
            values.append(np.concatenate([V, rng.standard_normal(2 * (n - 1) * bs)]))
        got = _factor(sizes, bs, values, precision)
        for s in list(range(7)) + ([255, 256, 257, 299] if len(sizes) > 7 else []):
            ref = host_factor(sizes[s], bs, values[s], precision)
            assert np.isfinite(ref).all() and np.array_equal(got[s], ref), (s, sizes[s])


@pytest.mark.parametrize('precision', [64, 32])
@pytest.mark.parametrize('bs', [17, 20, 21, 24, 31, 39, 40, 41])
def test_inverse_solve_of_few_and_many_systems_is_bitwise_the_same(bs, precision):
    """Few systems share each chain among four waves, many have a wave per chain (up to 40 unknowns): the same sums in the same order,
    for every remainder of four columns, chains from one block to some more than the loads in flight, the right-hand side apart
    from and in place of the solution. Tolerance: none."""
    import torch
    from spitfire_amd import _native
    rng = np.random.default_rng(bs)
    sizes = [1, 2, 3, 4, 5, 6, 9, 12]
    values = [rng.standard_normal(n * bs * bs + 2 * (n - 1) * bs) for n in sizes]
    inverses = [0.1 * rng.standard_normal(n * bs * bs) for n in sizes]
    rhs = [rng.standard_normal(n * bs) for n in sizes]
    dev, lib = torch.device('cuda:0'), _native.lib()
    st = torch.cuda.current_stream().cuda_stream
    got = []
    for copies in (1, 80):
        nb = np.asarray(sizes * copies)
        vo, do, xo = [torch.tensor(np.cumsum(np.r_[0, a])[:-1].astype(np.int64), device=dev)
                      for a in (nb * bs * bs + 2 * (nb - 1) * bs, nb * bs * bs, nb * bs)]
        V, D, b = (torch.tensor(np.tile(np.concatenate(a), copies), device=dev) for a in (values, inverses, rhs))
        D = D.to(torch.float64 if precision == 64 else torch.float32)
        n, x = torch.tensor(nb.astype(np.int32), device=dev), torch.full_like(b, 7.)
        in_place = b.clone()
        for r, out in ((b, x), (in_place, in_place)):
            _native.check(lib.gf_batch_btddod_inverse_solve(nb.size, n.data_ptr(), bs, V.data_ptr(), vo.data_ptr(),
                                                            D.data_ptr(), do.data_ptr(), precision, r.data_ptr(),
                                                            out.data_ptr(), xo.data_ptr(), st))
        assert torch.equal(x, in_place)
        got.append(x.cpu().numpy().reshape(copies, -1))
    assert np.isfinite(got[0]).all() and (got[1] == got[0]).all()


def test_lapack_l_blocks_have_one_rounding_an_operation():
    """L_1 = diag(sub) D_0^{-1} of upper triangular 2x2 blocks: 1/u and a product on the diagonal, two divisions and a product off it,
    and no further roundings (reciprocals in place of divisions would have two more). Tolerance: two and three half units in
    the last place against long double, and their squares."""
    import torch
    from spitfire_amd import _native
    n = 4000
    rng = np.random.default_rng(4)
    u0, u1, r, s0, s1 = rng.uniform(1., 2., (5, n)) * 2. ** rng.integers(-3, 4, (5, n))
    zero, one = np.zeros(n), np.ones(n)
    dev = torch.device('cuda:0')
    # blocks column by column, then the sub- and super-diagonals
    V = torch.tensor(np.stack([u0, zero, r, u1, one, zero, zero, one, s0, s1, zero, zero], axis=1).ravel(), device=dev)
    nb = torch.full((n,), 2, dtype=torch.int32, device=dev)
    vo, lo, po = (torch.arange(n, dtype=torch.int64, device=dev) * k for k in (12, 8, 4))
    L = torch.zeros(8 * n, dtype=torch.float64, device=dev)
    P = torch.zeros(4 * n, dtype=torch.int32, device=dev)
    _native.check(_native.lib().gf_batch_btddod_full_factorize(n, nb.data_ptr(), 2, V.data_ptr(), vo.data_ptr(), L.data_ptr(),
                                                               lo.data_ptr(), P.data_ptr(), po.data_ptr(),
                                                               torch.cuda.current_stream().cuda_stream))
    l = L.cpu().numpy().reshape(n, 2, 2, 2)[:, 1].transpose(0, 2, 1).astype(np.longdouble)
    u0, u1, r, s0, s1 = (a.astype(np.longdouble) for a in (u0, u1, r, s0, s1))
    half = 2. ** -53 * (1. + 1e-6)
    assert (l[:, 1, 0] == 0).all()
    for got, ref, k in ((l[:, 0, 0], s0 / u0, 2), (l[:, 1, 1], s1 / u1, 2), (l[:, 0, 1], -s0 * r / u1 / u0, 3)):
        assert np.max(np.abs((got - ref) / ref)) <= k * half
