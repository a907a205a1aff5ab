"""Parity of the HIP kernels against NumPy FP64 on seeded inputs (GPU)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def L():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from tncontract_amd import _lib
    _lib.lib()
    assert len(_lib.loaded_hip_runtimes()) == 1, _lib.loaded_hip_runtimes()
    return _lib


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def test_permute_matches_numpy(L):
    rng = np.random.default_rng(0)
    a = rng.standard_normal((7, 33, 65, 3))
    for perm in [(0, 1, 2, 3), (3, 2, 1, 0), (0, 2, 1, 3), (2, 0, 3, 1), (1, 3, 0, 2)]:
        t = dev(a).permute(perm)
        out = L.materialize(t)
        np.testing.assert_array_equal(out.cpu().numpy(), np.transpose(a, perm))
    b = rng.standard_normal((130, 70)).astype(np.float32)
    out = L.materialize(dev(b).t())
    np.testing.assert_array_equal(out.cpu().numpy(), b.T)


@pytest.mark.parametrize("shape", [(5, 7, 3), (64, 64, 64), (130, 257, 70), (300, 200, 1000),
                                   (16, 4096, 2), (1024, 1, 2048), (1, 1, 1)])
def test_contract_fp64_matches_numpy(L, shape):
    from tncontract_amd import tensor as T
    M, K, N = shape
    rng = np.random.default_rng(M * 7 + N)
    a = rng.standard_normal((M, K))
    b = rng.standard_normal((K, N))
    c = T._contract_data(dev(a), [1], dev(b), [0]).cpu().numpy()
    ref = a @ b
    assert np.abs(c - ref).max() <= 1e-12 * max(1.0, np.abs(ref).max()) * np.sqrt(K)


def test_contract_permuted_operands_fused(L):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(5)
    a = rng.standard_normal((6, 40, 5, 30))
    b = rng.standard_normal((30, 7, 6, 9))
    # contract a's axes (3, 0) with b's (0, 2); a and b are also permuted views
    da = dev(np.transpose(a, (2, 0, 3, 1))).permute(1, 3, 0, 2)  # == a as a strided view
    db = dev(np.transpose(b, (1, 3, 0, 2))).permute(2, 0, 3, 1)  # == b
    c = T._contract_data(da, [3, 0], db, [0, 2]).cpu().numpy()
    ref = np.tensordot(a, b, ([3, 0], [0, 2]))
    np.testing.assert_allclose(c, ref, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("prec,tol", [("fp32", 2e-5), ("bf16x3", 2e-4)])
def test_contract_mixed_precision(L, prec, tol):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(11)
    a = rng.standard_normal((300, 513))
    b = rng.standard_normal((513, 250))
    c = T._contract_data(dev(a), [1], dev(b), [0], precision=prec).cpu().numpy().astype(np.float64)
    ref = a @ b
    rel = np.linalg.norm(c - ref) / np.linalg.norm(ref)
    assert rel < tol, rel


@pytest.mark.parametrize("m,n", [(1, 1), (3, 5), (8, 8), (37, 13), (13, 37), (200, 64), (64, 200),
                                 (300, 300), (1280, 640), (2100, 90), (90, 2100)])
def test_qr_matches_lapack(L, m, n):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(m * 1000 + n)
    a = rng.standard_normal((m, n))
    q, r = T._qr_device(dev(a), 1)
    q, r = q.cpu().numpy(), r.cpu().numpy()
    k = min(m, n)
    assert q.shape == (m, k) and r.shape == (k, n)
    np.testing.assert_allclose(q @ r, a, atol=1e-12 * np.sqrt(n) * np.abs(a).max() * 10)
    np.testing.assert_allclose(q.T @ q, np.eye(k), atol=1e-13 * np.sqrt(m) * 10)
    assert np.all(np.tril(r, -1) == 0)
    # same Householder sign convention as LAPACK: Q and R agree with numpy
    qn, rn = np.linalg.qr(a, mode="reduced")
    np.testing.assert_allclose(r, rn, atol=1e-10 * np.abs(rn).max())


@pytest.mark.parametrize("m,n", [(1, 1), (4, 3), (3, 4), (32, 32), (33, 17), (17, 33), (100, 64),
                                 (64, 100), (256, 640), (640, 256), (300, 300)])
def test_svd_matches_lapack(L, m, n):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(m * 31 + n)
    a = rng.standard_normal((m, n))
    u, s, vt = T._svd_device(dev(a), 1)
    u, s, vt = u.cpu().numpy(), s.cpu().numpy(), vt.cpu().numpy()
    k = min(m, n)
    sref = np.linalg.svd(a, compute_uv=False)
    np.testing.assert_allclose(s, sref, rtol=1e-12, atol=1e-13 * sref[0])
    np.testing.assert_allclose((u * s) @ vt, a, atol=1e-12 * sref[0] * np.sqrt(k))
    np.testing.assert_allclose(u.T @ u, np.eye(k), atol=1e-12 * np.sqrt(k))
    np.testing.assert_allclose(vt @ vt.T, np.eye(k), atol=1e-12 * np.sqrt(k))


def test_svd_graded_spectrum(L):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(3)
    m, n = 200, 120
    uu, _ = np.linalg.qr(rng.standard_normal((m, n)))
    vv, _ = np.linalg.qr(rng.standard_normal((n, n)))
    s = np.exp(-np.arange(n) / 8.0)
    a = (uu * s) @ vv.T
    u, sg, vt = T._svd_device(dev(a), 1)
    sg = sg.cpu().numpy()
    np.testing.assert_allclose(sg, s, rtol=1e-9, atol=1e-14)


def test_eigh_psd_ties_across_sort_tiles(L):
    """The device rank sort with repeated keys and more keys than one LDS
    tile (2304 > 2048): the PSD eigensolver of a diagonal matrix whose 2304
    entries take 24 distinct values sorts them twice (the static pivot and
    the final order).  Eigenvalues must be the sorted diagonal and U a
    signed permutation matching them."""
    from tncontract_amd import tensor as T
    n = 2304
    rng = np.random.default_rng(5)
    diag = rng.permutation(np.repeat(np.arange(1.0, 25.0), n // 24))
    u, lam = T._eigh_psd_device(dev(np.diag(diag)), 1)
    u, lam = u.cpu().numpy(), lam.cpu().numpy()
    np.testing.assert_allclose(lam, np.sort(diag)[::-1], rtol=1e-14, atol=0)
    au = np.abs(u)
    np.testing.assert_allclose(au.max(axis=0), np.ones(n), rtol=0, atol=1e-14)
    np.testing.assert_allclose(au.sum(axis=0), np.ones(n), rtol=0, atol=1e-12)
    np.testing.assert_array_equal(diag[np.argmax(au, axis=0)], np.sort(diag)[::-1])
    assert len(set(np.argmax(au, axis=0).tolist())) == n  # a permutation


def test_svd_repeated_singular_values(L):
    """Equal singular values (a scaled orthogonal block beside a graded one)
    through the Jacobi's per-sweep norm sort and the final rank sort."""
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(6)
    m, n = 700, 520
    uu, _ = np.linalg.qr(rng.standard_normal((m, n)))
    vv, _ = np.linalg.qr(rng.standard_normal((n, n)))
    s = np.concatenate([np.full(300, 2.0), np.exp(-np.arange(220) / 40.0)])
    a = (uu * s) @ vv.T
    u, sg, vt = T._svd_device(dev(a), 1)
    u, sg, vt = u.cpu().numpy(), sg.cpu().numpy(), vt.cpu().numpy()
    np.testing.assert_allclose(sg, np.sort(s)[::-1], rtol=1e-12, atol=1e-13 * 2.0)
    np.testing.assert_allclose((u * sg) @ vt, a, atol=1e-12 * 2.0 * np.sqrt(n))
    np.testing.assert_allclose(u.T @ u, np.eye(n), atol=1e-12 * np.sqrt(n))


def test_sumsq_and_scale(L):
    rng = np.random.default_rng(9)
    a = rng.standard_normal(1000003)
    t = dev(a)
    assert abs(L.sumsq(t) - np.sum(a * a)) < 1e-9 * np.sum(a * a)
    L.scale_(t, 0.5)
    np.testing.assert_allclose(t.cpu().numpy(), 0.5 * a)


@pytest.mark.parametrize("prec,tol", [("native", 1e-12), ("fp32", 2e-5)])
def test_contract_with_non_fusing_operands(L, prec, tol):
    # environment-style products whose contracted axes are not neighbours in
    # one operand (GEMM-sized, so the operand is first copied into dense
    # (free, contracted) order): F = E(a,al,a',al') . C(a,k,al,t) over (a, al),
    # then K = C . F over (a, al), with C on the left
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(7)
    E = rng.standard_normal((128, 5, 128, 5))
    C = rng.standard_normal((128, 128, 5, 2))
    F_ref = np.tensordot(E, C, axes=([0, 1], [0, 2]))
    F = T._contract_data(dev(E), [0, 1], dev(C), [0, 2], prec)
    scale = np.abs(F_ref).max()
    assert F.shape == F_ref.shape
    assert np.abs(F.double().cpu().numpy() - F_ref).max() <= tol * scale * 10
    K_ref = np.tensordot(C, F_ref, axes=([0, 2], [0, 1]))
    K = T._contract_data(dev(C), [0, 2], dev(F_ref), [0, 1], prec)
    assert K.shape == K_ref.shape
    assert np.abs(K.double().cpu().numpy() - K_ref).max() <= tol * np.abs(K_ref).max() * 10
    # a strided (transposed) view as the operand
    Ct = dev(C.transpose(1, 0, 3, 2).copy()).permute(1, 0, 3, 2)
    F2 = T._contract_data(dev(E), [0, 1], Ct, [0, 2], prec)
    assert np.abs(F2.double().cpu().numpy() - F_ref).max() <= tol * scale * 10


# The split-bf16 product on its 16-byte-load path and beside it: edges of the
# 128 x 128 x 32 tile, the four operand layouts, odd row pitches and bases
# that are only 4-byte aligned.  Per product of x and y the split keeps
# |x y| (1 + d) with |d| <= 3 * 2^-18 (each half rounds to 8 bits, lo * lo is
# dropped), FP32 accumulation adds at most (3 K + 8) 2^-24 of sum |x y|.
@pytest.mark.parametrize("M,K,N", [(128, 128, 128), (129, 97, 131), (127, 33, 257), (300, 31, 70),
                                   (70, 1000, 41), (1030, 64, 1021)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_contract_bf16x3_tiles(L, M, K, N, layout):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(M + 3 * K + 7 * N)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = rng.standard_normal((K, N)).astype(np.float32)

    def strided(x, t):  # x as a view into a larger buffer, row pitch + 3, base + 1
        y = x.T if t else x
        buf = torch.zeros(y.shape[0] * (y.shape[1] + 3) + 1, dtype=torch.float32, device="cuda")
        v = buf[1:].view(y.shape[0], y.shape[1] + 3)[:, :y.shape[1]]
        v.copy_(torch.from_numpy(np.ascontiguousarray(y)))
        return v.T if t else v

    c = T._contract_data(strided(a, layout[0] == "t"), [1], strided(b, layout[1] == "t"), [0],
                         precision="bf16x3").cpu().numpy().astype(np.float64)
    a, b = a.astype(np.float64), b.astype(np.float64)
    bound = (3 * 2.0 ** -18 + (3 * K + 8) * 2.0 ** -24) * (np.abs(a) @ np.abs(b))
    assert np.all(np.abs(c - a @ b) <= bound)


# Small and few-output contractions with more than eight terms: every lane
# count (4 to 256 per output), ranges split over blocks, several contracted
# modes, permuted views.  A sum of K products in any order is within
# (K + 4) u sum |a b| of the exact one.
@pytest.mark.parametrize("shape_a,ax_a,shape_b,ax_b", [
    ((3, 9), [1], (9, 5), [0]), ((16, 16), [1], (2, 16, 16), [1]), ((7, 63), [1], (63, 2), [0]),
    ((5, 64), [1], (64, 3), [0]), ((4, 3, 5, 17), [3, 1], (3, 17, 6), [1, 0]),
    ((13, 300), [1], (300, 11), [0]), ((2, 40, 3, 50), [1, 3], (40, 50, 4), [0, 1]),
    ((4097,), [0], (4097,), [0]), ((3, 8191), [1], (8191, 1), [0]),
    ((1, 70001), [1], (70001, 2), [0]), ((30, 40, 50), [0, 1, 2], (50, 30, 40), [1, 2, 0]),
    ((600000,), [0], (600000,), [0])])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_contract_many_lanes_per_output(L, shape_a, ax_a, shape_b, ax_b, dtype):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(sum(shape_a) + sum(shape_b))
    a, b = rng.standard_normal(shape_a).astype(dtype), rng.standard_normal(shape_b).astype(dtype)
    # b as a view with its axes stored in reverse order
    db = dev(b.transpose()).permute(*range(b.ndim - 1, -1, -1))
    c = T._contract_data(dev(a), ax_a, db, ax_b).cpu().numpy()
    a, b = a.astype(np.float64), b.astype(np.float64)
    K = int(np.prod([shape_a[i] for i in ax_a]))
    ref, mag = np.tensordot(a, b, (ax_a, ax_b)), np.tensordot(np.abs(a), np.abs(b), (ax_a, ax_b))
    # (plus the oracle's own FP64 rounding)
    bound = (K + 4) * (np.finfo(dtype).eps / 2 + 2.0 ** -53) * mag
    assert c.shape == ref.shape and np.all(np.abs(c - ref) <= bound)


# QR blocks through their orthonormal factor (64 columns, at least 256 rows
# below the diagonal), beside the panels: ragged edges of both, columns of very
# different lengths, and the inputs that have to stay with the panels -- zero
# and unit columns, triangular and rank-deficient matrices, zero pivots, NaN.
# LAPACK's R is reached to rounding, its diagonal's signs with it.
@pytest.mark.parametrize("m,n", [(256, 64), (257, 65), (319, 64), (320, 128), (700, 129),
                                 (1285, 643), (500, 1500)])
@pytest.mark.parametrize("scale", ["flat", "graded"])
def test_qr_blocks_match_lapack(L, m, n, scale):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal((m, n))
    if scale == "graded":
        a *= 2.0 ** rng.integers(-300, 300, size=n)
    q, r = (x.cpu().numpy() for x in T._qr_device(dev(a), 1))
    k = min(m, n)
    ref = np.linalg.qr(a)[1]
    norms = np.linalg.norm(a, axis=0)
    assert np.abs(q.T @ q - np.eye(k)).max() <= 1e-13
    assert (np.linalg.norm(q @ r - a, axis=0) <= 1e-13 * norms).all()
    assert (np.abs(r - ref).max(axis=0) <= 1e-11 * norms).all()
    assert not np.tril(r, -1).any()


@pytest.mark.parametrize("case", ["eye", "triu", "zero", "zero_column", "rank", "zero_pivot", "nan"])
def test_qr_blocks_leave_special_inputs_to_the_panels(L, case):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(3)
    m, n = 700, 200
    a = rng.standard_normal((m, n))
    if case == "eye":
        a = np.eye(m, n)
    elif case == "triu":
        a = np.triu(a)
    elif case == "zero":
        a[:] = 0.0
    elif case == "zero_column":
        a[:, 70] = 0.0
    elif case == "rank":
        a = a[:, :40] @ rng.standard_normal((40, n))
    elif case == "zero_pivot":
        a[:64, :64] = 0.0
    elif case == "nan":
        a[300, 100] = np.nan
    q, r = (x.cpu().numpy() for x in T._qr_device(dev(a), 1))
    if case == "nan":
        assert np.isnan(q).any() and np.isnan(r).any()
        return
    assert np.abs(q.T @ q - np.eye(n)).max() <= 1e-13
    assert np.abs(q @ r - a).max() <= 1e-12 * max(1.0, np.abs(a).max()) * np.sqrt(n)
    if case in ("eye", "triu", "zero"):
        # no reflection at all: R is the matrix, with its own signs
        np.testing.assert_array_equal(r, a[:n])
    elif case in ("zero_pivot", "zero_column"):
        ref = np.linalg.qr(a)[1]
        keep = 70 if case == "zero_column" else n  # (past it the signs are rounding's)
        assert np.abs(r[:keep] - ref[:keep]).max() <= 1e-11 * np.abs(ref).max()


# SVDs that one workgroup does in one launch (at most 32 vectors of at most
# 256), at both limits and just past them, full, graded and rank-deficient,
# FP64 and FP32 in; bounds as for test_svd_matches_lapack's sizes: k eps for
# the values, a few sweeps' rounding for the factors.
@pytest.mark.parametrize("m,n", [(1, 7), (2, 2), (15, 256), (256, 16), (17, 257), (31, 31),
                                 (32, 32), (32, 33), (256, 32), (257, 32), (32, 256)])
@pytest.mark.parametrize("case", ["full", "graded", "rank", "zero_vectors"])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_svd_in_one_workgroup(L, m, n, case, dtype):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(m * 300 + n)
    a, k = rng.standard_normal((m, n)), min(m, n)
    if case == "graded":
        a = (a[:, :1] if n == 1 else a) * (10.0 ** -np.linspace(0, 12, n))
    elif case == "rank":
        r = max(1, k // 3)
        a = a[:, :r] @ rng.standard_normal((r, n))
    elif case == "zero_vectors":
        a[:, ::2] = 0.0
    a = a.astype(dtype)
    u, s, vt = (x.cpu().numpy().astype(np.float64) for x in T._svd_device(dev(a), 1))
    a = a.astype(np.float64)
    ref = np.linalg.svd(a, compute_uv=False)
    eps = 2e-13 if dtype == np.float64 else 2e-6
    assert np.abs(s - ref).max() <= 1e-13 * max(ref[0], 1e-300)
    assert np.all(np.diff(s) <= 0)
    assert np.linalg.norm((u * s) @ vt - a) <= eps * max(ref[0], 1e-300) * np.sqrt(k)
    big = int(np.count_nonzero(ref > 1e-10 * ref[0]))
    assert np.abs(u[:, :big].T @ u[:, :big] - np.eye(big)).max() <= eps
    assert np.abs(vt[:big] @ vt[:big].T - np.eye(big)).max() <= eps


# Jacobi with the inner pairs at every fourth step (more than four blocks of
# 16 vectors), from the last size without to a few past a whole block: the SVD
# (rotations accumulated) and the PSD eigensolver; bounds as above.
@pytest.mark.parametrize("n", [64, 65, 96, 97, 130, 257])
@pytest.mark.parametrize("case", ["full", "graded", "clusters", "rank"])
def test_jacobi_inner_pairs_every_fourth_step(L, n, case):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    if case != "full":
        u, v = np.linalg.qr(a)[0], np.linalg.qr(rng.standard_normal((n, n)))[0]
        s = {"graded": np.logspace(0, -12, n), "clusters": 10.0 ** -(np.arange(n) % 3),
             "rank": np.where(np.arange(n) < n // 3, 1.0, 0.0)}[case]
        a = (u * s) @ v
    ref = np.linalg.svd(a, compute_uv=False)
    u, s, vt = (x.cpu().numpy() for x in T._svd_device(dev(a), 1))
    assert np.abs(s - ref).max() <= 2e-13 * ref[0]
    assert np.linalg.norm((u * s) @ vt - a) <= 4e-13 * ref[0] * np.sqrt(n)
    big = int(np.count_nonzero(ref > 1e-10 * ref[0]))
    assert np.abs(u[:, :big].T @ u[:, :big] - np.eye(big)).max() <= 4e-13
    assert np.abs(vt[:big] @ vt[:big].T - np.eye(big)).max() <= 4e-13
    K = a.T @ a
    w, lam = (x.cpu().numpy() for x in T._eigh_psd_device(dev(K), 1)[:2])
    assert np.linalg.norm((w * lam) @ w.T - K) <= 4e-13 * ref[0] ** 2 * np.sqrt(n)
    big = int(np.count_nonzero(ref > 1e-5 * ref[0]))
    assert np.abs(w[:, :big].T @ w[:, :big] - np.eye(big)).max() <= 4e-13


# One-launch Jacobi steps (vectors of length at most 256), from the first size
# past one pair of blocks to the last: odd lengths, a last block of one vector,
# zero vectors (pairs that are copied); bounds as above.
@pytest.mark.parametrize("n", [33, 47, 129, 255, 256])
def test_jacobi_one_launch_steps(L, n):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    a[:, n // 2:n // 2 + 16] = 0.0
    ref = np.linalg.svd(a, compute_uv=False)
    for m in (a, a.T):
        u, s, vt = (x.cpu().numpy() for x in T._svd_device(dev(m.copy()), 1))
        assert np.abs(s - ref).max() <= 2e-13 * ref[0]
        assert np.linalg.norm((u * s) @ vt - m) <= 4e-13 * ref[0] * np.sqrt(n)
        k = n - 16
        assert np.abs(u[:, :k].T @ u[:, :k] - np.eye(k)).max() <= 4e-13
        assert np.abs(vt[:k] @ vt[:k].T - np.eye(k)).max() <= 4e-13
    K = a.T @ a
    w, lam = (x.cpu().numpy() for x in T._eigh_psd_device(dev(K), 1)[:2])
    assert np.linalg.norm((w * lam) @ w.T - K) <= 4e-13 * ref[0] ** 2 * np.sqrt(n)


# QR by one workgroup (at most 64 columns and 256 rows): both variants' edges in
# rows and columns, wide and tall, and the first sizes past them, FP64 and FP32
# in, through transposed strides; R against LAPACK's (the same reflectors), the
# bounds of a backward-stable factorisation.
@pytest.mark.parametrize("m,n", [(1, 1), (1, 64), (64, 1), (2, 3), (15, 16), (16, 15), (17, 33),
                                 (32, 32), (64, 32), (65, 32), (32, 64), (64, 64), (65, 33),
                                 (256, 32), (255, 63), (256, 64), (257, 64), (256, 65)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_qr_in_one_workgroup(L, m, n, dtype):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(64 * m + n)
    a = rng.standard_normal((m, n)).astype(dtype)
    eps = 1e-13 if dtype == np.float64 else 2e-6
    for d in (dev(a), dev(np.ascontiguousarray(a.T)).T):
        q, r = (x.cpu().numpy().astype(np.float64) for x in T._qr_device(d, 1))
        ref = np.linalg.qr(a.astype(np.float64))[1]
        size = np.linalg.norm(a)
        assert np.abs(np.tril(r, -1)).max(initial=0.0) == 0.0
        assert np.linalg.norm(q @ r - a) <= eps * size
        assert np.abs(q.T @ q - np.eye(min(m, n))).max() <= eps
        # R's condition: well within 1e3 eps away from the square sizes
        if abs(m - n) > 16:
            assert np.abs(r - ref).max() <= 1e2 * eps * size
    # zero columns: no reflector, the sign of the diagonal as LAPACK leaves it
    a[:, n // 2] = 0.0
    q, r = (x.cpu().numpy().astype(np.float64) for x in T._qr_device(dev(a), 1))
    assert np.linalg.norm(q @ r - a) <= eps * max(np.linalg.norm(a), 1.0)
    assert np.abs(q.T @ q - np.eye(min(m, n))).max() <= eps


# Columns that earlier reflectors leave with rounding only (rows equal up to
# rounding, 1e-16 smaller from column to column): their squares underflow, and
# the reflectors stay orthogonal all the same.
@pytest.mark.parametrize("scale", [1.0, 1e-150, 1e-300])
@pytest.mark.parametrize("m,n", [(64, 32), (40, 64), (200, 64)])
def test_small_qr_of_shrinking_columns(L, m, n, scale):
    from tncontract_amd import tensor as T
    from tncontract_amd.batched import batched_svd
    rng = np.random.default_rng(m + n)
    a = np.zeros((m, n))
    a[-1] = rng.standard_normal(n) * scale
    q, r = (x.cpu().numpy() for x in T._qr_device(dev(a), 1))
    assert np.abs(q.T @ q - np.eye(min(m, n))).max() <= 1e-13
    assert np.abs(q @ r - a).max() <= 1e-13 * scale
    if scale == 1.0:
        for u, s, vt in (T._svd_device(dev(a), 1), [x[0] for x in batched_svd([dev(a)])[:3]]):
            u, s, vt = (x.cpu().numpy() for x in (u, s, vt))
            assert abs(s[0] - np.linalg.norm(a)) <= 1e-13 * s[0]
            assert np.abs((u * s) @ vt - a).max() <= 1e-13 * s[0]


# Products of few 32 x 32 tiles (one workgroup each, K over its waves): tile
# edges, K around a wave's eights and the last K taken, one and several modes,
# every operand order.  Bound: K rounding errors of the absolute products.
@pytest.mark.parametrize("m,n,k", [(33, 31, 300), (16, 1024, 17), (128, 130, 63), (64, 64, 64),
                                   (95, 97, 65), (512, 511, 511), (256, 300, 512), (300, 256, 513),
                                   (1000, 1024, 128), (5, 2000, 40)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_contract_few_tiles(L, m, n, k, dtype):
    import tncontract_amd as tn
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(dtype), rng.standard_normal((k, n)).astype(dtype)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    bound = k * np.finfo(dtype).eps * (np.abs(a).astype(np.float64) @ np.abs(b)) + 1e-300
    for x, lx in ((a, ["m", "k"]), (a.T, ["k", "m"])):
        for y, ly in ((b, ["k", "n"]), (b.T, ["n", "k"])):
            z = tn.contract(tn.Tensor(dev(np.ascontiguousarray(x)), lx),
                            tn.Tensor(dev(np.ascontiguousarray(y)), ly), "k", "k")
            z.move_indices(["m", "n"], 0)
            assert (np.abs(z.data.cpu().numpy() - ref) <= bound).all()
    # both operands with two modes in every group that divides
    if m % 4 == 0 and n % 4 == 0 and k % 4 == 0:
        x = dev(np.ascontiguousarray(a.reshape(m // 4, 4, k // 4, 4).transpose(2, 0, 3, 1)))
        y = dev(np.ascontiguousarray(b.reshape(k // 4, 4, n // 4, 4).transpose(1, 3, 0, 2)))
        z = tn.contract(tn.Tensor(x, ["k0", "m0", "k1", "m1"]),
                        tn.Tensor(y, ["k1", "n1", "k0", "n0"]), ["k0", "k1"], ["k0", "k1"])
        z.move_indices(["m0", "m1", "n0", "n1"], 0)
        assert (np.abs(z.data.cpu().numpy().reshape(m, n) - ref) <= bound).all()


# Permuted copies: the general gather and the tiled transpose (whole and ragged
# tiles), element for element.
@pytest.mark.parametrize("shape,perm", [((3, 5), (1, 0)), ((2, 3, 5, 7), (2, 0, 3, 1)),
                                        ((5, 51, 2), (2, 1, 0)), ((509, 2, 5, 52), (1, 3, 0, 2)),
                                        ((7, 1, 9, 2, 3, 5), (5, 1, 0, 4, 2, 3)),
                                        ((64, 128), (1, 0)), ((65, 3, 130), (2, 1, 0)),
                                        ((1000, 2, 700), (1, 2, 0)), ((2, 600, 5, 400), (2, 1, 3, 0))])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_permuted_copies(L, shape, perm, dtype):
    from tncontract_amd import _lib
    x = torch.arange(int(np.prod(shape)), dtype=dtype, device="cuda").reshape(shape)
    y = x.permute(perm)
    assert torch.equal(_lib.contiguous(y), y.contiguous())
    z = x[tuple(slice(0, None, 2) for _ in shape)].permute(perm)
    assert torch.equal(_lib.contiguous(z), z.contiguous())


# FP64 matrices whose squared entries leave the range (2^(+-511) and beyond),
# beside the last that need no scaling: one workgroup's sizes, vectors without
# the preconditioning QR, one-launch and two-launch Jacobi steps, the batched
# SVD.  The power of two is exact, so the bounds are those at 2^0 (plus the
# rounding of singular values below 2^-1022).
MAGNITUDES = [-1030, -530, -517, -505, -190, 190, 505, 530, 1000]


def check_svd_at(a, u, s, vt, exp):
    ref = np.linalg.svd(a, compute_uv=False)
    s = np.ldexp(s, -exp)
    assert np.abs(s - ref).max() <= (2e-13 + 2.0 ** (-1074 - exp)) * ref[0]
    assert np.linalg.norm((u * s) @ vt - a) <= 4e-13 * ref[0] * np.sqrt(len(ref)) \
        + 2.0 ** (-1074 - exp) * len(ref)
    big = int(np.count_nonzero(ref > 1e-10 * ref[0]))
    assert np.abs(u[:, :big].T @ u[:, :big] - np.eye(big)).max() <= 4e-13
    assert np.abs(vt[:big] @ vt[:big].T - np.eye(big)).max() <= 4e-13


@pytest.mark.parametrize("exp", MAGNITUDES)
@pytest.mark.parametrize("m,n", [(24, 16), (32, 256), (300, 20), (40, 70), (130, 129), (300, 290)])
def test_svd_at_any_magnitude(L, m, n, exp):
    from tncontract_amd import tensor as T
    from tncontract_amd.batched import batched_svd
    rng = np.random.default_rng(m + n)
    low = rng.standard_normal((m, 7)) @ rng.standard_normal((7, n))
    sparse = low * (rng.random(n) < 0.5)
    one = rng.standard_normal((20, 30))
    for g in (rng.standard_normal((m, n)), low, sparse):
        x = np.ldexp(g, exp)
        a = np.ldexp(x, -exp)  # (what is left of g in subnormals)
        u, s, vt = (t.cpu().numpy() for t in T._svd_device(dev(x), 1))
        check_svd_at(a, u, s, vt, exp)
        if g is not sparse:  # each job of a batch has its own scale
            U, S, Vt, _ = batched_svd([dev(x), dev(one)])
            check_svd_at(a, U[0].cpu().numpy(), S[0].cpu().numpy(), Vt[0].cpu().numpy(), exp)
            check_svd_at(one, U[1].cpu().numpy(), S[1].cpu().numpy(), Vt[1].cpu().numpy(), 0)


@pytest.mark.parametrize("m,n", [(24, 16), (300, 20), (100, 100)])
@pytest.mark.parametrize("big", [1e200, 1e-200])
def test_svd_with_one_large_entry(L, m, n, big):
    from tncontract_amd import tensor as T
    a = np.random.default_rng(m).standard_normal((m, n)) * min(big, 1.0)
    a[m // 2, n // 3] = big * 1e3
    u, s, vt = (t.cpu().numpy() for t in T._svd_device(dev(a), 1))
    check_svd_at(a / big, u, s / big, vt, 0)


@pytest.mark.parametrize("scale", [1e-150, 1e-300, 1e150])
def test_svd_of_shrinking_columns_at_any_magnitude(L, scale):
    from tncontract_amd import tensor as T
    from tncontract_amd.batched import batched_svd
    for m, n in [(64, 32), (40, 64), (200, 64), (31, 20)]:
        a = np.zeros((m, n))
        a[-1] = np.random.default_rng(m + n).standard_normal(n)
        for u, s, vt in (T._svd_device(dev(a * scale), 1),
                         [x[0] for x in batched_svd([dev(a * scale)])[:3]]):
            u, s, vt = (x.cpu().numpy() for x in (u, s, vt))
            s = s / scale
            assert abs(s[0] - np.linalg.norm(a)) <= 1e-13 * s[0]
            assert np.abs((u * s) @ vt - a).max() <= 1e-13 * s[0]


# Blocks that pass the tests of the orthonormal-factor path although two of
# their columns are nearly dependent on others (smallest singular value about
# 1 / c): the factorisation is backward stable column by column all the same.
@pytest.mark.parametrize("m,n", [(256, 64), (1280, 64), (1280, 200)])
@pytest.mark.parametrize("c", [1, 30, 100, 300, 1000, 3000])
def test_qr_of_nearly_dependent_columns(L, m, n, c):
    from tncontract_amd import tensor as T
    for seed in range(3):
        rng = np.random.default_rng(1000 * seed + c)
        a = rng.standard_normal((m, n))
        for j in range(10, n, 64):
            w = rng.standard_normal(m)
            a[:, j] = a[:, j - 10:j] @ (rng.standard_normal(10) / 10) + w / c
            a[:, j + 1] = w + 0.3 * rng.standard_normal(m)
        q, r = (x.cpu().numpy() for x in T._qr_device(dev(a), 1))
        assert np.abs(q.T @ q - np.eye(n)).max() <= 1e-13
        res = np.linalg.norm(q @ r - a, axis=0) / np.linalg.norm(a, axis=0)
        assert res.max() <= 1e-14


# The rotations keep lengths: a singular vector has met about ten rotations per
# other vector, whose cosines and sines are rounded without bias, so the vectors
# that accumulate them stay within a random walk of 10 n steps of 2^-53 of length
# one (their mean well within).
@pytest.mark.parametrize("m,n", [(32, 32), (64, 32), (64, 64), (254, 636), (300, 290), (300, 20)])
def test_rotations_keep_lengths(L, m, n):
    from tncontract_amd import tensor as T
    from tncontract_amd.batched import batched_svd
    a = np.random.default_rng(m + n).standard_normal((m, n))
    k = min(m, n)
    for u, s, vt in (T._svd_device(dev(a), 1), [x[0] for x in batched_svd([dev(a)])[:3]]):
        for v in (u.cpu().numpy(), vt.cpu().numpy().T):
            w = v.astype(np.longdouble)
            assert abs(float(((w * w).sum(axis=0) - 1).mean())) <= np.sqrt(10 * k) * 2.0 ** -53


# One-launch Jacobi steps: sweeps are enqueued ahead of their outcomes, which
# reach the host through a word of pinned memory (tn_svd) or by copies
# (tn_svd_noalloc).  Both count and stop alike, at every limit.
@pytest.mark.parametrize("limit", [1, 2, 5, 6, 7, 8, 40])
@pytest.mark.parametrize("case", ["identity", "full"])
def test_sweep_counts_of_one_launch_steps(L, limit, case):
    from tncontract_amd import tensor as T
    n = 100
    a = np.eye(n) if case == "identity" else np.random.default_rng(1).standard_normal((n, n))
    d = dev(a)
    rows, cols, _, _ = T._matrix_modes(d, 1)
    lib = L.lib()
    ws = L.workspace(lib.tn_svd_workspace(n, n, 0))
    got = []
    for noalloc in (False, True):
        u, s, vt = L.empty((n, n)), L.empty((n,)), L.empty((n, n))
        sweeps = ctypes.c_int(-1)
        args = [L.ptr(d), ctypes.byref(rows), ctypes.byref(cols), n, n, L.ptr(u), L.ptr(s),
                L.ptr(vt), 0, 0.0, limit, ctypes.byref(sweeps)]
        rc = lib.tn_svd_noalloc(*args, L.stream_ptr()) if noalloc else \
            lib.tn_svd(*args, L.ptr(ws), ws.numel(), L.stream_ptr())
        got.append((rc, sweeps.value, u.cpu().numpy(), s.cpu().numpy(), vt.cpu().numpy()))
    (rc, used, u, s, vt), other = got
    assert other[:2] == (rc, used) and all(np.array_equal(x, y) for x, y in zip(got[0][2:], other[2:]))
    assert used <= limit
    if case == "identity":
        assert rc == L.TN_OK and used == 1
    elif limit <= 2:
        assert rc == L.TN_ERR_NOCONV and used == limit
    if rc == L.TN_OK:
        assert np.linalg.norm((u * s) @ vt - a) <= 4e-13 * s[0] * np.sqrt(n)


def test_svds_of_threads_with_their_own_streams(L):
    import threading
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(2)
    mats = [rng.standard_normal((m, n)) for m, n in [(100, 100), (64, 200), (250, 130), (40, 40)] * 3]
    errs = [None] * len(mats)

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            d = dev(mats[i])
            for _ in range(4):
                u, s, vt = (x.cpu().numpy() for x in T._svd_device(d, 1))
                e = np.linalg.norm((u * s) @ vt - mats[i]) / s[0]
                errs[i] = max(errs[i] or 0.0, e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(mats))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(e is not None and e <= 4e-13 * np.sqrt(200) for e in errs), errs


# Split-bf16 products with one row or column, and with operands that repeat one
# (stride 0) or are sliced (no unit stride: the tables).  A bf16 has an 8-bit
# significand, so a half's rounding is 2^-8 of it: x y is kept but for 3 * 2^-16.
@pytest.mark.parametrize("M,K,N", [(1, 300, 2000), (2000, 300, 1), (1, 4000, 70), (128, 64, 128),
                                   (200, 130, 300)])
@pytest.mark.parametrize("kind", ["dense", "rows_of_a", "columns_of_b", "k_of_a", "k_of_b", "sliced"])
def test_contract_bf16x3_broadcast_operands(L, M, K, N, kind):
    from tncontract_amd import tensor as T
    rng = np.random.default_rng(M + 3 * K + 7 * N)
    a, b = (dev(rng.standard_normal(s).astype(np.float32)) for s in ((M, K), (K, N)))
    if kind == "rows_of_a":
        a = a[:1].expand(M, K)
    elif kind == "columns_of_b":
        b = b[:, :1].expand(K, N)
    elif kind == "k_of_a":
        a = a[:, :1].expand(M, K)
    elif kind == "k_of_b":
        b = b[:1].expand(K, N)
    elif kind == "sliced":
        a, b = dev(rng.standard_normal((M, 2 * K)).astype(np.float32))[:, ::2], \
            dev(rng.standard_normal((K, 3 * N)).astype(np.float32))[:, ::3]
    c = T._contract_data(a, [1], b, [0], precision="bf16x3").cpu().numpy().astype(np.float64)
    a, b = a.cpu().numpy().astype(np.float64), b.cpu().numpy().astype(np.float64)
    bound = (3 * 2.0 ** -16 + (3 * K + 8) * 2.0 ** -24) * (np.abs(a) @ np.abs(b))
    assert np.all(np.abs(c - a @ b) <= bound)


# Products of few tiles allocate their result alone; a product that splits K
# gets the same partial sums in every precision.
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_contract_allocates_no_unused_buffer(L, dtype):
    from tncontract_amd import tensor as T
    for n, k, splits in [(512, 512, False), (256, 128, False), (256, 2000, True)]:
        a, b = (torch.ones(s, dtype=dtype, device="cuda") for s in ((n, k), (k, n)))
        torch.cuda.synchronize()
        base = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        c = T._contract_data(a, [1], b, [0])
        used = torch.cuda.max_memory_allocated() - base
        sums = L.lib().tn_contract_workspace(n, n, k, L.dtype_code(a)) if splits else 0
        assert used <= c.numel() * c.element_size() + sums + 1024
        assert splits == (used > 2 * c.numel() * c.element_size())
        assert (c == k).all()
