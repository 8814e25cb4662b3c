"""GPU parity of the C-ABI primitives against the oracle (tests/../oracle).

Tolerances: complex128 paths to 1e-12 relative (contraction rounding only);
complex64 (mixed) contractions to 2e-5 relative, the FP32 round-off of sums of
up to a few thousand terms.
"""
import ctypes

import numpy as np
import pytest

from conftest import crand

import qca_native as qn
from oracle import automaton as AU, local as LOC

pytestmark = pytest.mark.gpu


def dev(torch, a, dtype):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=dtype)).cuda()


def herm_env(rng, chi, D):
    E = crand(rng, chi, D, chi)
    return 0.5 * (E + np.conj(np.transpose(E, (2, 1, 0))))


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


W_CASES = [(1, range(1, 2)), (2, range(2, 5)), (2, range(1, 5)), (1, range(2, 3))]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("chil,chir,rule", [(1, 1, 0), (3, 5, 1), (16, 16, 0), (37, 29, 2),
                                            (64, 64, 1), (128, 96, 3)])
def test_heff_apply(gpu, prec, kind, chil, chir, rule):
    import torch
    rng = np.random.default_rng(chil * 131 + chir * 7 + kind)
    d, iv = W_CASES[rule]
    W = AU.bulk_tensor(d, iv)
    D = W.shape[2]
    if kind == 2:
        chir = chil if kind == 2 and rule % 2 == 0 else chir
        x = crand(rng, chil, chir)
        L, R = herm_env(rng, chil, D), herm_env(rng, chir, D)
        ref = LOC.bond_apply(x, L, R)
        Wd = None
    elif kind == 1:
        x = crand(rng, 2, chil, chir)
        L, R = herm_env(rng, chil, D), herm_env(rng, chir, D)
        ref = LOC.heff_apply(x, L, R, W)
        Wd = W
    else:
        x = crand(rng, 4, chil, chir)
        L, R = herm_env(rng, chil, D), herm_env(rng, chir, D)
        Wd = LOC.merge_w(W, W)
        ref = LOC.heff_apply(x, L, R, Wd)
    dt = np.complex128 if prec == 0 else np.complex64
    xd, Ld, Rd = dev(torch, x, dt), dev(torch, L, dt), dev(torch, R, dt)
    yd = torch.zeros_like(xd)
    Wh = np.ascontiguousarray(Wd if Wd is not None else np.zeros(1), dtype=np.complex128)
    qn.call("qca_heff_apply", prec, kind, qn.ptr(xd), qn.ptr(yd), qn.ptr(Ld), qn.ptr(Rd),
            Wh.ctypes.data if Wd is not None else None, D, D, chil, chir, None)
    got = yd.cpu().numpy().astype(np.complex128)
    assert rel(got, ref) < (1e-12 if prec == 0 else 2e-5)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("chil,chir,rule", [(31, 33, 1), (33, 64, 3), (65, 31, 1), (96, 97, 1), (160, 129, 3)])
def test_heff_apply_tiles(gpu, prec, kind, chil, chir, rule):
    """Blocks around the 32- and 64-wide tiles, on both sides of the choice between
    them and with and without K splits, with MPO channels that no row reads."""
    test_heff_apply(gpu, prec, kind, chil, chir, rule)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("chil,chir", [(1, 2), (5, 7), (32, 64), (128, 128)])
def test_env_update(gpu, prec, side, chil, chir):
    import torch
    rng = np.random.default_rng(chil + 17 * chir + side)
    Ws = AU.mpo_tensors(6, 2, range(2, 5))
    W = Ws[2]
    Dl, Dr = W.shape[2], W.shape[3]
    A = crand(rng, 2, chil, chir)
    dt = np.complex128 if prec == 0 else np.complex64
    if side == 0:
        E = herm_env(rng, chil, Dl)
        ref = LOC.env_left(E, A, W)
        out = torch.zeros((chir, Dr, chir), dtype=torch.complex128 if prec == 0 else torch.complex64, device="cuda")
    else:
        E = herm_env(rng, chir, Dr)
        ref = LOC.env_right(E, A, W)
        out = torch.zeros((chil, Dl, chil), dtype=torch.complex128 if prec == 0 else torch.complex64, device="cuda")
    Ad, Ed = dev(torch, A, dt), dev(torch, E, dt)
    Wh = np.ascontiguousarray(W, dtype=np.complex128)
    qn.call("qca_env_update", prec, side, qn.ptr(Ad), qn.ptr(Ed), qn.ptr(out), Wh.ctypes.data,
            Dl, Dr, chil, chir, None)
    got = out.cpu().numpy().astype(np.complex128)
    assert rel(got, ref) < (1e-12 if prec == 0 else 2e-5)


def test_env_update_golden(gpu):
    """Reference _assemble_new_layer_H_eff outputs (golden, reference tdvp.py:328-347)."""
    import torch
    from conftest import golden
    g = golden("units")
    W = g["W"]
    A, Lp, Rp = g["env_A"], g["env_Lprev"], g["env_Rprev"]
    chil, chir = A.shape[1], A.shape[2]
    Dl = Dr = W.shape[2]
    Wh = np.ascontiguousarray(W)
    for side, E, ref, shape in ((0, Lp, g["env_Lnew"], (chir, Dr, chir)), (1, Rp, g["env_Rnew"], (chil, Dl, chil))):
        out = torch.zeros(shape, dtype=torch.complex128, device="cuda")
        Ad, Ed = dev(torch, A, np.complex128), dev(torch, E, np.complex128)  # keep both alive
        qn.call("qca_env_update", 0, side, qn.ptr(Ad), qn.ptr(Ed), qn.ptr(out), Wh.ctypes.data,
                Dl, Dr, chil, chir, None)
        assert rel(out.cpu().numpy(), ref) < 1e-12


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind,chil,chir,delta", [(1, 4, 6, 0.05), (1, 4, 6, -0.05), (0, 3, 4, 0.05),
                                                 (2, 5, 5, -0.05), (0, 24, 24, 0.05), (1, 48, 40, -0.05)])
def test_krylov_expm(gpu, prec, kind, chil, chir, delta):
    import torch
    rng = np.random.default_rng(kind * 1000 + chil)
    W = AU.bulk_tensor(2, range(2, 5))
    D = W.shape[2]
    L, R = herm_env(rng, chil, D), herm_env(rng, chir, D)
    if kind == 0:
        Wk = LOC.merge_w(W, W)
        x = crand(rng, 4, chil, chir)
        Hm = LOC.dense_heff(L, R, Wk)
    elif kind == 1:
        Wk = W
        x = crand(rng, 2, chil, chir)
        Hm = LOC.dense_heff(L, R, Wk)
    else:
        Wk = None
        x = crand(rng, chil, chir)
        Hm = LOC.dense_keff(L, R)
    x /= np.linalg.norm(x)
    ref = LOC.expm_dense(Hm, x.reshape(-1), delta).reshape(x.shape)
    dt = np.complex128 if prec == 0 else np.complex64
    xd = dev(torch, x, np.complex128)
    Ld, Rd = dev(torch, L, dt), dev(torch, R, dt)
    Wh = np.ascontiguousarray(Wk if Wk is not None else np.zeros(1), dtype=np.complex128)
    it = ctypes.c_int(0)
    qn.call("qca_krylov_expm", prec, kind, qn.ptr(xd), qn.ptr(Ld), qn.ptr(Rd),
            Wh.ctypes.data if Wk is not None else None, D, D, chil, chir, delta, 0.0,
            ctypes.byref(it), None)
    got = xd.cpu().numpy()
    assert it.value >= 2
    assert np.abs(got - ref).max() < (1e-12 if prec == 0 else 2e-5)
    assert abs(np.linalg.norm(got) - 1.0) < (1e-12 if prec == 0 else 1e-5)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind,chil,chir,delta", [(2, 1, 1, 0.05), (2, 15, 17, -0.05), (2, 16, 16, 0.1),
                                                 (2, 1, 257, 0.05), (1, 9, 57, 0.1), (0, 1, 2, 0.05),
                                                 (2, 16, 16, 0.0)])
def test_krylov_expm_blocks(gpu, prec, kind, chil, chir, delta):
    """Vectors just below, at and above one and several 256-element blocks, a zero
    step, and steps long enough that the convergence bound does not apply (phase
    widths of 19 and 28, against 2.8)."""
    if delta == 0.0 or chil * chir == 1:
        # one iteration at least: the state itself, up to a phase
        import torch
        rng = np.random.default_rng(chil)
        D = AU.bulk_tensor(2, range(2, 5)).shape[2]
        x = crand(rng, chil, chir)
        x /= np.linalg.norm(x)
        L, R = herm_env(rng, chil, D), herm_env(rng, chir, D)
        dt = np.complex128 if prec == 0 else np.complex64
        xd = dev(torch, x, np.complex128)
        Ld, Rd = dev(torch, L, dt), dev(torch, R, dt)
        it = ctypes.c_int(0)
        qn.call("qca_krylov_expm", prec, kind, qn.ptr(xd), qn.ptr(Ld), qn.ptr(Rd), None, D, D, chil, chir, delta,
                0.0, ctypes.byref(it), None)
        ref = LOC.expm_dense(LOC.dense_keff(L, R), x.reshape(-1), delta).reshape(x.shape)
        assert np.abs(xd.cpu().numpy() - ref).max() < (1e-12 if prec == 0 else 2e-5)
    else:
        test_krylov_expm(gpu, prec, kind, chil, chir, delta)


@pytest.mark.parametrize("right", [1, 0])
@pytest.mark.parametrize("chil,chir,chi_max,eps", [(1, 1, 4, 1e-10), (2, 4, 8, 1e-10), (8, 8, 16, 1e-10),
                                                   (8, 8, 5, 1e-10), (16, 32, 64, 1e-3),
                                                   # one workgroup with four 16-column blocks,
                                                   # full and ragged (34..48 columns)
                                                   (32, 32, 64, 1e-10), (24, 20, 64, 1e-10),
                                                   (17, 20, 64, 1e-10),
                                                   (64, 64, 128, 1e-10), (128, 128, 128, 1e-10),
                                                   # the widest split (512 columns) and a
                                                   # ragged 400 x 272 one capped at 128
                                                   (256, 256, 256, 1e-10), (200, 136, 128, 1e-10)])
def test_svd_split(gpu, right, chil, chir, chi_max, eps):
    import torch
    rng = np.random.default_rng(chil * 3 + chir + right)
    th = crand(rng, 4, chil, chir)
    # graded spectrum so that truncation tails span many orders of magnitude
    M = th.reshape(2, 2, chil, chir).transpose(0, 2, 1, 3).reshape(2 * chil, 2 * chir)
    u, s, vh = np.linalg.svd(M, full_matrices=False)
    s = np.logspace(0, -14, len(s))
    M = (u * s) @ vh
    M /= np.linalg.norm(M)
    th = M.reshape(2, chil, 2, chir).transpose(0, 2, 1, 3).reshape(4, chil, chir)
    refAl, refs, refAr = LOC.split_theta(th, chil, chir, chi_max, eps)
    k_ref = len(refs)
    thd = dev(torch, th, np.complex128)
    kmax = min(chi_max, 2 * chil, 2 * chir)
    Al = torch.zeros((2, chil, kmax), dtype=torch.complex128, device="cuda")
    Ar = torch.zeros((2, kmax, chir), dtype=torch.complex128, device="cuda")
    k = ctypes.c_int(0)
    sig = np.zeros(min(2 * chil, 2 * chir))
    qn.call("qca_svd_split", qn.ptr(thd), qn.ptr(Al), qn.ptr(Ar), chil, chir, chi_max, eps, right,
            ctypes.byref(k), sig.ctypes.data, None)
    assert k.value == k_ref
    kk = k.value
    Al = Al.flatten()[: 2 * chil * kk].reshape(2, chil, kk).cpu().numpy()
    Ar = Ar.flatten()[: 2 * kk * chir].reshape(2, kk, chir).cpu().numpy()
    s_np = np.linalg.svd(M, compute_uv=False)
    assert np.abs(sig - s_np).max() < 1e-13
    # truncated state and isometry, gauge independent
    ref_th = np.einsum("pak,k,qkc->pqac", refAl, refs, refAr)
    got_th = np.einsum("pak,qkc->pqac", Al, Ar)
    assert np.abs(got_th - ref_th).max() < 1e-12
    if right:
        I = np.einsum("pak,pal->kl", Al.conj(), Al)
    else:
        I = np.einsum("pkc,plc->kl", Ar, Ar.conj())
    # Householder products and accumulated rotations lose orthogonality like
    # n * eps in the isometry's length n (512 at the widest split)
    n = 2 * chil if right else 2 * chir
    assert np.abs(I - np.eye(kk)).max() < max(1e-13, 2 * n * np.finfo(float).eps)


@pytest.mark.parametrize("spectrum", ["flat", "pairs", "steps"])
@pytest.mark.parametrize("chil,chir,right", [(17, 17, 1), (24, 24, 0), (24, 25, 1), (40, 25, 0), (45, 77, 0),
                                             (64, 65, 1), (128, 128, 0), (200, 20, 1)])
def test_svd_split_closing_steps(gpu, spectrum, chil, chir, right):
    """Splits whose last sweeps are products on the matrix cores, at column counts
    around the 16-column tiles (34..256): a flat spectrum (all pairs close),
    pairs 1e-6 apart and degenerate plateaus 1e-2 apart, against LAPACK within
    the bounds of test_svd_split."""
    import torch
    rng = np.random.default_rng(chil * 3 + chir + right)
    m, n = 2 * chil, 2 * chir
    U, _ = np.linalg.qr(crand(rng, m, min(m, n)))
    V, _ = np.linalg.qr(crand(rng, n, min(m, n)))
    i = np.arange(min(m, n))
    s = {"flat": 1 + 0.01 * i / len(i), "pairs": 0.93 ** (i // 2) * (1 + 1e-6 * (i % 2)),
         "steps": 10.0 ** (-2 * (i // (len(i) // 4 + 1))),
         "graded": 10.0 ** (-14 * i / len(i)), "rank1": 1.0 * (i == 0)}[spectrum]
    M = (U * s) @ V.conj().T
    M /= np.linalg.norm(M)
    ref = np.linalg.svd(M, compute_uv=False)
    th = dev(torch, M.reshape(2, chil, 2, chir).transpose(0, 2, 1, 3).reshape(4, chil, chir), np.complex128)
    kmax = min(m, n)
    Al = torch.zeros(2 * chil * kmax, dtype=torch.complex128, device="cuda")
    Ar = torch.zeros(2 * kmax * chir, dtype=torch.complex128, device="cuda")
    k = ctypes.c_int(0)
    sig = np.zeros(kmax)
    qn.call("qca_svd_split", qn.ptr(th), qn.ptr(Al), qn.ptr(Ar), chil, chir, kmax, 1e-10, right,
            ctypes.byref(k), sig.ctypes.data, None)
    kk = k.value
    assert kk == LOC.truncation_rank(ref, kmax, 1e-10)
    assert np.abs(sig - ref).max() < 1e-13
    A = Al[: m * kk].cpu().numpy().reshape(m, kk)
    B = Ar[: n * kk].cpu().numpy().reshape(2, kk, chir).transpose(1, 0, 2).reshape(kk, n)
    Q = A if right else B.conj().T
    assert np.abs(Q.conj().T @ Q - np.eye(kk)).max() < max(1e-13, 2 * len(Q) * np.finfo(float).eps)
    # the truncated state, normalised (reference tdvp.py:286-296)
    u, _, vh = np.linalg.svd(M, full_matrices=False)
    kept = (u[:, :kk] * ref[:kk] / np.linalg.norm(ref[:kk])) @ vh[:kk]
    assert np.abs(A @ B - kept).max() < 1e-12


@pytest.mark.parametrize("right", [1, 0])
@pytest.mark.parametrize("spectrum", ["flat", "graded", "rank1"])
@pytest.mark.parametrize("chil,chir", [(1, 1), (1, 2), (2, 2), (2, 1), (4, 4), (5, 4), (8, 8), (8, 9), (16, 16),
                                       (12, 16), (16, 17), (16, 33), (16, 64), (1, 64),
                                       # just past one workgroup's range: 130 and 200 long
                                       (16, 65), (3, 100)])
def test_svd_split_one_workgroup(gpu, spectrum, chil, chir, right):
    """Splits up to 32 x 128 take one workgroup: every half of the round-robin
    (2..32 columns), tall and wide, at the register sizes of the QR (32, 64, 128
    long), against LAPACK within the bounds of test_svd_split."""
    test_svd_split_closing_steps(gpu, spectrum, chil, chir, right)


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("chil,chir,target", [(1, 1, 2), (2, 2, 4), (4, 8, 8), (8, 8, 8), (32, 32, 32),
                                              (8, 4, 4), (16, 64, 32), (128, 256, 256)])
def test_qr_site_matches_lapack(gpu, side, chil, chir, target):
    """Complete QR with LAPACK's conventions: Q and R equal numpy.linalg.qr's,
    including the complement columns (reference mps.py:83-98, tdvp.py:74-78, 95-99)."""
    import torch
    from oracle import mps as OM
    if side == 1:
        target = min(target, 2 * chir)
    else:
        target = min(target, 2 * chil)
    rng = np.random.default_rng(chil + chir + target)
    A = crand(rng, 2, chil, chir)
    if side == 0:
        Q, R = OM.left_qr(A, reduced=False)
        refA = OM.truncate_pad(Q, (2, chil, target))
        refC = OM.truncate_pad(R, (target, chir))
        An = torch.zeros((2, chil, target), dtype=torch.complex128, device="cuda")
        C = torch.zeros((target, chir), dtype=torch.complex128, device="cuda")
    else:
        Q, R = OM.right_qr(A, reduced=False)
        refA = OM.truncate_pad(Q, (2, target, chir))
        refC = OM.truncate_pad(R, (chil, target))
        An = torch.zeros((2, target, chir), dtype=torch.complex128, device="cuda")
        C = torch.zeros((chil, target), dtype=torch.complex128, device="cuda")
    qn.call("qca_qr_site", side, qn.ptr(dev(torch, A, np.complex128)), chil, chir, target,
            qn.ptr(An), qn.ptr(C), None)
    assert np.abs(An.cpu().numpy() - refA).max() < 1e-12
    assert np.abs(C.cpu().numpy() - refC).max() < 1e-12


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n,d,iv", [(6, 1, range(1, 2)), (9, 2, range(2, 5)), (12, 2, range(1, 3)),
                                    (16, 1, range(2, 3))])
def test_exact_apply(gpu, prec, n, d, iv):
    import torch
    rng = np.random.default_rng(n)
    psi = crand(rng, 1 << n)
    ref = AU.apply_h(psi, n, d, iv)
    dt = np.complex128 if prec == 0 else np.complex64
    pd = dev(torch, psi, dt)
    out = torch.zeros_like(pd)
    qn.call("qca_exact_apply_h", prec, qn.ptr(pd), qn.ptr(out), n, d, iv.start, iv.stop, None)
    assert rel(out.cpu().numpy().astype(np.complex128), ref) < (1e-15 if prec == 0 else 1e-6)


def test_exact_expm_and_rho(gpu):
    import torch
    from oracle import exact as OE, mps as OM
    n, d, iv, dt = 10, 2, range(2, 5), 0.2
    pl = [0.0] * n
    pl[4] = pl[5] = pl[6] = 1.0
    ex = OE.ExactOracle(OM.product_state(pl), n, d, iv, dt)
    psi = dev(torch, OM.as_vector(OM.product_state(pl)), np.complex128)
    for _ in range(5):
        it = ctypes.c_int(0)
        qn.call("qca_exact_expm", qn.ptr(psi), n, d, iv.start, iv.stop, dt, 0.0, ctypes.byref(it), None)
        ex.do_time_step()
        assert np.abs(psi.cpu().numpy() - ex.psi).max() < 1e-12
    rho = np.zeros((n, 2, 2), dtype=np.complex128)
    qn.call("qca_exact_rho", qn.ptr(psi), n, rho.ctypes.data, None)
    assert np.abs(rho[:, 1, 1].real - ex.populations()).max() < 1e-13
    assert np.abs(np.trace(rho, axis1=1, axis2=2) - 1).max() < 1e-12


@pytest.mark.parametrize("n,d,iv", [(1, 1, range(0, 1)), (2, 1, range(1, 2)), (7, 3, range(2, 5)),
                                    (8, 2, range(0, 3)), (9, 9, range(3, 40)), (11, 5, range(1, 7)),
                                    (18, 2, range(2, 5)), (19, 4, range(3, 6)), (20, 1, range(-1, 2))])
def test_exact_apply_tiles(gpu, n, d, iv):
    """Tile edges of the state-vector Hamiltonian (256- and 1024-state tiles,
    shorter vectors, neighbourhoods reaching above the tile or beyond the
    chain).  At most n terms per amplitude: n roundings."""
    import torch
    psi = crand(np.random.default_rng(n), 1 << n)
    iv_np = range(max(iv.start, 0), iv.stop)
    ref = AU.apply_h(psi, n, d, iv_np)
    pd = dev(torch, psi, np.complex128)
    out = torch.zeros_like(pd)
    qn.call("qca_exact_apply_h", 0, qn.ptr(pd), qn.ptr(out), n, d, iv.start, iv.stop, None)
    assert np.abs(out.cpu().numpy() - ref).max() <= n * np.finfo(float).eps * max(np.abs(ref).max(), 1)


@pytest.mark.parametrize("n,d,dt,tol", [(2, 1, 0.3, 1e-12), (9, 3, -0.4, 1e-12), (10, 2, 0.0, 1e-14),
                                        # 628 units of tau * N: two substeps
                                        (8, 1, 50.0, 1e-10)])
def test_exact_expm_series(gpu, n, d, dt, tol):
    """The Chebyshev evolution against the dense propagator: backward steps, no
    step, and one longer than a single series; rounding of ~1000 terms and the
    dense phases (eps * tau * N) stay below 1e-10."""
    import torch
    from oracle import exact as OE, mps as OM
    As = OM.product_state([0.1 + 0.08 * i for i in range(n)])
    ex = OE.ExactOracle(As, n, d, range(1, 3), dt)
    psi = dev(torch, ex.psi, np.complex128)
    it = ctypes.c_int(0)
    qn.call("qca_exact_expm", qn.ptr(psi), n, d, 1, 3, dt, 0.0, ctypes.byref(it), None)
    ex.do_time_step()
    assert it.value >= 2
    assert np.abs(psi.cpu().numpy() - ex.psi).max() < tol


def test_exact_expm_refuses_non_finite(gpu):
    """A state with a NaN is refused and left as it was."""
    import torch
    psi = torch.zeros(1 << 10, dtype=torch.complex128, device="cuda")
    psi[3], psi[700] = 1.0, float("nan")
    before = psi.cpu().numpy()
    with pytest.raises(qn.QcaError) as e:
        qn.call("qca_exact_expm", qn.ptr(psi), 10, 1, 1, 2, 0.2, 0.0, None, None)
    assert e.value.code == -4
    assert np.array_equal(psi.cpu().numpy(), before, equal_nan=True)


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("chi_row,chi_col,target", [
    # panel edges: one column more than a panel, ragged last panels, single rows left
    (9, 9, 9), (8, 16, 16), (17, 17, 17), (33, 31, 31),
    # fewer rows than columns: a last panel of 10 or 8 reflectors with columns beside and right of it
    (5, 24, 10), (12, 40, 24), (3, 17, 6),
    # every register block of the panel (64-row chunks), complement columns up to a square Q
    (40, 20, 80), (90, 64, 180), (150, 100, 100), (200, 33, 48), (256, 40, 512)])
def test_qr_panels_match_lapack(gpu, side, chi_row, chi_col, target):
    """The blocked QR at its panel and register-block edges, against numpy.linalg.qr
    in LAPACK's conventions (as test_qr_site_matches_lapack)."""
    import torch
    from oracle import mps as OM
    rng = np.random.default_rng(chi_row * 7 + chi_col + side)
    chil, chir = (chi_row, chi_col) if side == 0 else (chi_col, chi_row)
    A = crand(rng, 2, chil, chir)
    if side == 0:
        Q, R = OM.left_qr(A, reduced=False)
        refA, refC = OM.truncate_pad(Q, (2, chil, target)), OM.truncate_pad(R, (target, chir))
    else:
        Q, R = OM.right_qr(A, reduced=False)
        refA, refC = OM.truncate_pad(Q, (2, target, chir)), OM.truncate_pad(R, (chil, target))
    An = torch.zeros(refA.shape, dtype=torch.complex128, device="cuda")
    C = torch.zeros(refC.shape, dtype=torch.complex128, device="cuda")
    Ad = dev(torch, A, np.complex128)
    qn.call("qca_qr_site", side, qn.ptr(Ad), chil, chir, target, qn.ptr(An), qn.ptr(C), None)
    assert np.abs(An.cpu().numpy() - refA).max() < 1e-12
    assert np.abs(C.cpu().numpy() - refC).max() < 1e-12


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("chi_row,chi_col,col", [(1, 2, 0), (9, 9, 3), (40, 20, 17), (150, 33, 32), (260, 5, 2)])
@pytest.mark.parametrize("scale", [1e-156, 1e-160, 1e-170, 1e-300, 0.0, 1e160])
def test_qr_column_out_of_range(gpu, scale, side, chi_row, chi_col, col):
    """A column whose squares under- or overflow (a vanishing Schmidt direction):
    numpy.linalg.qr's factors within the bound of test_qr_panels_match_lapack,
    each column of R relative to its own size."""
    import torch
    from oracle import mps as OM
    rng = np.random.default_rng(chi_row + chi_col + side)
    chil, chir = (chi_row, chi_col) if side == 0 else (chi_col, chi_row)
    A = crand(rng, 2, chil, chir)
    (A[:, :, col] if side == 0 else A[:, col])[...] *= scale
    target = 2 * chi_row
    Q, R = OM.left_qr(A, reduced=False) if side == 0 else OM.right_qr(A, reduced=False)
    refA = OM.truncate_pad(Q, (2, chil, target) if side == 0 else (2, target, chir))
    refC = OM.truncate_pad(R, (target, chir) if side == 0 else (chil, target))
    An = torch.zeros(refA.shape, dtype=torch.complex128, device="cuda")
    C = torch.zeros(refC.shape, dtype=torch.complex128, device="cuda")
    Ad = dev(torch, A, np.complex128)
    qn.call("qca_qr_site", side, qn.ptr(Ad), chil, chir, target, qn.ptr(An), qn.ptr(C), None)
    assert np.abs(An.cpu().numpy() - refA).max() < 1e-12
    got, ref = (C.cpu().numpy(), refC) if side == 0 else (C.cpu().numpy().T, refC.T)
    size = np.abs(ref).max(axis=0)
    assert (np.abs(got - ref).max(axis=0) <= 1e-12 * size).all()


@pytest.mark.parametrize("right", [1, 0])
@pytest.mark.parametrize("chil,chir", [(4, 5), (12, 16), (16, 40), (40, 33)])
@pytest.mark.parametrize("scale", [1e-156, 1e-160, 0.0])
def test_svd_split_column_out_of_range(gpu, scale, chil, chir, right):
    """Splits with a column and a row whose squares underflow, against LAPACK within
    the bounds of test_svd_split."""
    import torch
    rng = np.random.default_rng(chil + chir)
    m, n = 2 * chil, 2 * chir
    M = crand(rng, m, n)
    M[:, 1] *= scale
    M[2] *= scale
    M /= np.linalg.norm(M)
    th = dev(torch, M.reshape(2, chil, 2, chir).transpose(0, 2, 1, 3).reshape(4, chil, chir), np.complex128)
    kmax = min(m, n)
    Al = torch.zeros(m * kmax, dtype=torch.complex128, device="cuda")
    Ar = torch.zeros(n * kmax, dtype=torch.complex128, device="cuda")
    k = ctypes.c_int(0)
    sig = np.zeros(kmax)
    qn.call("qca_svd_split", qn.ptr(th), qn.ptr(Al), qn.ptr(Ar), chil, chir, kmax, 1e-10, right, ctypes.byref(k),
            sig.ctypes.data, None)
    u, ref, vh = np.linalg.svd(M, full_matrices=False)
    kk = k.value
    assert kk == LOC.truncation_rank(ref, kmax, 1e-10)
    assert np.abs(sig - ref).max() < 1e-13
    A = Al[: m * kk].cpu().numpy().reshape(m, kk)
    B = Ar[: n * kk].cpu().numpy().reshape(2, kk, chir).transpose(1, 0, 2).reshape(kk, n)
    Q = A if right else B.conj().T
    assert np.abs(Q.conj().T @ Q - np.eye(kk)).max() < 1e-13
    kept = (u[:, :kk] * ref[:kk] / np.linalg.norm(ref[:kk])) @ vh[:kk]
    assert np.abs(A @ B - kept).max() < 1e-12


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind,chil,chir", [(0, 3, 4), (1, 24, 24), (2, 33, 17)])
@pytest.mark.parametrize("where", ["L", "R", "x", "huge"])
def test_krylov_expm_refuses_non_finite(gpu, where, kind, chil, chir, prec):
    """A NaN in an environment or in the state, or a state whose norm overflows, is
    QCA_ERR_NOT_CONVERGED, and the state is left as it was."""
    import torch
    rng = np.random.default_rng(chil)
    W = AU.bulk_tensor(2, range(2, 5))
    D = W.shape[2]
    Wk = None if kind == 2 else np.ascontiguousarray(LOC.merge_w(W, W) if kind == 0 else W, dtype=np.complex128)
    x = crand(rng, {0: 4, 1: 2, 2: 1}[kind], chil, chir)
    L, R = herm_env(rng, chil, D), herm_env(rng, chir, D)
    if where == "huge":
        x *= 1e200
    else:
        # channel 0 of an environment carries the finished terms: it is always read
        {"L": L[:, 0], "R": R[:, -1], "x": x[0]}[where][0, 0] = float("nan")
    dt = np.complex128 if prec == 0 else np.complex64
    xd, Ld, Rd = dev(torch, x, np.complex128), dev(torch, L, dt), dev(torch, R, dt)
    with pytest.raises(qn.QcaError) as e:
        qn.call("qca_krylov_expm", prec, kind, qn.ptr(xd), qn.ptr(Ld), qn.ptr(Rd),
                Wk.ctypes.data if Wk is not None else None, D, D, chil, chir, 0.05, 0.0, None, None)
    assert e.value.code == -4
    assert np.array_equal(xd.cpu().numpy(), x, equal_nan=True)


def exact_h(n, d, lo, hi):
    """The rule Hamiltonian on vectors of any numpy type."""
    x = np.arange(1 << n)
    bits = [x >> (n - 1 - i) & 1 for i in range(n)]
    alive = [sum(bits[j] for j in range(max(0, i - d), min(n, i + d + 1)) if j != i) for i in range(n)]
    return lambda v: sum(v[x ^ (1 << (n - 1 - i))] * ((alive[i] >= lo) & (alive[i] < hi)) for i in range(n))


@pytest.mark.parametrize("n,d,lo,hi,dt", [(12, 2, 2, 5, 0.1), (13, 2, 2, 4, 0.1), (13, 1, 1, 3, 0.2), (14, 2, 1, 5, 0.5)])
def test_exact_expm_rounding(gpu, n, d, lo, hi, dt):
    """At the default tolerance nothing but the rounding of the series' K terms is
    left: sqrt(K) unit roundoffs in the 2-norm (they add up like a random walk),
    against a Taylor series in extended precision."""
    import torch
    rng = np.random.default_rng(n)
    psi = np.ones(1)
    for alive in rng.random(n) < 0.3:
        p = abs(float(alive) - 0.2 * rng.random())
        psi = np.kron(psi, [np.sqrt(1 - p), np.sqrt(p)])
    H = exact_h(n, d, lo, hi)
    ref = psi.astype(np.clongdouble)
    steps = int(np.ceil(np.pi / 2 * dt * n))
    h = -1j * np.longdouble(1.5707963267948966 * dt) / steps
    for _ in range(steps):
        term = ref
        for k in range(1, 30):
            term = H(term) * (h / k)
            ref = ref + term
    pd = dev(torch, psi, np.complex128)
    it = ctypes.c_int(0)
    qn.call("qca_exact_expm", qn.ptr(pd), n, d, lo, hi, dt, 0.0, ctypes.byref(it), None)
    err = np.sqrt(float((np.abs(pd.cpu().numpy() - ref) ** 2).sum()))
    assert err < np.sqrt(it.value) * 1.1102230246251565e-16


def test_exact_expm_tolerance_of_a_long_step(gpu):
    """The tolerance holds for the whole of a step of 12566 units of tau * N (25
    substeps), not for each of them."""
    import torch
    n, d, lo, hi, dt, tol = 8, 1, 1, 3, 1000.0, 1e-4
    H = exact_h(n, d, lo, hi)
    Hm = np.stack([H(e) for e in np.eye(1 << n)])
    lam, U = np.linalg.eigh(Hm)
    psi = crand(np.random.default_rng(0), 1 << n)
    psi /= np.linalg.norm(psi)
    ref = U @ (np.exp(-1j * np.pi / 2 * dt * lam) * (U.T @ psi))
    pd = dev(torch, psi, np.complex128)
    qn.call("qca_exact_expm", qn.ptr(pd), n, d, lo, hi, dt, tol, None, None)
    # eigenvalues to a few eps N, phases 1570 times as much: 1e-11
    assert np.linalg.norm(pd.cpu().numpy() - ref) < tol


def extended_qr(M):
    """Complete-QR factors (Q's first columns, R) by Householder reflectors with
    LAPACK's signs, in extended precision."""
    m, n = M.shape
    A = M.astype(np.clongdouble)
    refl = []
    for j in range(min(m, n)):
        x = A[j:, j]
        norm = np.sqrt((np.abs(x) ** 2).sum())
        beta = -norm if x[0].real >= 0 else norm
        tau, v = (beta - x[0]) / beta, x / (x[0] - beta)
        v[0] = 1
        A[j:, j:] -= np.outer(v, np.conj(tau) * (v.conj()[:, None] * A[j:, j:]).sum(axis=0))
        refl.append((v, tau))
    Q = np.eye(m, n, dtype=np.clongdouble)
    for j in reversed(range(len(refl))):
        v, tau = refl[j]
        Q[j:] -= np.outer(v, tau * (v.conj()[:, None] * Q[j:]).sum(axis=0))
    return Q, np.triu(A[:n])


@pytest.mark.parametrize("side,chil,chir", [(0, 180, 200), (0, 256, 256), (1, 256, 256)])
def test_qr_rounding(gpu, side, chil, chir):
    """Each of up to 16 block reflectors rounds a column of Q once at its own size
    and brings the rounding of 16 reflectors as a unit of about the same: 8 unit
    roundoffs in the 2-norm, 4 in R, whose columns take part in fewer of them."""
    import torch
    A = crand(np.random.default_rng(chil), 2, chil, chir)
    A *= np.logspace(0, -2, chir if side == 0 else chil)[(None, None, slice(None)) if side == 0 else (None, slice(None), None)]
    M = A.reshape(2 * chil, chir) if side == 0 else A.transpose(0, 2, 1).reshape(2 * chir, chil)
    Q, R = extended_qr(M)
    t = M.shape[1]
    An = torch.zeros((2, chil, t) if side == 0 else (2, t, chir), dtype=torch.complex128, device="cuda")
    C = torch.zeros((t, t), dtype=torch.complex128, device="cuda")
    Ad = dev(torch, A, np.complex128)
    qn.call("qca_qr_site", side, qn.ptr(Ad), chil, chir, t, qn.ptr(An), qn.ptr(C), None)
    gotq = An.cpu().numpy().reshape(len(M), t) if side == 0 else An.cpu().numpy().transpose(0, 2, 1).reshape(len(M), t)
    gotr = C.cpu().numpy() if side == 0 else C.cpu().numpy().T
    u = 1.1102230246251565e-16
    assert np.sqrt(float((np.abs(gotq - Q) ** 2).sum() / t)) < 8 * u
    assert np.sqrt(float((np.abs(gotr - R) ** 2).sum() / (np.abs(R) ** 2).sum())) < 4 * u


@pytest.mark.parametrize("op,chil,chir", [("left", 128, 128), ("right", 128, 128), ("left", 160, 200), ("right", 200, 160),
                                          (1, 100, 128), (2, 100, 100), (2, 160, 200)])
def test_fp32_sums_stay_short(gpu, op, chil, chir):
    """FP32 contractions in 32x32 tiles, random operands: over a chain of 64 additions
    the partial sum grows like sqrt(i), and so does its rounding error (u / sqrt(3) of
    it at each one) like a random walk: u sqrt(64 / 2) / sqrt(3) = 2.0e-7 of the sum
    in each of the two products, 2.8e-7 together in the 2-norm."""
    import torch
    rng = np.random.default_rng(chil + chir)
    W = AU.bulk_tensor(2, range(2, 5))
    D = W.shape[2]
    c64 = lambda a: np.ascontiguousarray(a, dtype=np.complex64)
    L, R = c64(crand(rng, chil, D, chil) / chil), c64(crand(rng, chir, D, chir) / chir)
    Wh = np.ascontiguousarray(W, dtype=np.complex128)
    if op in ("left", "right"):
        side = int(op == "right")
        A = c64(crand(rng, 2, chil, chir) / np.sqrt(chil + chir))
        E = R if side else L
        ref = (LOC.env_right if side else LOC.env_left)(*[a.astype(np.complex128) for a in (E, A)], W)
        out = torch.zeros(ref.shape, dtype=torch.complex64, device="cuda")
        Ad, Ed = dev(torch, A, np.complex64), dev(torch, E, np.complex64)
        qn.call("qca_env_update", 1, side, qn.ptr(Ad), qn.ptr(Ed), qn.ptr(out), Wh.ctypes.data, D, D, chil, chir, None)
    else:
        x = c64(crand(rng, chil, chir) if op == 2 else crand(rng, 2, chil, chir))
        args = [a.astype(np.complex128) for a in (x, L, R)]
        ref = LOC.bond_apply(*args) if op == 2 else LOC.heff_apply(*args, W)
        out = torch.zeros(ref.shape, dtype=torch.complex64, device="cuda")
        xd, Ld, Rd = dev(torch, x, np.complex64), dev(torch, L, np.complex64), dev(torch, R, np.complex64)
        qn.call("qca_heff_apply", 1, op, qn.ptr(xd), qn.ptr(out), qn.ptr(Ld), qn.ptr(Rd),
                None if op == 2 else Wh.ctypes.data, D, D, chil, chir, None)
    assert np.linalg.norm(out.cpu().numpy() - ref) < 2.8e-7 * np.linalg.norm(ref)


@pytest.mark.parametrize("right", [1, 0])
@pytest.mark.parametrize("chi", [4, 6, 8, 10, 16])
def test_svd_split_small_isometry_is_normalised(gpu, chi, right):
    """The isometry's columns are divided by their own norms: 6 unit roundoffs in the
    squared norm (the division, and sum and root of the norm, twice each)."""
    import torch
    for seed in range(4):
        rng = np.random.default_rng(100 * chi + seed)
        w = np.logspace(0, -7, chi)
        th = crand(rng, 4, chi, chi) * w[:, None] * w
        th /= np.linalg.norm(th)
        Al = torch.zeros(4 * chi * chi, dtype=torch.complex128, device="cuda")
        Ar = torch.zeros(4 * chi * chi, dtype=torch.complex128, device="cuda")
        k = ctypes.c_int(0)
        thd = dev(torch, th, np.complex128)
        qn.call("qca_svd_split", qn.ptr(thd), qn.ptr(Al), qn.ptr(Ar), chi, chi, 2 * chi, 1e-10, right,
                ctypes.byref(k), None, None)
        kk = k.value
        n = 2 * chi * kk
        Q = Al[:n].cpu().numpy().reshape(2 * chi, kk) if right else \
            Ar[:n].cpu().numpy().reshape(2, kk, chi).transpose(0, 2, 1).reshape(2 * chi, kk)
        norm2 = (np.abs(Q.astype(np.clongdouble)) ** 2).sum(axis=0)
        assert np.abs(norm2 - 1).max() < 6 * 1.1102230246251565e-16


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("chi_row,chi_col,target", [(1, 1, 1), (64, 1, 1), (256, 2, 4), (1, 64, 2), (1, 65, 2), (2, 3, 4),
                                                    (256, 3, 3)])
def test_qr_few_reflectors(gpu, side, chi_row, chi_col, target):
    """On both sides of the choice between the one-workgroup and the blocked QR: one,
    two and three reflectors, few and many columns beside them."""
    test_qr_panels_match_lapack(gpu, side, chi_row, chi_col, target)


@pytest.mark.parametrize("spectrum", ["flat", "graded", "rank1"])
@pytest.mark.parametrize("chil,chir", [(65, 1), (65, 8), (72, 9), (128, 16), (129, 4), (256, 16)])
def test_svd_split_tall(gpu, spectrum, chil, chir):
    """Splits with more than 128 rows and up to 32 columns (one and two QR panels,
    up to 256 and up to 512 rows), against LAPACK within the bounds of
    test_svd_split."""
    test_svd_split_closing_steps(gpu, spectrum, chil, chir, 1)
    test_svd_split_closing_steps(gpu, spectrum, chir, chil, 0)


@pytest.mark.parametrize("dt", [0.3, -1.0, 5.0])
@pytest.mark.parametrize("n,d,lo,hi,states,few", [
    (10, 1, 2, 3, [0], True),                                   # dead: H psi = 0
    (10, 1, 2, 3, [0b0001110000], True),                        # a blinker
    (10, 2, 2, 5, [0, 1, 0b1000000001], True),                  # still lives in superposition
    (10, 1, 2, 3, [0b0111000111, 0b1110000000], True),          # blinkers side by side
    (10, 1, 1, 3, [0b0000100000], False),                       # spreads over more than 64 states
    (6, 2, 1, 4, list(range(64)), True),                        # every state, and just that many
    (7, 2, 1, 4, list(range(64)), False), (7, 2, 1, 4, list(range(65)), False),
    (10, 1, 0, 1, list(range(70)), False)])
def test_exact_expm_few_states(gpu, n, d, lo, hi, states, few, dt):
    """States on few basis states, closed under the Hamiltonian or not, against the
    dense propagator (rounding of the phases: eps * tau * N); a closed set takes no
    more applications than a series for its own few states."""
    import torch
    H = exact_h(n, d, lo, hi)
    lam, U = np.linalg.eigh(np.stack([H(e) for e in np.eye(1 << n)]))
    psi = np.zeros(1 << n, dtype=complex)
    psi[states] = crand(np.random.default_rng(len(states)), len(states))
    psi /= np.linalg.norm(psi)
    ref = U @ (np.exp(-1j * np.pi / 2 * dt * lam) * (U.T @ psi))
    pd = dev(torch, psi, np.complex128)
    it = ctypes.c_int(0)
    qn.call("qca_exact_expm", qn.ptr(pd), n, d, lo, hi, dt, 0.0, ctypes.byref(it), None)
    assert np.abs(pd.cpu().numpy() - ref).max() < 1e-12
    if few:
        degree = max(int((H(np.eye(1 << n)[x]) != 0).sum()) for x in range(1 << n)) if n < 8 else 4
        assert it.value <= np.pi / 2 * abs(dt) * degree * 2 + 30
    if states == [0]:
        assert it.value == 1


@pytest.mark.parametrize("n,d,iv", [(1, 1, range(0, 1)), (7, 3, range(2, 5)), (8, 2, range(0, 3)), (9, 9, range(3, 40)),
                                    (18, 2, range(2, 5)), (19, 4, range(3, 6)), (20, 1, range(0, 2))])
def test_exact_apply_tiles_fp32(gpu, n, d, iv):
    """The edges of test_exact_apply_tiles in complex64: at most n terms per
    amplitude, n roundings."""
    import torch
    psi = crand(np.random.default_rng(n), 1 << n).astype(np.complex64)
    ref = AU.apply_h(psi.astype(np.complex128), n, d, iv)
    pd = dev(torch, psi, np.complex64)
    out = torch.zeros_like(pd)
    qn.call("qca_exact_apply_h", 1, qn.ptr(pd), qn.ptr(out), n, d, iv.start, iv.stop, None)
    assert np.abs(out.cpu().numpy() - ref).max() <= n * np.finfo(np.float32).eps * max(np.abs(ref).max(), 1)
