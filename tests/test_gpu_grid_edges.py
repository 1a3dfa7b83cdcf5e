"""GPU tests of the operator and the solves at grid edges where their kernels
change: odd and even edges, every radix (up to 13), the smallest grids, the
last edge of each elements-per-thread class of the slab kernels (88), of the
slab kernels (126) and the first beyond them, and the edges where
tangent_homo's contraction gets a launch of its own (40) or shares
fft_grid.hip's kernels with the large-grid plans (64).

G_K_dF against the same projection through numpy's FFT (1e-12 of the largest
value, as the oracle comparison of test_gpu_parity); the CG solution through
its residual, formed again by a separate operator application; tangent_homo
against one cpfft_pcg solve per column (1e-9)."""
import numpy as np
import pytest

import cpfft_amd as C
import oracle_lib as O
from cpfft_amd.microstructure import polycrystal

pytestmark = pytest.mark.gpu


def _solver(N, mode):
    _, ang = polycrystal(N, 4, 5 * N)
    return C.Solver(N, ang, C.Material(), dt=0.25, gamma_mode=mode)


def _project(A, N):
    h = np.fft.rfftn(A.reshape(9, N, N, N), axes=(1, 2, 3))
    f = np.fft.fftfreq(N, 1.0 / N)
    q = [f[:, None, None], f[None, :, None], np.arange(N // 2 + 1.0)[None, None, :]]
    qq = q[0] ** 2 + q[1] ** 2 + q[2] ** 2
    w = np.where(qq > 0, 1.0 / np.maximum(qq, 1.0), 0.0)
    if N % 2 == 0:
        for v in q:
            w = w * (abs(v) != N // 2)
    out = np.empty_like(h)
    for i in range(3):
        aq = (h[3 * i] * q[0] + h[3 * i + 1] * q[1] + h[3 * i + 2] * q[2]) * w
        for j in range(3):
            out[3 * i + j] = aq * q[j]
    return np.fft.irfftn(out, s=(N, N, N), axes=(1, 2, 3)).reshape(9, -1)


@pytest.mark.parametrize("N", [2, 3, 9, 10, 11, 13, 14, 16, 25, 26, 32, 33, 45, 48, 52, 81, 88, 90,
                               125, 126, 130])
def test_gkdf_edges(N):
    V = N ** 3
    rng = np.random.default_rng(N)
    F = rng.standard_normal((9, V))
    K = rng.standard_normal((81, V)) if N <= 52 else None
    want = _project(F, N)
    for mode in (0, 1) if N % 2 else (1,):
        s = _solver(N, mode)
        s.upload(C.DFM, F)
        s.gkdf(C.DFM, C.B, 0)
        got = s.download(C.B)
        assert abs(got - want).max() <= 1e-12 * max(abs(want).max(), 1e-300)
        if K is not None:
            s.upload(C.K4, K)
            s.gkdf(C.DFM, C.B, 1)
            wk = _project(np.stack([(K[9 * r:9 * r + 9] * F).sum(0) for r in range(9)]), N)
            assert abs(s.download(C.B) - wk).max() <= 1e-12 * max(abs(wk).max(), 1e-300)
        s.close()


@pytest.mark.parametrize("N,mode", [(3, 0), (9, 0), (9, 1), (10, 1), (39, 0), (40, 1), (88, 1),
                                    (90, 1), (126, 1), (130, 1), (135, 0)])
def test_cg_edges(N, mode):
    s = _solver(N, mode)
    s.drive_eps_sig(1, 0)
    rng = np.random.default_rng(7 * N)
    s.upload(C.DFM, 1e-3 * rng.standard_normal((9, N ** 3)))
    s.gkdf(C.DFM, C.B, 1)
    s.dscal(-1.0, C.B)
    b = s.download(C.B)
    tol = 1e-8
    out = []
    for graphs in (False, True):
        s.set_graphs(graphs)
        rc, it, relres = s.pcg(C.B, C.WORK, tol)
        assert rc == 0 and it > 1
        out.append((it, relres, s.download(C.WORK)))
    assert out[0][:2] == out[1][:2] and np.array_equal(out[0][2], out[1][2])
    s.gkdf(C.WORK, C.DFM, 1)
    true_rel = np.linalg.norm(b - s.download(C.DFM)) / np.linalg.norm(b)
    assert true_rel <= tol
    assert abs(true_rel - out[0][1]) <= 1e-3 * tol
    s.close()


@pytest.mark.parametrize("N,mode", [(9, 0), (9, 1), (16, 1), (39, 0), (39, 1), (40, 1), (45, 0),
                                    (64, 1)])
def test_tangent_homo_edges(N, mode):
    s = _solver(N, mode)
    s.drive_eps_sig(1, 0)
    K = s.download(C.K4)
    got = s.tangent_homo(1e-8).reshape(9, 9)  # [j][i]
    for i in range(9):
        E = np.zeros(9)
        E[i] = 1.0
        s.fill9(C.DFM, E)
        s.gkdf(C.DFM, C.B, 1)
        s.dscal(-1.0, C.B)
        assert s.pcg(C.B, C.WORK, 1e-8)[0] in (0, 1)
        x = s.download(C.WORK)
        x[i] += 1.0
        want = np.array([(K[9 * j:9 * j + 9] * x).sum(0).mean() for j in range(9)])
        assert abs(got[:, i] - want).max() <= 1e-9 * abs(want).max()
    s.close()


@pytest.mark.parametrize("N,tol", [(20, 1e-2), (40, 1e-2), (48, 1e-1)])
def test_solves_with_the_references_even_operator(N, tol):
    """The reference's operator on even edges, where it is no projection (CG
    converges to a loose tolerance only): p.q from the inverse pass and an
    update of its own, for one system and for nine, these with the contraction in
    the forward pass (20) and in a launch of its own whose result the inverse
    pass overwrites (40, 48), over two host round trips (20, 40).  Against the
    oracle: equal iteration counts, 1e-9 as test_pcg_and_tangent_homo."""
    V = N ** 3
    _, ang = polycrystal(N, 4, 5 * N)
    s = C.Solver(N, ang, C.Material(), dt=0.25, gamma_mode=0)
    s.drive_eps_sig(1, 0)
    K = s.download(C.K4)
    fo = O.FFT(N, 0)
    b = -fo.gkdf(np.ascontiguousarray(K.reshape(9, 9, V)[:, 1]))
    xo, rco, ito, _ = fo.pcg(K, b, tol)
    s.upload(C.B, b)
    rc, it, _ = s.pcg(C.B, C.DFM, tol)
    x = s.download(C.DFM)
    assert rc == rco == 0 and it == ito
    assert abs(x - xo).max() <= 1e-9 * abs(xo).max()
    want = fo.tangent_homo(K, tol)
    for graphs in (False, True):
        s.set_graphs(graphs)
        assert abs(s.tangent_homo(tol) - want).max() <= 1e-9 * abs(want).max()
    s.close()
