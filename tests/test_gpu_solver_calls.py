"""GPU tests of what the solver's calls leave behind beside their results: the
recorded kernel times, the time of a solve with nothing to do, the device
memory a context holds, and the launch shapes it reports."""
import ctypes
import time

import numpy as np
import pytest
import torch

import cpfft_amd as C
from cpfft_amd.microstructure import polycrystal

pytestmark = pytest.mark.gpu


def _solver(N, mode=1):
    _, ang = polycrystal(N, 4, 5 * N)
    return C.Solver(N, ang, C.Material(), dt=0.25, gamma_mode=mode)


def _rhs(s, seed):
    """tangent of the explicit update in K4, a right-hand side in B"""
    s.drive_eps_sig(1, 0)
    rng = np.random.default_rng(seed)
    s.upload(C.DFM, 1e-3 * rng.standard_normal((9, s.V)))
    s.gkdf(C.DFM, C.B, 1)
    s.dscal(-1.0, C.B)


@pytest.mark.parametrize("N,mode", [(16, 1), (9, 0), (64, 1)])
def test_zero_right_hand_side_keeps_recorded_times(N, mode):
    """a solve with nothing to do records nothing and drops nothing"""
    s = _solver(N, mode)
    _rhs(s, N)
    s.set_timing(1)
    rc, it, _ = s.pcg(C.B, C.WORK, 1e-8)
    assert rc == 0 and it > 0
    s.fill9(C.B, np.zeros(9))
    assert s.pcg(C.B, C.WORK, 1e-8) == (1, 0, 0.0)
    assert not s.download(C.WORK).any()
    _, cnt = s.kernel_times()
    assert cnt[0] == it and cnt[2] == it
    s.close()


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("mode", [0, 1])
def test_zero_right_hand_side_returns_early(mode, graphs):
    """Nothing but the norm of b is formed for it: under 0.4 of the time of a
    solve stopped after the eight iterations of a host round trip (a solve whose
    iterations are all enqueued and return one by one takes 0.45 to 0.7)."""
    s = _solver(16, mode)
    _rhs(s, 16)
    s.set_graphs(graphs)
    s.set_cg_maxit(8)
    s.fill9(C.DFM, np.zeros(9))

    def median(f):
        for _ in range(5):
            f()
        v = []
        for _ in range(41):
            t0 = time.perf_counter()
            f()
            s.sync()
            v.append(time.perf_counter() - t0)
        return np.median(v)

    def solve():
        with pytest.raises(C.CpfftError):
            s.pcg(C.B, C.WORK, 1e-12)

    def zero():
        assert s.pcg(C.DFM, C.WORK, 1e-12) == (1, 0, 0.0)

    a = median(zero)
    assert not s.download(C.WORK).any()
    b = median(solve)
    print(f"\n[zero] mode {mode} graphs {graphs}: {a * 1e6:.0f} of {b * 1e6:.0f} us", flush=True)
    assert a < 0.4 * b
    s.close()


@pytest.mark.parametrize("N,systems", [(96, 9), (126, 5), (130, 3)])
def test_tangent_spectra_are_allocated_at_first_use(N, systems):
    """The spectra of tangent_homo's systems, 700 MB at most (twice that above
    126), are not part of what a context that only solves holds.  (The device
    hands out 2 MiB pages, so the free memory tells the size to that much at
    either end.)"""
    free = lambda: torch.cuda.mem_get_info()[0]  # noqa: E731

    def one():
        s = _solver(N)
        s.drive_eps_sig(1, 0)
        s.set_cg_maxit(1)
        s.sync()
        a = free()
        with pytest.raises(C.CpfftError):
            s.tangent_homo(1e-8)
        b = free()
        with pytest.raises(C.CpfftError):
            s.tangent_homo(1e-8)
        assert free() == b
        s.close()
        return a - b

    one()  # loads the kernels
    grown = one()
    want = systems * (9 if N <= 126 else 18) * N * N * (N // 2 + 1) * 16
    assert abs(grown - want) <= 4 << 20
    assert want <= (700 if N <= 126 else 1400) << 20


@pytest.mark.parametrize("N,mode,graphs", [(96, 1, True), (126, 1, False), (130, 1, True),
                                           (135, 0, False)])
def test_tangent_homo_in_groups(N, mode, graphs):
    """tangent_homo where nine systems share a launch with more than 64 KiB of
    LDS a block (96), where five and four do (126) and where fewer share the
    five kernels above 126: two columns, of the first and the last group,
    against a cpfft_pcg solve each (1e-9, as test_tangent_homo_edges)."""
    s = _solver(N, mode)
    s.drive_eps_sig(1, 0)
    s.set_graphs(graphs)
    got = s.tangent_homo(1e-8).reshape(9, 9)  # [j][i]
    K = s.download(C.K4)
    for i in (1, 8):
        E = np.zeros(9)
        E[i] = 1.0
        s.fill9(C.DFM, E)
        s.gkdf(C.DFM, C.B, 1)
        s.dscal(-1.0, C.B)
        assert s.pcg(C.B, C.WORK, 1e-8)[0] == 0
        x = s.download(C.WORK)
        x[i] += 1.0
        want = np.array([np.einsum("cv,cv->", K[9 * j:9 * j + 9], x) for j in range(9)]) / s.V
        assert abs(got[:, i] - want).max() <= 1e-9 * abs(want).max()
    s.close()


@pytest.mark.parametrize("N", [20, 64, 96])
def test_displacements_into_any_memory(N):
    """cpfft_f2disp into pageable, pinned and device memory: the same bytes (20^3
    fits one direct copy), and into pinned memory, which needs no staging, in
    under 0.9 of the time (staged, the two differ by a few per cent)."""
    s = _solver(N)
    rng = np.random.default_rng(N)
    s.upload(C.FN1, np.eye(3).reshape(9, 1) + 1e-3 * rng.standard_normal((9, s.V)))
    ln = np.array([1.0, 1.25, 0.8])
    n = 3 * (N + 1) ** 3
    page = np.full(n, np.nan)
    pin = torch.full((n,), float("nan"), dtype=torch.float64).pin_memory()
    dev = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()

    def call(p):
        assert C.lib().cpfft_f2disp(s.h, s.field(C.FN1), C._p(ln), ctypes.cast(p, C._dp)) == 0

    def median(p):
        v = []
        for _ in range(25):
            t0 = time.perf_counter()
            call(p)
            v.append(time.perf_counter() - t0)
        return np.median(v[4:])

    a, b = median(page.ctypes.data), median(pin.data_ptr())
    call(dev.data_ptr())
    print(f"\n[f2disp] {N}: pageable {a * 1e6:.0f}, pinned {b * 1e6:.0f} us", flush=True)
    assert np.isfinite(page).all()
    assert np.array_equal(page, pin.numpy()) and np.array_equal(page, dev.cpu().numpy())
    if N == 96:
        assert b < 0.9 * a
    s.close()


@pytest.mark.parametrize("N,mode", [(90, 1), (45, 0)])
def test_times_of_a_solve_are_the_operators(N, mode):
    """The operator's time within a solve is that of all its kernels: at least
    0.9 of an application's own (it also forms the direction), and with the
    textbook operator, whose inverse pass updates the vectors too, what is left
    for the update is under a fifth of it."""
    s = _solver(N, mode)
    _rhs(s, N)
    s.set_timing(1)
    for _ in range(20):
        s.gkdf(C.DFM, C.WORK, 1)
    gk, n = s.kernel_times()
    assert n[0] == 20
    s.set_timing(1)
    assert s.pcg(C.B, C.WORK, 1e-8)[0] == 0
    cg, _ = s.kernel_times()
    print(f"\n[times] {N}: G_K_dF {gk[0] * 1e3:.1f}, in a solve {cg[0] * 1e3:.1f} + {cg[2] * 1e3:.1f} us",
          flush=True)
    assert cg[0] >= 0.9 * gk[0]
    if mode == 1:
        assert cg[2] < 0.2 * cg[0]
    s.close()


@pytest.mark.parametrize("N,mode", [(16, 1), (45, 0), (96, 1), (126, 1), (128, 1)])
def test_times_count_applications(N, mode):
    """tangent_homo's right-hand sides are nine applications, however many share
    a launch; the average is an application's (launched together they take less
    than alone)."""
    s = _solver(N, mode)
    s.drive_eps_sig(1, 0)
    s.set_timing(1)
    s.gkdf(C.DFM, C.B, 0)
    for _ in range(20):
        s.gkdf(C.DFM, C.B, 0)
    one, _ = s.kernel_times()
    s.set_cg_maxit(1)
    with pytest.raises(C.CpfftError):
        s.tangent_homo(1e-8)
    s.set_timing(1)
    with pytest.raises(C.CpfftError):
        s.tangent_homo(1e-8)
    avg, cnt = s.kernel_times()
    print(f"\n[times] {N}: alone {one[3] * 1e3:.1f}, in tangent_homo {avg[3] * 1e3:.1f} us", flush=True)
    assert cnt[3] == 9
    assert 0.0 < avg[3] < 1.5 * one[3]
    s.close()


def _shapes(s):
    """every shape cpfft_set_tune takes that differs from the one set in one place"""
    now = s.tune()
    for k in range(4):
        for v in range(1, 65):
            shape = list(now)
            shape[k] = v
            if v == now[k]:
                continue
            try:
                s.set_tune(shape)
            except C.CpfftError:
                continue
            assert s.tune() == shape
            yield shape
    s.set_tune(now)


@pytest.mark.parametrize("N,mode,waves", [(16, 1, 2), (32, 1, 2), (48, 1, 3), (16, 0, 3), (32, 0, 3),
                                          (48, 0, 5)])
def test_reported_shapes_are_the_launched_ones(N, mode, waves):
    """out[3] of cpfft_get_tune: wavefronts of the x pass, whose blocks take eight
    x lines of two (textbook operator) or three (reference's) components, two
    points a thread below N = 32, else four; and with the reference's operator
    the shapes change no result either"""
    s = _solver(N, mode)
    assert s.tune()[3] == waves
    if mode == 0:
        _rhs(s, N)
        s.set_cg_maxit(20)

        def run():
            s.gkdf(C.DFM, C.WORK, 0)
            g = s.download(C.WORK)
            C.lib().cpfft_pcg(s.h, s.field(C.B), s.field(C.WORK), 1e-8, None, None)
            return g, s.download(C.WORK)

        ref = run()
        tried = 0
        for shape in _shapes(s):
            got = run()
            assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1]), shape
            tried += 1
        assert tried >= 3
    s.close()


def test_shapes_are_tuned_for_each_operator():
    """a choice timed with one operator, whose x pass is another kernel, is not
    taken over by the other: 200 repetitions of eight or more launches take
    longer than a millisecond, a look at the stored choice does not"""
    a, b = _solver(48, 1), _solver(48, 0)
    t0 = time.perf_counter()
    a.autotune(reps=200, force=True)
    t1 = time.perf_counter()
    b.autotune(reps=200)
    t2 = time.perf_counter()
    b.autotune(reps=200)
    t3 = time.perf_counter()
    assert t1 - t0 > 1e-3 and t2 - t1 > 1e-3 and t3 - t2 < 1e-3
    a.close()
    b.close()


@pytest.mark.parametrize("N", [16, 48, 64, 96])
def test_tangent_homo_under_every_shape(N):
    """No shape changes a tangent (the large grids: their systems take none of them)."""
    s = _solver(N)
    s.drive_eps_sig(1, 0)
    ref = s.tangent_homo(1e-6)
    for shape in _shapes(s):
        assert np.array_equal(s.tangent_homo(1e-6), ref), shape
    s.close()


@pytest.mark.parametrize("N,why", [(17, "prime factor above 13"), (34, "prime factor above 13"),
                                   (169, "13 twice"), (228, "above 227 but 256"),
                                   (250, "above 227 but 256")])
def test_refused_edges_and_why(N, why):
    """edges that no kernel serves are refused with -3 and the true reason"""
    m = C.Material()
    cm = C.CMaterial(**{k: getattr(m, k) for k, _ in C.CMaterial._fields_})
    ang = np.zeros((3, N ** 3))
    h = ctypes.c_void_p()
    assert C.lib().cpfft_create(N, ctypes.byref(cm), C._p(ang), 0.25, 1, ctypes.byref(h)) == -3
    assert why in C.lib().cpfft_last_error().decode()
    if N <= 48:
        assert C.lib().cpfft_gkdf_noalloc(N, 1, 8, None, 16, None) == -3


@pytest.mark.parametrize("N,former", [(16, [16, 8, 4, 18]), (32, [32, 16, 2, 9]), (48, [16, 12, 6, 18])])
def test_shapes_a_program_kept_are_taken(N, former):
    """launch shapes of 16, 32 and 48 from before these edges had kernels of their
    own: taken, returned, without a change of results, and gone once tuned"""
    s = _solver(N)
    now = s.tune()
    _rhs(s, N)
    s.gkdf(C.B, C.WORK, 1)
    ref = s.download(C.WORK)
    s.set_tune(former)
    assert s.tune() == former
    s.gkdf(C.B, C.WORK, 1)
    assert np.array_equal(s.download(C.WORK), ref)
    s.set_tune(now)
    assert s.tune() == now
    with pytest.raises(C.CpfftError):
        s.set_tune([7, *now[1:]])
    assert s.tune() == now
    s.set_tune(former)
    assert s.autotune(reps=1, force=True)[3] < 9
    s.close()
