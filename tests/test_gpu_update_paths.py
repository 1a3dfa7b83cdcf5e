"""GPU tests of the stress update's instantiations (explicit update, Newton
iteration with and without warm-start candidates, integral and other rate
exponents, Voce exponent one and other) against the oracle, on 5^3 = 125
voxels (a full wavefront and one of 61).

Bars: 1e-9 per output field as in test_gpu_parity for the plain start; for
the warm start, which stops at another point within the local tolerances,
|R| <= max(1e-5 MPa, 5e-5 |R_0|) with |R_0| below a few MPa leaves the stress
within 2e-4 MPa at most of about 40, i.e. 1e-5."""
import numpy as np
import pytest

import cpfft_amd as C
import oracle_lib as O
from cpfft_amd.microstructure import polycrystal

pytestmark = pytest.mark.gpu


def rel(a, b):
    return abs(a - b).max() / max(abs(b).max(), 1e-300)


@pytest.mark.parametrize("slip_set,rate_n,voche_m", [(1, 20.0, 1.0), (1, 17.5, 1.0), (80, 20.0, 0.8),
                                                     (80, 9.0, 1.0), (8, 12.5, 1.2)])
def test_update_instantiations(slip_set, rate_n, voche_m):
    N, dt = 5, 0.25
    V = N ** 3
    _, ang = polycrystal(N, 6, 31)
    rng = np.random.default_rng(slip_set)
    mat = C.Material(slip_set=slip_set, rate_n=rate_n, voche_m=voche_m)
    s = C.Solver(N, ang, mat, dt=dt, gamma_mode=1)
    oc = O.crystal(slip_set=slip_set, rate_n=rate_n, voche_m=voche_m, jac_exact=1)
    Fn = np.zeros((9, V))
    Fn[[0, 4, 8]] = 1.0
    Fn1 = Fn + 5e-5 * rng.standard_normal((9, V))
    Fn1[0] += 2.5e-4
    Fn1[[4, 8]] -= 1.2e-4
    sn = O.state_init(oc, V)
    for step in (1, 2):
        for it in (0, 1):
            s.upload(C.FN, Fn)
            s.upload(C.FN1, Fn1)
            s.upload(C.STATE_N, sn)
            nf = s.drive_eps_sig(step, it)
            Po, Ko, so, st = O.drive_eps_sig(oc, ang, step, it, dt, Fn, Fn1, sn)
            assert nf == st[3]
            assert rel(s.download(C.PN1), Po) < 1e-9, (step, it)
            assert rel(s.download(C.K4), Ko) < 1e-9, (step, it)
            sg = s.download(C.STATE_NP1)
            ns = oc.nslip
            for w0, w1 in [(0, 6), (6, 15), (15, 17), (17, 23), (23, 23 + ns), (23 + ns, 23 + 2 * ns),
                           (23 + 2 * ns, 26 + 2 * ns)]:
                assert rel(sg[w0:w1], so[w0:w1]) < 1e-9, (step, it, w0)
        # again from the iterate just found, at a slightly corrected F
        F2 = Fn1 + 1e-7 * rng.standard_normal((9, V))
        s.upload(C.FN1, F2)
        s.set_warm_start(C.WARM_PREVIOUS)
        l0 = s.local_stats()
        assert s.drive_eps_sig(step, 2) == 0
        l1 = s.local_stats()
        s.set_warm_start(0)
        P2, _, _, st = O.drive_eps_sig(oc, ang, step, 2, dt, Fn, F2, sn)
        assert rel(s.download(C.PN1), P2) < 1e-5
        print(f"\n[warm] step {step}: {l1[0] - l0[0]} local iterations", flush=True)
        sn, Fn = so, Fn1
        Fn1 = Fn + 3e-5 * rng.standard_normal((9, V))
        Fn1[0] += 2.5e-4
        Fn1[[4, 8]] -= 1.2e-4
    s.close()
