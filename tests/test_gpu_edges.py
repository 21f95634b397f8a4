"""Kernels at the edges of their tiles, against the oracle: relative 2-norm of
the derivative, 1e-11 in FP64 (the L = 0 Poisson operator's conditioning) and
1e-5 with the complex64 mean field, as in test_gpu_parity."""
import numpy as np
import pytest

import td1c_amd
from oracle.oracle import Oracle
from td1c_amd.abi import Problem
from tests import cases as C

pytestmark = pytest.mark.gpu


def hprod_error(prob, lf, path=0):
    import torch

    o = Oracle(prob)
    w = C.wfn_for(prob, o.lcic)
    o.set_wfn0(w)
    ref = o.htot(1.0, lf, w)
    hp = td1c_amd.HProd(prob)
    hp.set_transform_path(path)
    hp.set_wfn0(w)
    out = hp.htot(1.0, lf, hp.to_device(w))
    torch.cuda.synchronize()
    return np.linalg.norm(out.cpu().numpy() - ref) / np.linalg.norm(ref)


# the matrix-core Legendre transform: column tiles of 16 per parity class
# (lmax 14..17, 31..33 around one and two tiles), odd and even numbers of
# theta points (the middle point), orders m whose classes swap, rows that end
# inside a tile of 8 or 16 (nfe * 20 - 1 points)
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("lmax1,lmax2,nlat,mval", [
    (1, 2, 0, [0, 1]), (6, 13, 0, [0, 1]), (7, 14, 16, [0, 1]), (15, 31, 0, [0, -1]), (16, 30, 33, [1, -1]),
    (17, 33, 0, [0, 0]), (31, 63, 0, [0, 1]), (32, 64, 66, [0, 0])])
def test_legendre_tiles(gpu_lib, lmax1, lmax2, nlat, mval, precision):
    prob = Problem(nfe=3, ndvr=20, rmax=9.0, lmax1=lmax1, lmax2=lmax2, nlat=nlat, znuc=4.0, ndcore=2, nel_alpha=2,
                   nel_beta=2, mval=mval, precision=precision)
    assert hprod_error(prob, C.LF_LEN, path=2) < (1e-5 if precision else 1e-11)


# the register-resident mean-field kernels of each orbital partition (frozen
# cores, dynamical cores, active orbitals), one beyond them on either side
# (the generic kernel), and the CI launches of long CI vectors (5 and more
# active orbitals): one determinant short of the LDS budget up to 4900
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nfc,ndc,nact,nel", [
    (0, 5, 0, 0), (0, 12, 0, 0), (0, 0, 2, 2), (0, 0, 3, 2), (1, 0, 2, 2), (1, 0, 3, 4), (0, 1, 3, 2), (1, 1, 2, 2),
    (1, 1, 4, 4), (0, 2, 2, 2), (0, 1, 4, 2), (0, 0, 5, 2), (0, 0, 5, 4), (1, 0, 5, 6), (0, 1, 5, 4), (1, 0, 6, 8),
    (0, 0, 6, 2), (1, 1, 6, 2), (1, 0, 7, 2), (0, 0, 8, 8), (1, 0, 8, 2)])
def test_partitions(gpu_lib, nfc, ndc, nact, nel, precision):
    n = nfc + ndc + nel // 2
    prob = Problem(nfe=3, ndvr=20, rmax=9.0, lmax1=3, lmax2=6, znuc=4.0, nfcore1=nfc, ndcore=ndc, nact=nact, nel_alpha=n,
                   nel_beta=n, lval=[0] * (nfc + ndc + nact), igauge=1, precision=precision)
    assert hprod_error(prob, C.LF_VEL) < (1e-5 if precision else 1e-11)


# occupations graded over ten decades (the CI coefficients of orbital i scaled by
# 10^(-5 i / (n - 1))), for the regularised inverse of the 1-RDM: the weakly
# occupied orbitals dominate the derivative, and a Jacobi sweep that stops at a
# fraction of the largest occupation leaves 5e-11 in it (seed 87)
@pytest.mark.parametrize("n,seed", [(8, 87), (8, 91), (6, 31), (4, 125)])
def test_graded_occupations(gpu_lib, n, seed):
    import torch

    prob = Problem(nfe=3, ndvr=20, rmax=9.0, lmax1=3, lmax2=6, znuc=2.0, nact=n, nel_alpha=1, nel_beta=1, lval=[0] * n,
                   igauge=1)
    o = Oracle(prob)
    w = C.wfn_for(prob, o.lcic)
    rng = np.random.default_rng(seed)
    scale = 10.0 ** np.linspace(0, -5, n)
    ci = scale[:, None] * (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) * scale
    w[-o.lcic:] = ci.ravel() / np.linalg.norm(ci)
    ref = o.htot(1.0, C.LF_VEL, w)
    hp = td1c_amd.HProd(prob)
    got = hp.htot(1.0, C.LF_VEL, hp.to_device(w))
    torch.cuda.synchronize()
    assert np.linalg.norm(got.cpu().numpy() - ref) < 1e-11 * np.linalg.norm(ref)


# the element one-body kernel at orders other than 20 (rows padded to 16, 24
# and 32) and element counts that end inside a block, both gauges, a frozen
# core beside m = 0 and 1; the half step's right-hand sides with it
@pytest.mark.parametrize("igauge", [0, 1])
@pytest.mark.parametrize("ndvr,nfe", [(2, 5), (5, 24), (15, 4), (16, 13), (17, 3), (20, 13), (24, 7), (25, 2), (32, 8)])
def test_onebody_orders(gpu_lib, ndvr, nfe, igauge):
    import torch

    prob = Problem(nfe=nfe, ndvr=ndvr, rmax=1.5 * nfe, lmax1=3, lmax2=6, znuc=5.0, nfcore1=1, ndcore=2, nel_alpha=3,
                   nel_beta=3, mval=[0, 0, 1], lval=[0, 0, 1], igauge=igauge, isplit=1)
    lf = C.LF_VEL if igauge else C.LF_LEN
    assert hprod_error(prob, lf) < 1e-11
    o = Oracle(prob)
    w = C.smooth_wfn_for(prob, o.lcic)
    o.set_wfn0(w)
    o.h1itr_gen(0.005)
    ref, _ = o.h1itr_prop(lf, 0.005, w)
    hp = td1c_amd.HProd(prob)
    hp.set_wfn0(w)
    hp.h1itr_gen(0.01)
    got = hp.h1itr_prop(lf, hp.to_device(w))
    torch.cuda.synchronize()
    assert np.linalg.norm(got.cpu().numpy() - ref) < 1e-11 * np.linalg.norm(ref)


# the observables without frozen cores read the state in place: after an hprod
# of another state, and with rows below l = |m| that no orbital has
@pytest.mark.parametrize("igauge,nact", [(0, 0), (1, 0), (1, 2)])
def test_observables_in_place(gpu_lib, igauge, nact):
    prob = Problem(nfe=5, ndvr=20, rmax=15.0, lmax1=4, lmax2=8, znuc=4.0, ndcore=2 - nact // 2, nact=nact, nel_alpha=2,
                   nel_beta=2, mval=[0, 1] if nact == 0 else [0, 0, 1], igauge=igauge)
    lf = C.LF_VEL if igauge else C.LF_LEN
    o = Oracle(prob)
    w = C.wfn_for(prob, o.lcic)
    rows = w[:prob.nfun * 5 * prob.nr].reshape(prob.nfun, 5, prob.nr)
    ref, ref_p = o.dipole3(lf, w), o.ipx(2, 4.0, lf, w)
    rows[-1, 0] = 7.0
    hp = td1c_amd.HProd(prob)
    d = hp.to_device(w)
    hp.htot(1.0, lf, hp.to_device(w * 0.5))
    scale = max(1.0, np.abs(ref).max())
    assert np.abs(hp.dipole3(lf, d) - ref).max() <= 1e-11 * scale
    assert np.abs(hp.ipx(2, 4.0, lf, d) - ref_p).max() <= 1e-11
    assert np.array_equal(d.cpu().numpy(), w)


# the factors of the exponential propagators, made on the device: one to 31
# interior points per element, 2 elements (one bridge, no reduction step) to
# 161 (the most), with and without a frozen core; made again in
# the buffers of another step size's and another scheme's factors
@pytest.mark.parametrize("ndvr,nfe,nfc", [(2, 2, 0), (2, 161, 1), (5, 24, 0), (20, 2, 1), (20, 9, 0), (32, 5, 1)])
def test_etd_factors(gpu_lib, ndvr, nfe, nfc):
    import torch

    prob = Problem(nfe=nfe, ndvr=ndvr, rmax=max(9.0, 0.2 * nfe), lmax1=2, lmax2=4, znuc=4.0, nfcore1=nfc, ndcore=2 - nfc,
                   nel_alpha=2, nel_beta=2, lval=[0, 0], igauge=1, isplit=1)
    o = Oracle(prob)
    w = C.smooth_wfn_for(prob, o.lcic)
    o.set_wfn0(w)
    o.etdrb_gen(0.01)
    lf = np.zeros(54)
    lf[:27] = np.tile(C.LF_VEL, 3)
    ref = o.etdrb_step(lf, w.copy(), apply_mask=False)
    hp = td1c_amd.HProd(prob)
    hp.set_wfn0(w)
    td1c_amd.ETDRB(hp, 0.02)
    for again in range(2):
        etd = td1c_amd.ETDRB(hp, 0.01)
        d = hp.to_device(w)
        etd.prop(d, lfields=lf, apply_mask=False)
        torch.cuda.synchronize()
        assert np.linalg.norm(d.cpu().numpy() - ref) < 1e-10 * np.linalg.norm(ref)
        td1c_amd.ETDRK4(hp, 0.02)
    hp.close()
