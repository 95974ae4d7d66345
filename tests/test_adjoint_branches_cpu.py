"""The FP64 adjoint body (abt_amd/csrc/adjbody.h) at the edges of its branches, against a plain
torch.autograd model of one triangular aperture and one bin.

The model forms the aperture integral by quadrature (Gauss-Legendre on the collapsed square, 64 x 64
points: exact to rounding for the phases below 70 rad used here), so it knows nothing of edges, series or
divided differences.  Bins are placed by their q (a bin's direction from the centre follows from q, the
aperture's frame and the propagation vector): on and beside the nulls of an edge, where the one denominator hands
over to the edge form and its series; either side of the series about q = 0, and at q = 0; near
enough to the origin that the far geometry does not hold; in the forward fallback; within the k_y clamp.

Tolerances, of the largest gradient component of the group of bins: the exponentials' rounding enters the
gradient of the form factor as at most 1.7e-13 of 2 A, and the form factor falls to ~1e-3 of 2 A at the phases used
here, so 1e-10.  Within the clamp, at 1 - |k_y| = 2e-7, 1 - k_y^2 carries 3e-10 of rounding, squared in the
derivative's denominators: 1e-8.
"""
import numpy as np
import pytest
import torch

from abt_amd import lib
from abt_amd.beams import BeamSet
from tests import emu

LAM = 0.532
K2CLAMP, FWD = float(np.float32(0.999999)), float(np.float32(0.999))
WN = 2.0 * float(np.float32(3.14159265358979)) / LAM


def _unit(a):
    return a / np.linalg.norm(a)


def _frame(v, P):
    n = np.cross(v[1] - v[0], v[2] - v[0])
    ez = -_unit(n)
    ey = _unit(np.cross(ez, P))
    return np.cross(ey, ez), ey, ez


def _aperture(seed, centre, clockwise=False):
    rng = np.random.default_rng(seed)
    v = np.array([[0.0, 0.0, 0.0], [2.1, 0.2, 0.0], [0.7, 1.6, 0.0]]) * 1.3
    R = np.linalg.qr(rng.normal(size=(3, 3)))[0]
    R *= np.sign(np.linalg.det(R))
    v = (v - v.mean(0)) @ R.T + centre
    if clockwise:
        v = v[::-1].copy()
    n = _unit(np.cross(v[1] - v[0], v[2] - v[0]))
    P = _unit(n + 0.6 * rng.normal(size=3))
    vk7 = _unit(np.cross(P, rng.normal(size=3)))
    ampl = rng.normal(size=(1, 8))
    bs = BeamSet(ampl, vk7[None], P[None], np.array([np.pi]), np.array([0, 3]), v)
    return bs, v, P


def _direction(v, P, q1, q2, side=1.0):
    """khat whose (P - khat) has the in-plane components q1, q2."""
    ex, ey, ez = _frame(v, P)
    k1, k2 = P @ ex - q1, P @ ey - q2
    return k1 * ex + k2 * ey + side * np.sqrt(1.0 - k1 * k1 - k2 * k2) * ez


def _model(v, C, P, x, xt, Lam, fb, clamp):
    """Re sum conj(Lam') A' of one bin: A' = s (g I + h J) C, the bin's T_phi folded into Lam'."""
    cross = torch.linalg.cross
    c = v.mean(0)
    N = cross(v[1] - v[0], v[2] - v[0])
    n = N / N.norm()
    ez = -n
    ey = cross(ez, P)
    ey = ey / ey.norm()
    ex = cross(ey, ez)
    d = x - c
    rho, r0 = d.norm(), x.norm()
    kh = d / rho
    ph = WN * ((c @ c - 2.0 * x @ c) / (rho + r0)) + 2 * np.pi * ((WN * float(r0) / (2 * np.pi)) % 1.0)
    q = WN * (P - kh)
    g, w = np.polynomial.legendre.leggauss(64)
    g, w = torch.tensor(0.5 * (g + 1)), torch.tensor(0.5 * w)
    s, t = g[:, None], g[None, :]
    u = (v[0] - c) + s[..., None] * ((v[1] - v[0]) + t[..., None] * (v[2] - v[1]))
    F = N.norm() * ((w[:, None] * w[None, :] * s) * torch.exp(1j * (u @ q))).sum()
    k1, k2, k3, Kz = kh @ ex, kh @ ey, kh @ ez, P @ ez
    k2c = torch.sign(k2.detach()) * K2CLAMP if clamp else k2
    sq, s13 = torch.sqrt(1 - k2c * k2c), torch.sqrt(1 - k2 * k2)
    inc = torch.tensor([0.0, 0.0, -1.0], dtype=torch.float64)
    hv = cross(inc, (xt - c) if fb else kh)
    hv = torch.cat([hv[:2], torch.zeros(1, dtype=torch.float64)])
    hc = hv / hv.norm()
    p, qh = hc @ ((ey - k2c * kh) / sq), hc @ (cross(kh, ey) / s13)
    da, db = -(Kz * sq + k3 / sq) / 2, -k1 * k2c / (2 * sq)
    gg, hh = p * da + qh * db, p * db - qh * da
    M = torch.stack([torch.stack([gg, hh]), torch.stack([-hh, gg])])
    A = torch.exp(1j * ph) * (1j / LAM) * F * (M.to(torch.complex128) @ C)
    return (Lam.conj() * A).real.sum()


def _check(bs, v, P, dirs, rho, tol, fb=False, clamp=False):
    rng = np.random.default_rng(5)
    recs, _ = lib.prepare_beams_host(bs, LAM)
    sigma = np.asarray(recs).reshape(1, -1)[0, 94]
    xt = np.array([2e5, -3e5, 0.0])
    got, want = [], []
    for kh in dirs:
        x = v.mean(0) + rho * kh
        assert fb == (not abs(kh[2]) < FWD)
        Lam = rng.normal(size=(2, 2)) + 1j * rng.normal(size=(2, 2))
        r = np.linalg.norm(x)
        b = np.array([[*x, xt[0], xt[1], r, WN * r / (2 * np.pi)]])
        lp = np.array([[z for col in (0, 1) for row in (0, 1) for z in (Lam[row, col].real, Lam[row, col].imag)]])
        gv, ga = emu.adjoint(recs, b, lp, LAM)
        V = torch.tensor(v, requires_grad=True)
        a = torch.tensor(bs.ampl.reshape(8), requires_grad=True)
        C = sigma * torch.complex(a[0::2], a[1::2]).reshape(2, 2).T
        L = _model(V, C, torch.tensor(P), torch.tensor(x), torch.tensor(xt), torch.tensor(Lam), fb, clamp)
        L.backward()
        got.append((gv.reshape(9), ga.reshape(8)))
        want.append((V.grad.numpy().reshape(9), a.grad.numpy()))
    for j in (0, 1):
        g, w = np.array([z[j] for z in got]), np.array([z[j] for z in want])
        e = np.abs(g - w).max(1) / np.abs(w).max()
        assert np.isfinite(g).all() and (e <= tol).all(), (j, e)


@pytest.mark.parametrize("clockwise", [False, True])
@pytest.mark.parametrize("edge", [0, 1, 2])
def test_edge_nulls(edge, clockwise):
    bs, v, P = _aperture(edge, np.array([4.0, -7.0, 3.0]), clockwise)
    ex, ey, _ = _frame(v, P)
    e = np.roll(v, -1, 0)[edge] - v[edge]
    e = np.array([e @ ex, e @ ey])
    nrm = np.array([-e[1], e[0]]) / np.linalg.norm(e)
    nrm *= np.sign(nrm[0] * (P @ ex)) or 1.0              # towards the directions that exist
    dirs = []
    for K in (0.0, 1e-9, 1e-5, 1e-3, 3e-3, 1e-2, 0.1, 0.99, 1.01, 3.0):
        q = nrm * 0.5 + e / (e @ e) * (K / WN)
        dirs.append(_direction(v, P, *q, side=np.sign(P @ _frame(v, P)[2])))
    _check(bs, v, P, dirs, 1e6, 1e-10)


@pytest.mark.parametrize("centre,rho", [((0.1, 0.0, -0.1), 1e6), ((60.0, -40.0, 50.0), 1e6), ((5.0, 4.0, -6.0), 400.0)])
def test_series_border_and_geometry(centre, rho):
    """q a from 0 through the series' border to an ordinary bin, centres in the far geometry and beyond it."""
    bs, v, P = _aperture(7, np.array(centre))
    ex, ey, ez = _frame(v, P)
    a = np.linalg.norm(v - v.mean(0), axis=1).max()
    dirs = []
    for qa in (0.0, 1e-9, 1e-3, 0.3, 1.4999, 1.5001, 1.8, 4.0, 12.0):
        for ang in (0.4, 2.9):
            q = qa / (a * WN) * np.array([np.cos(ang), np.sin(ang)])
            dirs.append(_direction(v, P, *q, side=np.sign(P @ ez)))
    _check(bs, v, P, dirs, rho, 1e-10)


def test_forward_fallback():
    bs, v, P = _aperture(9, np.array([1.0, 2.0, 3.0]))
    t = np.array([0.0, 1e-4, 0.01, 0.044])
    dirs = [np.array([np.sin(a), 0.0, s * np.cos(a)]) for a in t for s in (1.0, -1.0)]
    _check(bs, v, P, dirs, 1e6, 1e-10, fb=True)


def test_within_the_clamp():
    bs, v, P = _aperture(11, np.array([1.0, -2.0, 0.5]))
    ex, ey, ez = _frame(v, P)
    dirs = [s * np.sqrt(1 - h * h) * ey + h * (np.cos(a) * ex + np.sin(a) * ez)
            for s in (1.0, -1.0) for a in (0.3, 2.0, 4.4) for h in (np.sqrt(4e-7),)]
    assert all(abs(d @ ey) > K2CLAMP for d in dirs)
    _check(bs, v, P, dirs, 1e6, 1e-8, clamp=True)
