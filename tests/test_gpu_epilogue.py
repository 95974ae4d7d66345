"""The epilogue's one pass over the bins (a workgroup per theta, a lane per phi, weighted sums) at the edges of
its shapes: fewer phi than a wave, one more and one less than whole waves and than a workgroup, several passes of
a workgroup; odd and even counts (simpne's last panel); uneven angles; amplitudes aligned to one double only.
Against the oracle's finalise.  A weighted sum of n terms in any order differs from the reference's by at most
~n 1.1e-16 of the sum of their magnitudes: 7e-14 at 600 terms, so 1e-13 of the largest value of each
array and 1e-12 of the theta integrals, the asymmetry parameters' in absolute terms (they are at most 1)."""
import numpy as np
import pytest

from abt_amd import lib

pytestmark = pytest.mark.gpu
LAM = 0.532


def _angles(nth, nph, seed):
    rng = np.random.default_rng(seed)
    a = lambda n, top: np.cumsum(rng.uniform(0.5, 1.5, n)) * (top / (1.6 * n))
    return a(nth, np.pi), a(nph, 2 * np.pi)


@pytest.mark.parametrize("scaling", [False, True])
@pytest.mark.parametrize("nth,nph", [(3, 3), (4, 63), (5, 64), (300, 65), (7, 192), (6, 255), (9, 256), (257, 257),
                                     (3, 600)])
def test_epilogue_shapes(orc, nth, nph, scaling):
    import torch
    th, ph = _angles(nth, nph, nth + nph)
    rng = np.random.default_rng(nph)
    nb = nth * nph
    rb, re = rng.normal(size=8 * nb), 0.3 * rng.normal(size=8 * nb)
    ref = orc.finalise(th, ph, LAM, rb, re)
    kw = dict(scaling=scaling, beam_energy_out=abs(ref["scatt_beam"]) * 0.9,
              ext_energy_out=abs(ref["scatt_ext_diff"]) * 1.1) if scaling else {}
    if scaling:
        ref = orc.finalise(th, ph, LAM, rb, re, **kw)
    g = lib.DeviceGrid(th, ph, LAM)
    f64 = dict(dtype=torch.float64, device="cuda")
    # one double into its allocation: 8-byte alignment
    ab, ae = (torch.cat([torch.zeros(1, **f64), torch.from_numpy(a).cuda()])[1:] for a in (rb, re))
    m, m1, par = torch.full((48 * nb,), np.nan, **f64), torch.full((48 * nth,), np.nan, **f64), torch.zeros(9, **f64)
    lib.finalise_dev(g, ab, ae, m, m1, par, **kw)
    m, m1, par = m.cpu().numpy().reshape(3, 16, nb), m1.cpu().numpy().reshape(3, 16, nth), par.cpu().numpy()
    for i, s in enumerate(("", "_beam", "_ext")):
        for got, want in ((m[i], ref["mueller" + s]), (m1[i], ref["mueller_1d" + s])):
            np.testing.assert_allclose(got, want, rtol=0, atol=1e-13 * np.abs(want).max())
    np.testing.assert_allclose(par[:3], [ref["scatt"], ref["scatt_beam"], ref["scatt_ext_diff"]], rtol=1e-12)
    np.testing.assert_allclose(par[3:6], [ref["asymmetry"], ref["asymmetry_beam"], ref["asymmetry_ext_diff"]],
                               rtol=0, atol=1e-12)
    np.testing.assert_allclose(par[6], ref["back_scatt"], rtol=1e-12)
    np.testing.assert_allclose(ab.cpu().numpy(), ref["ampl_beam"], rtol=1e-12)
    np.testing.assert_allclose(ae.cpu().numpy(), ref["ampl_ext"], rtol=1e-12)
