"""The multishift solver holds back the updates of its shift vectors for four
iterations and handles four shifts at a time: shift counts that leave a
remainder, shifts that converge at different iterations (and so inside a
group of four), one to three right-hand sides, half volumes that are no
multiple of a wavefront.  Every solution must meet its own equation."""
import numpy as np
import pytest

from oracle import BC_ANTIPERIODIC
from test_gpu_parity import setup, src_field

pytestmark = pytest.mark.gpu
yh = pytest.importorskip("yahmc_amd")


@pytest.mark.parametrize("model,nshift,nrhs", [("su3_fund", 1, 1), ("su2_adj", 5, 2), ("su2_fund", 13, 3),
                                               ("su3_sym", 4, 1)])
def test_every_shift_meets_its_equation(model, nshift, nrhs):
    o, lat, rng = setup(model, dims=(4, 2, 6, 6), bc=BC_ANTIPERIODIC)
    mass, prec = 0.1, 1e-22
    shifts = list(np.geomspace(1e-4, 50.0, nshift))
    srcs = [lat.field("f64").upload(src_field(o, rng, even_only=True)) for _ in range(nrhs)]
    dsts = [[lat.field("f64") for _ in shifts] for _ in srcs]
    its = lat.cg_mshift_batched(lat.inv_par(mass, prec), shifts, dsts, srcs)
    print(f"\n[case] {model} iterations {its}", flush=True)
    ax = lat.field("f64")
    for b, row in zip(srcs, dsts):
        nb = lat.spinor_sqnorm(b)
        for s, x in zip(shifts, row):
            lat.Hphi_sq(mass, ax, x)
            lat.spinor_mulr_add_assign(ax, s, x)
            lat.spinor_mulr_add_assign(ax, -1.0, b)
            # the recurrence's residual, plus the rounding of as many steps
            assert lat.spinor_sqnorm(ax) < 10 * prec * nb, s
    # one right-hand side alone, launched eagerly, takes the same steps; its
    # norms are summed in another order than a batch's (the check above
    # writes odd halves)
    alone = [lat.field("f64") for _ in shifts]
    lat.tune(yh.TUNE_GRAPHS, 0)
    it = lat.cg_mshift(lat.inv_par(mass, prec), shifts, alone, srcs[0])
    assert abs(it - its[0]) <= 1
    for x, y in zip(alone, dsts[0]):
        a, b = x.download(yh.EVEN)[: o.VH], y.download(yh.EVEN)[: o.VH]
        assert np.abs(a - b).max() < (1e-11 if nrhs > 1 else 1e-15) * np.abs(b).max()
