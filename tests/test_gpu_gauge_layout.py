"""The gauge kernels on lattices whose half volume is no multiple of a
wavefront or a workgroup, against the oracle: the transposition of host links
to component planes and back, the Wilson and improved forces, the link
update, and the represented links and clover term built from the moved links."""
import numpy as np
import pytest

from fields import random_gauge
from oracle import BC_ANTIPERIODIC, BC_OPEN, Oracle

pytestmark = pytest.mark.gpu
yh = pytest.importorskip("yahmc_amd")

# half volumes 8 (less than a wavefront), 144 = 2 * 64 + 16 and 720 = 11 * 64 + 16
DIMS = [(2, 2, 2, 2), (4, 2, 6, 6), (6, 4, 6, 10)]
MODELS = [("su2_fund", 2, "fundamental"), ("su3_fund", 3, "fundamental"), ("su3_sym", 3, "symmetric"),
          ("su4_asym", 4, "antisymmetric")]


@pytest.mark.parametrize("model,nc,rep", MODELS)
@pytest.mark.parametrize("dims,bc", [(d, "antiperiodic") for d in DIMS] + [(d, "open") for d in DIMS[1:]])
def test_ragged_lattices(model, nc, rep, dims, bc):
    print(f"\n[case] gauge kernels {model} {dims} {bc}", flush=True)
    o = Oracle(model).init(dims, bc=BC_OPEN if bc == "open" else BC_ANTIPERIODIC, csw=1.0)
    rng = np.random.default_rng(71)
    links = random_gauge(rng, o.V, nc)
    P = rng.normal(size=(4 * o.V, nc * nc - 1))
    o.set_gauge(links)
    lat = yh.Lattice(dims, nc=nc, repr=rep, bc=bc, csw=1.0)
    lat.set_gauge(links)
    assert np.array_equal(lat.get_gauge(), links)
    o.apply_bcs_on_gauge()
    lat.apply_bcs_on_gauge_field()
    for x in (o, lat):
        x.set_momenta(P)
        x.wilson_gauge_force(0.37, 5.6)
        x.improved_gauge_force(0.21, 5.6, 5.0 / 3.0, -1.0 / 12.0)
    got, want = lat.get_momenta(), o.get_momenta()
    # sums of at most 3 * 14 products of unitary matrices in 64 bits
    assert np.abs(got - want).max() < 1e-13 * np.abs(want).max()
    # the same momenta on both sides, so that the links compare to rounding
    lat.set_momenta(want)
    for x in (o, lat):
        x.update_links(0.05)
    o.represent()
    lat.represent_gauge_field()
    assert np.abs(lat.get_gauge() - o.get_gauge()).max() < 1e-13
    assert np.abs(lat.gauge_repr().reshape(o.get_repr().shape) - o.get_repr()).max() < 1e-13
    want = o.get_clover()
    assert np.abs(lat.clover_term().reshape(want.shape) - want).max() < 1e-13 * max(1.0, np.abs(want).max())
