"""The gauge kernels on lattices whose half volume is no multiple of a
wavefront or a workgroup, against the oracle: the transposition of host links
to component planes and back, the Wilson and improved forces, the link
update, the represented links and the clover term built from the moved links,
and its inverse (log det, and the operator in every storage precision)."""
import numpy as np
import pytest

from fields import gaussian_spinor, random_gauge
from oracle import BC_ANTIPERIODIC, BC_OPEN, Oracle

pytestmark = pytest.mark.gpu
yh = pytest.importorskip("yahmc_amd")

# half volumes 8 (less than a wavefront), 144 = 2 * 64 + 16 and 720 = 11 * 64 + 16
DIMS = [(2, 2, 2, 2), (4, 2, 6, 6), (6, 4, 6, 10)]
MODELS = [("su2_fund", 2, "fundamental"), ("su3_fund", 3, "fundamental"), ("su3_sym", 3, "symmetric"),
          ("su4_asym", 4, "antisymmetric"), ("su2_adj", 2, "adjoint"), ("su3_adj", 3, "adjoint"),
          ("su4_fund", 4, "fundamental"), ("su2_sym", 2, "symmetric")]


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
    mass = 0.3
    assert abs(lat.clover_logdet(mass) - o.clover_logdet(mass)) < 1e-12 * abs(o.clover_logdet(mass))
    src = gaussian_spinor(rng, o.V, o.dr)
    want = np.zeros_like(src)
    o.Hphi(mass, want, src.copy())
    # 64-bit, 32-bit and 16-bit fixed-point storage of links, clover term and inverse
    for prec, tol in (("f64", 1e-13), ("f32", 2e-6), ("f16", 2e-4)):
        fs, fd = lat.field(prec).upload(src), lat.field(prec)
        lat.Hphi(mass, fd, fs)
        got = fd.download(yh.EVEN)[: o.VH]
        assert np.abs(got - want[: o.VH]).max() < tol * np.abs(want).max(), prec


FORCE_MODELS = [("su2_fund", 2, "fundamental"), ("su3_fund", 3, "fundamental"), ("su4_asym", 4, "antisymmetric"),
                ("su3_sym", 3, "symmetric"), ("su4_fund", 4, "fundamental"), ("su2_adj", 2, "adjoint")]


@pytest.mark.parametrize("model,nc,rep", FORCE_MODELS)
@pytest.mark.parametrize("dims,bc", [((4, 2, 6, 6), "antiperiodic"), ((6, 4, 6, 10), "open")])
def test_ragged_fermion_forces(model, nc, rep, dims, bc):
    """The force sequence of a two-flavour monomial (packed clover-force
    matrices up to D_R = 4, full ones at 6), and the matrices themselves."""
    print(f"\n[case] fermion forces {model} {dims} {bc}", flush=True)
    o = Oracle(model).init(dims, bc=BC_OPEN if bc == "open" else BC_ANTIPERIODIC, csw=1.0)
    rng = np.random.default_rng(72)
    links = random_gauge(rng, o.V, nc)
    P = rng.normal(size=(4 * o.V, nc * nc - 1))
    o.set_gauge(links)
    o.apply_bcs_on_gauge()
    o.represent()
    lat = yh.Lattice(dims, nc=nc, repr=rep, bc=bc, csw=1.0)
    lat.set_gauge(o.get_gauge())
    src = gaussian_spinor(rng, o.V, o.dr)
    field = lat.field("f64").upload(src)
    for x, y in ((o, src.copy()), (lat, field)):
        x.set_momenta(P)
        x.begin_fermion_force()
        x.wilson_fermion_force_q(0.3, 0.2, 1.0, y)
        x.clover_logdet_force(0.2, 2.0)
    want = o.get_clover_force()
    got = lat.get_clover_force().reshape(want.shape)
    assert np.abs(got - want).max() < 1e-12 * np.abs(want).max()
    for x in (o, lat):
        x.end_fermion_force(0.3)
    got, want = lat.get_momenta(), o.get_momenta()
    assert np.abs(got - want).max() < 1e-12 * np.abs(want).max()


@pytest.mark.parametrize("nc,rep,dims", [(2, "fundamental", (34, 26, 26, 26)), (3, "fundamental", (26, 22, 18, 26)),
                                         (4, "antisymmetric", (14, 18, 26, 22))])
def test_host_links_in_pieces(nc, rep, dims):
    """Links of more than 128 MiB cross to the device and back in pieces: these
    volumes are no multiple of a piece, pieces cross the parity boundary, and
    so does a block of 16 sites where the half volume is 8 past a multiple."""
    V = int(np.prod(dims))
    assert V * 64 * nc * nc > 128 << 20
    print(f"\n[case] host links in pieces nc={nc} {dims}", flush=True)
    lat = yh.Lattice(dims, nc=nc, repr=rep, bc="antiperiodic", csw=0.0)
    rng = np.random.default_rng(73)
    links = rng.random(size=(4 * V, 2 * nc * nc))  # any numbers: they are only moved
    lat.set_gauge(links)
    assert np.array_equal(lat.get_gauge(), links)
    if rep == "fundamental":
        # represented links are copies in the same planes, but for the antiperiodic sign of direction 0 at t = 0
        got = lat.gauge_repr().reshape(V, 4, -1)
        want = links.reshape(V, 4, -1).copy()
        assert np.array_equal(got[:, 1:], want[:, 1:]) and np.array_equal(np.abs(got), np.abs(want))
