"""Small lattices put a site's eight directions on eight waves; with
YH_TUNE_HOP_SPLIT off they take the kernels of one thread per site.  FP64 and FP32
operators must agree bit for bit (the same sums in the same order), the 16-bit
ones to the rounding of one multiplication before the fixed-point store, and
FP64 must meet the oracle; half volumes below, at and past a workgroup of 64
sites, every boundary condition, D_R = 2, 3, 4 and 6, and every
reconstruction.  A lattice just past the line between the two runs the
kernels of one thread per site by default."""
import numpy as np
import pytest

from oracle import BC_ANTIPERIODIC, BC_OPEN, BC_PERIODIC, BC_SF
from test_gpu_parity import rel, setup, src_field

pytestmark = pytest.mark.gpu
yh = pytest.importorskip("yahmc_amd")

CASES = [("su3_fund", (2, 2, 2, 2), BC_ANTIPERIODIC), ("su3_fund", (4, 2, 6, 6), BC_PERIODIC),
         ("su3_fund", (6, 4, 4, 4), BC_OPEN), ("su2_fund", (6, 4, 6, 10), BC_SF),
         ("su2_adj", (4, 2, 6, 6), BC_ANTIPERIODIC), ("su3_sym", (4, 2, 6, 6), BC_OPEN),
         ("su4_asym", (4, 4, 2, 4), BC_ANTIPERIODIC), ("su4_fund", (4, 2, 6, 6), BC_ANTIPERIODIC),
         ("su4_fund", (6, 4, 6, 10), BC_SF)]


@pytest.mark.parametrize("model,dims,bc", CASES)
def test_split_hop_matches_one_thread_per_site(model, dims, bc):
    o, lat, rng = setup(model, dims=dims, bc=bc, csw=1.0, cf=1.1)
    mass = 0.2
    s = src_field(o, rng)
    got = {}
    for split in (True, False):
        for prec in ("f64", "f32", "f16"):
            fs, fd = lat.field(prec).upload(s), lat.field(prec)
            outs = []
            lat.Dphi_oe(fd, fs)
            outs.append(fd.download()[o.VH:])
            lat.Dphi_eo(fd, fs)
            outs.append(fd.download()[: o.VH])
            lat.Hphi_sq(mass, fd, fs)
            outs.append(fd.download()[: o.VH])
            got[split, prec] = outs
        lat.tune(yh.TUNE_HOP_SPLIT, 0)
    want = np.zeros_like(s)
    o.Hphi_sq(mass, want, s.copy())
    assert rel(got[True, "f64"][2], want[: o.VH]) < 1e-13
    for prec in ("f64", "f32"):
        for a, b in zip(got[True, prec], got[False, prec]):
            assert np.array_equal(a, b), prec
    # one unit of the 16-bit store (2^-15 of the site's largest component) per
    # hop, of which H^2 has four
    for n, (a, b) in enumerate(zip(got[True, "f16"], got[False, "f16"])):
        assert rel(a, b) < (4 if n == 2 else 1) * 2.0**-15 * 4


@pytest.mark.parametrize("model", ["su3_fund", "su3_sym"])
def test_split_solves_match(model):
    """CG with its norms from the split kernels, FP64 and mixed 16-bit."""
    o, lat, rng = setup(model, dims=(4, 2, 6, 6), bc=BC_ANTIPERIODIC)
    fb = lat.field("f64").upload(src_field(o, rng, even_only=True))
    res = []
    for split in (True, False):
        x, y = lat.field("f64"), lat.field("f64")
        it = lat.cg_inverter(lat.inv_par(0.1, 1e-24), x, fb)
        it16, _ = lat.cg_mixed(lat.inv_par(0.1, 1e-24, sloppy="f16", reliable_every=50), y, fb)
        res.append((it, x.download()[: o.VH], it16, y.download()[: o.VH]))
        lat.tune(yh.TUNE_HOP_SPLIT, 0)
    assert abs(res[0][0] - res[1][0]) <= 1 and rel(res[0][1], res[1][1]) < 1e-11
    assert abs(res[0][2] - res[1][2]) <= 4 and rel(res[0][3], res[1][3]) < 1e-11


@pytest.mark.parametrize("key,prec,tol", [("TUNE_RECON12_F64", "f64", 1e-13), ("TUNE_HALF_LINKS", "f32", 5e-3)])
@pytest.mark.parametrize("dims,bc", [((2, 2, 2, 2), BC_PERIODIC), ((4, 2, 6, 6), BC_ANTIPERIODIC),
                                     ((6, 4, 6, 10), BC_OPEN)])
def test_other_reconstructions(key, prec, tol, dims, bc):
    """FP64 12-real links, and 16-bit links under FP32 spinors: by default they
    are read as 18 and 12 reals of the spinors' precision."""
    o, lat, rng = setup("su3_fund", dims=dims, bc=bc, csw=1.0, cf=1.1)
    s = src_field(o, rng)
    want = np.zeros_like(s)
    o.Hphi_sq(0.2, want, s.copy())
    got = {}
    for on, split in ((0, 1), (1, 1), (1, 0)):
        lat.tune(getattr(yh, key), on)
        lat.tune(yh.TUNE_HOP_SPLIT, split)
        fs, fd = lat.field(prec).upload(s), lat.field(prec)
        lat.Dphi_oe(fd, fs)
        lat.Dphi_eo(fd, fs)
        hop = fd.download()
        lat.Hphi_sq(0.2, fd, fs)
        got[on, split] = (hop, fd.download()[: o.VH])
    assert rel(got[1, 1][1], want[: o.VH]) < tol
    for a, b in zip(got[1, 1], got[1, 0]):
        assert np.array_equal(a, b)
    assert not np.array_equal(got[0, 1][1], got[1, 1][1])  # the links asked for are in use


@pytest.mark.parametrize("model,dims,bc", [("su3_fund", (18, 16, 16, 16), BC_ANTIPERIODIC),
                                           ("su3_fund", (6, 12, 32, 32), BC_OPEN),
                                           ("su2_fund", (18, 16, 16, 16), BC_OPEN),
                                           ("su4_fund", (18, 16, 16, 16), BC_ANTIPERIODIC),
                                           ("su3_sym", (18, 16, 16, 16), BC_PERIODIC)])
def test_just_past_the_line(model, dims, bc):
    """36,864 sites a parity: the default kernels are those of one thread per
    site, staged where a (t, x) plane is a multiple of 256 sites."""
    o, lat, rng = setup(model, dims=dims, bc=bc, csw=1.0, cf=1.1)
    s = src_field(o, rng)
    want = {k: np.zeros_like(s) for k in ("Hphi_sq", "Dphi_oe")}
    o.Hphi_sq(0.2, want["Hphi_sq"], s.copy())
    o.Dphi_oe(want["Dphi_oe"], s.copy())
    keys = [None] + ([yh.TUNE_RECON12_F64, yh.TUNE_HALF_LINKS] if model == "su3_fund" else [])
    for key in keys:
        if key:
            lat.tune(key, 1)
        for prec, tol in (("f64", 1e-13), ("f32", 5e-3 if key == yh.TUNE_HALF_LINKS else 2e-6), ("f16", 4e-4)):
            out = []
            for split in (1, 0):  # of no effect at this size
                lat.tune(yh.TUNE_HOP_SPLIT, split)
                fs, fd = lat.field(prec).upload(s), lat.field(prec)
                lat.Dphi_oe(fd, fs)
                hop = fd.download()[o.VH:]
                lat.Hphi_sq(0.2, fd, fs)
                out.append((hop, fd.download()[: o.VH]))
            assert rel(out[0][0], want["Dphi_oe"][o.VH:]) < tol, prec
            assert rel(out[0][1], want["Hphi_sq"][: o.VH]) < tol, prec
            assert all(np.array_equal(a, b) for a, b in zip(*out)), prec
