"""Small lattices put a site's eight directions on eight waves; with
YH_TUNE_HOP_SPLIT off they take the kernels of one thread per site.  FP64 and FP32
operators must agree bit for bit (the same sums in the same order), the 16-bit
ones to the rounding of one multiplication before the fixed-point store, and
FP64 must meet the oracle; half volumes below, at and past a workgroup of 64
sites, every boundary condition, representation and reconstruction."""
import numpy as np
import pytest

from oracle import BC_ANTIPERIODIC, BC_OPEN, BC_PERIODIC, BC_SF
from test_gpu_parity import rel, setup, src_field

pytestmark = pytest.mark.gpu
yh = pytest.importorskip("yahmc_amd")

CASES = [("su3_fund", (2, 2, 2, 2), BC_ANTIPERIODIC), ("su3_fund", (4, 2, 6, 6), BC_PERIODIC),
         ("su3_fund", (6, 4, 4, 4), BC_OPEN), ("su2_fund", (6, 4, 6, 10), BC_SF),
         ("su2_adj", (4, 2, 6, 6), BC_ANTIPERIODIC), ("su3_sym", (4, 2, 6, 6), BC_OPEN),
         ("su4_asym", (4, 4, 2, 4), BC_ANTIPERIODIC)]


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
