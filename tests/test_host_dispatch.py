"""Host logic of the C ABI without a GPU: which kernels a call launches, with
which grid and arguments, and how much device memory it takes, read from a HIP
runtime that only records (hip_stub.c).  Each case runs in a process of its
own, which loads that runtime before libyahmc.so."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "yahmc_amd", "lib", "libyahmc.so")
pytestmark = pytest.mark.skipif(not os.path.exists(LIB), reason="libyahmc.so not built")

PRELUDE = """
import ctypes, json, re, sys
sys.path.insert(0, {root!r})
stub = ctypes.CDLL({stub!r}, ctypes.RTLD_GLOBAL)
stub.stub_name.restype = ctypes.c_char_p
stub.stub_in_use.restype = stub.stub_peak.restype = ctypes.c_size_t
import numpy as np
import yahmc_amd as yh

def lattice(dims, nc=3, repr="fundamental"):
    lat = yh.Lattice(dims, nc=nc, repr=repr)
    lat.set_gauge(np.zeros((4 * lat.V, 2 * nc * nc)))
    return lat

def launches(f):
    "[kernel, grid, watched argument] of every launch of f()"
    stub.stub_reset()
    f()
    out = []
    for i in range(stub.stub_launches()):
        g = (ctypes.c_uint32 * 3)()
        stub.stub_grid(i, g)
        name = re.match(r"_ZN2yh\\d+(k_[a-z0-9_]+?)(?:I|E|P|R|K|$)", stub.stub_name(i).decode()).group(1)
        out.append([name, list(g), stub.stub_arg(i)])
    return out

def names(f):
    return sorted({{n for n, _, _ in launches(f)}})
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "hip_stub.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "hip_stub.c")], check=True)
    return so


def run(stub, body):
    """what `body` prints last, as JSON"""
    out = subprocess.run([sys.executable, "-c", PRELUDE.format(root=ROOT, stub=stub) + body], capture_output=True,
                         text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    return json.loads(out.stdout.splitlines()[-1])


@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
def test_split_hop_has_a_key_of_its_own(stub, prec):
    """Setting the staging mask, to its default or to another value, does not
    change which kernels a small lattice runs; YH_TUNE_HOP_SPLIT does, both ways."""
    got = run(stub, f"""
lat = lattice((8, 4, 4, 4))
s, d = lat.field({prec!r}), lat.field({prec!r})
hop = lambda: names(lambda: lat.Dphi_eo(d, s))
out = [hop()]
for key, value in ((yh.TUNE_HOP_STAGE, 3), (yh.TUNE_HOP_STAGE, 0), (yh.TUNE_HOP_SPLIT, 0), (yh.TUNE_HOP_STAGE, 7),
                   (yh.TUNE_HOP_SPLIT, 1)):
    lat.tune(key, value)
    out.append(hop())
print(json.dumps(out))
""")
    split, one = ["k_hop_split"], ["k_hop"]
    assert got == [split, split, split, one, one, split]


def test_autotune_times_the_kernels_that_read_the_chunk(stub):
    """On a small lattice the autotuner times the hop of one thread per site,
    whose block order the chunk sets, and leaves the eight-wave hop in use."""
    got = run(stub, """
lat = lattice((8, 8, 8, 8))
s, d = lat.field("f64"), lat.field("f64")
tuned = names(lambda: lat.autotune(reps=1))
after = names(lambda: lat.Dphi_eo(d, s))
lat.tune(yh.TUNE_HOP_SPLIT, 0)
lat.autotune(reps=1)
print(json.dumps([tuned, after, names(lambda: lat.Dphi_eo(d, s))]))
""")
    assert got == [["k_hop"], ["k_hop_split"], ["k_hop"]]


@pytest.mark.parametrize("nc,rep,own", [(3, "fundamental", 64), (2, "fundamental", 64), (3, "symmetric", 0)])
def test_force_order_reaches_every_clover_force_kernel(stub, nc, rep, own):
    """YH_TUNE_FORCE_ORDER sets the grid (four rows for -1) and the run length,
    the last argument, of the clover-force kernel of every representation."""
    body = f"""
lat = lattice((8, 4, 4, 4), {nc}, {rep!r})
lat.set_momenta(np.zeros((4 * lat.V, lat.ng)))
def core():
    lat.begin_fermion_force()
    return [[g[1], a] for n, g, a in launches(lambda: lat.end_fermion_force(0.1)) if "k_force_clover" in n]
out = [core()]
for order in (0, 5, -1):
    lat.tune(yh.TUNE_FORCE_ORDER, order)
    out.append(core())
print(json.dumps(out))
"""
    assert [o[0][0] for o in run(stub, body)] == [1, 1, 1, 4]
    assert run(stub, 'stub.stub_watch(b"k_force_clover_", 6)' + body) == [[[1, own]], [[1, 0]], [[1, 5]], [[4, -1]]]


@pytest.mark.parametrize("nrhs,num", [(1, 1), (1, 12), (4, 3)])
def test_multishift_takes_half_fields(stub, nrhs, num):
    """The multishift's working fields are even or odd halves: four residuals,
    p, q and a direction per shift, two operator temporaries when batched."""
    got = run(stub, f"""
lat = lattice((8, 8, 8, 8))
srcs = [lat.field("f64") for _ in range({nrhs})]
dsts = [[lat.field("f64") for _ in range({num})] for _ in srcs]
def solve():
    try:
        lat.cg_mshift_batched(lat.inv_par(0.1, 1e-20, max_iter=16), [0.1] * {num}, dsts, srcs)
    except yh.YahmcError as e:
        assert e.code == -4
solve()  # the context's own temporaries
before = stub.stub_in_use()
stub.stub_reset()
solve()
half = 64 * lat.dr * ((lat.VH + 63) // 64 * 64 + 64)
print(json.dumps([(stub.stub_peak() - before) / half, stub.stub_in_use() - before]))
""")
    halves = nrhs * (6 + num + (2 if nrhs > 1 else 0))
    assert halves <= got[0] < halves + 1 and got[1] == 0


@pytest.mark.parametrize("nc", [2, 4])
def test_links_are_held_once(stub, nc):
    """A context keeps its fundamental links once; the buffer that their host
    transfers go through is bounded."""
    used = run(stub, f"""
lat = yh.Lattice((64, 48, 48, 48), nc={nc})
print(json.dumps(stub.stub_in_use()))
""")
    V = 64 * 48**3
    assert used < 64 * nc * nc * V + (144 << 20)
