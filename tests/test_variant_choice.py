"""Which kernel a call launches, on a HIP runtime without a device: a variant
named in the call, by tdbp_set_variant or in the environment is the one that
runs, on a burst small enough for the split tiles too; unnamed, those run."""
import pytest

from fakehip import run

SETUP = """
T.init(0)
sc = synth.make_burst(130, 2600, 17, 5, aperture=31, dem="flat", ntargets=0, seed=1)
g = sc.geom
d = T.DeviceArray((g.L, g.S), np.complex64)
sat, dem = T.DeviceArray.from_host(sc.satloc), T.DeviceArray.from_host(sc.dem)
out = T.DeviceArray((g.nlines, g.demwidth), np.complex64)


def single(precision, variant=None):
    T.backproject(g, T.samples(d), sat, dem, out, precision, variant=variant)


def noalloc(precision):
    T.backproject_noalloc(g, T.samples(d), sat, dem, out, precision)


def batch(precision, variant=-1):
    b = T.Batch(precision, variant)
    b.add(g, T.samples(d), sat, dem, out)
    b.run()


def kernel(call, *a, **k):
    F.fake_clear()
    call(*a, **k)
    names = [c[2] for c in log() if c[0] == "hipLaunchKernel"]
    one, = [n for n in names if any(k in n for k in ("k_plainI", "k_mixedI", "k_batch_plainI",
                                                     "k_batch_mixedI"))]
    return one


fp64, mixed = T.PLAIN_FP64, T.MIXED
"""


@pytest.mark.parametrize("how", ["set", "environment"])
def test_a_named_variant_runs(how):
    run(SETUP + f"how = {how!r}" + """
split = [kernel(f, p) for p in (fp64, mixed) for f in (single, noalloc, batch)]
named = [kernel(single, fp64, 1), kernel(batch, fp64, 1), kernel(single, mixed, 5),
         kernel(batch, mixed, 5)]
os.environ["TDBP_PLAIN_VARIANT"] = "1"
if how == "set":
    T.check(T.lib().tdbp_set_variant(5))
else:
    os.environ["TDBP_VARIANT"] = "5"
assert [kernel(single, fp64), kernel(batch, fp64), kernel(single, mixed),
        kernel(batch, mixed)] == named
assert [kernel(noalloc, fp64), kernel(noalloc, mixed)] == named[::2]
T.check(T.lib().tdbp_set_variant(-1))
for v in ("TDBP_PLAIN_VARIANT", "TDBP_VARIANT"):
    os.environ[v] = "99"    # no such variant: as if unset
assert [kernel(f, p) for p in (fp64, mixed) for f in (single, noalloc, batch)] == split
assert not set(split) & set(named)
""")
