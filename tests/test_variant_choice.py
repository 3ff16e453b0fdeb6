"""Which kernel a call launches, on a HIP runtime without a device: a variant
named in the call, by tdbp_set_variant or in the environment is the one that
runs, on a burst small enough for the split tiles too; unnamed, those run.  The
autotuners time the kernel that runs unnamed, and leave the choice to the rule
where that is the fastest."""
import pytest

from fakehip import run

SETUP = """
T.init(0)
sc = synth.make_burst(130, 2600, 17, 5, aperture=31, dem="flat", ntargets=0, seed=1)
large = synth.make_burst(420, 3400, 400, 420, aperture=64, dem="flat", ntargets=0, seed=2)
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


COSTS = """
F.fake_cost(b"k_", 0.0, 0.0)                 # fits and fills
for k in (b"k_mixedI", b"k_batch_mixedI", b"k_plainI", b"k_batch_plainI", b"_ldsI"):
    F.fake_cost(k, 3.0, 3.0)
SPLIT, WHOLE = (b"%s_mixedILi4ELi2E", b"%s_mixedILi4ELi1E")


def buffers(sc):
    g = sc.geom
    return (g, T.samples(T.DeviceArray((g.L, g.S), np.complex64)),
            T.DeviceArray.from_host(sc.satloc), T.DeviceArray.from_host(sc.dem),
            T.DeviceArray((g.nlines, g.demwidth), np.complex64))


def batched():
    return [c[2] for c in log() if c[0] == "hipLaunchKernel" and "k_batch_mixed" in c[2]]


small, big = buffers(sc), buffers(large)
"""


def test_autotune_times_the_split_tiles():
    run(SETUP + COSTS + """
F.fake_cost(SPLIT % b"k", 1.0, 1.0)
F.fake_cost(WHOLE % b"k", 2.0, 2.0)
best, ms = T.autotune(*small)
assert (best, ms[11], ms[5]) == (11, 1.0, 2.0)
assert SPLIT.decode() % "k" in kernel(single, mixed)
assert WHOLE.decode() % "k" in kernel(T.backproject, *big, mixed)   # not the small burst's
F.fake_cost(WHOLE % b"k", 0.5, 0.5)
best, ms = T.autotune(*small)
assert (best, ms[11], ms[5]) == (5, 1.0, 0.5)
assert WHOLE.decode() % "k" in kernel(single, mixed)                # what was timed
""")


def test_batch_autotune_times_the_split_tiles():
    run(SETUP + COSTS + """
F.fake_cost(SPLIT % b"k_batch", 1.0, 0.1)    # alone: on the large burst too
F.fake_cost(WHOLE % b"k_batch", 2.0, 0.5)
for bursts, want in (([small, small], 11), ([small, big], -1), ([big, big], 11)):
    b, fresh = T.Batch(mixed), T.Batch(mixed)
    for x in bursts:
        b.add(*x)
        fresh.add(*x)
    best, ms = b.autotune()
    assert best == want and len(ms) == T.lib().tdbp_variant_count(), (best, ms)
    F.fake_clear()
    b.run()
    got = batched()
    named = T.Batch(mixed, best)
    for x in bursts:
        named.add(*x)
    named.run()
    F.fake_clear()
    named.run()
    assert got == batched() and len(got) == 1 + (best < 0)
    if best < 0:
        F.fake_clear()
        fresh.run()
        fresh.run()
        assert batched()[-2:] == got
""")
