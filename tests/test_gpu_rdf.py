"""RDF bins on the GPU (mgpu_rdf) against the oracle's rdf_inner/rdf_accum
restatement: bit-identical float bins, including accumulation into bins that
already hold values (Moldy accumulates over RDF steps)."""
import numpy as np
import pytest

from test_gpu_parity import CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", list(CASES))
def test_rdf_bitwise(case):
    from moldy_amd import engine as E
    from oracle.oracle import Oracle
    s = CASES[case]()
    o = Oracle(s)
    xyz = o.make_sites()
    limit = min(0.45 * float(np.diag(s.h).min()), 10.0)
    nbins = 100
    rc, ref = o.rdf(xyz, limit, nbins)
    assert rc == 0
    e = E.ForceEngine(s)
    got = e.rdf(s.h, xyz, limit, nbins)
    print(case, "pairs binned:", int(np.rint(ref.sum() * s.nsites / np.linalg.det(s.h))))
    assert np.array_equal(got, ref)
    # second RDF step accumulates
    rc, ref2 = o.rdf(xyz, limit, nbins, rdf=ref.copy())
    got2 = e.rdf(s.h, xyz, limit, nbins, rdf=got)
    assert np.array_equal(got2, ref2)
    e.close()


@pytest.mark.parametrize("nbins", [1, 60, 5000])
def test_rdf_preloaded_bins(nbins):
    """Bins that already hold values of every kind (zero, values around powers
    of two where the float spacing doubles, values that an addition no longer
    changes, and negative ones), few bins with large counts, and so many
    that the counts do not fit in LDS: the reference's one-by-one float
    additions, bit for bit."""
    from moldy_amd import engine as E, system
    from oracle.oracle import Oracle
    s = system.salt_water(nwater=300, nmg=6, ncl=12, seed=5, cutoff=7.0, alpha=0.38)
    o = Oracle(s)
    xyz = o.make_sites()
    nblk = (s.max_id - 1) * s.max_id // 2
    rng = np.random.default_rng(nbins)
    p2 = np.ldexp(1.0, rng.integers(-4, 27, (nblk, nbins)))
    kinds = [0.0 * p2, p2 * (1 - 2.0 ** -24), p2 * rng.uniform(1, 2, p2.shape), -p2, 1e9 * p2, 1e-40 + 0 * p2]
    rdf0 = np.choose(rng.integers(0, len(kinds), p2.shape), kinds).astype(np.float32)
    rc, ref = o.rdf(xyz, 6.9, nbins, rdf=rdf0.copy())
    assert rc == 0
    e = E.ForceEngine(s)
    got = e.rdf(s.h, xyz, 6.9, nbins, rdf=rdf0.copy())
    assert np.array_equal(got, ref)
    e.close()
