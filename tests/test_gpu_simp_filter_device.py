"""The density filter built on the device: H and Hs equal the oracle's
sequential loop to the bit, whatever the radius is to the mesh (each element
alone, bins of one element, a few, all in one bin), on meshes whose element
order follows no row order, on a sliver of a domain and at sizes around a
slice of 64 rows and a workgroup of 256.  Rows beyond the layout's 65,535
entries are refused as before."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _shuffled(p):
    t = p.conn.reshape(-1, 3)[np.random.default_rng(5).permutation(p.N_elem)]
    return dataclasses.replace(p, conn=t.ravel().copy())


def _case(name):
    from nbots_amd import synth
    if name == "shuffled":
        return _shuffled(synth.cantilever_point(33, 17, jitter=0.3))
    if name == "shifted":
        p = synth.cantilever_point(40, 20, jitter=0.2)
        return dataclasses.replace(p, nod=p.nod * 1e-3 - 7.25)
    nx, ny = (int(v) for v in name.split("x"))
    return synth.cantilever_point(nx, ny, jitter=0.1)


@pytest.mark.parametrize("name,rmin", [
    ("8x4", 1.5), ("8x4", 100.0), ("8x4", 1e-3), ("43x3", 2.4), ("16x8", 1.5), ("200x1", 3.0),
    ("shuffled", 1.5), ("shuffled", 4.7), ("shuffled", 40.0), ("shifted", 2.4e-3),
    ("64x33", 0.5), ("64x33", 1e-9)])
def test_device_filter_equals_the_oracles(name, rmin):
    import oracle
    from nbots_amd import synth
    from nbots_amd.fem import Fem, Simp
    p = _case(name)
    f = Fem.from_problem(p)
    print(f"[simp filter] {name} {rmin}", flush=True)
    s = Simp(f, rmin=rmin)
    got = s.filter()
    s.destroy()
    f.destroy()
    cx, cy = synth.elem_centroids(p)
    n = p.N_elem
    if rmin < 1e-6:   # too many bins for the oracle; each element is alone
        want = np.arange(n + 1), np.arange(n), np.full(n, rmin), np.full(n, rmin)
    else:
        want = oracle.filter_build(cx, cy, rmin)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def test_too_long_rows_are_refused():
    from nbots_amd import synth
    from nbots_amd.fem import Fem, Simp
    p = synth.cantilever_point(260, 130)     # 67,600 elements
    f = Fem.from_problem(p)
    print("[simp filter] rows of 67,600", flush=True)
    with pytest.raises(Exception, match="filter row"):
        Simp(f, rmin=1e4)
    s = Simp(f, rmin=1.5)
    s.destroy()
    f.destroy()
