"""Becke weights and compaction of the device rebuild where their kernels have
edges: one to three nuclei (a product of no factor, of one, of a pair),
groups of 63 to 66 nuclei (either side of the nearest 64 whose distances are
kept, odd and even remainders of the factor pairs), groups of several
thousand points (several steps of the walk and a remainder), all points kept
or those of weight zero dropped, and two nuclei at one place, whose pair has
no reciprocal.

The host's weights come from the same arithmetic and its sums run in the same
order, so the groups and their sums are equal bit for bit (a sum that is not
a number on one side is not one on the other).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("drop", [1, 0])
@pytest.mark.parametrize("natoms", [1, 2, 3, 63, 64, 65, 66, -5])
def test_device_weights_equal_the_hosts(natoms, drop):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lio_amd import g2g, systems
    n = abs(natoms)
    Z, pos = systems.random_molecule_ang(n, 70 + n) if n > 1 else (np.array([8]), np.zeros((1, 3)))
    pos = np.array(pos, dtype=float)
    if natoms < 0:
        pos[-1] = pos[0]  # two nuclei at one place
    s = systems.make_system("edge%d" % natoms, Z, pos, seed=n)
    opts = dict(little_cube_size=30.0, assign_all_functions=1, remove_zero_weights=drop)
    print("natoms", natoms, "drop", drop, flush=True)
    out = []
    for mode in ("host", "device"):
        ctx = g2g.Context(s, grid_mode=mode, **opts)
        ctx.build_grid()
        out.append(ctx.groups())
        ctx.close()
    host, dev = out
    assert len(host) == len(dev) > 0
    for a, b in zip(host, dev):
        for key in ("kind", "npoints", "nfuncs", "fhash"):
            assert a[key] == b[key]
        for key in ("wsum", "xsum"):
            assert np.array_equal(a[key], b[key], equal_nan=True)


@pytest.mark.parametrize("precision", ["fp64", "bf16x6"])
def test_reloads_of_changing_size_equal_a_fresh_one(precision):
    """One engine takes systems of growing and shrinking size in turn, with
    the host's and the device's grids, so that its pinned buffer of host
    tables is written again after other sizes and is passed by for tables too
    large for it (the 30-atom host grid's points): each solve equals that of
    an engine that held nothing before, bit for bit."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lio_amd import g2g, systems
    made = {}
    for n in (2, 8, 30):
        Z, pos = systems.random_molecule_ang(n, 70 + n)
        made[n] = systems.make_system("reload%d" % n, Z, pos, seed=n)
    kept = g2g.Context(made[2], precision=precision)
    for n, mode in [(2, "device"), (30, "device"), (8, "host"), (30, "host"), (2, "host"),
                    (8, "device"), (30, "device")]:
        print("atoms", n, mode, flush=True)
        kept.set_grid_mode(mode)
        kept.set_system(made[n])
        kept.build_grid()
        kept.build_grid()  # the tables are written again at once
        fresh = g2g.Context(made[n], precision=precision, grid_mode=mode)
        fresh.build_grid()
        E0, F0, _ = fresh.solve()
        E1, F1, _ = kept.solve()
        assert E0 == E1 and np.array_equal(F0, F1)
        fresh.close()
    kept.close()
