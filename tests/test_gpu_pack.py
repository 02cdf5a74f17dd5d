"""The forms of the Fock packing (a map of F_g's rows by group, of local indices
by group, of these for some groups at a time), which the number of a
molecule's groups chooses: up to 8192, up to 16384, above.  Four waters on a fine cube lattice have that many
groups; their quadrature points are the same on every lattice."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = [(1.0, 0, 8192), (0.8, 8192, 16384), (0.5, 8192, 16384), (0.4, 16384, 1 << 30)]


def _torch():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _waters(n):
    from lio_amd import systems
    if n == 1:
        return systems.config0()
    Z, pos = systems.water_cluster_ang(n, box=5.0, seed=1)
    return systems.make_system("w%d" % n, Z, pos, seed=1)


def _options(cube):
    # every function in every group, so that the lattice only groups the sums
    return dict(little_cube_size=cube, assign_all_functions=1, sphere_radius=0.0)


def test_fock_of_many_groups():
    """Sums of 86180 points of order one, in FP64, grouped otherwise: 1e-10."""
    _torch()
    from lio_amd import g2g
    s = _waters(4)
    ref = None
    for cube, lo, hi in [(30.0, 0, 8192)] + FORMS:
        ctx = g2g.Context(s, grid_mode="device", **_options(cube))
        info = ctx.build_grid()
        E, F, si = ctx.solve()
        ctx.close()
        print("cube", cube, "groups", info["ngroups"], "pack ms", si["kernel_ms"][3], flush=True)
        assert lo < info["ngroups"] <= hi
        if ref is None:
            ref = E, F
        assert abs(E - ref[0]) <= 1e-10 and np.max(np.abs(F - ref[1])) <= 1e-10


@pytest.mark.parametrize("cube", [f[0] for f in FORMS])
def test_forms_sum_in_one_order(cube):
    """The largest molecule of a batch chooses the form for all: the small
    one's Fock matrix is bitwise the one it gives alone, by rows."""
    torch = _torch()
    from lio_amd import g2g

    def fock(mols):
        b = g2g.Batch(mols, precision="fp64", grid_mode="device", **_options(cube))
        rho = torch.from_numpy(b.packed_density()).cuda()
        F = torch.zeros_like(rho)
        torch.cuda.synchronize()
        b.solve_device(rho.data_ptr(), F.data_ptr())
        b.energies()
        torch.cuda.synchronize()
        out = F[:int(b.offsets[1])].cpu().numpy()
        b.close()
        return out

    print("cube", cube, flush=True)
    assert np.array_equal(fock([_waters(1)]), fock([_waters(1), _waters(4)]))
