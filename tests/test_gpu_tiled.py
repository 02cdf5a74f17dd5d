"""Tiled value planes and operand-ordered P_g of the chunked split-BF16
density (variants 10 and 11), on the GPU, at the sizes where the layouts have
edges: groups of one 32-function block, row counts that end inside a chunk,
point counts that are not multiples of 64.

The tiled layout holds the values of the point-major planes, P_g the same
pieces, so every product is variant 8's; the FP64 epilogue sums differ in
grouping only: 1e-10 on Exc, N, F and the forces, as for the chunked form's
other comparisons.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SAME = 1e-10


def _molecule(name):
    from lio_amd import systems
    if name == "water":
        return systems.config0()
    n, iexch = name
    Z, pos = systems.random_molecule_ang(n, 50 + n)
    return systems.make_system("mol%d" % n, Z, pos, seed=n, iexch=iexch)


@pytest.mark.parametrize("grid_type", [0, 2])
@pytest.mark.parametrize("name", ["water", (2, 9), (5, 9), (9, 9), (14, 3), (22, 9)])
def test_tiled_layout_equals_point_major(name, grid_type):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lio_amd import g2g
    s = _molecule(name)
    out = {}
    for variant in (8, 10, 11):
        ctx = g2g.Context(s, precision="bf16x6")
        ctx.set_schedule(density_variant=variant)
        ctx.build_grid(grid_type)
        F = np.zeros(s.M * (s.M + 1) // 2)
        E, f, info = ctx.solve_forces(fock=F)
        out[variant] = (E, info["electrons"], F, f)
        ctx.close()
    print("case", name, grid_type, out[10][0], out[10][0] - out[8][0], flush=True)
    for a, b in zip(out[8], out[10]):
        assert np.max(np.abs(np.asarray(a) - np.asarray(b))) <= SAME
    for a, b in zip(out[10], out[11]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("grid_type", [0, 2])
@pytest.mark.parametrize("name", ["water", (2, 9), (5, 9), (9, 9), (14, 3), (22, 9)])
def test_fp64_chunks_against_the_oracle(name, grid_type):
    """FP64 density in (point tile, 64-function chunk) blocks with the
    gradient forms up to the diagonal, at row counts of one to several chunks
    (and parts of them).  Oracle and library differ by FP64 round-off of sums
    of at most 1e5 terms of order one: 1e-10."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import os
    import sys
    sys.path.insert(0, os.path.join(os.path.dirname(__file__), "..", "oracle"))
    from pyxc import Oracle
    from lio_amd import g2g
    import dataclasses
    s = dataclasses.replace(_molecule(name), grid_type=grid_type)
    o = Oracle()
    o.setup(s)
    Eo, Fo, _ = o.solve()
    ctx = g2g.Context(s)
    ctx.build_grid()
    F = np.zeros(s.M * (s.M + 1) // 2)
    E, f, info = ctx.solve_forces(fock=F)
    fo = o.solve_forces()
    ctx.close()
    fo = fo[1] if isinstance(fo, tuple) else fo
    print("case", name, grid_type, E - Eo, np.max(np.abs(F - Fo)), flush=True)
    assert abs(E - Eo) <= SAME and abs(info["electrons"] - o.electrons()) <= SAME
    assert np.max(np.abs(F - Fo)) <= SAME
    assert np.max(np.abs(f - np.asarray(fo).reshape(f.shape))) <= SAME


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("opened", [False, True])
def test_forces_from_stored_y_equal_recomputed(precision, opened):
    """FP64 and FP32 forces with Y = P phi left by the density kernel and with
    Y recomputed (the entry point that allocates nothing, before a Y buffer
    exists): the same operations, so bitwise the same, at group sizes of one
    row tile to several chunks."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lio_amd import g2g, systems
    mols = [_molecule(n) for n in ((2, 9), (5, 9), (22, 9))]
    if opened:
        mols = [systems.open_shell(m) for m in mols]
    b = g2g.Batch(mols, precision=precision)
    rho = torch.from_numpy(b.packed_density()).cuda()
    F = torch.zeros_like(rho)
    f = torch.zeros((2, 3 * int(b.atoms()[-1])), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    b.solve_forces_static(rho.data_ptr(), F.data_ptr(), f[0].data_ptr())
    b.energies()
    b.solve_forces(rho.data_ptr(), F.data_ptr(), f[1].data_ptr())
    b.energies()
    torch.cuda.synchronize()
    b.close()
    assert float(f[0].abs().max()) > 0.0
    assert torch.equal(f[0], f[1])
