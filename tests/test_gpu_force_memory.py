"""The memory of the FP64 and FP32 force passes.

Y = P_g phi lies where the grid's allocation has room (the Fock matrix's
buffers, not yet in use, and the bytes to spare) and is formed again for the
groups that do not fit there, to the same bits.  So a forces call takes no
device memory, whatever was loaded before, and its results do not depend on
how much of Y was kept.
"""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _torch():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _system(n, opened=False, iexch=9):
    from lio_amd import systems
    Z, pos = systems.random_molecule_ang(n, 50 + n)
    s = systems.make_system("mol%d" % n, Z, pos, seed=n, iexch=iexch)
    return systems.open_shell(s) if opened else s


def _child(code):
    r = subprocess.run([sys.executable, "-u", "-c", code % {"root": ROOT}], capture_output=True,
                       text=True, timeout=200)
    print(r.stdout[-2000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0
    line = [x for x in r.stdout.splitlines() if x.startswith("RESULT ")][-1]
    return json.loads(line[len("RESULT "):])


FREE = r"""
import json, sys
sys.path.insert(0, %(root)r)
import torch
from lio_amd import g2g, systems

def run(ctx, s, forces):
    if s.open:
        ctx.solve_open(fock=True, forces=forces)
    elif forces:
        ctx.solve_forces(s.rho_packed)
    else:
        ctx.solve(s.rho_packed)

out = []
for prec in ("fp64", "fp32"):
    for opened in (False, True):
        for n in (5, 45):          # the small one loads every kernel
            Z, pos = systems.random_molecule_ang(n, 50 + n)
            s = systems.make_system("mol", Z, pos, seed=n)
            if opened:
                s = systems.open_shell(s)
            ctx = g2g.Context(s, precision=prec, grid_mode="device")
            ctx.build_grid()
            run(ctx, s, False)
            free = torch.cuda.mem_get_info()[0]
            run(ctx, s, True)
            out.append([prec, opened, n, free - torch.cuda.mem_get_info()[0]])
            print(out[-1], flush=True)
            ctx.close()
print("RESULT " + json.dumps(out), flush=True)
"""


def test_forces_take_no_device_memory():
    """In a process whose pool holds nothing, the free device memory is the
    same before and after the first forces call of a grid (45 atoms: Y is
    some 100 MB in FP64, of two spins twice that)."""
    _torch()
    for prec, opened, n, taken in _child(FREE):
        if n == 45:
            assert taken <= 0, (prec, opened, taken)


def _forces(ctx, s):
    if s.open:
        E, Fa, Fb, f, _ = ctx.solve_open(fock=True, forces=True)
        return E, np.asarray(f), np.concatenate([Fa, Fb])
    F = np.zeros(s.M * (s.M + 1) // 2)
    E, f, _ = ctx.solve_forces(s.rho_packed, fock=F)
    return E, np.asarray(f), F


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_forces_across_reloads_equal_recomputed(precision):
    """One engine takes grids of growing and shrinking size, one and two
    spins, both kinds of functional and both precisions in turn, so that Y
    lies in an allocation of an earlier grid, whole, in part or not at all:
    energies, forces and Fock matrices equal bit for bit those of the entry
    point that forms all of Y again."""
    torch = _torch()
    from lio_amd import g2g
    other = "fp32" if precision == "fp64" else "fp64"
    kept = g2g.Context(_system(2), precision=precision)
    seen = []
    for n, opened, iexch, prec in [(9, False, 9, precision), (9, True, 9, precision),
                                   (22, True, 9, precision), (22, False, 2, precision),
                                   (22, False, 9, other), (5, False, 9, precision),
                                   (9, True, 9, other), (30, False, 9, precision),
                                   (30, True, 9, precision), (9, False, 2, precision)]:
        s = _system(n, opened, iexch)
        kept.set_precision(prec)
        kept.set_system(s)
        kept.build_grid()
        held, total = kept.force_y()
        print("atoms", n, "open", opened, "iexch", iexch, prec, "held %d of %d" % (held, total),
              flush=True)
        seen.append((held, total))
        for _ in range(2):
            E, f, Fk = _forces(kept, s)
            b = g2g.Batch([s], precision=prec)
            rho = torch.from_numpy(b.packed_density()).cuda()
            F = torch.zeros_like(rho)
            g = torch.zeros(3 * s.natom, dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            b.solve_forces_static(rho.data_ptr(), F.data_ptr(), g.data_ptr())
            E0, _ = b.energies()
            torch.cuda.synchronize()
            b.close()
            assert E == E0[0]
            assert np.array_equal(Fk, F.cpu().numpy())
            assert np.array_equal(f.reshape(-1, 3)[:s.natom], g.cpu().numpy().reshape(-1, 3))
    kept.close()
    # a closed shell's Y is a tenth of its planes, the headroom an eighth
    fresh = g2g.Context(_system(22), precision=precision)
    fresh.build_grid()
    held, total = fresh.force_y()
    fresh.close()
    assert held == total > 0


SLAB = r"""
import json, sys
import numpy as np
sys.path.insert(0, %(root)r)
from lio_amd import g2g, systems
g2g.reserve_slab(3 << 30)
out = []
for prec in ("fp64", "fp32"):
    for opened in (False, True):
        Z, pos = systems.random_molecule_ang(22, 72)
        s = systems.make_system("mol22", Z, pos, seed=22)
        if opened:
            s = systems.open_shell(s)
        ctx = g2g.Context(s, precision=prec)
        ctx.build_grid()
        f = ctx.solve_open(fock=True, forces=True)[3] if opened else ctx.solve_forces()[1]
        out.append([prec, opened, ctx.force_y()[0], np.asarray(f).tolist()])
        ctx.close()
print("RESULT " + json.dumps(out), flush=True)
"""


def test_forces_from_a_slab_equal_those_with_more_y_kept():
    """A grid carved from the slab has no bytes to spare: solve_forces and
    solve_open form more of Y again, to the bits of a grid that keeps it."""
    _torch()
    from lio_amd import g2g
    for prec, opened, held, f in _child(SLAB):
        s = _system(22, opened)
        ctx = g2g.Context(s, precision=prec)
        ctx.build_grid()
        E, f0, _ = _forces(ctx, s)
        mine = ctx.force_y()[0]
        ctx.close()
        print(prec, opened, "held", held, "here", mine, flush=True)
        assert held < mine
        assert np.array_equal(np.asarray(f), f0)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("iexch", [9, 2])
def test_bytes_of_a_grid(precision, iexch):
    """A grid's bytes are its planes, P_g and F_g per group, the slices'
    partial Fock tiles, the density's partial sums (ten per point and chunk of
    64 functions, one in LDA), the force sums, six values per point, and lists
    of under 32 MB."""
    _torch()
    from lio_amd import g2g
    b = g2g.Batch([_system(45, iexch=iexch)], precision=precision)
    m, p = (x.astype(np.int64) for x in b.group_sizes())
    item = 8 if precision == "fp64" else 4
    planes = (10 if iexch == 9 else 4) * item * int((m * p).sum())
    blocks = int((m * m).sum())
    tiles, chunks = (m + 63) // 64, (p + 63) // 64 * ((m + 63) // 64)
    sl = np.array([g2g.auto_slice(precision, x) for x in m])
    fpart = int((tiles * (tiles + 1) // 2 * ((p + sl - 1) // sl)).sum()) * 64 * 64 * 8
    cpart = int(chunks.sum()) * (10 if iexch == 9 else 1) * 64 * 8
    force = 24 * int(((p + 63) // 64 * m).sum())
    bound = planes + item * blocks + 8 * blocks + fpart + cpart + force \
        + 48 * int(p.sum()) + (32 << 20)
    print(precision, iexch, "arena", b.arena_bytes(), "bound", bound, "sums", cpart, flush=True)
    got = b.arena_bytes()
    b.close()
    assert got <= bound


GROW = r"""
import json, sys
sys.path.insert(0, %%(root)r)
from lio_amd import g2g, systems
def system(n):
    Z, pos = systems.random_molecule_ang(n, 50 + n)
    return systems.make_system("mol", Z, pos, seed=n)
small, large = system(22), system(30)
g2g.reserve_slab(%(slab)d)
ctx = g2g.Context(small, precision="bf16x6")
ctx.build_grid()
ctx.solve_forces()
ctx.set_precision("%(prec)s")
ctx.set_system(large)
ctx.build_grid()
print("RESULT " + json.dumps(ctx.solve()[0]), flush=True)
"""


@pytest.mark.parametrize("prec", ["bf16x6", "fp32"])
def test_a_larger_grid_takes_the_place_of_an_old_y(prec):
    """The Y buffer of split-BF16 forces that a larger grid, or one of another
    precision, cannot use is given back before that grid is placed: a slab
    that holds the new grid alone takes it."""
    _torch()
    from lio_amd import g2g
    ctx = g2g.Context(_system(22), precision="bf16x6")
    first = ctx.build_grid()["arena_bytes"] + 4 * ctx.force_y()[1] + 1024
    ctx.set_precision(prec)
    middle = ctx.grid_info()["arena_bytes"]
    ctx.set_system(_system(30))
    second = ctx.build_grid()["arena_bytes"]
    E = ctx.solve()[0]
    ctx.close()
    slab = max(first, middle, second) + (1 << 20)
    print("arena and Y %d, then %d and %d, slab %d" % (first, middle, second, slab), flush=True)
    assert second > first  # so old Y and new grid do not fit together
    assert _child(GROW % {"slab": slab, "prec": prec}) == E


@pytest.mark.parametrize("opened", [False, True])
def test_captured_forces_replay(opened):
    """An FP64 forces call allocates nothing, so it can be captured: every
    replay, with eager builds of another density between them, equals the
    eager call."""
    torch = _torch()
    from lio_amd import g2g
    s = _system(9, opened)
    b = g2g.Batch([s], precision="fp64")
    rho = torch.from_numpy(b.packed_density()).cuda()
    other = 0.5 * rho
    F = torch.zeros_like(rho)
    f = torch.zeros(3 * s.natom, dtype=torch.float64, device="cuda")
    g = torch.zeros_like(f)
    torch.cuda.synchronize()
    b.solve_forces(rho.data_ptr(), F.data_ptr(), f.data_ptr())
    b.energies()
    want, wantF = f.clone(), F.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.ExternalStream(b.stream())
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        b.solve_forces(rho.data_ptr(), F.data_ptr(), f.data_ptr())
    for k in range(3):
        f.fill_(-7.0)
        F.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(f, want) and torch.equal(F, wantF)
        b.solve_forces(other.data_ptr(), F.data_ptr(), g.data_ptr())
        b.energies()
        assert not torch.equal(g, want)
    b.close()
