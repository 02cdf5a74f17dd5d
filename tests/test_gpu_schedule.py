"""The schedule knobs say what runs: knobs that were read can be set again
without changing the build, the automatic Fock slices can be restored, and
the tuner can choose them.

Another slice length sums the Fock matrix in another order, so equal bits mean
the same slices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _torch():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _batch(precision):
    from lio_amd import g2g, systems
    mols = []
    for n in (3, 12, 45):  # groups of some 30 to some 400 functions
        Z, pos = systems.random_molecule_ang(n, 50 + n)
        mols.append(systems.make_system("mol%d" % n, Z, pos, seed=n))
    return g2g.Batch(mols, precision=precision)


def _fock(b, rho, torch):
    F = torch.zeros_like(rho)
    torch.cuda.synchronize()
    b.solve_device(rho.data_ptr(), F.data_ptr())
    b.energies()
    torch.cuda.synchronize()
    return F.cpu().numpy()


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x6"])
def test_schedule_read_and_set_again(precision):
    torch = _torch()
    from lio_amd import g2g
    b = _batch(precision)
    rho = torch.from_numpy(b.packed_density()).cuda()
    F0 = _fock(b, rho, torch)
    m, _ = b.group_sizes()
    print(precision, "functions", m.min(), m.max(), b.schedule(), flush=True)
    assert b.schedule()["fock_slice"] == (1024 if precision == "bf16x6" else g2g.AUTO_SLICE)
    read = b.schedule()
    b.set_schedule(fock_slice=read["fock_slice"], density_variant=read["density_variant"])
    assert np.array_equal(_fock(b, rho, torch), F0)
    b.set_schedule(fock_slice=2048)
    assert b.schedule()["fock_slice"] == 2048
    assert not np.array_equal(_fock(b, rho, torch), F0)
    b.set_schedule(fock_slice=g2g.AUTO_SLICE)
    assert b.schedule() == read
    assert np.array_equal(_fock(b, rho, torch), F0)
    # groups above the buckets: the automatic slice of their size
    bounds = [64, 128, 192, 384, 100000]
    b.set_bucket_slices(bounds, [g2g.auto_slice(precision, x) for x in bounds])
    assert np.array_equal(_fock(b, rho, torch), F0)
    b.set_bucket_slices(bounds[:2], [512, 512])
    F1 = _fock(b, rho, torch)
    b.set_bucket_slices(bounds, [512, 512] + [g2g.auto_slice(precision, x) for x in bounds[2:]])
    assert np.array_equal(_fock(b, rho, torch), F1)
    b.close()


@pytest.mark.parametrize("precision", ["fp64", "bf16x6"])
def test_tuner_can_choose_the_automatic_slices(precision):
    torch = _torch()
    from lio_amd import g2g
    b = _batch(precision)
    rho = torch.from_numpy(b.packed_density()).cuda()
    F0 = _fock(b, rho, torch)
    F = torch.zeros_like(rho)
    torch.cuda.synchronize()
    best, table = b.tune(rho.data_ptr(), F.data_ptr(), reps=2)
    print(precision, best, table, flush=True)
    assert (g2g.AUTO_SLICE, None) in table
    best, table = b.tune(rho.data_ptr(), F.data_ptr(), slices=(g2g.AUTO_SLICE,), reps=1)
    assert best == (g2g.AUTO_SLICE, None)
    assert np.array_equal(_fock(b, rho, torch), F0)
    # the tuner per size bucket starts from the automatic slices or from 1024
    sched = b.autotune(rho.data_ptr(), F.data_ptr(), slices=(), reps=1, persistent=(False,))
    auto = [g2g.auto_slice(precision, e) for e in sched["bucket_mhi"]]
    print(sched["bucket_slice"], sched["table"], flush=True)
    assert sched["bucket_slice"] in (auto, [1024] * len(auto)) and "automatic" in sched["table"]
    if sched["bucket_slice"] == auto:
        assert np.array_equal(_fock(b, rho, torch), F0)
    b.close()
