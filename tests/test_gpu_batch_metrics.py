"""Batches whose members have metrics of one kind and of different kinds, with
the heights that the contexts choose (GPU, through the C ABI)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def rel_l2(a, b):
    return float((a - b).norm() / b.norm())


def varying(disc):
    """The grid with a metric whose components vary with the level."""
    scale = 1.0 + 1e-3 * np.sin(0.7 * np.arange(disc.nz))
    disc.dXdxI = disc.dXdxI * scale[None, :, None, None, None, None]
    return disc


def alone(pkg, torch, disc, seed, precision):
    host, phys = pkg.host, pkg.discretization.Phys()
    FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, device="cuda", precision=precision)
    ctx = host.init_context(FE, Metric, phys, Global)
    V = torch.as_tensor(pkg.state.jet_state(disc, seed=seed), device="cuda").clone()
    host.TimeStepper(V, 100.0, 2, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    info = ctx.info()[2]
    ctx.close()
    return V.cpu(), info


def batch(pkg, torch, discs, seeds, precision):
    host = pkg.host
    ens = host.ensemble_setup(discs, precision=precision)
    V = torch.as_tensor(pkg.state.ensemble_state(discs, seeds), device="cuda").clone()
    host.TimeStepper(V, 100.0, 2, ens.FE[0], ens.Metric[0], pkg.discretization.Phys(), ens.Cache, ens.JCache, ens.Global)
    torch.cuda.synchronize()
    return ens, V.cpu()


@pytest.mark.parametrize("nes,p,nz,precision", [
    ([3, 2, 4], 4, 64, "fp64"), ([3, 2], 4, 57, "fp64"), ([3, 2], 3, 48, "fp64"), ([3, 2], 4, 64, "mixed"),
    ([10, 10, 10, 10], 4, 32, "fp64"),  # together enough workgroups for 16 levels in pass 1, alone not
])
def test_members_of_one_kind(pkg, torch_cuda, nes, p, nz, precision):
    print(f"batch of one kind nes={nes} p={p} nz={nz} {precision}", flush=True)
    grids = {ne: pkg.discretization.build(ne, p, nz, 512.0 * nz) for ne in set(nes)}
    discs, seeds = [grids[ne] for ne in nes], list(range(len(nes)))
    ens, V = batch(pkg, torch_cuda, discs, seeds, precision)
    assert ens.Global._ctx.info()[2]
    if len(nes) == 4:
        assert ens.Global._ctx.launch_shape()["pass1_chunk_levels"] == 16
    for m, (disc, seed) in enumerate(zip(discs, seeds)):
        want, compact = alone(pkg, torch_cuda, disc, seed, precision)
        assert compact and torch_cuda.equal(ens.member(V, m), want), f"member {m}"


@pytest.mark.parametrize("nz,precision", [(20, "fp64"), (64, "fp64"), (20, "mixed"), (72, "fp64")])
def test_members_of_different_kinds(pkg, torch_cuda, monkeypatch, nz, precision):
    """One member whose metric varies with the level: all have the bits of
    their own contexts in the full layout, and agree to rounding (1e-12; the
    mixed mode's kernels of both layouts read the same values) with their
    default ones."""
    print(f"batch of two kinds nz={nz} {precision}", flush=True)
    build = pkg.discretization.build
    discs, seeds = [build(3, 4, nz, 512.0 * nz), varying(build(2, 4, nz, 512.0 * nz)), build(2, 4, nz, 512.0 * nz)], [0, 1, 2]
    ens, V = batch(pkg, torch_cuda, discs, seeds, precision)
    assert not ens.Global._ctx.info()[2]
    for m, (disc, seed) in enumerate(zip(discs, seeds)):
        want, compact = alone(pkg, torch_cuda, disc, seed, precision)
        assert compact == (m != 1)
        monkeypatch.setenv("CGD_METRIC", "full")
        full, _ = alone(pkg, torch_cuda, disc, seed, precision)
        monkeypatch.delenv("CGD_METRIC")
        got = ens.member(V, m)
        assert torch_cuda.equal(got, full), f"member {m}"
        for c in range(5):
            assert rel_l2(got[c], want[c]) <= 1e-12, f"member {m} V{c + 1}"
