"""Values that are not numbers, in the tendency of a regular metric against the
general kernel on the same metric (GPU, through the C ABI)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("p,nz,level", [(4, 20, 7), (4, 20, 8), (4, 64, 33), (3, 9, 0), (3, 9, 8)])
def test_nonfinite_theta_reaches_the_same_points(pkg, monkeypatch, p, nz, level, bad):
    """rho*theta of one point NaN or infinite (rho, the wind and the pressure
    finite): the upwind flux of theta through both of its level's interfaces
    is not a number whichever side is upwind, in both kernels."""
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    host = pkg.host
    print(f"nonfinite p={p} nz={nz} level={level} {bad}", flush=True)
    disc = pkg.discretization.build(2, p, nz, 512.0 * nz)
    phys = pkg.discretization.Phys()
    eq = host.CompressibleShallow()
    out = []
    for metric in ("regular", "compact"):
        monkeypatch.setenv("CGD_METRIC", metric)
        FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, device="cuda")
        ctx = host.init_context(FE, Metric, phys, Global)
        assert ctx.info()[2]
        U0 = pkg.state.jet_state(disc, seed=3)
        rng = np.random.default_rng(3)
        U0[1:4] += rng.standard_normal(U0[1:4].shape)
        U0[3][:, -1] = 0.0
        U = torch.as_tensor(U0, device="cuda")
        host.FcnPrepareGPU(U, FE, Metric, phys, Cache, None, Global, None, eq)
        U[4, ::7, level] = bad
        F = torch.zeros_like(U)
        host.FcnGPU(F, U, FE, Metric, phys, Cache, None, Global, None, eq)
        torch.cuda.synchronize()
        out.append(torch.isfinite(F).cpu())
        ctx.close()
    for v in range(5):
        assert torch.equal(out[0][v], out[1][v]), f"F{v + 1}: {int((out[0][v] != out[1][v]).sum())} points differ"
    for other in (level - 1, level + 1):
        if 0 <= other < nz:
            assert not out[0][4][::7, other].any()
