"""CGD_THOMAS=1: the serial recurrence of the column solve in its own order, at
every height (GPU, through the C ABI).

The expected solution is triSolve!'s recurrence on the tri matrix and the
right-hand side that the call leaves, in exact rational arithmetic rounded where
the kernel rounds (a - q b is one fused multiply-add): the same bits.
"""
from fractions import Fraction

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def thomas(t0, t1, t2, rhs):
    n = len(rhs)
    fma = lambda q, x, y: float(Fraction(y) - Fraction(q) * Fraction(x))  # noqa: E731
    x, b = [float(t1[0])], [float(rhs[0])]
    for j in range(n - 1):
        q = float(t2[j]) / x[j]
        x.append(fma(q, float(t0[j + 1]), float(t1[j + 1])))
        b.append(fma(q, b[j], float(rhs[j + 1])))
    sol = [0.0] * n
    sol[-1] = b[-1] / x[-1]
    for j in range(n - 2, -1, -1):
        sol[j] = fma(float(t0[j + 1]), sol[j + 1], b[j]) / x[j]
    return np.array(sol)


@pytest.mark.parametrize("nz", [20, 64, 65, 70, 129, 256])
def test_serial_recurrence(pkg, oracle_mod, monkeypatch, nz):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    host = pkg.host
    print(f"thomas nz={nz}", flush=True)
    disc = pkg.discretization.build(2, 3, nz, 30000.0)
    phys = pkg.discretization.Phys()
    eq = host.CompressibleShallow()
    U0 = pkg.state.jet_state(disc, seed=8)
    monkeypatch.setenv("CGD_THOMAS", "1")
    FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, device="cuda")
    host.init_context(FE, Metric, phys, Global)
    U = torch.as_tensor(U0, device="cuda")
    host.FcnPrepareGPU(U, FE, Metric, phys, Cache, None, Global, None, eq)
    host.JacSchurGPU(JCache, U, FE, Metric, phys, Cache, Global, None, eq)
    JCache.CompTri = True
    for solve in range(2):  # the second reuses tri
        v = torch.as_tensor(np.random.default_rng(solve).standard_normal(U0.shape), device="cuda")
        k = torch.zeros_like(v)
        host.SchurSolveGPU(k, v, JCache, 150.0, Cache, Global)
        torch.cuda.synchronize()
        tri, rhs, k4 = JCache.tri.cpu().numpy(), v[3].cpu().numpy(), k[3].cpu().numpy()
        for ig in (0, 7, disc.num_g - 1):
            assert np.array_equal(k4[ig, :-1], thomas(*tri[ig].T, rhs[ig, :-1])) and k4[ig, -1] == 0.0
    V = U.clone()
    host.TimeStepper(V, 100.0, 2, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    hd = host.hyperdiffusion_for(2)
    orc = oracle_mod.Oracle(disc, phys, (hd, hd, hd))
    Vo = U0.copy()
    orc.rw_step(Vo, 100.0, 2)
    for c in range(5):
        d = np.linalg.norm(V[c].cpu().numpy() - Vo[c]) / np.linalg.norm(Vo[c])
        assert d <= 1e-12, f"V{c + 1} {d:.3e}"
