"""The element kernels and the column kernels at the sizes where they can go
wrong (edges of level chunks and of wavefronts, both orders), through the C
ABI, against the CPU oracle.

FP64 results are held to 1e-12 relative L2 per component on a state with
noise in the wind: the sums have a few dozen terms of 1.1e-16 relative
rounding each, with cancellation of up to 1e2 in the noisy state.  Steps of
the mixed mode are held to 1e-5, the bar of that mode's FP32 tendency.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12


def rel_l2(a, b):
    den = np.linalg.norm(np.ravel(b))
    return float(np.linalg.norm(np.ravel(a - b)) / (den if den > 0 else 1.0))


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def noisy_state(pkg, disc, seed):
    U = pkg.state.jet_state(disc, seed=seed)
    rng = np.random.default_rng(seed)
    U[1] += 5.0 * rng.standard_normal(U[1].shape)
    U[2] += 5.0 * rng.standard_normal(U[2].shape)
    U[3] += 0.5 * rng.standard_normal(U[3].shape)
    U[3][:, -1] = 0.0
    return U


def setup(pkg, oracle_mod, ne, p, nz, H=30000.0, **kw):
    disc = pkg.discretization.build(ne, p, nz, H)
    phys = pkg.discretization.Phys()
    dev = pkg.host.device_setup(disc, phys, device="cuda", **kw)
    hd = pkg.host.hyperdiffusion_for(ne)
    kw.pop("precision", None)
    orc = oracle_mod.Oracle(disc, phys, (hd, hd, hd), **kw)
    return disc, phys, dev, orc


def tendency(torch, host, phys, dev, U0):
    FE, Metric, Global, Cache, JCache = dev
    U = torch.as_tensor(U0, device="cuda")
    F = torch.full_like(U, 7.0)
    eq = host.CompressibleShallow()
    host.FcnPrepareGPU(U, FE, Metric, phys, Cache, None, Global, None, eq)
    host.FcnGPU(F, U, FE, Metric, phys, Cache, None, Global, None, eq)
    torch.cuda.synchronize()
    return F.cpu().numpy(), Cache.Temp1.cpu().numpy()


@pytest.mark.parametrize("metric", ["regular", "compact", "full"])
@pytest.mark.parametrize("H", [30000.0, None])
@pytest.mark.parametrize("p,nz,chunk", [(4, 3, 8), (4, 8, 8), (4, 9, 8), (4, 17, 16), (4, 31, 16), (3, 7, 8),
                                        (3, 16, 8), (3, 25, 8)])
def test_tendency_metric_kernels(pkg, oracle_mod, torch_cuda, monkeypatch, metric, p, nz, chunk, H):
    """The tendency kernel of a regular metric, the general one on the same
    metric, and the full layout; every face, edge and corner of the sphere
    sums its element copies (ne = 2: every element touches a corner).  With
    layers of 512 m (H = None) the metric for p = 4 is the same at all levels
    to the bit, as the regular and the compact layout ask."""
    if metric != "regular":
        monkeypatch.setenv("CGD_METRIC", metric)
    print(f"tendency {metric} p={p} nz={nz} chunk={chunk}", flush=True)
    disc, phys, dev, orc = setup(pkg, oracle_mod, 2, p, nz, H=H or 512.0 * nz)
    ctx = pkg.host.init_context(dev[0], dev[1], phys, dev[2])
    ctx.set_launch_shape(chunk_levels=chunk)
    if metric == "full" or (H is None and p == 4):
        assert ctx.info()[2] == (metric != "full")
    U0 = noisy_state(pkg, disc, 3)
    F, T1 = tendency(torch_cuda, pkg.host, phys, dev, U0)
    Fo, T1o = orc.fcn(U0.copy(), orc.prepare(U0.copy()))
    for v in range(5):
        assert rel_l2(T1[v], T1o[v]) <= TOL, f"Temp1[{v}] {rel_l2(T1[v], T1o[v]):.3e}"
        assert rel_l2(F[v], Fo[v]) <= TOL, f"F{v + 1} {rel_l2(F[v], Fo[v]):.3e}"
    assert np.all(F[3][:, -1] == 0.0)


@pytest.mark.parametrize("chunk", [0, 8])
@pytest.mark.parametrize("p,nz", [(4, 47), (4, 48), (4, 63), (3, 48), (3, 64)])
def test_pass1_columns(pkg, oracle_mod, torch_cuda, p, nz, chunk):
    """Pass 1 over whole columns (48 <= nz <= 64 unless a chunk height is set)
    and in level chunks, and in the mixed mode's steps."""
    torch, host = torch_cuda, pkg.host
    print(f"pass 1 p={p} nz={nz} chunk={chunk}", flush=True)
    disc, phys, dev, orc = setup(pkg, oracle_mod, 2, p, nz)
    ctx = host.init_context(dev[0], dev[1], phys, dev[2])
    if chunk:
        ctx.set_launch_shape(pass1_chunk_levels=chunk)
    U0 = noisy_state(pkg, disc, 4)
    F, T1 = tendency(torch, host, phys, dev, U0)
    Fo, T1o = orc.fcn(U0.copy(), orc.prepare(U0.copy()))
    for v in range(5):
        assert rel_l2(T1[v], T1o[v]) <= TOL, f"Temp1[{v}] {rel_l2(T1[v], T1o[v]):.3e}"
        assert rel_l2(F[v], Fo[v]) <= TOL, f"F{v + 1} {rel_l2(F[v], Fo[v]):.3e}"
    disc, phys, dev, orc = setup(pkg, oracle_mod, 2, p, nz, precision="mixed")
    FE, Metric, Global, Cache, JCache = dev
    ctx = host.init_context(FE, Metric, phys, Global)
    if chunk:
        ctx.set_launch_shape(pass1_chunk_levels=chunk)
    U0 = pkg.state.jet_state(disc, seed=5)
    V = torch.as_tensor(U0, device="cuda").clone()
    host.TimeStepper(V, 300.0, 2, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    Vo = U0.copy()
    orc.rw_step(Vo, 300.0, 2)
    for c in range(5):
        e = rel_l2(V[c].cpu().numpy(), Vo[c])
        assert e <= 1e-5, f"mixed V{c + 1} {e:.3e}"


@pytest.mark.parametrize("p,nz,ntr", [(3, 7, 0), (4, 11, 0), (3, 50, 2)])
def test_hooks_with_the_copies(pkg, oracle_mod, torch_cuda, p, nz, ntr):
    """Forcing and damping where the copies are summed (point counts that no
    workgroup divides), in the tendency and in the step."""
    torch, host = torch_cuda, pkg.host
    damping = (30000.0, 12000.0, 0.05)
    print(f"hooks p={p} nz={nz} NumTr={ntr}", flush=True)
    disc = pkg.discretization.build(2, p, nz, 30000.0)
    phys = pkg.discretization.Phys()
    dev = host.device_setup(disc, phys, device="cuda", NumTr=ntr, damping=damping, forcing=True)
    FE, Metric, Global, Cache, JCache = dev
    hd = host.hyperdiffusion_for(2)
    orc = oracle_mod.Oracle(disc, phys, (hd, hd, hd), NumTr=ntr, damping=damping, forcing=host.held_suarez_param())
    U0 = noisy_state(pkg, disc, 6)
    U0 = np.concatenate([U0] + [0.01 * (t + 1) * U0[0:1] for t in range(ntr)], axis=0)
    F, _ = tendency(torch, host, phys, dev, U0)
    Fo, _ = orc.fcn(U0.copy(), orc.prepare(U0.copy()))
    for v in range(5 + ntr):
        assert rel_l2(F[v], Fo[v]) <= TOL, f"F{v + 1} {rel_l2(F[v], Fo[v]):.3e}"
    V = torch.as_tensor(U0, device="cuda").clone()
    host.TimeStepper(V, 100.0, 2, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    Vo = U0.copy()
    orc.rw_step(Vo, 100.0, 2)
    for v in range(5 + ntr):
        assert rel_l2(V[v].cpu().numpy(), Vo[v]) <= TOL, f"V{v + 1} {rel_l2(V[v].cpu().numpy(), Vo[v]):.3e}"


@pytest.mark.parametrize("nz,precision", [(65, "fp64"), (128, "fp64"), (129, "fp64"), (256, "fp64"), (65, "mixed")])
def test_tall_columns(pkg, oracle_mod, torch_cuda, nz, precision):
    """Columns taller than a wavefront: the Schur solve (with and without a
    new tri) and the steps, which are FP64 in the mixed mode too."""
    torch, host = torch_cuda, pkg.host
    print(f"tall columns nz={nz} {precision}", flush=True)
    disc, phys, dev, orc = setup(pkg, oracle_mod, 2, 3, nz, precision=precision)
    FE, Metric, Global, Cache, JCache = dev
    U0 = pkg.state.jet_state(disc, seed=8)
    U = torch.as_tensor(U0, device="cuda")
    eq = host.CompressibleShallow()
    host.FcnPrepareGPU(U, FE, Metric, phys, Cache, None, Global, None, eq)
    host.JacSchurGPU(JCache, U, FE, Metric, phys, Cache, Global, None, eq)
    blocks = orc.jac(U0.copy(), orc.prepare(U0.copy()))
    JCache.CompTri = True
    for solve in range(2):  # the second reuses tri
        v0 = np.random.default_rng(solve).standard_normal(U0.shape)
        v = torch.as_tensor(v0, device="cuda")
        k = torch.zeros_like(v)
        host.SchurSolveGPU(k, v, JCache, 150.0, Cache, Global)
        torch.cuda.synchronize()
        vo = v0.copy()
        ko, trio = orc.schur(vo, blocks, 150.0)
        assert rel_l2(JCache.tri.cpu().numpy(), trio) <= TOL
        for c in range(5):
            assert rel_l2(k[c].cpu().numpy(), ko[c]) <= TOL, f"k[{c}] {rel_l2(k[c].cpu().numpy(), ko[c]):.3e}"
            assert rel_l2(v[c].cpu().numpy(), vo[c]) <= TOL, f"v[{c}]"
    V = U.clone()
    host.TimeStepper(V, 100.0, 2, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    Vo = U0.copy()
    orc.rw_step(Vo, 100.0, 2)
    for c in range(5):
        e = rel_l2(V[c].cpu().numpy(), Vo[c])
        assert e <= TOL, f"V{c + 1} {e:.3e}"


@pytest.mark.parametrize("scale", [1.0, 1.01])
def test_prepare_theta(pkg, torch_cuda, scale):
    """theta of the prepare kernel: the quotient where kappa = Rd/Cpd, the
    power of the pressure elsewhere and where the pressure is not a positive
    number.  A handful of roundings: 1e-14."""
    torch, host = torch_cuda, pkg.host

    class P(pkg.discretization.Phys):
        @property
        def kappa(self):
            return scale * (self.Rd / self.Cpd)

    phys = P()
    disc = pkg.discretization.build(2, 3, 11, 30000.0)
    print(f"prepare theta scale={scale}", flush=True)
    FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, device="cuda")
    U = torch.as_tensor(pkg.state.jet_state(disc, seed=2), device="cuda")
    U[4, 0, :3] = torch.tensor([-1.0, 0.0, float("nan")], dtype=U.dtype, device="cuda")
    host.FcnPrepareGPU(U, FE, Metric, phys, Cache, None, Global, None, host.CompressibleShallow())
    torch.cuda.synchronize()
    p, T, th = Cache.AuxG[0], Cache.AuxG[1], Cache.AuxG[2]
    want = (phys.p0 / p) ** (phys.Rd / phys.Cpd) * p / (phys.Rd * U[0])
    bad = torch.zeros_like(p, dtype=torch.bool)
    bad[0, :3] = True
    assert torch.equal(torch.isnan(th), torch.isnan(want)) and torch.isnan(th[bad]).all()
    assert float(((th - want) / want)[~bad].abs().max()) <= 1e-14


@pytest.mark.parametrize("limited", [False, True])
@pytest.mark.parametrize("metric", ["compact", "full"])
@pytest.mark.parametrize("p,nz,chunk,ntr", [(4, 3, 8, 1), (4, 9, 8, 3), (4, 17, 16, 2), (3, 8, 8, 2), (3, 25, 8, 1)])
def test_tracer_passes(pkg, oracle_mod, torch_cuda, monkeypatch, p, nz, chunk, ntr, metric, limited):
    """The tracers' element copies, halo levels and upwind fluxes, with equal
    and with general layer volumes, in steps (and in the plain transport's
    tendency and caches)."""
    torch, host = torch_cuda, pkg.host
    if metric == "full":
        monkeypatch.setenv("CGD_METRIC", "full")
    print(f"tracers p={p} nz={nz} chunk={chunk} NumTr={ntr} {metric} limited={limited}", flush=True)
    disc, phys, dev, orc = setup(pkg, oracle_mod, 2, p, nz, H=512.0 * nz, NumTr=ntr, horlimit=limited)
    FE, Metric, Global, Cache, JCache = dev
    host.init_context(FE, Metric, phys, Global).set_launch_shape(chunk_levels=chunk)
    U0 = noisy_state(pkg, disc, 9)
    q = 0.01 * (1.0 + 0.5 * np.random.default_rng(9).random((ntr,) + U0[0].shape))
    U0 = np.concatenate([U0, q * U0[0:1]], axis=0)
    if not limited:
        F, T1 = tendency(torch, host, phys, dev, U0)
        Fo, T1o = orc.fcn(U0.copy(), orc.prepare(U0.copy()))
        for v in range(5 + ntr):
            assert rel_l2(F[v], Fo[v]) <= TOL, f"F{v + 1} {rel_l2(F[v], Fo[v]):.3e}"
            assert rel_l2(T1[v], T1o[v]) <= TOL, f"Temp1[{v}] {rel_l2(T1[v], T1o[v]):.3e}"
    V = torch.as_tensor(U0, device="cuda").clone()
    host.TimeStepper(V, 100.0, 2, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    Vo = U0.copy()
    orc.rw_step(Vo, 100.0, 2)
    for v in range(5 + ntr):
        assert rel_l2(V[v].cpu().numpy(), Vo[v]) <= TOL, f"V{v + 1} {rel_l2(V[v].cpu().numpy(), Vo[v]):.3e}"


@pytest.mark.parametrize("nz", [44, 48, 60, 77])
def test_taller_chunks(pkg, torch_cuda, nz):
    """Both passes in chunks of 16 levels, which the context takes by itself,
    against 8 (44 and 60: a ragged last chunk)."""
    torch, host = torch_cuda, pkg.host
    print(f"taller chunks nz={nz}", flush=True)
    disc = pkg.discretization.build(16, 4, nz, 512.0 * nz)
    phys = pkg.discretization.Phys()
    dev = host.device_setup(disc, phys, device="cuda")
    FE, Metric, Global, Cache, JCache = dev
    ctx = host.init_context(FE, Metric, phys, Global)
    U0 = noisy_state(pkg, disc, 10)
    out = []
    for shape in ({}, {"chunk_levels": 8, "pass1_chunk_levels": 8}):
        ctx.set_launch_shape(**shape)
        F, T1 = tendency(torch, host, phys, dev, U0)
        V = torch.as_tensor(U0, device="cuda").clone()
        host.TimeStepper(V, 100.0, 2, FE, Metric, phys, Cache, JCache, Global)
        torch.cuda.synchronize()
        out.append((F, T1, V.cpu().numpy()))
    for x, y in zip(*out):
        for v in range(5):
            assert rel_l2(x[v], y[v]) <= TOL, f"{v + 1} {rel_l2(x[v], y[v]):.3e}"
    if nz < 48 or nz > 64:  # no columns: pass 1's chunk height changes no bit
        assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("nz", [3, 33, 64])
def test_column_calls_alignment(pkg, torch_cuda, nz):
    """The Jacobian and the column solve on J blocks that take 16-byte
    accesses and on ones that do not: the same bits."""
    torch, host = torch_cuda, pkg.host
    print(f"column alignment nz={nz}", flush=True)
    disc = pkg.discretization.build(2, 3, nz, 30000.0)
    phys = pkg.discretization.Phys()
    FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, device="cuda")
    U = torch.as_tensor(pkg.state.jet_state(disc, seed=11), device="cuda")
    eq = host.CompressibleShallow()
    names = ("JRhoW", "JWRho", "JWRhoTh", "JRhoThW")
    out = []
    for shift in (0, 1):
        for name in names:
            J = getattr(JCache, name)
            view = torch.zeros(J.numel() + 2, dtype=J.dtype, device="cuda")[shift:shift + J.numel()].view(J.shape)
            assert view.data_ptr() % 16 == 8 * shift
            setattr(JCache, name, view)
        host.FcnPrepareGPU(U, FE, Metric, phys, Cache, None, Global, None, eq)
        host.JacSchurGPU(JCache, U, FE, Metric, phys, Cache, Global, None, eq)
        v = torch.as_tensor(np.random.default_rng(11).standard_normal(tuple(U.shape)), device="cuda")
        k = torch.zeros_like(v)
        JCache.CompTri = True
        host.SchurSolveGPU(k, v, JCache, 150.0, Cache, Global)
        torch.cuda.synchronize()
        out.append([getattr(JCache, n).cpu() for n in names] + [JCache.tri.cpu(), k.cpu(), v.cpu()])
    assert all(torch.equal(x, y) for x, y in zip(*out))
