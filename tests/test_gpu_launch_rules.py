"""Which kernels run: the shape that a context reports, sets and tunes names
them (GPU, through the C ABI).  The kernels are read off torch's profiler.

The layers are 512 m thick, so that the metric has the same bits at all levels
(the compact layout, regular) at the level counts used here.
"""
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def kernels_of(torch, fn):
    """The names, without arguments, of the kernels that fn launches."""
    from torch.profiler import ProfilerActivity, profile

    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    names = {re.sub(r"^void |\(.*", "", e.key) for e in prof.key_averages()}
    return {n for n in names if n.startswith("k_")}


class Case:
    def __init__(self, pkg, torch, ne, p, nz, precision="fp64", ntr=0, thickness=512.0):
        self.host, self.torch = pkg.host, torch
        disc = pkg.discretization.build(ne, p, nz, thickness * nz)
        self.phys = pkg.discretization.Phys()
        self.dev = pkg.host.device_setup(disc, self.phys, device="cuda", precision=precision, NumTr=ntr)
        self.ctx = pkg.host.init_context(self.dev[0], self.dev[1], self.phys, self.dev[2])
        U0 = pkg.state.jet_state(disc, seed=1)
        U0 = np.concatenate([U0] + [0.01 * (t + 1) * U0[0:1] for t in range(ntr)], axis=0)
        self.U0 = torch.as_tensor(U0, device="cuda")

    def step(self, n=1):
        FE, Metric, Global, Cache, JCache = self.dev
        V = self.U0.clone()
        self.host.TimeStepper(V, 100.0, n, FE, Metric, self.phys, Cache, JCache, Global)
        self.torch.cuda.synchronize()
        return V

    def kernels(self):
        return {k for k in kernels_of(self.torch, self.step) if k.startswith(("k_fcn", "k_tr1", "k_tr2", "k_stage"))}


def heights(shape):
    return shape["chunk_levels"], shape["pass1_chunk_levels"]


@pytest.mark.parametrize("ne,p,nz,precision,ntr,shape,names", [
    (3, 4, 64, "fp64", 0, (16, 64), {"k_fcn1c<5, double>", "k_fcn2r<5, 16>"}),
    (3, 4, 62, "fp64", 1, (16, 64), {"k_fcn1c<5, double>", "k_fcn2r<5, 16>", "k_tr1<5, 8, true>", "k_tr2<5, 8, true>"}),
    (3, 4, 64, "mixed", 0, (8, 64), {"k_fcn1c<5, float>", "k_fcn2<5, 8, true, float, false>"}),
    (3, 3, 48, "fp64", 0, (8, 64), {"k_fcn1c<4, double>", "k_fcn2r<4, 8>"}),
    (19, 4, 32, "fp64", 0, (8, 16), {"k_fcn1<5, 16, true, double, 1>", "k_fcn2r<5, 8>"}),
    (3, 4, 32, "fp64", 0, (8, 8), {"k_fcn1<5, 8, true, double, 1>", "k_fcn2r<5, 8>"}),
    (3, 4, 72, "fp64", 0, (8, 8), {"k_fcn1<5, 8, true, double, 1>", "k_fcn2r<5, 8>"}),
    (3, 4, 80, "mixed", 0, (16, 8), {"k_fcn1<5, 8, true, double, 1>", "k_fcn2r<5, 16>"}),
    (3, 4, 50, "fp64", 0, (8, 8), {"k_fcn1<5, 8, false, double, 1>", "k_fcn2<5, 8, false, double, false>"}),
])
def test_shape_names_what_runs(pkg, torch_cuda, ne, p, nz, precision, ntr, shape, names):
    """The reported heights are those of the kernels that run; setting the
    reported shape, here or on a fresh context, changes neither; a height
    that is set runs, and the reported shape brings the first ones back."""
    print(f"shape ne={ne} p={p} nz={nz} {precision} NumTr={ntr}", flush=True)
    c = Case(pkg, torch_cuda, ne, p, nz, precision, ntr)
    first = c.ctx.launch_shape()
    assert heights(first) == shape and c.ctx.info()[1] == 8
    assert c.kernels() == names
    V = c.step(2)
    c.ctx.set_launch_shape(**first)
    assert c.ctx.launch_shape() == first and c.kernels() == names
    assert torch_cuda.equal(c.step(2), V)
    c.ctx.set_launch_shape(chunk_levels=8, pass1_chunk_levels=8)
    if shape != (8, 8):
        assert heights(c.ctx.launch_shape()) == (8, 8)
        ran = c.kernels()
        assert ran != names and not any(k.startswith("k_fcn1c") or ", 16" in k for k in ran)
    c.ctx.set_launch_shape(**first)
    assert c.ctx.launch_shape() == first and c.kernels() == names
    d = Case(pkg, torch_cuda, ne, p, nz, precision, ntr)
    d.ctx.set_launch_shape(**first)
    assert d.ctx.launch_shape() == first and d.kernels() == names
    assert torch_cuda.equal(d.step(2), V)


def test_columns_refused(pkg, torch_cuda, monkeypatch):
    """Whole columns need the compact metric and at most 64 levels."""
    print("columns refused", flush=True)
    for nz, metric, ok in ((64, "", True), (20, "", True), (72, "", False), (20, "full", False)):
        monkeypatch.setenv("CGD_METRIC", metric)
        c = Case(pkg, torch_cuda, 2, 4, nz)
        if ok:
            V = c.step(2)
            c.ctx.set_launch_shape(pass1_chunk_levels=64)
            assert "k_fcn1c<5, double>" in c.kernels()
            assert torch_cuda.equal(c.step(2), V)
        else:
            with pytest.raises(pkg.host.CGDError):
                c.ctx.set_launch_shape(pass1_chunk_levels=64)
        with pytest.raises(pkg.host.CGDError):
            c.ctx.set_launch_shape(chunk_levels=64)


@pytest.mark.parametrize("ne,nz,precision", [(3, 64, "fp64"), (19, 32, "fp64"), (3, 64, "mixed")])
def test_autotune_runs_its_candidates(pkg, torch_cuda, ne, nz, precision):
    """Every height that the context admits is timed, and the chosen shape is
    the one that runs, here and set on a fresh context."""
    print(f"autotune candidates ne={ne} nz={nz} {precision}", flush=True)
    c = Case(pkg, torch_cuda, ne, 4, nz, precision)
    FE, Metric, Global, Cache, JCache = c.dev
    got = {}
    V = c.U0.clone()
    ran = kernels_of(torch_cuda, lambda: got.update(s=c.ctx.autotune(V, 100.0, Cache, JCache, reps=1)))
    R = "float" if precision == "mixed" else "double"
    for z in (8, 16):
        assert f"k_fcn1<5, {z}, true, {R}, 1>" in ran and f"k_fcn1<5, {z}, true, {R}, 2>" in ran
        assert (f"k_fcn2<5, {z}, true, float, false>" if R == "float" else f"k_fcn2r<5, {z}>") in ran
    assert f"k_fcn1c<5, {R}>" in ran
    shape = got["s"][0]
    assert c.ctx.launch_shape() == shape and torch_cuda.equal(V, c.U0)
    names, V = c.kernels(), c.step(2)
    d = Case(pkg, torch_cuda, ne, 4, nz, precision)
    d.ctx.set_launch_shape(**shape)
    assert d.ctx.launch_shape() == shape and d.kernels() == names
    assert torch_cuda.equal(d.step(2), V)


def test_persistent_stands_in_for_the_chosen_heights(pkg, torch_cuda):
    """A persistent launch has chunks of 8 levels; the heights that the context
    chose stand again when it is turned off, and set ones are refused."""
    print("persistent heights", flush=True)
    c = Case(pkg, torch_cuda, 3, 4, 64)
    first = c.ctx.launch_shape()
    c.ctx.set_launch_shape(persistent=1)
    assert heights(c.ctx.launch_shape()) == (8, 8) and c.ctx.info()[1] == 8
    assert c.kernels() == {"k_stage_persist<5, true, double, 64, true>"}
    FE, Metric, Global, Cache, _ = c.dev
    F = torch_cuda.empty_like(c.U0)
    fcn = lambda: pkg.host.FcnGPU(F, c.U0, FE, Metric, c.phys, Cache, None, Global, None,  # noqa: E731
                                  pkg.host.CompressibleShallow())
    assert "k_fcn1c<5, double>" in kernels_of(torch_cuda, fcn)  # a separate tendency
    c.ctx.check_device()
    c.ctx.set_launch_shape(persistent=-1)
    assert c.ctx.launch_shape() == first
    with pytest.raises(pkg.host.CGDError):
        c.ctx.set_launch_shape(persistent=1, chunk_levels=16)
    c = Case(pkg, torch_cuda, 3, 4, 32)
    c.ctx.set_launch_shape(chunk_levels=16)
    with pytest.raises(pkg.host.CGDError):
        c.ctx.set_launch_shape(persistent=1)
    assert c.ctx.launch_shape()["chunk_levels"] == 16


@pytest.mark.parametrize("p,nz", [(4, 64), (4, 62), (4, 57), (4, 48), (4, 20), (3, 48)])
def test_heights_change_no_bit_of_a_regular_metric(pkg, torch_cuda, p, nz):
    """On a regular metric the tendency and the steps have the same bits at
    every height, and in persistent launches whichever heights the separate
    ones have (57, 62, 20: ragged last chunks)."""
    torch = torch_cuda
    print(f"heights p={p} nz={nz}", flush=True)
    c = Case(pkg, torch, 3, p, nz)
    FE, Metric, Global, Cache, JCache = c.dev
    eq = pkg.host.CompressibleShallow()
    U = c.U0 + torch.randn(c.U0.shape, generator=torch.Generator("cuda").manual_seed(1), device="cuda",
                           dtype=c.U0.dtype) * torch.tensor([0.0, 3.0, 3.0, 0.3, 0.0], device="cuda")[:, None, None]
    U[3, :, -1] = 0.0
    c.U0 = U

    def results():
        F = torch.empty_like(U)
        pkg.host.FcnPrepareGPU(U, FE, Metric, c.phys, Cache, None, Global, None, eq)
        pkg.host.FcnGPU(F, U, FE, Metric, c.phys, Cache, None, Global, None, eq)
        return F, Cache.Temp1[:5].clone(), c.step(3)

    want = results()
    assert all(bool(torch.isfinite(x).all()) for x in want)
    heights_ = [(8, 8)] + ([(16, 16), (8, 16), (16, 8)] if p == 4 else []) + [(8, 64)]
    for z2, z1 in heights_:
        c.ctx.set_launch_shape(chunk_levels=z2, pass1_chunk_levels=z1)
        for v, (x, y) in enumerate(zip(results(), want)):
            assert torch.equal(x, y), f"heights {z2}, {z1}, result {v}"
    d = Case(pkg, torch, 3, p, nz)
    d.U0 = U
    d.ctx.set_launch_shape(persistent=1, col_block=((p + 1) ** 2 * 8 + 63) // 64 * 64)
    assert torch.equal(d.step(3), want[2])
    d.ctx.check_device()
    d.ctx.set_launch_shape(persistent=-1)
    assert torch.equal(d.step(3), want[2])


def rel_l2(a, b):
    return float(np.linalg.norm(np.ravel(a - b)) / np.linalg.norm(np.ravel(b)))


@pytest.mark.parametrize("p,nz", [(4, 48), (4, 57), (4, 63), (3, 48), (3, 61)])
def test_columns_against_the_oracle(pkg, oracle_mod, torch_cuda, p, nz):
    """Pass 1 over whole columns of fewer levels than lanes: the caches and
    tendencies in FP64 to 1e-12 relative L2 (a few dozen terms of 1.1e-16 each,
    cancellation of up to 1e2), the mixed mode's steps to that mode's 1e-5."""
    torch, host = torch_cuda, pkg.host
    print(f"columns against the oracle p={p} nz={nz}", flush=True)
    disc = pkg.discretization.build(2, p, nz, 512.0 * nz)
    phys = pkg.discretization.Phys()
    hd = host.hyperdiffusion_for(2)
    orc = oracle_mod.Oracle(disc, phys, (hd, hd, hd))
    c = Case(pkg, torch, 2, p, nz)
    assert f"k_fcn1c<{p + 1}, double>" in c.kernels()
    rng = np.random.default_rng(4)
    U0 = c.U0.cpu().numpy()
    U0[1:4] += np.array([5.0, 5.0, 0.5])[:, None, None] * rng.standard_normal(U0[1:4].shape)
    U0[3][:, -1] = 0.0
    FE, Metric, Global, Cache, _ = c.dev
    U = torch.as_tensor(U0, device="cuda")
    F = torch.empty_like(U)
    eq = host.CompressibleShallow()
    host.FcnPrepareGPU(U, FE, Metric, phys, Cache, None, Global, None, eq)
    host.FcnGPU(F, U, FE, Metric, phys, Cache, None, Global, None, eq)
    torch.cuda.synchronize()
    Fo, T1o = orc.fcn(U0.copy(), orc.prepare(U0.copy()))
    for v in range(5):
        assert rel_l2(Cache.Temp1[v].cpu().numpy(), T1o[v]) <= 1e-12, f"Temp1[{v}]"
        assert rel_l2(F[v].cpu().numpy(), Fo[v]) <= 1e-12, f"F{v + 1}"
    m = Case(pkg, torch, 2, p, nz, "mixed")
    assert f"k_fcn1c<{p + 1}, float>" in m.kernels()
    Vo = m.U0.cpu().numpy().copy()
    orc.rw_step(Vo, 100.0, 2)
    V = m.step(2).cpu().numpy()
    for v in range(5):
        assert rel_l2(V[v], Vo[v]) <= 1e-5, f"mixed V{v + 1}"


@pytest.mark.parametrize("nz,precision", [(70, "fp64"), (130, "fp64"), (70, "mixed")])
def test_hooks_above_64_levels(pkg, oracle_mod, torch_cuda, nz, precision):
    """Forcing and damping in the fused stage of columns taller than a
    wavefront (FP64 in either mode), to 1e-12 relative L2 of the oracle."""
    torch, host = torch_cuda, pkg.host
    print(f"hooks above 64 levels nz={nz} {precision}", flush=True)
    damping = (30000.0, 12000.0, 0.05)
    disc = pkg.discretization.build(2, 3, nz, 30000.0)
    phys = pkg.discretization.Phys()
    FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, device="cuda", damping=damping, forcing=True,
                                                          precision=precision)
    hd = host.hyperdiffusion_for(2)
    orc = oracle_mod.Oracle(disc, phys, (hd, hd, hd), damping=damping, forcing=host.held_suarez_param())
    U0 = pkg.state.jet_state(disc, seed=6)
    V = torch.as_tensor(U0, device="cuda").clone()
    host.TimeStepper(V, 100.0, 2, FE, Metric, phys, Cache, JCache, Global)
    torch.cuda.synchronize()
    Vo = U0.copy()
    orc.rw_step(Vo, 100.0, 2)
    for v in range(5):
        assert rel_l2(V[v].cpu().numpy(), Vo[v]) <= 1e-12, f"V{v + 1}"


@pytest.mark.parametrize("shift", [0, 1])
def test_column_solve_streams_on_large_grids(pkg, torch_cuda, shift):
    """The column solve of 2^21 points and more streams past the cache; its
    columns are those of a small grid with the same inputs, to the bit, with
    J blocks that take 16-byte accesses and without."""
    torch, host = torch_cuda, pkg.host
    print(f"column streams shift={shift}", flush=True)
    phys = pkg.discretization.Phys()
    gen = torch.Generator("cuda").manual_seed(5)
    solves, inputs = [], None
    for ne in (25, 3):
        FE, Metric, Global, Cache, JCache, _ = host.device_build(ne, 3, 64, 30000.0)
        ctx = host.init_context(FE, Metric, phys, Global)
        g, nz = Global.NumG, Global.Nz
        assert (g * nz >= 1 << 21) == (ne == 25)
        if inputs is None:
            blocks = [1e-3 * torch.randn((g, nz - 1, 2), generator=gen, device="cuda", dtype=torch.float64)
                      for _ in range(4)]
            inputs = blocks, torch.randn((5, g, nz), generator=gen, device="cuda", dtype=torch.float64)
        for name, J in zip(("JRhoW", "JWRho", "JWRhoTh", "JRhoThW"), inputs[0]):
            buf = torch.zeros(J[:g].numel() + 1, device="cuda", dtype=torch.float64)[shift:]
            setattr(JCache, name, buf[:J[:g].numel()].view(g, nz - 1, 2).copy_(J[:g]))
        v = inputs[1][:, :g].clone()  # the solve overwrites its right-hand side
        k = torch.zeros_like(v)
        JCache.CompTri = True

        def solve():
            host.SchurSolveGPU(k, v, JCache, 1.0, Cache, Global)

        names = kernels_of(torch, solve)
        want = f"k_schur_col<{'false' if shift else 'true'}, {'true' if ne == 25 else 'false'}>"
        assert names == {want}
        solves.append((k, v, JCache.tri))
        ctx.close()
    small = solves[1][0].shape[1]
    assert torch.isfinite(solves[0][0]).all()
    assert torch.equal(solves[0][0][:, :small], solves[1][0]) and torch.equal(solves[0][1][:, :small], solves[1][1])
    assert torch.equal(solves[0][2][:small], solves[1][2])
