"""One context on several streams (GPU, through the C ABI): tendencies and steps
use arrays of the context, so calls on different streams run one after the other
and give the bits of the same calls on one stream."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("nz,precision", [(8, "fp64"), (8, "mixed"), (20, "fp64")])
def test_calls_on_two_streams(pkg, torch_cuda, nz, precision):
    """Two states, each with work arrays of its own, in turn on two streams
    without a wait between; small grids, so that nothing but the order of the
    calls keeps the kernels of both apart."""
    torch, host = torch_cuda, pkg.host
    print(f"two streams nz={nz} {precision}", flush=True)
    disc = pkg.discretization.build(4, 4, nz, 512.0 * nz)
    phys = pkg.discretization.Phys()
    eq = host.CompressibleShallow()
    FE, Metric, Global, _, _ = host.device_setup(disc, phys, device="cuda", precision=precision)
    ctx = host.init_context(FE, Metric, phys, Global)
    works = [host.device_setup(disc, phys, device="cuda", precision=precision)[3:] for _ in range(2)]
    U = [torch.as_tensor(pkg.state.jet_state(disc, seed=s), device="cuda") for s in range(2)]

    def run(streams):
        F = [torch.zeros_like(u) for u in U]
        V = [u.clone() for u in U]
        for i, (Cache, _) in enumerate(works):
            host.FcnPrepareGPU(U[i], FE, Metric, phys, Cache, None, Global, None, eq)
        torch.cuda.synchronize()
        for _ in range(20):
            for i, (Cache, JCache) in enumerate(works):
                with torch.cuda.stream(streams[i]):
                    host.FcnGPU(F[i], U[i], FE, Metric, phys, Cache, None, Global, None, eq)
        torch.cuda.synchronize()
        for _ in range(10):
            for i, (Cache, JCache) in enumerate(works):
                with torch.cuda.stream(streams[i]):
                    host.TimeStepper(V[i], 100.0, 1, FE, Metric, phys, Cache, JCache, Global)
        torch.cuda.synchronize()
        return F + V

    one = torch.cuda.Stream()
    want = run([one, one])
    got = run([torch.cuda.Stream(), torch.cuda.Stream()])
    assert all(bool(torch.isfinite(x).all()) for x in want)
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    got = run([torch.cuda.current_stream(), one])
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    ctx.close()


def test_graph_and_eager_streams(pkg, torch_cuda):
    """A captured step replayed on one stream, eager steps of another state on
    a second one in between."""
    torch, host = torch_cuda, pkg.host
    print("graph and eager streams", flush=True)
    disc = pkg.discretization.build(4, 4, 8, 512.0 * 8)
    phys = pkg.discretization.Phys()
    FE, Metric, Global, Cache, JCache = host.device_setup(disc, phys, device="cuda")
    ctx = host.init_context(FE, Metric, phys, Global)
    Cache2, JCache2 = host.device_setup(disc, phys, device="cuda")[3:]
    U = [torch.as_tensor(pkg.state.jet_state(disc, seed=s), device="cuda") for s in range(2)]
    out = []
    for streams in ([torch.cuda.Stream()] * 2, [torch.cuda.Stream(), torch.cuda.Stream()]):
        G, E = U[0].clone(), U[1].clone()
        ctx.graph_create(G, 100.0, Cache, JCache, nsteps=1)
        torch.cuda.synchronize()
        for _ in range(10):
            with torch.cuda.stream(streams[0]):
                ctx.graph_launch()
            with torch.cuda.stream(streams[1]):
                host.TimeStepper(E, 100.0, 1, FE, Metric, phys, Cache2, JCache2, Global)
        torch.cuda.synchronize()
        out.append((G.clone(), E.clone()))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


def test_calls_in_a_capture(pkg, torch_cuda):
    """A tendency captured by the caller replays with the eager bits, with eager
    calls on other streams between the replays."""
    torch, host = torch_cuda, pkg.host
    print("calls in a capture", flush=True)
    disc = pkg.discretization.build(3, 4, 8, 512.0 * 8)
    phys = pkg.discretization.Phys()
    eq = host.CompressibleShallow()
    FE, Metric, Global, Cache, _ = host.device_setup(disc, phys, device="cuda")
    host.init_context(FE, Metric, phys, Global)
    U = torch.as_tensor(pkg.state.jet_state(disc, seed=0), device="cuda")
    F, W = torch.zeros_like(U), torch.zeros_like(U)
    host.FcnPrepareGPU(U, FE, Metric, phys, Cache, None, Global, None, eq)
    host.FcnGPU(W, U, FE, Metric, phys, Cache, None, Global, None, eq)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        host.FcnGPU(F, U, FE, Metric, phys, Cache, None, Global, None, eq)
    for _ in range(3):
        F.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(F, W)
        W.zero_()
        with torch.cuda.stream(torch.cuda.Stream()):
            host.FcnGPU(W, U, FE, Metric, phys, Cache, None, Global, None, eq)
        torch.cuda.synchronize()
        assert torch.equal(F, W)
