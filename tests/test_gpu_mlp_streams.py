"""The network's calls on streams of the caller's: what has ended when a call
returns, and what a later call may overwrite."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rc():
    import radiancecascade_amd as rc
    if rc.device_count() < 1:
        pytest.skip("no HIP device")
    return rc


def _net(rc, seed):
    rng = np.random.default_rng(seed)
    return ((rng.standard_normal(rc._abi.MLP_PARAMS) * 0.1).astype(np.float32),
            rng.standard_normal(64).astype(np.float32), rng.uniform(0.5, 2.0, 64).astype(np.float32), 1.5)


def _busy(stream):
    """Some 20 ms of work on the stream."""
    with torch.cuda.stream(stream):
        a = torch.ones((8192, 8192), device="cuda:0")
        for _ in range(10):
            a = torch.mm(a, a).clamp_(max=1.0)
    return a


def test_gradient_has_ended_when_the_call_returns(rc):
    """On a stream of the caller's, behind other work on it: the stream is idle
    when the call returns, so another stream reads the gradient and the loss,
    and the next gradient of the context may go to another stream."""
    n = 5000
    rng = np.random.default_rng(0)
    x = torch.from_numpy(rng.standard_normal((n, 64)).astype(np.float32)).cuda()
    t = torch.from_numpy(rng.standard_normal((n, 48)).astype(np.float32)).cuda()
    out = [(torch.zeros(rc._abi.MLP_PARAMS, device="cuda:0"), torch.zeros(1, device="cuda:0")) for _ in range(3)]
    with rc.RadianceCascadeStage(64, 64, levels=3) as st:
        st.mlp_set(*_net(rc, 1))
        st.mlp_gradient(x, t, *out[0])
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        for s, (g, lo) in zip(streams, out[1:]):
            keep = _busy(s)
            st.mlp_gradient(x, t, g, lo, stream=s)
            assert s.query()
            assert torch.equal(g, out[0][0]) and torch.equal(lo, out[0][1])
            del keep


def test_gradient_after_one_on_the_null_stream(rc):
    """A gradient that still runs on the null stream keeps its partial sums
    when the next one goes to another stream."""
    n = 40000
    rng = np.random.default_rng(5)
    x = [torch.from_numpy(rng.standard_normal((n, 64)).astype(np.float32)).cuda() for _ in range(2)]
    t = torch.from_numpy(rng.standard_normal((n, 48)).astype(np.float32)).cuda()
    g = [torch.zeros(rc._abi.MLP_PARAMS, device="cuda:0") for _ in range(4)]
    lo = torch.zeros(1, device="cuda:0")
    side = torch.cuda.Stream()
    with rc.RadianceCascadeStage(64, 64, levels=3) as st:
        st.mlp_set(*_net(rc, 4))
        for k in range(2):
            st.mlp_gradient(x[k], t, g[k], lo)
            torch.cuda.synchronize()
        keep = _busy(torch.cuda.default_stream())
        st.mlp_gradient(x[0], t, g[2], lo)
        st.mlp_gradient(x[1], t, g[3], lo, stream=side)
        torch.cuda.synchronize()
        del keep
    assert torch.equal(g[2], g[0]) and torch.equal(g[3], g[1])


def test_gradient_in_a_captured_graph(rc):
    """A captured gradient is computed by each replay."""
    n = 300
    rng = np.random.default_rng(2)
    x = torch.from_numpy(rng.standard_normal((n, 64)).astype(np.float32)).cuda()
    t = torch.from_numpy(rng.standard_normal((n, 48)).astype(np.float32)).cuda()
    g, lo = torch.empty(rc._abi.MLP_PARAMS, device="cuda:0"), torch.empty(1, device="cuda:0")
    ge, le = torch.empty_like(g), torch.empty_like(lo)
    with rc.RadianceCascadeStage(64, 64, levels=3) as st:
        st.mlp_set(*_net(rc, 3))
        st.mlp_gradient(x, t, g, lo)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            st.mlp_gradient(x, t, g, lo)
        for k in range(3):
            x.mul_(-0.75)
            g.fill_(7.0)
            graph.replay()
            torch.cuda.synchronize()
            st.mlp_gradient(x, t, ge, le)
            assert torch.equal(g, ge) and torch.equal(lo, le), k


@pytest.mark.parametrize("call", ["forward", "gradient", "frame"])
def test_a_new_network_waits_for_the_old_ones_work(rc, call):
    """Work queued on another stream before mlp_set uses the network it was
    given."""
    n = 20000
    rng = np.random.default_rng(6)
    x = torch.from_numpy(rng.standard_normal((n, 64)).astype(np.float32)).cuda()
    t = torch.from_numpy(rng.standard_normal((n, 48)).astype(np.float32)).cuda()
    W, H = 320, 200
    e = torch.from_numpy((rng.uniform(size=(3, H, W)) < 0.01).astype(np.float32)).cuda()
    d = torch.full((H, W), 0.5, device="cuda:0")
    with rc.RadianceCascadeStage(W, H, levels=4) as st:
        st.set_surrogate(True)

        def go(stream):
            if call == "forward":
                out = torch.zeros((n, 64), device="cuda:0")
                torch.cuda.synchronize()
                return lambda: st.mlp_forward(x, out, stream=stream), [out]
            if call == "gradient":
                out = [torch.zeros(rc._abi.MLP_PARAMS, device="cuda:0"), torch.zeros(1, device="cuda:0")]
                torch.cuda.synchronize()
                return lambda: st.mlp_gradient(x, t, *out, stream=stream), out
            out = torch.zeros_like(e)
            torch.cuda.synchronize()
            return lambda: st.run_device(d, e, out, stream=stream), [out]

        side = torch.cuda.Stream()
        st.mlp_set(*_net(rc, 7))
        run, want = go(side)
        run()
        torch.cuda.synchronize()
        run, got = go(side)
        keep = _busy(side)
        run()
        st.mlp_set(*_net(rc, 8))
        torch.cuda.synchronize()
        del keep
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        run, other = go(side)
        run()
        torch.cuda.synchronize()
        assert not torch.equal(other[0], want[0])
