"""The forward's two builds (two waves per SIMD up to 9 worlds a CU, three beyond): the same bits on both sides of the
line, in every output and in the tape, for standing and contact-heavy worlds (contacts between robot bodies included), at
the default options and away from them. The three-wave build, which keeps some registers in scratch memory, also against
the float64 oracle, in a captured graph, compiled, and on two streams at once."""
import numpy as np
import pytest

import oracle
from nablaengine_amd import synthetic

pytestmark = pytest.mark.gpu
KEYS = ("qpos", "qvel", "warm", "ctrl", "friction", "com")


def _line():
    import torch
    return 9 * torch.cuda.get_device_properties(0).multi_processor_count


def _inputs(n, config=1, seed=31):
    import torch
    st = synthetic.states(n, config=config, seed=seed)
    return st, [torch.from_numpy(st[k]).cuda() for k in KEYS]


def _equal(a, b):
    return all(np.array_equal(x.cpu().numpy().view(np.uint8), y.cpu().numpy().view(np.uint8)) for x, y in zip(a, b))


@pytest.mark.parametrize("config", [1, 4])
@pytest.mark.parametrize("substeps,iterations", [(4, 10), (1, 50), (7, 3), (2, 0)])
def test_both_builds_give_the_same_bits(config, substeps, iterations):
    from nablaengine_amd import torch_ffi
    n = _line()
    _, args = _inputs(n + 1, config)
    kw = dict(tape=True, substeps=substeps, iterations=iterations)
    three = torch_ffi.forward(*args, **kw)
    assert _equal([x[:n] for x in three], torch_ffi.forward(*(x[:n] for x in args), **kw))
    assert _equal([x[n:] for x in three], torch_ffi.forward(*(x[n:] for x in args), **kw))


def test_three_waves_vs_oracle():
    """Config-1 worlds, past the line, at the engine's settings: the gates of the two-wave build's comparison (qvel median
    <= 2e-6 and p99 <= 2e-5, qpos median <= 2e-7 and p99 <= 2e-6)."""
    from nablaengine_amd import torch_ffi
    st, args = _inputs(_line() + 256)
    q1, v1 = (x.cpu().numpy().astype(np.float64) for x in torch_ffi.forward(*args)[:2])
    oq, ov, _, _ = oracle.step_mt(16, **{k: st[k].astype(np.float64) for k in st}, **oracle.ENGINE)
    ev, eq = (np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1) for a, b in ((v1, ov), (q1, oq)))
    print(f"qvel median {np.median(ev):.3g} p99 {np.percentile(ev, 99):.3g}; qpos median {np.median(eq):.3g} p99 "
          f"{np.percentile(eq, 99):.3g}")
    assert np.median(ev) <= 2e-6 and np.percentile(ev, 99) <= 2e-5
    assert np.median(eq) <= 2e-7 and np.percentile(eq, 99) <= 2e-6


def test_three_waves_in_a_graph():
    """forward(tape=True) and backward captured past the line; three replays on new inputs with eager work of both builds
    between them, each bitwise the eager result."""
    import torch
    from nablaengine_amd import torch_ffi
    n = _line() + 1
    _, static = _inputs(n)
    cots = [torch.from_numpy(x).cuda() for x in synthetic.cotangents(n)]
    torch_ffi.forward(*static, tape=True)  # warm the caching allocator outside the capture
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = torch_ffi.forward(*static, tape=True)
        grads = torch_ffi.backward(out[4], static[4], static[5], *cots)
    for rep in range(3):
        _, new = _inputs(n, config=(4, 1, 4)[rep], seed=100 + rep)
        for a, b in zip(static, new):
            a.copy_(b)
        torch_ffi.step(*_inputs(n + rep, seed=200 + rep)[1])
        torch_ffi.step(*_inputs(300, seed=300 + rep)[1])
        g.replay()
        torch.cuda.synchronize()
        e = torch_ffi.forward(*new, tape=True)
        assert _equal(out, e) and _equal(grads, torch_ffi.backward(e[4], new[4], new[5], *cots)), f"replay {rep}"


def test_three_waves_compiled():
    """torch.compile(fullgraph=True, aot_eager) of a loss through step past the line: loss and gradients bitwise eager's."""
    import torch
    from nablaengine_amd import torch_ffi
    n = _line() + 1
    _, args = _inputs(n)
    cq, cv = (torch.from_numpy(x).cuda() for x in synthetic.cotangents(n))

    def loss(*x):
        q1, v1, _ = torch_ffi.step(*x)
        return (q1 * cq).sum() + (v1 * cv).sum()

    torch._dynamo.reset()
    got = []
    for f in (loss, torch.compile(loss, fullgraph=True, backend="aot_eager")):
        x = [t.clone().requires_grad_(i in (0, 1, 3)) for i, t in enumerate(args)]
        value = f(*x)
        value.backward()
        got.append([value.detach().reshape(1), x[0].grad, x[1].grad, x[3].grad])
    assert _equal(*got)


def test_three_waves_on_two_streams():
    """Launches past the line in flight on two streams at once, each bitwise its own on an idle GPU."""
    import torch
    from nablaengine_amd import torch_ffi
    args = [_inputs(_line() + 1 + i, config=c, seed=40 + i)[1] for i, c in enumerate((1, 4))]
    alone = [torch_ffi.forward(*a, tape=True) for a in args]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in args]
    out = [[], []]
    for _ in range(3):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                out[i].append(torch_ffi.forward(*args[i], tape=True))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(_equal(alone[i], r) for r in out[i]), i
