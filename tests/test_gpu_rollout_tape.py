"""A rollout's forward on a context that has run a reverse records its last
segment for the next reverse. Its states, lists and gradients equal, bit for bit,
those of a fresh context (which records nothing), whatever runs on the context
between the forward and the reverse."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import dev, say  # noqa: E402

N = 3000


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def block(scene, seed):
    return scene.jittered_lattice((20, 15, 10), (0.3, 0.5, 0.3), 0.0042, 0.1, seed=seed)


def forward(ctx, x0, double, nsteps, every):
    dt = torch.float64 if double else torch.float32
    x = dev(x0).to(dt)
    v = torch.zeros_like(x)
    return x, v, ctx.rollout_forward(x, v, None, nsteps, every)


def reverse(ctx, x, token):
    xb = torch.linspace(-1, 1, 3 * N, dtype=x.dtype, device="cuda:0").reshape(N, 3)
    vb = xb.flip(0) * 1e-3
    ctx.rollout_backward(xb, vb, token)
    return xb, vb


def lists(ctx):
    nl = ctx.step_neighbors(N)
    return nl.index, nl.elements


def other_step(ctx, scene):  # a larger search: the context's buffers grow
    x = dev(scene.jittered_lattice((24, 20, 20), (0.3, 0.5, 0.3), 0.0042, 0.1, seed=9))
    ctx.step(x, torch.zeros_like(x), None, 4)


def other_precision(ctx, scene, double):
    x, _, token = forward(ctx, block(scene, 8), not double, 3, 3)
    reverse(ctx, x, token)


BETWEEN = {
    "nothing": lambda ctx, scene, double: None,
    "lists": lambda ctx, scene, double: lists(ctx),
    "a step": lambda ctx, scene, double: other_step(ctx, scene),
    "the other precision": other_precision,
}


@pytest.mark.parametrize("between", list(BETWEEN))
@pytest.mark.parametrize("nsteps,every", [(1, 1), (5, 2), (4, 4), (3, 10)])
@pytest.mark.parametrize("double", [False, True])
def test_recorded_forward(fluid, scene, double, nsteps, every, between):
    say(f"recorded forward, {'f64' if double else 'f32'}, {nsteps} steps, checkpoint {every}, {between} between")
    ctx = fluid.Context("cuda:0")
    for seed in (1, 2, 3):
        x0 = block(scene, seed)
        fresh = fluid.Context("cuda:0")
        x, v, token = forward(fresh, x0, double, nsteps, every)
        want = [x, v, *lists(fresh), *reverse(fresh, x, token)]
        pairs = fresh.stats()["neighbor_pairs"]
        x, v, token = forward(ctx, x0, double, nsteps, every)
        got = [x, v, *lists(ctx)]
        BETWEEN[between](ctx, scene, double)
        got += reverse(ctx, x, token)
        if between in ("nothing", "lists"):
            assert ctx.stats()["neighbor_pairs"] == pairs > 0
        again = reverse(ctx, x, token)
        for a, b in zip(got + list(again), want + want[-2:]):
            np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())


def test_recorded_forward_and_a_replayed_step(fluid, scene):
    """A step captured into a caller's graph searches without the host: lists
    exported after its replay are its own, and the reverse is the rollout's."""
    say("recorded forward, a replayed step between")
    ctx = fluid.Context("cuda:0")
    x, _, token = forward(ctx, block(scene, 1), False, 4, 2)
    reverse(ctx, x, token)
    xs, vs = dev(block(scene, 7)), torch.zeros(N, 3, device="cuda:0")
    ctx.step(xs, vs)
    torch.cuda.synchronize()
    ctx.stats()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="relaxed"):
        ctx.step(xs, vs)
    x0 = block(scene, 2)
    fresh = fluid.Context("cuda:0")
    fx, _, ftoken = forward(fresh, x0, False, 4, 2)
    want = reverse(fresh, fx, ftoken)
    x, _, token = forward(ctx, x0, False, 4, 2)
    xs.copy_(dev(block(scene, 7)))
    vs.zero_()
    graph.replay()
    got_lists = lists(ctx)
    got = reverse(ctx, x, token)
    one = fluid.Context("cuda:0")
    xo, vo = dev(block(scene, 7)), torch.zeros(N, 3, device="cuda:0")
    one.step(xo, vo)
    for a, b in zip([*got, *got_lists], [*want, *lists(one)]):
        np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())
