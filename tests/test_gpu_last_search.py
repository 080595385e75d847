"""Lists of a recorded forward when a call is captured before they are exported:
until the first replay step_neighbors gives the forward's, after it the step's,
and the gradients stay those of a fresh context, bit for bit."""
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


def forward(ctx, x0, dtype, every):
    x = dev(x0).to(dtype)
    v = torch.zeros_like(x)
    return x, ctx.rollout_forward(x, v, None, 4, every)


def reverse(ctx, x, token):
    xb = torch.linspace(-1, 1, 3 * N, dtype=x.dtype, device="cuda:0").reshape(N, 3)
    vb = xb.flip(0) * 1e-3
    ctx.rollout_backward(xb, vb, token)
    return xb, vb


def lists(ctx):
    nl = ctx.step_neighbors(N)
    return nl.index, nl.elements


def equal(got, want):
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())


@pytest.mark.parametrize("storage", [{}, {"list_slots": 4}])
@pytest.mark.parametrize("every", [2, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_lists_around_a_capture(fluid, scene, dtype, every, storage):
    say(f"lists of a recorded forward around a capture, {dtype}, checkpoint {every}, {storage}")
    ctx = fluid.Context("cuda:0", **storage)
    xs, vs = dev(block(scene, 7)), torch.zeros(N, 3, device="cuda:0")
    ctx.step(xs, vs)
    for seed in (1, 2):
        x, token = forward(ctx, block(scene, seed), dtype, every)
        if seed == 1:
            reverse(ctx, x, token)
    fresh = fluid.Context("cuda:0", **storage)
    fx, ftoken = forward(fresh, block(scene, 2), dtype, every)
    want_lists = lists(fresh)
    want = reverse(fresh, fx, ftoken)
    torch.cuda.synchronize()
    ctx.stats()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="relaxed"):
        ctx.step(xs, vs)
    equal(lists(ctx), want_lists)
    equal(reverse(ctx, x, token), want)
    one = fluid.Context("cuda:0", **storage)
    for _ in range(2):
        xs.copy_(dev(block(scene, 7)))
        vs.zero_()
        graph.replay()
        x, token = forward(ctx, block(scene, 2), dtype, every)
        equal(lists(ctx), want_lists)
        equal(reverse(ctx, x, token), want)
        xs.copy_(dev(block(scene, 7)))
        vs.zero_()
        graph.replay()
        ctx.step(xs, vs)
        xo, vo = dev(block(scene, 7)), torch.zeros(N, 3, device="cuda:0")
        one.step(xo, vo, None, 1)
        one.step(xo, vo, None, 1)
        equal((xs, vs, *lists(ctx)), (xo, vo, *lists(one)))
