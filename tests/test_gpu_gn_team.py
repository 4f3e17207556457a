"""GroupNorm(+SiLU) with the unit kept on chip between the passes, against
float64 and against the two-launch path over the forms that both accept, and
with every wait ending at once: each block then leaves its share to the launch
after unless the sums are there by then, or leaves it in any case."""
import time

import pytest
import torch

from test_gpu_parity import EPS

pytestmark = pytest.mark.gpu

CASES = [
    # (N, C, HW, G, silu, residual, affine)
    (1, 768, 8192, 8, True, False, True),        # one chunk per plane, 768 in all: the least
    (2, 768, 8192, 8, True, False, True),        # 1536: the least forward
    (4, 192, 8196, 4, True, True, True),         # a last chunk of one vector
    (4, 96, 25600, 8, False, False, True),       # plain GroupNorm, a ragged last chunk
    (2, 32, 262144, 32, True, False, False),     # one plane per unit, no affine
    (3, 64, 65536, 8, False, True, True),
    (2, 128, 73728, 16, True, True, True),       # forward only: backward above 2048 chunks
    (2, 512, 8196, 4, True, False, True),        # 128 planes per unit, the most
    (2, 96, 102400, 16, True, False, True),
    (1, 6, 2097152, 2, True, False, True),       # forward: three chunks per half-block (LDS)
    (4, 99, 28672, 3, True, False, True),        # odd channels per unit
]


def chunks(N, C, HW):
    return N * C * -(-HW // 8192)


def tensors(N, C, HW, affine, seed=3):
    g = torch.Generator(device="cuda").manual_seed(seed)
    new = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x, dy = new(N, C, HW) + 3.0, new(N, C, HW)
    x[0, 0, 5] += 40.0
    gamma = new(C) if affine else None
    beta = new(C) if affine else None
    return x, dy, gamma, beta


def both(gpu, x, dy, gamma, beta, G, silu, residual):
    y, st = gpu.gn_silu_forward(x, gamma, beta, G, eps=EPS, silu=silu, residual=residual)
    d = gpu.gn_silu_backward(dy, x, gamma, beta, st, G, silu=silu, residual=residual)
    return [y, st.mean, st.rstd, *d]


def float64(x, dy, gamma, beta, G, silu, residual):
    N, C, HW = x.shape
    t = [x.double().requires_grad_()]
    t += [(torch.ones(C) if v is None else v.cpu()).cuda().double().requires_grad_()
          for v in (gamma,)]
    t += [(torch.zeros(C) if v is None else v.cpu()).cuda().double().requires_grad_()
          for v in (beta,)]
    u = t[0].reshape(N, G, -1)
    mean = u.mean(2, keepdim=True)
    rstd = ((u - mean).square().mean(2, keepdim=True) + EPS).rsqrt()
    y = ((u - mean) * rstd).reshape(N, C, HW) * t[1][:, None] + t[2][:, None]
    if silu:
        y = y * torch.sigmoid(y)
    if residual:
        y = y + t[0]
    d = torch.autograd.grad(y, t, dy.double())
    return [y.detach(), mean.detach().reshape(-1), rstd.detach().reshape(-1), *d]


@pytest.fixture
def wait_us(gpu):
    old = gpu.tune_get(gpu.TUNE_TEAM_WAIT_US)
    yield lambda v: gpu.tune(gpu.TUNE_TEAM_WAIT_US, v)
    gpu.tune(gpu.TUNE_TEAM_WAIT_US, old)


@pytest.mark.parametrize("case", CASES)
def test_team_matches_float64_and_two_launches(gpu, wait_us, case):
    N, C, HW, G, silu, residual, affine = case
    x, dy, gamma, beta = tensors(N, C, HW, affine)
    args = (gpu, x, dy, gamma, beta, G, silu, residual)
    gpu.prof_summary()  # drop earlier records
    gpu.prof_enable(True)
    got = both(*args)
    torch.cuda.synchronize()
    names = {p["kernel"] for p in gpu.prof_summary()}
    gpu.prof_enable(False)
    assert any("team_fwd" in n for n in names) == (chunks(N, C, HW) >= 1536), names
    held = chunks(1, C // G, HW) <= 256 and not (silu and residual and chunks(N, C, HW) > 2048)
    assert any("team_bwd" in n for n in names) == held, names
    wait_us(-1)
    two = both(*args)
    wait_us(0)
    alone = both(*args)
    truth = float64(x, dy, gamma, beta, G, silu, residual)
    for a, b, c, t, what in zip(got, two, alone, truth, ("y", "mean", "rstd", "dx", "dgamma", "dbeta")):
        assert torch.equal(a, c), f"{what}: depends on who computed the sums"
        scale = t.abs().max()
        # both paths round float64 sums of the same terms: at most an ulp or
        # two of fp32 apart
        assert (a - b).abs().max() <= 4 * 2.0 ** -23 * scale, what
        assert (a.double() - t).abs().max() <= 1e-5 * scale, what


@pytest.mark.parametrize("case", CASES)
def test_every_block_may_leave(gpu, wait_us, case):
    """No block gets its unit's sums in time, so all of the output comes from
    the launch after: bit for bit a team's, every gradient added once."""
    N, C, HW, G, silu, residual, affine = case
    x, dy, gamma, beta = tensors(N, C, HW, affine)
    args = (gpu, x, dy, gamma, beta, G, silu, residual)
    want = both(*args)
    wait_us(-2)
    for a, b, what in zip(both(*args), want, ("y", "mean", "rstd", "dx", "dgamma", "dbeta")):
        assert torch.equal(a, b), what


def test_team_leaves_overlapping_outputs_alone(gpu):
    """In place, the two launches run, as they always did."""
    x, dy, gamma, beta = tensors(2, 128, 65536, True)
    y, st = gpu.gn_silu_forward(x, gamma, beta, 8, eps=EPS)
    inplace = x.clone()
    gpu.gn_silu_forward(inplace, gamma, beta, 8, eps=EPS, y=inplace)
    assert (inplace - y).abs().max() <= 4 * 2.0 ** -23 * y.abs().max()
    dx, _, _ = gpu.gn_silu_backward(dy, x, gamma, beta, st, 8)
    d = dy.clone()
    gpu.gn_silu_backward(d, x, gamma, beta, st, 8, dx=d)
    assert (d - dx).abs().max() <= 4 * 2.0 ** -23 * dx.abs().max()


@pytest.mark.parametrize("wait", [None, 0, -2])
def test_team_graph_replays(gpu, wait_us, wait):
    """Replays with other work between them, also where blocks leave their
    shares to the launch after."""
    if wait is not None:
        wait_us(wait)
    x, dy, gamma, beta = tensors(3, 64, 65536, True)
    ws = gpu.workspace(3, 64, 65536, 8)
    want = both(gpu, x, dy, gamma, beta, 8, True, False)
    y, dx = torch.empty_like(x), torch.empty_like(x)
    st = [torch.empty(24, device="cuda") for _ in range(3)]
    dg, db = torch.zeros(64, device="cuda"), torch.zeros(64, device="cuda")

    def step():
        dg.zero_()
        db.zero_()
        _, s = gpu.gn_silu_forward(x, gamma, beta, 8, eps=EPS, y=y, mean=st[0], rstd=st[1],
                                   mean_lo=st[2], ws=ws)
        gpu.gn_silu_backward(dy, x, gamma, beta, s, 8, dx=dx, dgamma=dg, dbeta=db, ws=ws)

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for _ in range(3):
        y.fill_(7.0)
        dx.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip((y, st[0], st[1], dx, dg, db), want):
            assert torch.equal(a, b)
        both(gpu, dy, x, gamma, beta, 8, True, False)  # other work between replays


def test_team_on_two_streams(gpu):
    """Teams of two launches share the chip; whichever blocks run first,
    every call ends with the results it has alone."""
    x, dy, gamma, beta = tensors(2, 64, 262144, True)
    want = both(gpu, x, dy, gamma, beta, 8, True, False)
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = [None, None]
    for _ in range(3):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i] = both(gpu, x, dy, gamma, beta, 8, True, False)
    torch.cuda.synchronize()
    for g in got:
        for a, b in zip(g, want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("shape", [(1, 16, 1048576, 8), (1, 32, 1048576, 8), (1, 24, 1048576, 4),
                                   (1, 64, 4194304, 16)])
@pytest.mark.parametrize("backward", [False, True])
def test_streams_cost_no_more_than_two_launches(gpu, wait_us, shape, backward):
    """Two streams' calls at once take no longer than where every call reads
    its tensor twice (bar: half more, for timing).  Where a team needed more
    than half of the chip, both streams' teams stood in each other's way: 3.7 to
    20 times as long."""
    N, C, HW, G = shape
    calls = []
    for i in range(2):
        x, dy, gamma, beta = tensors(N, C, HW, True, seed=i)
        y, dx, ws = torch.empty_like(x), torch.empty_like(x), gpu.workspace(N, C, HW, G)
        st = [torch.empty(N * G, device="cuda") for _ in range(3)]
        dg, db = torch.zeros(C, device="cuda"), torch.zeros(C, device="cuda")
        _, s = gpu.gn_silu_forward(x, gamma, beta, G, y=y, mean=st[0], rstd=st[1], mean_lo=st[2],
                                   ws=ws)
        # (default arguments: each call keeps its own tensors)
        if backward:
            calls.append(lambda dy=dy, x=x, ga=gamma, be=beta, s=s, dx=dx, dg=dg, db=db, ws=ws:
                         gpu.gn_silu_backward(dy, x, ga, be, s, G, dx=dx, dgamma=dg, dbeta=db,
                                              ws=ws))
        else:
            calls.append(lambda x=x, ga=gamma, be=beta, y=y, st=st, ws=ws: gpu.gn_silu_forward(
                x, ga, be, G, y=y, mean=st[0], rstd=st[1], mean_lo=st[2], ws=ws))
    streams = [torch.cuda.Stream() for _ in calls]

    def run():
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(10):
            for s, call in zip(streams, calls):
                with torch.cuda.stream(s):
                    call()
        torch.cuda.synchronize()
        return time.perf_counter() - t0

    default = gpu.tune_get(gpu.TUNE_TEAM_WAIT_US)
    best = {}
    for wait in (default, -1) * 4:
        wait_us(wait)
        t = run()
        best[wait] = min(t, best.get(wait, t))
    assert best[default] <= 1.5 * best[-1], best
