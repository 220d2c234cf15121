"""Serving loop through the C ABI: each result is the same alone and in a mix
(bit for bit), equals the plain per-call entry points, admission by HBM
budget queues requests instead of failing them, and a request that can
never fit is refused."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FIELDS = ("rho", "vfrac", "sie", "temp", "press")


@pytest.fixture(scope="module")
def setup(sgm, workloads, torch_gpu):
    ctx, table = workloads.pool_context()
    w = workloads.uneven(ctx, 1 << 15)
    yield ctx, w
    ctx.close()


def make_requests(w, seed, nreq=24):
    rng = np.random.default_rng(seed)
    off = w["offsets"]
    reqs = []
    for i in range(nreq):
        if i % 3 == 0:
            n = int(rng.integers(500, 6000))
            c0 = int(rng.integers(0, w["ncell"] - n))
            reqs.append(("pte", c0, n))
        else:
            m = int(rng.integers(0, 6))
            sel = np.flatnonzero(w["mat_ids"] == m)
            n = int(rng.integers(100, min(20000, len(sel))))
            s0 = int(rng.integers(0, len(sel) - n))
            reqs.append(("vec", m, sel[s0:s0 + n]))
    return reqs


def submit(srv, w, r):
    off = w["offsets"]
    if r[0] == "pte":
        _, c0, n = r
        e0, e1 = int(off[c0]), int(off[c0 + n])
        out = {k: np.full(e1 - e0, np.nan) for k in FIELDS}
        conv = np.full(n, -1, dtype=np.int32)
        t = srv.submit_pte(off[c0:c0 + n + 1].copy(), w["mat_ids"][e0:e1].copy(),
                           *[w[k][e0:e1].copy() for k in ("rho", "vfrac", "temp", "press")],
                           w["vfrac_tot"][c0:c0 + n].copy(), w["sie_tot"][c0:c0 + n].copy(),
                           out, conv)
        return t, (out, conv)
    _, m, idx = r
    P = np.full(len(idx), np.nan)
    T = np.full(len(idx), np.nan)
    t = srv.submit_vec(m, w["rho"][idx].copy(), w["sie"][idx].copy(), P_out=P, T_out=T)
    return t, (P, T)


def same(a, b):
    return np.array_equal(a, b, equal_nan=True)


def equal_results(x, y):
    if isinstance(x[0], dict):
        return all(same(x[0][k], y[0][k]) for k in FIELDS) and same(x[1], y[1])
    return same(x[0], y[0]) and same(x[1], y[1])


def test_alone_equals_mix_equals_plain(sgm, setup, torch_gpu):
    torch = torch_gpu
    ctx, w = setup
    params = sgm.mix_params(tight=True)
    reqs = make_requests(w, 7)
    # the mix: everything submitted at once, a budget small enough to queue
    srv = sgm.Server(ctx, budget_bytes=96 << 20, nlanes=4, max_group_requests=8,
                     max_group_cells=40000, params=params)
    sub = [submit(srv, w, r) for r in reqs]
    for t, _ in sub:
        assert srv.wait(t)[0] == 0
    st = srv.stats()
    srv.close()
    assert st["completed"] == len(reqs) and st["failed"] == 0
    assert st["groups"] < len(reqs)  # requests were merged into launch groups
    mix = [res for _, res in sub]
    # alone: one request in the server at a time
    srv = sgm.Server(ctx, budget_bytes=96 << 20, nlanes=4, params=params)
    alone = []
    for r in reqs:
        t, res = submit(srv, w, r)
        assert srv.wait(t)[0] == 0
        alone.append(res)
    srv.close()
    for i, (a, b) in enumerate(zip(mix, alone)):
        assert equal_results(a, b), (i, reqs[i][0])
    # the plain per-call entry points on device copies of the same inputs
    dev = torch.device("cuda")
    off = w["offsets"]
    for r, res in zip(reqs, mix):
        if r[0] == "pte":
            _, c0, n = r
            e0, e1 = int(off[c0]), int(off[c0 + n])
            d = {k: torch.tensor(w[k][e0:e1], device=dev) for k in FIELDS}
            o = torch.tensor(off[c0:c0 + n + 1] - e0, device=dev, dtype=torch.int32)
            m = torch.tensor(w["mat_ids"][e0:e1], device=dev)
            vt = torch.tensor(w["vfrac_tot"][c0:c0 + n], device=dev)
            s_ = torch.tensor(w["sie_tot"][c0:c0 + n], device=dev)
            conv = torch.zeros(n, dtype=torch.int32, device=dev)
            assert ctx.pte(0, n, e1 - e0, o, m, d["rho"], d["vfrac"], d["sie"], d["temp"],
                           d["press"], vt, s_, params=params, conv=conv) == 0
            torch.cuda.synchronize()
            for k in FIELDS:
                assert same(d[k].cpu().numpy(), res[0][k]), k
            assert same(conv.cpu().numpy(), res[1])
        else:
            _, mm, idx = r
            rho = torch.tensor(w["rho"][idx], device=dev)
            sie = torch.tensor(w["sie"][idx], device=dev)
            P = torch.empty_like(rho)
            T = torch.empty_like(rho)
            assert ctx.vec_eval(mm, sgm.F_P_RHO_SIE, rho, sie, P) == 0
            assert ctx.vec_eval(mm, sgm.F_T_RHO_SIE, rho, sie, T) == 0
            torch.cuda.synchronize()
            assert same(P.cpu().numpy(), res[0]) and same(T.cpu().numpy(), res[1])


def test_plain_server_matches_batched(sgm, setup, torch_gpu):
    ctx, w = setup
    reqs = make_requests(w, 11, nreq=9)
    out = []
    for plain in (False, True):
        srv = sgm.Server(ctx, budget_bytes=256 << 20, plain=plain)
        sub = [submit(srv, w, r) for r in reqs]
        for t, _ in sub:
            assert srv.wait(t)[0] == 0
        srv.close()
        out.append([res for _, res in sub])
    for a, b in zip(*out):
        assert equal_results(a, b)


def test_request_larger_than_budget_is_refused(sgm, setup, torch_gpu):
    ctx, w = setup
    srv = sgm.Server(ctx, budget_bytes=64 << 20)
    n = 3_000_000
    rho = np.ones(n)
    with pytest.raises(RuntimeError, match="-6"):
        srv.submit_vec(0, rho, rho, P_out=np.zeros(n), T_out=np.zeros(n))
    # the server keeps serving
    t, (P, T) = submit(srv, w, ("vec", 0, np.arange(100)))
    assert srv.wait(t)[0] == 0 and np.isfinite(P).all()
    srv.close()


@pytest.mark.parametrize("n", [1, 100, 3000, 20000])
def test_working_set_follows_the_request(sgm, setup, torch_gpu, n):
    """A closure request's share of the arena: about 0.9 KB a cell while every
    cell has a straggler record (a one-cell request once took 2.8 MB), records
    for a sixteenth of the cells per material count past that."""
    ctx, w = setup
    srv = sgm.Server(ctx, budget_bytes=64 << 20, params=sgm.mix_params(tight=True))
    t, _ = submit(srv, w, ("pte", 0, n))
    assert srv.wait(t)[0] == 0
    peak = srv.stats()["arena_peak_bytes"]
    srv.close()
    nnz = int(w["offsets"][n])
    # five doubles and an id per entry; 28 bytes of inputs and flags a cell, 24
    # of keys and lists and the sort's copy of a key and a value (12)
    state = 41 * nnz + 64 * n + (64 << 10)
    assert peak <= state + min(740 * n, 2780 * max(1024, n // 16))


def test_poisson_trace_completes(sgm, workloads, setup, torch_gpu):
    """A short open-loop trace through the load generator: every request
    completes and latencies are positive."""
    serving = __import__("importlib").import_module("singularity-eos_amd.serving")
    ctx, w = setup
    pools = serving.Pools(torch_gpu, w, npoint=1 << 16)
    tr = serving.make_trace(40, 400.0, 3, pool_cells=w["ncell"], nmax=2e4)
    res = serving.run(torch_gpu, ctx, pools, tr, budget=256 << 20, ring_bytes=256 << 20)
    assert (res["status"] == 0).all()
    assert (res["latency"] > 0).all()
