"""Triangular factors of A left in two halves (kfac_pi_damped_inverse_halves_batched,
kfac_precondition_halves_batched, kfac_factor_complete_batched) against float64.

With X = U^T U (U upper) and Y = U^-1, such a factor holds Y but for the block right of the cut, where
it has U's.  Bound of every comparison: the condition numbers here are below 200, and a float32 inverse or
product of triangular factors is off by at most about cond * sqrt(n) * 2^-24, below 1e-4 for n <= 1100."""
import pytest
import torch

from torchsso import _ops as ops

pytestmark = pytest.mark.gpu
TOL = 1e-4


def spd(n, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(2 * n + 8, n, generator=g, dtype=torch.float64)
    return a.t() @ a / a.shape[0] + 0.1 * torch.eye(n, dtype=torch.float64)


def cut_of(n):
    return 128 * (-(-n // 128) // 2)


def operand(x, form):
    """(the operand as the engine takes it, the inverse), float64; form: I inverse, F factor, H in halves"""
    u = torch.linalg.cholesky(x).t().contiguous()
    y = torch.linalg.solve_triangular(u, torch.eye(x.shape[0], dtype=x.dtype), upper=True).contiguous()
    inv = y @ y.t()
    if form == 'I':
        return inv, inv
    h = cut_of(x.shape[0])
    if form == 'H' and h > 0:
        y = y.clone()
        y[:h, h:] = u[:h, h:]
    return y, inv


def rel(a, b):
    return ((a.double().cpu() - b).norm() / b.norm()).item()


# (dG, dA, bias, forms of G and A) of the layers of one call
CASES = [
    [(300, 257, True, 'FH')],                                   # one layer: its reductions are cut into pieces
    [(64, 1025, True, 'IH')], [(1000, 384, False, 'IH')],       # beside an explicit inverse
    [(128, 128, True, 'FH'), (1, 2, True, 'FH')],               # one block: no halves
    [(256, 384, False, 'IF'), (129, 640, True, 'FH'), (385, 100, True, 'FI'), (10, 513, True, 'IH')],
    [(257 + 37 * i, 300 + 61 * i, i % 2 == 0, 'FI'[i % 2] + 'HHFI'[i % 4]) for i in range(12)],
    [(900, 1100, True, 'FH')] * 12,                             # enough tiles for no pieces
]


@pytest.mark.parametrize('case', range(len(CASES)))
def test_precondition(case):
    dev = torch.device('cuda', 0)
    gen = torch.Generator().manual_seed(case)
    Go, Ao, gw, gb, want = [], [], [], [], []
    seen = {}
    for dG, dA, bias, (gf, af) in CASES[case]:
        for d, f in ((dG, gf), (dA, af)):
            if (d, f) not in seen:
                seen[d, f] = operand(spd(d, d), f)
        v = torch.randn(dG, dA, generator=gen, dtype=torch.float64)
        (go, gi), (ao, ai) = seen[dG, gf], seen[dA, af]
        want.append(gi @ v @ ai)
        Go.append(go.float().contiguous().to(dev))
        Ao.append(ao.float().contiguous().to(dev))
        gw.append((v[:, :-1] if bias else v).float().contiguous().to(dev))
        gb.append(v[:, -1].float().contiguous().to(dev) if bias else None)
    before = [t.clone() for t in Go + Ao]
    forms = [c[3] for c in CASES[case]]
    ops.precondition_factored_batched(Go, Ao, gw, gb, [f[0] != 'I' for f in forms], [f[1] != 'I' for f in forms],
                                      a_halves=[f[1] == 'H' for f in forms])
    for w, b, ref in zip(gw, gb, want):
        got = w if b is None else torch.cat([w, b[:, None]], 1)
        assert rel(got, ref) < TOL
    assert all(torch.equal(a, b) for a, b in zip(before, Go + Ao))


def test_an_explicit_inverse_is_not_in_halves_whatever_the_list_says():
    """(reductions of this call are cut into pieces, and those over an explicit inverse are twice as long)"""
    dev = torch.device('cuda', 0)
    gen = torch.Generator().manual_seed(9)
    layers = [(300, 1025, 'I'), (129, 640, 'H'), (64, 385, 'I')]
    Go, Ao, gw, gb, want = [], [], [], [], []
    for dG, dA, form in layers:
        v = torch.randn(dG, dA, generator=gen, dtype=torch.float64)
        (go, gi), (ao, ai) = operand(spd(dG, dG), 'F'), operand(spd(dA, dA), form)
        want.append(gi @ v @ ai)
        Go.append(go.float().contiguous().to(dev))
        Ao.append(ao.float().contiguous().to(dev))
        gw.append(v[:, :-1].float().contiguous().to(dev))
        gb.append(v[:, -1].float().contiguous().to(dev))
    ops.precondition_factored_batched(Go, Ao, gw, gb, None, [f != 'I' for _, _, f in layers], a_halves=[True] * 3)
    for w, b, ref in zip(gw, gb, want):
        assert rel(torch.cat([w, b[:, None]], 1), ref) < TOL


# (22 matrices of 8 blocks are more than the sweep takes)
DIMS = [(1000, 1024), (1025, 897)] * 6


def test_inversion_leaves_halves_and_completes_them():
    dev = torch.device('cuda', 0)
    As64 = [spd(a, i) for i, (a, _) in enumerate(DIMS)]
    Gs64 = [spd(g, 50 + i) for i, (_, g) in enumerate(DIMS)]
    As, Gs = [a.float().to(dev) for a in As64], [g.float().to(dev) for g in Gs64]
    damp = [1e-2] * len(DIMS)
    none = [None] * len(DIMS)
    Af, Gf = [torch.full_like(a, float('nan')) for a in As], [torch.full_like(g, float('nan')) for g in Gs]
    halves = [i % 3 != 2 for i in range(len(DIMS))]
    asked = list(halves)
    info = ops.pi_damped_inverse_factored_batched(As, Gs, damp, none, none, Af, Gf, a_halves=halves)
    assert halves == asked and int(info.abs().sum()) == 0

    def damped(a, g):
        pi = ((a.trace() / a.shape[0]) / (g.trace() / g.shape[0])).sqrt()
        return (a + 0.1 * pi * torch.eye(a.shape[0], dtype=a.dtype),
                g + 0.1 / pi * torch.eye(g.shape[0], dtype=g.dtype))
    todo = []
    for i, (a, g) in enumerate(zip(As64, Gs64)):
        for x, f, half in zip(damped(a, g), (Af[i], Gf[i]), (halves[i], False)):
            assert rel(f, operand(x, 'H' if half else 'F')[0]) < TOL
            assert torch.equal(f, f.triu())
            if half:
                todo.append((x, f))
    ops.factor_complete_batched([f for _, f in todo])
    for x, f in todo:
        assert rel(f, operand(x, 'F')[0]) < TOL
        assert torch.equal(f, f.triu())


def test_small_batches_have_whole_factors():
    dev = torch.device('cuda', 0)
    a, g = spd(300, 1).float().to(dev), spd(100, 2).float().to(dev)
    af, gf = torch.empty_like(a), torch.empty_like(g)
    halves = [True]
    ops.pi_damped_inverse_factored_batched([a], [g], [1e-2], [None], [None], [af], [gf], a_halves=halves)
    assert halves == [False]
    want_a, want_g = torch.empty_like(a), torch.empty_like(g)
    ops.pi_damped_inverse_factored_batched([a], [g], [1e-2], [None], [None], [want_a], [want_g])
    assert torch.equal(af, want_a) and torch.equal(gf, want_g)


def test_optimizer_keeps_halves_where_inverses_are_used_once(monkeypatch):
    """Which form a layer's inverse has from step to step, what preconditioning makes of the halves, and
    `inv` of them."""
    import torch.nn as nn
    import torchsso
    from torchsso.curv.curvature import KronCurvature
    monkeypatch.setattr(KronCurvature, 'halved_inverse_min_dim', 256)
    monkeypatch.setattr(KronCurvature, 'halved_inverse_min_work', 1.)
    dev = torch.device('cuda', 0)
    torch.manual_seed(0)
    model = nn.Sequential(*[nn.Linear(1000, 1000, device=dev) for _ in range(13)])
    opt = torchsso.optim.SecondOrderOptimizer(model, 'Cov', {'Linear': 'Kron'}, {'damping': 1e-1}, lr=0.)
    x = torch.randn(256, 1000, device=dev)
    curv = opt.param_groups[3]['curv']

    def closure():
        opt.zero_grad()
        out = model(x)
        loss = out.pow(2).mean()
        loss.backward()
        closure.raw = [p.grad.clone() for p in model[3].parameters()]
        return loss, out

    def preconditioned():
        A, G = (e.double().cpu() for e in curv.ema)
        pi = ((A.trace() / A.shape[0]) / (G.trace() / G.shape[0])).sqrt()
        invs = [torch.linalg.inv(m + s * curv.damping ** 0.5 * torch.eye(m.shape[0], dtype=m.dtype))
                for m, s in ((A, pi), (G, 1 / pi))]
        u = invs[1] @ torch.cat([closure.raw[0], closure.raw[1][:, None]], 1).double().cpu() @ invs[0]
        assert rel(model[3].weight.grad, u[:, :-1]) < TOL and rel(model[3].bias.grad, u[:, -1]) < TOL
        return invs
    forms = []
    for inverse_renewed in (True, True, True, False, True, True):
        opt.update_inv = inverse_renewed
        opt.step(closure=closure)
        forms.append(curv._a_in_halves)
        if inverse_renewed:
            invs = preconditioned()
    # (nothing is known at the first; the third's inverses were used twice, the fifth's once)
    assert forms == [False, True, True, True, False, True]
    got = [p.grad.clone() for p in model[3].parameters()]
    for a, b in zip(curv.inv, invs):
        assert rel(a, b) < TOL
    assert curv._a_in_halves           # (reading the inverse changes nothing)
    for p, r in zip(model[3].parameters(), closure.raw):
        p.grad = r.clone()
    curv.precondition_grad(list(model[3].parameters()))
    for p, g in zip(model[3].parameters(), got):
        assert rel(p.grad, g.double().cpu()) < TOL


def test_one_factor_that_has_to_be_in_halves_takes_the_batch_with_it():
    """(alone it would be inverted whole; matrices of one block have no halves)"""
    dev = torch.device('cuda', 0)
    A64, G64 = spd(300, 1), spd(100, 2)
    pi = ((A64.trace() / 300) / (G64.trace() / 100)).sqrt()
    want = operand(A64 + 0.1 * pi * torch.eye(300, dtype=A64.dtype), 'H')[0]
    a, g = A64.float().to(dev), G64.float().to(dev)
    af, gf, af1, gf1 = torch.empty_like(a), torch.empty_like(g), torch.empty_like(g), torch.empty_like(g)
    halves = [2, 2]
    ops.pi_damped_inverse_factored_batched([a, g], [g, g], [1e-2] * 2, [None] * 2, [None] * 2, [af, af1], [gf, gf1],
                                           a_halves=halves)
    assert halves == [True, False]
    assert rel(af, want) < TOL


@pytest.mark.parametrize('form', ['whole', 'halves'])
def test_captured_graphs_find_the_form_they_were_captured_with(form, monkeypatch):
    """Graphs of a preconditioning and of an inversion, replayed between calls that choose a form anew."""
    import torch.nn as nn
    import torchsso
    from torchsso.curv import curvature
    monkeypatch.setattr(curvature.KronCurvature, 'halved_inverse_min_dim', 256)
    monkeypatch.setattr(curvature.KronCurvature, 'halved_inverse_min_work', 1.)
    dev = torch.device('cuda', 0)
    torch.manual_seed(0)
    model = nn.Sequential(*[nn.Linear(1000, 1000, device=dev) for _ in range(13)])
    opt = torchsso.optim.SecondOrderOptimizer(model, 'Cov', {'Linear': 'Kron'}, {'damping': 1e-1}, lr=0.)
    x = torch.randn(256, 1000, device=dev)

    def closure():
        opt.zero_grad(set_to_none=False)
        out = model(x)
        loss = out.pow(2).mean()
        loss.backward()
        return loss, out
    opt.step(closure=closure)
    curvs = [g['curv'] for g in opt.param_groups]
    pairs = [(g['curv'], g['params']) for g in opt.param_groups]
    for k, d in enumerate((1001, 1000)):     # (of a scale at which neither form passes for the other)
        factor = spd(d, d).float().to(dev)
        for c in curvs:
            c.ema[k].copy_(factor)
    if form == 'whole':
        curvature.precondition_all(pairs)    # (used twice)
    curvature.update_inv_all(curvs)
    assert [c._a_in_halves for c in curvs] == [form == 'halves'] * 13

    def restored():
        for i, (_, params) in enumerate(pairs):
            gen = torch.Generator(device=dev).manual_seed(i)
            for p in params:
                p.grad.copy_(torch.randn(p.shape, device=dev, generator=gen))

    def graph_of(run):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            run()
        return graph
    restored()
    A, G = (e.double().cpu() for e in curvs[3].ema)
    pi = ((A.trace() / A.shape[0]) / (G.trace() / G.shape[0])).sqrt()
    r = curvs[3].damping ** 0.5
    v = torch.cat([pairs[3][1][0].grad, pairs[3][1][1].grad[:, None]], 1).double().cpu()
    want = (torch.linalg.inv(G + r / pi * torch.eye(G.shape[0], dtype=G.dtype)) @ v
            @ torch.linalg.inv(A + r * pi * torch.eye(A.shape[0], dtype=A.dtype)))

    def check():
        w, b = (p.grad for p in pairs[3][1])
        assert rel(torch.cat([w, b[:, None]], 1), want) < TOL
    precondition = graph_of(lambda: curvature.precondition_all(pairs))
    invert = graph_of(lambda: curvature.update_inv_all(curvs))
    eager_inversions = [lambda: curvature.update_inv_all(curvs), lambda: curvature.update_inv_all([curvs[3]]),
                        lambda: None]
    for again in eager_inversions * 2:
        for inversion in (invert.replay, again):
            inversion()
            for run in (lambda: curvature.precondition_all(pairs), precondition.replay):
                restored()
                run()
                check()
    for c in curvs:
        c.inv = None             # (nothing of the graphs' memory is used behind them)


@pytest.mark.parametrize('form', ['whole', 'halves'])
def test_captured_reads_of_an_inverse_find_the_form_they_were_captured_with(form, monkeypatch):
    """A graph of `inv` alone (which multiplies the factor by its transpose, and completes a copy of one in halves
    first), replayed behind inversions that choose a form anew."""
    import torch.nn as nn
    import torchsso
    from torchsso.curv import curvature
    monkeypatch.setattr(curvature.KronCurvature, 'halved_inverse_min_dim', 256)
    monkeypatch.setattr(curvature.KronCurvature, 'halved_inverse_min_work', 1.)
    dev = torch.device('cuda', 0)
    torch.manual_seed(0)
    model = nn.Sequential(*[nn.Linear(1000, 1000, device=dev) for _ in range(13)])
    opt = torchsso.optim.SecondOrderOptimizer(model, 'Cov', {'Linear': 'Kron'}, {'damping': 1e-1}, lr=0.)
    x = torch.randn(256, 1000, device=dev)

    def closure():
        opt.zero_grad(set_to_none=False)
        out = model(x)
        loss = out.pow(2).mean()
        loss.backward()
        return loss, out
    opt.step(closure=closure)
    curvs = [g['curv'] for g in opt.param_groups]
    pairs = [(g['curv'], g['params']) for g in opt.param_groups]
    for k, d in enumerate((1001, 1000)):
        factor = spd(d, d).float().to(dev)
        for c in curvs:
            c.ema[k].copy_(factor)
    if form == 'whole':
        curvature.precondition_all(pairs)    # (used twice)
    curvature.update_inv_all(curvs)
    assert [c._a_in_halves for c in curvs] == [form == 'halves'] * 13
    A, G = (e.double().cpu() for e in curvs[3].ema)
    pi = ((A.trace() / A.shape[0]) / (G.trace() / G.shape[0])).sqrt()
    r = curvs[3].damping ** 0.5
    want = [torch.linalg.inv(m + s * torch.eye(m.shape[0], dtype=m.dtype)) for m, s in ((A, r * pi), (G, r / pi))]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        read = list(curvs[3].inv)
    for uses in (0, 1, 2, 1, 0):
        for _ in range(uses):
            curvature.precondition_all(pairs)
        curvature.update_inv_all(curvs)
        for t in read:
            t.fill_(float('nan'))
        graph.replay()
        for t, w in zip(read, want):
            assert rel(t, w) < TOL
    for c in curvs:
        c.inv = None             # (nothing of the graph's memory is used behind it)


def test_inverses_that_are_read_every_time_stay_whole(monkeypatch):
    """(to complete a factor in halves costs a read what the inversion was spared)"""
    import torch.nn as nn
    import torchsso
    from torchsso.curv.curvature import KronCurvature
    monkeypatch.setattr(KronCurvature, 'halved_inverse_min_dim', 256)
    monkeypatch.setattr(KronCurvature, 'halved_inverse_min_work', 1.)
    dev = torch.device('cuda', 0)
    torch.manual_seed(0)
    model = nn.Sequential(*[nn.Linear(1000, 1000, device=dev) for _ in range(13)])
    opt = torchsso.optim.SecondOrderOptimizer(model, 'Cov', {'Linear': 'Kron'}, {'damping': 1e-1}, lr=0.)
    x = torch.randn(256, 1000, device=dev)

    def closure():
        opt.zero_grad()
        out = model(x)
        loss = out.pow(2).mean()
        loss.backward()
        return loss, out
    forms = []
    for read in (True, True, True, False, False, True, True):
        opt.step(closure=closure)
        forms.append([g['curv']._a_in_halves for g in opt.param_groups[2:4]])
        if read:
            opt.param_groups[2]['curv'].inv
    # (the inverses of the third layer are in halves only behind a step without a read)
    assert forms == [[False, False], [False, True], [False, True], [False, True], [True, True], [True, True],
                     [False, True]]
