"""Shampoo on the GPU: the batched inverse-root kernel against the reference's golden outputs and the
fp64 closed form, and ShampooGradientMaker against the reference's golden multi-step runs and the CPU
oracle.  Tolerances: roots and preconditioned gradients 1e-3 relative Frobenius error (the iteration
stops at max|M - I| <= 1e-6, so two fp32 implementations agree to ~1e-5 on well-conditioned input)."""
import copy
import ctypes
import os

import numpy as np
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from asdl_amd import PreconditioningConfig, ShampooGradientMaker, kernels as K, compute_power, _lib
from conftest import GOLDEN
from models_small import GOLDEN_SHAMPOO, get_mlp
from oracle import cpu_ref as R
import bench_models

pytestmark = pytest.mark.gpu


def relerr(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return float((a - b).norm() / b.norm().clamp_min(1e-300))


def _closed_form_root(S, p):
    w, V = torch.linalg.eigh(S.double().cpu())
    if float(w[0]) <= 0:
        return None
    return V @ torch.diag(w ** (-1.0 / p)) @ V.T


def _check_root(mine, golden, stat_after, p, what):
    """The coupled Newton iteration in fp32 loses accuracy with cond(S): the reference's own output is up to
    5e-3 away from the exact root at cond ~ 1e6.  Both are therefore judged against the fp64 closed form of the
    (ridged) statistic; where the reference is accurate (< 1e-4) the two must also agree directly."""
    exact = _closed_form_root(stat_after, p)
    if exact is None:
        return None          # numerically indefinite input: no meaningful root to compare with
    e_ref, e_mine = relerr(golden, exact), relerr(mine, exact)
    assert e_mine <= max(4 * e_ref, 1e-4), (what, e_mine, e_ref)
    if e_ref < 1e-4:
        assert relerr(mine, golden) < 1e-3, (what, relerr(mine, golden))
    return e_ref


def test_inv_root_matches_reference_golden():
    z = np.load(os.path.join(GOLDEN, 'power.npz'))
    checked = 0
    for name in sorted({k.split('/')[0] for k in z.files}):
        mat = torch.from_numpy(z[f'{name}/in']).cuda()
        p, eps = int(z[f'{name}/p']), float(z[f'{name}/eps'])
        print(f'inv_root golden {name} p={p}', flush=True)
        root, stats = K.inv_root_newton(mat, p, eps, torch.from_numpy(z[f'{name}/v0']).cuda())
        after = torch.from_numpy(z[f'{name}/mat_after'])
        torch.testing.assert_close(mat.cpu(), after, rtol=1e-5, atol=1e-10)
        if _check_root(root, torch.from_numpy(z[f'{name}/root']), after, p, name) is not None:
            checked += 1
    assert checked >= 5


@pytest.mark.parametrize('n,p,batch', [(2, 4, 1), (16, 2, 3), (200, 4, 2), (768, 4, 1), (130, 8, 2), (64, 6, 1),
                                       (520, 4, 2), (1000, 6, 2), (600, 2, 3), (512, 3, 1)])
def test_inv_root_closed_form(n, p, batch):
    """(S + ridge I)^(-1/p) against the fp64 closed form, the power iteration and the iteration count against the
    oracle.  Statistics below 512 columns iterate on fp32 matrices, the others on 16-bit planes padded to a multiple
    of 192 (520 -> 576, 1000 -> 1152), here two fp16 planes each (the ridge of 1e-6 bounds the root below 4096; the
    bf16 planes have their own test below); p = 6 and p = 3 take the general power sequence (squares and a running product),
    p = 2, 4, 8 repeated squaring."""
    g = torch.Generator().manual_seed(n + p)
    S = torch.empty(batch, n, n)
    for b in range(batch):
        X = torch.randn(3 * n, n, generator=g)
        S[b] = X.T @ X / (3 * n)
    v0 = torch.rand(batch, n, generator=g) * 2 - 1
    Sg = S.cuda().clone()
    print(f'inv_root closed form n={n} p={p} batch={batch}', flush=True)
    root, stats = K.inv_root_newton(Sg, p, 1e-6, v0.cuda())
    stats = stats.cpu()
    for b in range(batch):
        # the power iteration stops on |change| <= 1e-6 or after 100 steps, not at convergence: compare with
        # the oracle's estimate from the same start vector, and loosely with the true lambda_max
        lam_orc, _ = R.power_iter(S[b], v0[b])
        assert abs(float(stats[b, 0]) - float(lam_orc)) / float(lam_orc) < 1e-3
        lam = torch.linalg.eigvalsh(S[b].double())[-1]
        assert abs(float(stats[b, 0]) - float(lam)) / float(lam) < 5e-2
        Sr = S[b].double() + 1e-6 * float(stats[b, 0]) * torch.eye(n, dtype=torch.float64)
        assert relerr(Sg[b], Sr) < 1e-6                       # the ridge stays in the statistic
        w, V = torch.linalg.eigh(Sr)
        ref = V @ torch.diag(w ** (-1.0 / p)) @ V.T
        assert relerr(root[b], ref) < 1e-3, (b, relerr(root[b], ref), stats[b])
        # same iteration count as the oracle run from the same start vector
        _, iters, _ = R.compute_power(S[b].clone(), p, v0[b], ridge_epsilon=1e-6)
        assert abs(int(stats[b, 2]) - iters) <= 1, (int(stats[b, 2]), iters)


@pytest.mark.parametrize('groups', [
    ((2, 4, 1), (31, 2, 1), (32, 3, 2), (33, 4, 1), (63, 8, 1), (65, 4, 3), (129, 6, 1)),      # fp32 matrices on 64-wide tiles
    ((255, 4, 40), (256, 4, 25), (511, 2, 3)),                                # fp32 on split products, and not enough for them
    ((512, 4, 1), (577, 4, 2), (640, 2, 1), (300, 4, 1)),                     # small tiles of planes beside fp32 ones
    ((513, 4, 45), (20, 4, 2)),                                               # 192-wide tiles of planes
])
def test_inv_root_group_of_several_sizes(groups):
    """Groups of different size and power in one call: each root symmetric (exactly on planes, which mirror their tiles) and
    against the fp64 closed form."""
    g = torch.Generator().manual_seed(5)
    items, before = [], []
    for n, p, batch in groups:
        X = torch.randn(batch, 2 * n, n, generator=g) * torch.logspace(0, -1, n)
        S = (X.transpose(1, 2) @ X / (2 * n)).cuda()
        items.append((S, p, (torch.rand(batch, n, generator=g) * 2 - 1).cuda(), None))
        before.append(S.clone())
    print(f'inv_root groups {groups}', flush=True)
    results = K.inv_root_group(items, 1e-6)
    for (n, p, batch), (S, _, _, _), old, (root, stats) in zip(groups, items, before, results):
        assert (stats[:, 2] > 0).all() and (stats[:, 3] <= 1e-6).all(), (n, p, stats)
        assert torch.equal(root, root.transpose(1, 2)) if n >= 512 else relerr(root, root.transpose(1, 2)) < 1e-3
        for b in (0, batch - 1):
            lam = float(stats[b, 0])
            assert relerr(S[b], old[b].double() + 1e-6 * lam * torch.eye(n, device='cuda')) < 1e-6
            assert relerr(root[b], _closed_form_root(S[b], p)) < 1e-3, (n, p, b)


def _classical_root_steps(S, p, ridge, tol=1e-6):
    """Steps of the reference's iteration (asdl/precondition/shampoo.py:508-521) by its effect on the eigenvalues, in 64 bits."""
    ev = torch.linalg.eigvalsh(S.double()).clamp_min(0.0)
    ev = ev + ridge * ev[-1]
    m = ev * (1 + p) / (2 * ev.norm())
    steps = 0
    while float((m - 1).abs().max()) > tol:
        m = m * (1 + 1 / p - m / p) ** p
        steps += 1
    return steps


def _with_eigenvalues(ev, g):
    """A symmetric matrix with these eigenvalues: three random reflections of the diagonal one."""
    S = torch.diag(ev.double())
    for _ in range(3):
        v = torch.randn(len(ev), generator=g, dtype=torch.float64, device=ev.device)
        v /= v.norm()
        Sv = S @ v
        S = S - 2 * torch.outer(v, Sv) - 2 * torch.outer(Sv, v) + 4 * (v @ Sv) * torch.outer(v, v)
    return ((S + S.T) / 2).float()


@pytest.mark.parametrize('n,kind,p', [(n, kind, p) for n in (130, 512) for p in (2, 4, 8) for kind in (
    '1 to 0.01', '1 to 0.0001', 'few tiny', 'rank 1/4', '3 batches', '10 batches', '40 batches')] +
    [(3072, '1 to 0.01', 4), (3072, 'rank 1/4', 4)])
def test_inv_root_takes_no_more_steps_than_the_classical_iteration(n, kind, p):
    """Full-rank statistics (summed over several batches of n / 4 rows, or with given eigenvalues) as well as rank-deficient ones:
    the schedule comes from the spectrum."""
    g = torch.Generator('cuda').manual_seed(n)
    if 'batches' in kind or 'rank' in kind:
        rows = n // 4 * (int(kind.split()[0]) if 'batches' in kind else 1)
        X = torch.randn(rows, n, generator=g, device='cuda')
        S = X.T @ X
    else:
        low = -4 if '0.0001' in kind else -2
        ev = torch.logspace(0, low, n, device='cuda')
        if kind == 'few tiny':
            ev[-3:] = 1e-7
        S = _with_eigenvalues(ev, g)
    v0 = torch.rand(1, n, generator=g, device='cuda') * 2 - 1
    classical = _classical_root_steps(S, p, 1e-6)
    print(f'inv_root steps n={n} {kind} p={p}: classical {classical}', flush=True)
    root, stats = K.inv_root_newton(S.unsqueeze(0).clone(), p, 1e-6, v0)
    steps, error = int(stats[0, 2]), float(stats[0, 3])
    print(f'  here {steps}', flush=True)
    assert error <= 1e-6 and steps <= classical, (steps, classical)
    if kind in ('rank 1/4', 'few tiny'):
        assert steps < classical - 2, (steps, classical)


@pytest.mark.parametrize('m,n,rank', [(512, 784, 128), (256, 300, 64), (300, 600, 16), (768, 1100, 200), (96, 700, 50)])
def test_inv_root_is_as_good_as_the_classical_one_where_the_gradient_lies(m, n, rank):
    """L^(-1/4) G R^(-1/4) for L = G G^T, R = G^T G of a rank-deficient G, what Shampoo does with a first gradient, against 64 bits:
    at most 1.3 times the error with the reference's steps throughout, which a limit of 31 steps asks for.  (The error of the
    whole root is the null space's and says nothing here.)"""
    g = torch.Generator('cuda').manual_seed(m)
    G = torch.randn(m, rank, generator=g, device='cuda') @ torch.randn(rank, n, generator=g, device='cuda') / rank
    roots = {'here': [], 'classical': [], 'exact': []}
    for S in (G @ G.T, G.T @ G):
        S = ((S + S.T) / 2).unsqueeze(0).contiguous()
        v0 = torch.rand(1, S.shape[1], generator=g, device='cuda') * 2 - 1
        for which, max_iter in (('here', 100), ('classical', 31)):
            ridged = S.clone()
            root, stats = K.inv_root_newton(ridged, 4, 1e-6, v0, max_iter=max_iter)
            assert float(stats[0, 3]) <= 1e-6
            roots[which].append(root[0].double())
        w, V = torch.linalg.eigh(ridged[0].double())
        roots['exact'].append((V * w.clamp_min(1e-30) ** -0.25) @ V.T)
    L, R_ = roots['exact']
    exact = L @ G.double() @ R_
    here, classical = (relerr(L @ G.double() @ R_, exact) for L, R_ in (roots['here'], roots['classical']))
    print(f'root on the range of G {m} x {n} rank {rank}: here {here:.2e}, classical {classical:.2e}', flush=True)
    assert here <= 1.3 * classical


@pytest.mark.parametrize('n,batch', [(33, 3), (255, 2), (511, 1), (512, 3), (513, 45), (577, 3), (1000, 1)])
def test_inv_root_steps_of_the_fourth_degree(n, batch):
    """Rank-deficient statistics beside a well-conditioned one (whose steps stay classical) on fp32 matrices, small tiles and 192-wide tiles
    (45 of 513 columns): far fewer steps than the first degree takes, each root the one that its matrix gets in a call of its own (on
    planes bit for bit, whichever tile it takes), and the exact one: 1e-5 for the well-conditioned one, 5 % for the others, whose
    smallest eigenvalues, 1e-6 of the largest, the rounding of fp32 moves by up to 2e-7 of the largest, a quarter of that in the root."""
    g = torch.Generator('cuda').manual_seed(n)
    S = torch.empty(batch + 1, n, n, device='cuda')
    for b in range(batch):
        X = torch.randn(max(2, n // (3 + b % 3)), n, generator=g, device='cuda')
        S[b] = X.T @ X
    S[batch] = _with_eigenvalues(torch.linspace(1, 2, n, device='cuda'), g)
    v0 = torch.rand(batch + 1, n, generator=g, device='cuda') * 2 - 1
    ridged = S.clone()
    print(f'inv_root fourth degree n={n} batch={batch}', flush=True)
    root, stats = K.inv_root_newton(ridged, 4, 1e-6, v0)
    assert (stats[:, 3] <= 1e-6).all() and (stats[:batch, 2] <= 13).all(), stats
    for b in {0, batch // 2, batch - 1, batch}:
        alone, st = K.inv_root_newton(S[b:b + 1].clone(), 4, 1e-6, v0[b:b + 1])
        assert torch.equal(st[0, :3], stats[b, :3]), (b, st, stats[b])
        # the final error is the same too, or (wide tiles, M not formed in the last step) an estimate from above, but for the rounding of M,
        # four products of 22 bits
        assert st[0, 3] == stats[b, 3] or (batch > 40 and st[0, 3] <= stats[b, 3] + 4 * 2.0 ** -22 and stats[b, 3] <= 0.625e-6), (b, st, stats[b])
        if n >= 512:
            assert torch.equal(alone[0], root[b]) and torch.equal(root[b], root[b].T), b
        else:
            assert relerr(alone[0], root[b]) < 1e-6, b
        assert relerr(root[b], _closed_form_root(ridged[b], 4)) < (1e-5 if b == batch else 5e-2), b


@pytest.mark.parametrize('groups,ridge', [
    (((2, 1, 1), (65, 3, 2), (130, 4, 1), (33, 5, 3), (40, 7, 1), (64, 11, 1)), 1e-6),
    (((512, 4, 1), (600, 2, 2), (577, 7, 1), (300, 8, 2), (520, 10, 1)), 1e-6),
    (((513, 4, 45), (20, 6, 2)), 1e-6),
    (((520, 4, 1), (600, 3, 2)), 0.0),
])
def test_inv_root_stays_within_its_workspace(groups, ridge, monkeypatch):
    """Storage by size, power and ridge: as many bytes again behind the workspace stay as they were, and the roots are right."""
    g = torch.Generator().manual_seed(9)
    items = []
    for n, p, batch in groups:
        X = torch.randn(batch, 3 * n, n, generator=g)
        items.append(((X.transpose(1, 2) @ X / (3 * n)).cuda(), p, (torch.rand(batch, n, generator=g) * 2 - 1).cuda(), None))
    made = []

    def workspace(nbytes, device):
        made.append((torch.full((2 * nbytes + 512,), 0xA5, dtype=torch.uint8, device=device), nbytes))
        return made[-1][0][:nbytes], nbytes

    monkeypatch.setattr(K, 'workspace', workspace)
    results = K.inv_root_group(items, ridge)
    (buf, nbytes), = made
    assert torch.all(buf[nbytes:] == 0xA5)
    for (S, p, _, _), (root, _) in zip(items, results):
        assert relerr(root[0], _closed_form_root(S[0], p)) < 1e-3, (S.shape, p)


def test_inv_root_of_more_columns_than_the_lds_holds():
    """A statistic whose Lanczos vectors do not fit the LDS (more than 32768 columns; 64-bit indices throughout): lambda_max against
    a power iteration here, the ridge, and two steps for p = 1, X_2 = z T_0 T_1 with T_0 = 2 I - z S, T_1 = 2 I - T_0 z S, applied to
    two vectors in 64 bits.  Three products of 7e13 operations."""
    n, p, eps = 32772, 1, 1e-3
    g = torch.Generator('cuda').manual_seed(1)
    u = torch.randn(n, generator=g, device='cuda')
    S = torch.outer(u, u) * (10 / float(u @ u))
    S.diagonal().add_(1 + torch.rand(n, generator=g, device='cuda'))
    before = S.diagonal().clone()
    v = torch.randn(n, generator=g, device='cuda')
    for _ in range(30):
        v = S @ (v / v.norm())
    lam = float(v.norm())
    try:
        root, stats = K.inv_root_newton(S, p, eps, torch.rand(1, n, generator=g, device='cuda') * 2 - 1, max_iter=2)
        assert int(stats[0, 2]) == 2
        assert abs(float(stats[0, 0]) - lam) < 1e-4 * lam
        assert relerr(S.diagonal() - before, torch.full((n,), eps * lam)) < 1e-3
        norm = float(sum(float((rows.double() ** 2).sum()) for rows in S.split(4096))) ** 0.5
        z = (1 + p) / (2 * norm)

        def times(x):
            return z * torch.cat([rows.double() @ x for rows in S.split(4096)])
        x = torch.randn(n, 2, generator=g, device='cuda').double()
        Sx = times(x)
        t1 = 2 * x - (2 * Sx - times(Sx))                 # T_1 x
        expected = z * (2 * t1 - times(t1))
        got = torch.cat([rows.double() @ x for rows in root.split(4096)])
        assert relerr(got, expected) < 1e-5, relerr(got, expected)
    finally:
        K.release_workspaces()


def test_inv_root_polled_and_unpolled_enqueue_give_the_same_result():
    """The host may stop enqueuing Newton iterations once the convergence flags are all zero (read every few
    iterations) or enqueue all of them blindly: bit-equal roots and the same iteration counts."""
    g = torch.Generator().manual_seed(77)
    S = torch.empty(3, 96, 96)
    for b in range(3):
        X = torch.randn(40 * (b + 1), 96, generator=g)        # one rank-deficient, two full-rank statistics
        S[b] = X.T @ X / X.shape[0]
    v0 = (torch.rand(3, 96, generator=g) * 2 - 1).cuda()
    r0, st0 = K.inv_root_newton(S.cuda().clone(), 4, 1e-6, v0, poll_every=0)
    r1, st1 = K.inv_root_newton(S.cuda().clone(), 4, 1e-6, v0, poll_every=3)
    r2, st2 = K.inv_root_newton(S.cuda().clone(), 4, 1e-6, v0)
    assert torch.equal(r0, r1) and torch.equal(r0, r2)
    assert torch.equal(st0, st1) and torch.equal(st0, st2)
    assert 1 <= float(st0[:, 2].max()) < 100
    # the same on 16-bit planes (576 columns; p = 4: two fp16 planes; p = 2 with a ridge of 1e-7: the ridge does not
    # bound the root below 4096, three bf16 planes): parts of an odd number of iterations end with the iterates in the second buffer pair,
    # from which they are brought back before the next part starts
    S = torch.empty(2, 576, 576)
    for b in range(2):
        X = torch.randn(400 * (b + 1), 576, generator=g)
        S[b] = X.T @ X / X.shape[0]
    v0 = (torch.rand(2, 576, generator=g) * 2 - 1).cuda()
    for p, eps, planes in ((4, 1e-6, 2), (2, 1e-7, 3)):
        assert _lib.load().ak_inv_root_plane_format(576, p, eps) == planes
        r0, st0 = K.inv_root_newton(S.cuda().clone(), p, eps, v0, poll_every=0)
        r1, st1 = K.inv_root_newton(S.cuda().clone(), p, eps, v0, poll_every=3)
        r2, st2 = K.inv_root_newton(S.cuda().clone(), p, eps, v0)
        assert torch.equal(r0, r1) and torch.equal(r0, r2)
        assert torch.equal(st0, st1) and torch.equal(st0, st2)
        assert 1 <= float(st0[:, 2].max()) < 100


def test_inv_root_plane_formats_and_their_fallbacks():
    """Which statistics iterate on which storage: fp32 matrices below 512 columns; two fp16 planes where ridge, power
    and size bound the root's largest eigenvalue below 4096; three bf16 planes else (no ridge, a small ridge with a
    low power, powers above 8).  A well-conditioned statistic without a ridge (bf16 planes) against the closed form."""
    fmt = _lib.load().ak_inv_root_plane_format
    assert fmt(130, 8, 1e-6) == 0 and fmt(511, 4, 1e-6) == 0
    assert fmt(768, 4, 1e-6) == 2 and fmt(3072, 4, 1e-6) == 2 and fmt(1000, 6, 1e-6) == 2 and fmt(512, 3, 1e-6) == 2
    assert fmt(600, 2, 1e-6) == 2 and fmt(768, 2, 1e-3) == 2 and fmt(3072, 4, 1e-13) == 2
    assert fmt(768, 2, 1e-6) == 3 and fmt(3072, 4, 1e-14) == 3
    assert fmt(768, 4, 0.0) == 3 and fmt(768, 4, 1e-30) == 3 and fmt(768, 10, 1e-6) == 3
    g = torch.Generator().manual_seed(5)
    n = 600
    X = torch.randn(4 * n, n, generator=g)
    S = (X.T @ X / (4 * n)).unsqueeze(0)
    v0 = torch.rand(1, n, generator=g) * 2 - 1
    for p, eps in ((4, 0.0), (4, 1e-6), (2, 1e-7)):
        assert fmt(n, p, eps) == (2 if eps == 1e-6 else 3)
        root, stats = K.inv_root_newton(S.cuda().clone(), p, eps, v0.cuda())
        lam = float(stats[0, 0])
        w, V = torch.linalg.eigh(S[0].double() + eps * lam * torch.eye(n, dtype=torch.float64))
        ref = V @ torch.diag(w ** (-1.0 / p)) @ V.T
        assert relerr(root[0], ref) < 1e-5, (p, eps, relerr(root[0], ref))


def test_compute_power_api_and_1x1():
    S = torch.tensor([[4.0]]).cuda()
    assert torch.equal(compute_power(S, 4).cpu(), torch.eye(1))
    d = torch.tensor([1.0, 16.0]).cuda()
    torch.testing.assert_close(compute_power(d, 4, ridge_epsilon=0.0).cpu(), torch.tensor([1.0, 0.5]))


def _reference_order_vectors(gm, generator):
    """Draws the power-iteration start vectors in the reference's order (parameter by parameter, axis by
    axis) and buckets them per statistic size, the order in which the maker's groups list their members."""
    per_n = {}
    for prec in gm.preconditioners:
        for n in prec.param.shape:
            per_n.setdefault(n, []).append(torch.rand(n, generator=generator) * 2 - 1)
    return per_n


@pytest.mark.parametrize('tag', sorted(GOLDEN_SHAMPOO))
def test_shampoo_gpu_matches_reference_golden(tag):
    damping, ema, ci, pi = GOLDEN_SHAMPOO[tag]
    z = np.load(os.path.join(GOLDEN, f'shampoo_{tag}.npz'))
    model = get_mlp()
    model.load_state_dict({k[len('init/'):]: torch.from_numpy(z[k]) for k in z.files if k.startswith('init/')})
    model = model.cuda()
    config = PreconditioningConfig(damping=damping, ema_decay=ema, curvature_upd_interval=ci,
                                   preconditioner_upd_interval=pi)
    gm = ShampooGradientMaker(model, config)
    gen = torch.Generator().manual_seed(int(z['seed']))
    opt = torch.optim.SGD(model.parameters(), lr=0.05)
    n_steps = len({k.split('/')[0] for k in z.files if k.startswith('step')})
    for step in range(n_steps):
        if gm.do_update_preconditioner(step):
            vecs = _reference_order_vectors(gm, gen)
            gm.start_vector_fn = lambda count, n, dev, _v=vecs: torch.stack(_v[n]).to(dev)
        opt.zero_grad(set_to_none=True)
        x, t = torch.from_numpy(z[f'step{step}/x']).cuda(), torch.from_numpy(z[f'step{step}/t']).cuda()
        gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(model, x), t)
        print(f'shampoo golden {tag} step {step}', flush=True)
        gm.forward_and_backward()
        worst_ref = 0.0
        for i, prec in enumerate(gm.preconditioners):
            for j in range(2):
                torch.testing.assert_close(prec.statistics[j].cpu(), torch.from_numpy(z[f'step{step}/stat/{i}/{j}']),
                                           rtol=1e-4, atol=1e-12)
                e_ref = _check_root(prec.preconditioners[j], torch.from_numpy(z[f'step{step}/prec/{i}/{j}']),
                                    torch.from_numpy(z[f'step{step}/stat/{i}/{j}']), 4, (tag, step, i, j))
                worst_ref = max(worst_ref, e_ref or 0.0)
        # gradients inherit the accuracy of the roots: 1e-3 when the reference's roots are accurate, else a
        # few times the reference's own distance from the exact roots
        tol = max(1e-3, 8 * worst_ref)
        for name, p in model.named_parameters():
            assert relerr(p.grad, torch.from_numpy(z[f'step{step}/grad/{name}'])) < tol, (tag, step, name, tol)
        # follow the reference's trajectory exactly: apply ITS preconditioned gradients, so that every step is
        # compared on identical parameters (ill-conditioned roots would otherwise compound through the optimizer)
        with torch.no_grad():
            for name, p in model.named_parameters():
                p.grad.copy_(torch.from_numpy(z[f'step{step}/grad/{name}']).cuda())
        opt.step()


def test_shampoo_gpt2_shaped_mini_vs_oracle():
    # config 5 geometry at a small width: d = 64, 2 layers, 4 heads, vocab 97, 2 x 32 tokens
    torch.manual_seed(0)
    model_cpu = bench_models.gpt2_small(vocab=97, d=64, n_layer=2, n_head=4, n_ctx=32)
    model_gpu = copy.deepcopy(model_cpu).cuda()
    idx = torch.randint(0, 97, (2, 32))
    tgt = torch.randint(0, 97, (2, 32))

    def loss_fn(logits, targets, reduction='mean'):
        return F.cross_entropy(logits.view(-1, logits.size(-1)), targets.view(-1), reduction=reduction)

    config = PreconditioningConfig(damping=1e-6, curvature_upd_interval=1, preconditioner_upd_interval=2)
    gm = ShampooGradientMaker(model_gpu, config)
    orc = R.ShampooOracle(model_cpu, damping=1e-6, curvature_upd_interval=1, preconditioner_upd_interval=2)
    gen = torch.Generator().manual_seed(3)
    for step in range(3):
        model_cpu.zero_grad(set_to_none=True)
        model_gpu.zero_grad(set_to_none=True)
        vecs = _reference_order_vectors(gm, gen)
        taken = {n: 0 for n in vecs}

        def cpu_vec(n):
            v = vecs[n][taken[n]]
            taken[n] += 1
            return v
        gm.start_vector_fn = lambda count, n, dev, _v=vecs: torch.stack(_v[n]).to(dev)
        orc.forward_and_backward(idx, tgt, loss_fn=loss_fn, start_vectors=cpu_vec)
        gm.setup_loss_call(loss_fn, gm.setup_model_call(model_gpu, idx.cuda()), tgt.cuda())
        gm.forward_and_backward()
        for (name, p_cpu), (_, p_gpu) in zip(model_cpu.named_parameters(), model_gpu.named_parameters()):
            if p_cpu.grad is None:
                continue
            e = relerr(p_gpu.grad, p_cpu.grad)
            assert e < 5e-3, (step, name, e)


@pytest.mark.parametrize('tag', ['mat_10x6_b4', 'mat_9x13_b5_ema', 'conv_5x4x3x3_b4'])
def test_block_partitioned_preconditioner_matches_reference_golden(tag):
    """Preconditioner(param, config, block_size=...) driven directly, as recorded from the reference
    (asdl/precondition/shampoo.py:300-367, 398-462)."""
    from asdl_amd.shampoo import Preconditioner
    z = np.load(os.path.join(GOLDEN, f'shampoo_blocks_{tag}.npz'))
    shape = tuple(int(v) for v in z['shape'])
    param = nn.Parameter(torch.zeros(*shape).cuda())
    config = PreconditioningConfig(damping=float(z['damping']), ema_decay=float(z['ema_decay']))
    prec = Preconditioner(param, config, block_size=int(z['block_size']))
    exp = 2 * len(shape)
    for step in range(3):
        grad = torch.from_numpy(z[f'step{step}/grad_in'])
        param.grad = grad.clone().cuda()
        print(f'shampoo blocks {tag} step {step}', flush=True)
        prec.update_statistics()
        gen = torch.Generator().manual_seed(1000 * int(z['seed']) + step)
        prec.start_vector_fn = lambda n, _g=gen: (torch.rand(n, generator=_g) * 2 - 1).cuda()
        prec.update_preconditioners()
        prec.precondition()
        worst_ref = 0.0
        for i, (st, pm) in enumerate(zip(prec.statistics, prec.preconditioners)):
            after = torch.from_numpy(z[f'step{step}/stat/{i}'])
            torch.testing.assert_close(st.cpu(), after, rtol=1e-4, atol=1e-12)
            if after.shape[0] > 1:
                worst_ref = max(worst_ref, _check_root(pm, torch.from_numpy(z[f'step{step}/prec/{i}']), after, exp,
                                                       (tag, step, i)) or 0.0)
        assert relerr(param.grad, torch.from_numpy(z[f'step{step}/grad_out'])) < max(1e-3, 8 * worst_ref), (tag, step)


def test_grouped_preconditioning_gives_the_per_parameter_result(monkeypatch):
    """shampoo.GROUPED_PRECONDITION: the products of all matrix-shaped parameters in two launches, against the
    per-parameter chain and against P_0^T G P_1 in fp64; a convolution weight and a matrix with an odd size in
    the same model take the per-parameter way."""
    import asdl_amd.shampoo as shampoo_mod

    def run(grouped):
        monkeypatch.setattr(shampoo_mod, 'GROUPED_PRECONDITION', grouped)
        torch.manual_seed(21)
        model = nn.Sequential(nn.Conv2d(3, 8, 3, padding=1), nn.Flatten(), nn.Linear(8 * 6 * 6, 132), nn.ReLU(),
                              nn.Linear(132, 260), nn.ReLU(), nn.Linear(260, 37), nn.ReLU(), nn.Linear(37, 8)).cuda()
        x, t = torch.randn(16, 3, 6, 6).cuda(), torch.randint(0, 8, (16,)).cuda()
        gm = ShampooGradientMaker(model, PreconditioningConfig(data_size=16, damping=1e-6))
        gm.start_vector_fn = lambda count, n, dev: torch.linspace(-1, 1, count * n, device=dev).reshape(count, n)
        out = {}
        for step in range(2):
            model.zero_grad(set_to_none=True)
            gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(model, x), t)
            raw = {}
            orig = gm.precondition

            def precondition_and_keep():
                for name, p in model.named_parameters():
                    raw[name] = p.grad.detach().double().clone()
                orig()
            gm.precondition = precondition_and_keep
            gm.forward_and_backward()
            gm.precondition = orig
            for (name, p), pc in zip([(n_, p_) for n_, p_ in model.named_parameters() if p_.ndim > 1], gm.preconditioners):
                out[(step, name)] = p.grad.detach().clone()
                for a, stat in enumerate(pc.statistics):
                    out[(step, name, a)] = stat.detach().clone()
                    assert torch.equal(stat, stat.T)
                if p.ndim == 2:
                    ref = pc.preconditioners[0].double().T @ raw[name] @ pc.preconditioners[1].double()
                    # the roots of nearly singular statistics span many decades: the terms of these sums cancel
                    assert relerr(p.grad, ref) < 1e-3, (grouped, step, name, relerr(p.grad, ref))
                    print(f'grouped={grouped} step {step} {name}: {relerr(p.grad, ref):.2e}', flush=True)
        return out

    single, grouped = run(False), run(True)
    assert single.keys() == grouped.keys()
    for key in single:
        if len(key) == 3:
            # statistics: same kernels either way; the convolution backward kernels of the library are not
            # reproducible bit for bit from run to run, so the raw gradients may differ in the last bits
            assert relerr(grouped[key], single[key].double()) < 1e-5, key
        else:
            assert relerr(grouped[key], single[key].double()) < 1e-3, key


def test_block_partitioner_and_dimension_merging():
    from asdl_amd.shampoo import BlockPartitioner, Preconditioner, _merge_small_dims
    assert _merge_small_dims([1, 2, 512, 1, 2048, 1, 3, 4], 1024) == [1024, 2048, 12]
    assert _merge_small_dims([1, 2, 768, 1, 2048], 1024) == [2, 768, 2048]
    g = torch.Generator().manual_seed(1)
    t = torch.randn(10, 6, 7, generator=g).cuda()
    bp = BlockPartitioner(t.shape, 4)
    parts = bp.partition(t)
    want = [t[b] for b in R.block_slices((10, 6, 7), 4)]
    assert len(parts) == len(want) == 12 and all(torch.equal(a, b) for a, b in zip(parts, want))
    assert bp.kronecker_factor_shapes()[:3] == [[4, 4], [4, 4], [4, 4]] and bp.num_splits() == 3
    assert torch.equal(bp.merge_partitions(parts), t)
    # merged dimensions: a (6, 3, 2, 2) weight with max_dim 8 is preconditioned as (6, 6, 2), against the oracle
    param = nn.Parameter(torch.zeros(6, 3, 2, 2).cuda())
    prec = Preconditioner(param, PreconditioningConfig(damping=1e-4, ema_decay=-1), block_size=8,
                          best_effort_shape_interpretation=True)
    orc = R.PartitionedShampooOracle((6, 3, 2, 2), 8, True, damping=1e-4)
    assert [tuple(s.shape) for s in prec.statistics] == [(6, 6), (6, 6), (2, 2)]
    for step in range(2):
        grad = torch.randn(6, 3, 2, 2, generator=g)
        param.grad = grad.clone().cuda()
        prec.update_statistics()
        orc.update_statistics(grad)
        vecs = [torch.rand(n, generator=g) * 2 - 1 for n in (6, 6, 2)]
        it_a, it_b = iter(vecs), iter(vecs)
        prec.start_vector_fn = lambda n: next(it_a).cuda()
        prec.update_preconditioners()
        orc.update_preconditioners(lambda n: next(it_b))
        prec.precondition()
        for a, b in zip(prec.statistics, orc.statistics):
            assert relerr(a, b) < 1e-5
        assert relerr(param.grad, orc.precondition(grad)) < 1e-3


def test_shampoo_gpt2_small_weight_shapes_full_size():
    """The transformer configuration at the real weight shapes of one decoder block (768 x 2304 attention input,
    768 x 768 attention output, 768 x 3072 and 3072 x 768 MLP): statistics against fp64 products of the very
    gradients, inverse fourth roots through the closed form of the ridged statistic, and the preconditioned
    gradient against P_L^T G P_R recomputed in fp64 from the stored roots."""
    torch.manual_seed(9)
    shapes = [(2304, 768), (768, 768), (3072, 768), (768, 3072)]
    model = nn.Sequential(*[nn.Linear(i, o, bias=False) for o, i in shapes]).cuda()
    params = [m.weight for m in model]
    gm = ShampooGradientMaker(model, PreconditioningConfig(damping=1e-6, ema_decay=-1))
    # statistics accumulated over five gradients, as in training: every statistic has full rank (a single gradient
    # leaves the larger side of each weight rank deficient, cond = 1e6 after the ridge, where no fp32 root is accurate)
    sums = [[torch.zeros(s[0], s[0], dtype=torch.float64, device='cuda'),
             torch.zeros(s[1], s[1], dtype=torch.float64, device='cuda')] for s in shapes]
    for _ in range(5):
        grads = [torch.randn(*s).cuda() * 1e-2 for s in shapes]
        for p, g, acc in zip(params, grads, sums):
            p.grad = g.clone()
            acc[0] += g.double() @ g.double().T
            acc[1] += g.double().T @ g.double()
        gm.update_curvature()
    for prec, acc in zip(gm.preconditioners, sums):
        for stat, ref in zip(prec.statistics, acc):
            assert relerr(stat, ref) < 1e-5, relerr(stat, ref)
    gm.update_preconditioner()
    for prec, acc in zip(gm.preconditioners, sums):
        for stat, root, ref in zip(prec.statistics, prec.preconditioners, acc):
            lam_max = float(torch.linalg.eigvalsh(ref)[-1])
            ridge = float((stat.double() - ref).diagonal().mean())      # the root computation leaves its ridge behind
            print(f'  n={stat.shape[0]}: ridge read back from the diagonal off by {abs(ridge - 1e-6 * lam_max) / (1e-6 * lam_max):.3f} of it',
                  flush=True)
            assert abs(ridge - 1e-6 * lam_max) < 0.1 * 1e-6 * lam_max
            exact = _closed_form_root(stat, 4)
            assert exact is not None and relerr(root, exact) < 5e-3, relerr(root, exact)
    gm.precondition()
    for prec, g, p in zip(gm.preconditioners, grads, params):
        ref = prec.preconditioners[0].double().T @ g.double() @ prec.preconditioners[1].double()
        assert relerr(p.grad, ref) < 1e-4


def test_shampoo_gpt2_small_full_decoder_bf16_real_gradients():
    """The transformer configuration as bench.py runs it: the 12-layer GPT-2-small-shaped decoder, 8 x 1024 random
    tokens, bf16 autocast, epsilon 1e-6, statistics and roots from the REAL gradients of two steps.  After one or two
    steps every statistic is rank deficient (a 768 x 2304 gradient leaves at least 1536 zero eigenvalues on its
    long side), so after the ridge cond = 1e6: the regime in which the coupled Newton iteration is slow and no fp32
    root is accurate.  Checked: every statistic against the fp64 sums of products of the captured gradients (1e-5);
    the roots of the 768-wide statistics of two blocks against the CPU oracle run on the same statistic with the same
    start vector, both measured against the fp64 closed form; one root of each larger size (2304, 3072, 1024) against
    the fp64 closed form; every preconditioned gradient against P_L^T G P_R in fp64 from the stored roots (1e-3)."""
    torch.manual_seed(13)
    model = bench_models.gpt2_small().cuda()
    x = torch.randint(0, 50257, (8, 1024)).cuda()
    t = torch.randint(0, 50257, (8 * 1024,)).cuda()
    gm = ShampooGradientMaker(model, PreconditioningConfig(damping=1e-6, curvature_upd_interval=1,
                                                           preconditioner_upd_interval=1))
    gen = torch.Generator().manual_seed(14)
    starts = {}

    def start_vectors(count, n, dev):
        v = torch.rand(count, n, generator=gen) * 2 - 1
        starts[n] = v
        return v.to(dev)
    gm.start_vector_fn = start_vectors

    def fwd(inp):
        with torch.autocast('cuda', dtype=torch.bfloat16):
            return model(inp).float()

    def token_loss(y, target):
        return F.cross_entropy(y.reshape(-1, y.shape[-1]), target)

    precs = gm.preconditioners
    assert len(precs) == 49
    sums = [[torch.zeros(n, n, dtype=torch.float64, device='cuda') for n in pc.param.shape] for pc in precs]
    opt = torch.optim.SGD([p for p in model.parameters() if p.requires_grad], lr=1e-3)
    for step in range(2):
        opt.zero_grad(set_to_none=True)
        gm.setup_loss_call(token_loss, gm.setup_model_call(fwd, x), t)
        print(f'shampoo gpt2 full step {step}', flush=True)
        # the template of forward_and_backward(), one phase at a time
        gm.forward()
        gm.backward()
        raw = [pc.param.grad.detach().clone() for pc in precs]
        for g, acc in zip(raw, sums):
            acc[0] += g.double() @ g.double().T
            acc[1] += g.double().T @ g.double()
        before = [[s_.clone() for s_ in pc.statistics] for pc in precs] if step == 1 else None
        gm.update_curvature()
        worst = 0.0
        for k, (pc, acc) in enumerate(zip(precs, sums)):
            for j, (stat, ref) in enumerate(zip(pc.statistics, acc)):
                if step == 0:
                    e = relerr(stat, ref + 1e-12 * torch.eye(ref.shape[0], dtype=torch.float64, device='cuda'))
                else:       # the first root update left its ridge in the stored statistic: compare the increment
                    g = raw[k].double()
                    inc = g @ g.T if j == 0 else g.T @ g
                    e = relerr(stat.double() - before[k][j].double(), inc)
                worst = max(worst, e)
                assert e < (1e-5 if step == 0 else 1e-4), (step, k, j, e)
        print(f'  statistics: worst relative error {worst:.1e}', flush=True)
        stats_in = [[s_.clone() for s_ in pc.statistics] for pc in precs]
        gm.update_preconditioner()
        iters = {key: st[:, 2].max().item() for key, st in gm.last_root_stats.items()}
        print(f'  Newton iterations (max per size group): {iters}', flush=True)
        # roots of 768-wide statistics against the CPU oracle on the same input (blocks 0 and 11: c_proj, both sides)
        members = {}
        for k, pc in enumerate(precs):
            for j, n in enumerate(pc.param.shape):
                members.setdefault(n, []).append((k, j))
        names = [n_ for n_, p_ in model.named_parameters() if p_.requires_grad and p_.ndim > 1]
        picks = [(k, j) for k, nm in enumerate(names) if nm in ('h.0.c_proj.weight', 'h.11.c_proj.weight') for j in (0, 1)]
        worst_ratio = 0.0
        for k, j in picks:
            n = precs[k].param.shape[j]
            slot = members[n].index((k, j))
            S = stats_in[k][j].cpu()
            root_ref, it_ref, err_ref = R.compute_power(S.clone(), 4, starts[n][slot].clone(), ridge_epsilon=1e-6)
            exact = _closed_form_root(precs[k].statistics[j], 4)      # the stored statistic holds the ridge now
            e_ref, e_mine = relerr(root_ref, exact), relerr(precs[k].preconditioners[j], exact)
            print(f'  root {names[k]} axis {j}: oracle {e_ref:.2e} ({it_ref} iterations), here {e_mine:.2e}', flush=True)
            worst_ratio = max(worst_ratio, e_mine / max(e_ref, 1e-30))
            assert e_mine <= max(4 * e_ref, 1e-4), (names[k], j, e_mine, e_ref)
        # one root of each larger size: distance from the fp64 closed form, and (first update; the CPU run of the
        # 3072-wide iteration takes a minute) the oracle's distance on the same input with the same start vector
        for n in (1024, 2304, 3072):
            k, j = members[n][0]
            exact = _closed_form_root(precs[k].statistics[j], 4)
            e = relerr(precs[k].preconditioners[j], exact)
            if step == 0:
                root_ref, it_ref, _ = R.compute_power(stats_in[k][j].cpu().clone(), 4, starts[n][0].clone(), ridge_epsilon=1e-6)
                e_ref = relerr(root_ref, exact)
                print(f'  root n={n} ({names[k]} axis {j}): oracle {e_ref:.2e} ({it_ref} iterations), here {e:.2e}', flush=True)
                assert e <= max(4 * e_ref, 1e-4), (n, e, e_ref)
            else:
                print(f'  root n={n} ({names[k]} axis {j}): distance from the fp64 closed form {e:.2e}', flush=True)
                assert e < 1e-2, (n, e)
        gm.precondition()
        worst = 0.0
        for pc, g in zip(precs, raw):
            ref = pc.preconditioners[0].double().T @ g.double() @ pc.preconditioners[1].double()
            e = relerr(pc.param.grad, ref)
            worst = max(worst, e)
            assert e < 1e-3, e
        print(f'  preconditioned gradients: worst relative error {worst:.1e}', flush=True)
        gm.state['step'] += 1
        opt.step()


def test_state_dict_resume_continues_the_run():
    """Save after three of six steps (step + statistics + inverse roots of every parameter), load into a fresh
    maker on a fresh copy of the model, continue: roots are taken every 4th step, so steps 3 precondition with
    loaded roots and the root update of step 4 works on statistics that were accumulated across the save."""
    import io
    torch.manual_seed(31)
    data = [(torch.randn(16, 12).cuda(), torch.randint(5, (16,)).cuda()) for _ in range(6)]

    def net():
        torch.manual_seed(32)
        return nn.Sequential(nn.Linear(12, 16), nn.ReLU(), nn.Linear(16, 8), nn.ReLU(), nn.Linear(8, 5)).cuda()

    def make(model):
        config = PreconditioningConfig(damping=1e-6, curvature_upd_interval=1, preconditioner_upd_interval=4)
        gm = ShampooGradientMaker(model, config)
        gen = torch.Generator().manual_seed(33)
        gm.start_vector_fn = lambda count, n, device: (torch.rand(count, n, generator=gen) * 2 - 1).to(device)
        return gm, torch.optim.SGD(model.parameters(), lr=0.05), gen

    def step(model, gm, opt, x, t):
        opt.zero_grad(set_to_none=True)
        gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(model, x), t)
        gm.forward_and_backward()
        grads = [p.grad.clone() for p in model.parameters()]
        opt.step()
        return grads

    model = net()
    gm, opt, gen = make(model)
    straight = [step(model, gm, opt, x, t) for x, t in data]
    model = net()
    gm, opt, gen = make(model)
    resumed = [step(model, gm, opt, x, t) for x, t in data[:3]]
    buf = io.BytesIO()
    torch.save({'model': model.state_dict(), 'shampoo': gm.state_dict(), 'rng': gen.get_state()}, buf)
    del model, gm, opt
    buf.seek(0)
    ckpt = torch.load(buf, weights_only=True)
    model = net()
    model.load_state_dict(ckpt['model'])
    gm, opt, gen = make(model)
    gen.set_state(ckpt['rng'])
    gm.load_state_dict(ckpt['shampoo'])
    assert gm.state['step'] == 3 and len(ckpt['shampoo']['shampoo']) == 3
    resumed += [step(model, gm, opt, x, t) for x, t in data[3:]]
    for k, (a, b) in enumerate(zip(straight, resumed)):
        for ga, gb in zip(a, b):
            assert torch.equal(ga, gb), f'step {k}'


# A matrix has the same bits whichever launch shape its products take: alone (32 x 32 fp32 tiles; 64 x 64 plane tiles by 16
# waves), beside planes (64 x 64 fp32 tiles by 16 waves), in a call of more tiles than CUs (8 waves); sizes around the chunks of 128 k
# (fp32) and 256 k (planes), with and without fp16 planes.
@pytest.mark.parametrize('p,eps', [(4, 1e-6), (2, 1e-6), (1, 1e-6), (3, 0.0)])
def test_roots_have_the_same_bits_in_every_launch_shape(p, eps):
    from asdl_amd import kernels as K
    sizes = [3, 31, 33, 127, 128, 129, 257, 385, 511, 512, 513, 769, 1025]
    g = torch.Generator().manual_seed(p)
    stats, starts = {}, {}
    for n in sizes:
        x = torch.randn(2, n + 20, n, generator=g) * torch.logspace(0, -1, n)
        stats[n], starts[n] = x.transpose(1, 2) @ x / n, torch.rand(2, n, generator=g) * 2 - 1

    def roots(*take):
        items = [(stats[n][:b].cuda(), p, starts[n][:b].cuda(), None) for n, b in take]
        return {n: (out[0].cpu(), st[0].cpu()) for (n, _), (out, st) in zip(take, K.inv_root_group(items, eps))}
    alone = {n: roots((n, 1))[n] for n in sizes}
    many = roots(*[(n, 2) for n in sizes])
    few = [roots((n, 1), (512, 1)) for n in sizes if n < 512]
    for n, (root, st) in alone.items():
        assert torch.isfinite(root).all() and int(st[2]) > 0
        assert torch.equal(root, many[n][0]) and torch.equal(st, many[n][1]), n
    for got in few:
        for n, (root, _) in got.items():
            assert torch.equal(root, alone[n][0]), n


@pytest.mark.parametrize("widths", [(5, 3), (64, 65, 1), (784, 512, 512, 10), (33, 1000, 7)])
def test_small_matrices_precondition_in_two_launches(widths):
    torch.manual_seed(0)
    model = nn.Sequential(*(nn.Linear(a, b) for a, b in zip(widths, widths[1:])), nn.Unflatten(1, (1, widths[-1], 1)),
                          nn.Conv2d(1, 2, 1)).cuda()
    maker = ShampooGradientMaker(model, PreconditioningConfig(damping=1e-6))
    expected = []
    for pc in maker.preconditioners:
        for q in pc.preconditioners:
            x = torch.randn_like(q)
            q.copy_(x @ x.T / len(x) + torch.eye(len(x), device="cuda"))
            q.copy_(0.5 * (q + q.T))
        pc.param.grad = torch.randn_like(pc.param)
        g = pc.param.grad.double()
        for q in pc.preconditioners:
            g = torch.tensordot(g, q.double(), dims=([0], [0]))
        expected.append(g)
    maker.precondition()
    for pc, g in zip(maker.preconditioners, expected):
        assert relerr(pc.param.grad, g) < 1e-5


def test_models_whose_products_go_to_the_grouped_path_are_not_asked_at_every_step(monkeypatch):
    """The sizes decide between the two-launch form and the split products (one rule, the library's): a declined model pays for the
    question once, without a call that walks its gradients or takes a workspace."""
    model = nn.Sequential(nn.Linear(1440, 1440), nn.Linear(1440, 1440)).cuda()
    assert not K.kron_precond_deep_pays([(1440, 1440)] * 2) and K.kron_precond_deep_pays([(512, 784), (512, 512), (10, 512)])
    maker = ShampooGradientMaker(model, PreconditioningConfig(damping=1e-6))
    calls = []
    monkeypatch.setattr(K, 'kron_precond_deep', lambda *a, **k: calls.append(a))
    for _ in range(2):
        for pc in maker.preconditioners:
            pc.param.grad = torch.randn_like(pc.param)
        expected = [pc.param.grad.clone() for pc in maker.preconditioners]
        maker.precondition()                     # (the preconditioners are identities)
        assert not calls
        assert all(relerr(pc.param.grad, g) < 1e-5 for pc, g in zip(maker.preconditioners, expected))


def test_inv_root_lanczos_on_half_the_statistics():
    """The Lanczos steps of 128 MB of statistics read the lower triangles by tiles, here of ragged sizes, against the same statistics in
    calls small enough for whole rows."""
    gen = torch.Generator('cuda').manual_seed(7)
    items = []
    for n, batch in ((2817, 4), (1700, 2), (513, 40), (65, 3), (256, 2)):
        x = torch.randn(batch, 2 * n, n, device='cuda', generator=gen) * torch.logspace(0, -2, n, device='cuda')
        S = torch.stack([m.t() @ m for m in x])
        S = torch.tril(S) + torch.tril(S, -1).transpose(1, 2)
        items.append((S.contiguous(), 4, torch.rand(batch, n, device='cuda', generator=gen), None))
    def halves(batches):
        n, b = [S.shape[1] for S, *_ in items], batches
        return _lib.load().ak_inv_root_lanczos_halves((ctypes.c_int64 * len(n))(*n), (ctypes.c_int * len(b))(*b), len(n))
    assert halves([S.shape[0] for S, *_ in items]) == 1 and halves([1] * len(items)) == 0
    together = K.inv_root_group([(S.clone(), p, v, out) for S, p, v, out in items], 1e-6)
    for (S, p, v, _), (out, stats) in zip(items, together):
        for z in range(0, S.shape[0], 7):
            one, alone = K.inv_root_group([(S[z:z + 1].clone(), p, v[z:z + 1], None)], 1e-6)[0]
            # the largest eigenvalue: T's entries round in another order, by a few 2^-24 a step
            assert float((stats[z, 0] - alone[0, 0]).abs() / alone[0, 0].abs()) < 32 * 4 * 2.0 ** -24
            root = out[z].double()
            for _ in range(2):
                root = root @ root
            exact = torch.linalg.inv(S[z].double() + 1e-6 * float(alone[0, 0]) * torch.eye(S.shape[1], device='cuda', dtype=torch.float64))
            own = one[0].double()
            for _ in range(2):
                own = own @ own
            assert float((root - exact).norm()) <= 1.5 * float((own - exact).norm()) + 1e-6 * float(exact.norm())
