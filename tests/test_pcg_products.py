"""The forms of the reduced system's conjugate gradient against each other and against the oracle's loop.

A random block-sparse system at image level (unknowns that several images share, parameters that are no
unknown, images without partners) goes through every form that accepts it; few iterations, so that the
iterates agree to rounding."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import solver as osol

DEV = 'cuda:0'


def block_system(m, d, shared, seed, density=0.5, dtype=np.float64, drop=0.0):
    """m images of d parameters, the first `shared` of them one unknown for all images; each image pair is a
    block with probability `density`; a share `drop` of the other parameters is no unknown.  Returns the plan
    arrays and the dense system at unknown level (S without damping, rhs, camera diagonal)."""
    rng = np.random.Generator(np.random.PCG64(seed))
    pairs = [(i, j) for i in range(m) for j in range(i, m) if i == j or rng.random() < density]
    full = rng.normal(0, 0.3, (m * d, m * d))
    full = full @ full.T / (m * d) + np.diag(rng.uniform(1, 3, m * d))
    S_pairs = np.stack([full[i * d:(i + 1) * d, j * d:(j + 1) * d] for i, j in pairs]).astype(dtype)
    umap = np.full((m, d), -1, dtype=np.int64)
    umap[:, :shared] = np.arange(shared)
    n = shared
    for i in range(m):
        for j in range(shared, d):
            if rng.random() >= drop:
                umap[i, j] = n
                n += 1
    flat = umap.reshape(-1)
    P = np.zeros((m * d, n))
    ok = flat >= 0
    P[np.nonzero(ok)[0], flat[ok]] = 1
    img = np.zeros((m * d, m * d))
    for b, (i, j) in zip(S_pairs.astype(np.float64), pairs):
        img[i * d:(i + 1) * d, j * d:(j + 1) * d] = b
        img[j * d:(j + 1) * d, i * d:(i + 1) * d] = b.T
    rows = [[] for _ in range(m)]
    for q, (i, j) in enumerate(pairs):
        rows[i].append(q << 1)
        if j != i:
            rows[j].append((q << 1) | 1)
    e = rng.normal(0, 1, (m, d)).astype(dtype)
    dg = (rng.uniform(0.5, 2, (m, d))).astype(dtype)
    return dict(m=m, d=d, n=n, pairs=pairs, S_pairs=S_pairs, umap=umap, rows=rows, e=e, dg=dg,
                S=P.T @ img @ P, rhs=P.T @ e.reshape(-1).astype(np.float64), diag=P.T @ dg.reshape(-1).astype(np.float64))


def pcg_args(sysm, maxiter, tol, real32, dampen=1e-3):
    """ba_pcg_args of a block_system with its workspace (row copies included), and the tensors it points into."""
    from blast3r_amd._lib import PCG_BLOCK, PCG_LONG_LIST, BaPcgArgs, lib
    m, d, n, pairs, rows = (sysm[k] for k in ('m', 'd', 'n', 'pairs', 'rows'))
    R = torch.float32 if real32 else torch.float64
    i32 = torch.int32
    t = lambda a, dt: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device=DEV)
    flat = sysm['umap'].reshape(-1)
    valid = np.nonzero(flat >= 0)[0]
    order = np.argsort(flat[valid], kind='stable')
    counts = np.bincount(flat[valid], minlength=n)
    inv_ptr = np.concatenate([[0], np.cumsum(counts)])
    long_u = np.nonzero(counts > PCG_LONG_LIST)[0]
    nblk = (n + PCG_BLOCK - 1) // PCG_BLOCK
    long_ptr = np.searchsorted(long_u, np.arange(nblk + 1) * PCG_BLOCK)
    long_idx = np.full(n, -1)
    long_idx[long_u] = np.arange(len(long_u)) - long_ptr[long_u // PCG_BLOCK]
    row_ptr = np.cumsum([0] + [len(r) for r in rows])
    n_ent, gw = int(row_ptr[-1]), 16 if d <= 16 else 32
    keep = dict(umap=t(sysm['umap'], i32), inv_ptr=t(inv_ptr, i32), inv_src=t(valid[order], i32), leaf=t(np.zeros(n), i32),
                row_ptr=t(row_ptr, i32), row_ent=t(np.concatenate([np.array(r, dtype=np.int64) for r in rows]), i32),
                pair_i1=t([q[0] for q in pairs], i32), pair_i2=t([q[1] for q in pairs], i32),
                S_pairs=t(sysm['S_pairs'], R), e_img=t(sysm['e'], R), dg_img=t(sysm['dg'], R),
                long_u=t(long_u if len(long_u) else np.zeros(1), i32), long_ptr=t(long_ptr, i32), long_idx=t(long_idx, i32),
                row_u=torch.zeros(n_ent * gw, dtype=i32, device=DEV), istate=torch.zeros(8, dtype=i32, device=DEV))
    for name, size in dict(rhs=n, diagA=n, damp=n, x=n, xbest=n, r=n, z=n, p=2 * n, y_img=m * d, img_part=m,
                           partials=int(lib().ba_pcg_partials_size(n)), state=16, S_rows=n_ent * d * d).items():
        keep[name] = torch.zeros(size, dtype=R, device=DEV)
    pa = BaPcgArgs()
    pa.n_u, pa.n_imgs, pa.d, pa.real32 = n, m, d, int(real32)
    pa.dampen, pa.adaptive, pa.maxiter, pa.tol = dampen, 0, int(maxiter), float(tol)
    pa.n_row_ent, pa.n_long = n_ent, len(long_u)
    for name, v in keep.items():
        setattr(pa, name, v.data_ptr())
    return pa, keep


def oracle_iterate(sysm, maxiter, tol, dampen=1e-3):
    S = torch.from_numpy(sysm['S']) + dampen * torch.eye(sysm['n'], dtype=torch.float64)
    dA = torch.from_numpy(sysm['diag']) + dampen
    x, it, conv = osol.pcg(lambda v: S @ v, torch.from_numpy(sysm['rhs']), M_mv=lambda v: v / dA, tol=tol, maxiter=maxiter)
    return x, it, conv


SHAPES = [(1, 13, 2), (3, 1, 0), (7, 13, 2), (40, 13, 2), (41, 16, 0), (300, 9, 0), (515, 13, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize('real32', [False, True], ids=['fp64', 'fp32'])
@pytest.mark.parametrize('m,d,shared', SHAPES)
def test_pair_block_product(m, d, shared, real32):
    """ba_pcg_solve_pairs_range against ba_pcg_solve and the oracle's loop after 8 updates: the products differ
    in the order of their sums only.  A sum of k terms is off by at most k eps of its terms' magnitudes; 8
    updates on a system of condition number below 100 keep that below 1e4 eps."""
    from blast3r_amd._lib import BaPcgPairs, check, lib, stream_ptr
    eps = 1.2e-7 if real32 else 2.3e-16
    for drop in (0.0, 0.3):
        sysm = block_system(m, d, shared, seed=m * 100 + d, density=0.6 if m < 100 else 0.03, drop=drop,
                            dtype=np.float32 if real32 else np.float64)
        print(f'pair-block product m={m} d={d} shared={shared} drop={drop} n={sysm["n"]}', flush=True)
        if sysm['n'] == 0:
            continue
        pa, keep = pcg_args(sysm, 8, 0.0, real32)
        check(lib().ba_pcg_solve(ctypes.byref(pa), stream_ptr(DEV)))
        x_rows, ist_rows = keep['x'].clone(), keep['istate'].cpu()
        R, gw = keep['x'].dtype, 16
        t = torch.full((len(sysm['pairs']), gw), float('nan'), dtype=R, device=DEV)
        p_img = torch.full((m, gw), float('nan'), dtype=R, device=DEV)
        up = torch.full((m + 1,), -7, dtype=torch.int32, device=DEV)
        pw = BaPcgPairs(t=t.data_ptr(), p_img=p_img.data_ptr(), up_ptr=up.data_ptr(), n_pairs=len(sysm['pairs']))
        pa.S_rows = pa.row_u = None                    # not used by this form
        for _ in range(2):                             # a second solve starts afresh
            check(lib().ba_pcg_solve_pairs_range(ctypes.byref(pa), ctypes.byref(pw), 0, 8, 1, None, stream_ptr(DEV)))
        torch.cuda.synchronize()
        x, it, conv = oracle_iterate(sysm, 8, 0.0)
        for got in (x_rows, keep['x']):
            assert float((got.cpu().double() - x).norm() / x.norm()) < 1e4 * eps
        assert keep['istate'].cpu()[2:6].tolist() == ist_rows[2:6].tolist()


@pytest.mark.gpu
def test_pair_block_product_stops_where_the_loop_converges():
    """The same outcome and iterate as the row copies where the loop converges before its cap, launched in
    ranges whose stopped flag the host reads."""
    from blast3r_amd._lib import BaPcgPairs, check, lib, stream_ptr
    sysm = block_system(40, 13, 2, seed=5)
    pa, keep = pcg_args(sysm, 60, 1e-10, False)
    check(lib().ba_pcg_solve(ctypes.byref(pa), stream_ptr(DEV)))
    x_rows, ist_rows = keep['x'].clone(), keep['istate'].cpu()
    t = torch.zeros((len(sysm['pairs']), 16), dtype=torch.float64, device=DEV)
    p_img = torch.zeros((40, 16), dtype=torch.float64, device=DEV)
    up = torch.zeros(41, dtype=torch.int32, device=DEV)
    flag = torch.zeros(1, dtype=torch.int32, device=DEV)
    pw = BaPcgPairs(t=t.data_ptr(), p_img=p_img.data_ptr(), up_ptr=up.data_ptr(), n_pairs=len(sysm['pairs']))
    st = stream_ptr(DEV)
    end = 0
    for it0 in range(0, 60, 20):
        check(lib().ba_pcg_solve_pairs_range(ctypes.byref(pa), ctypes.byref(pw), it0, it0 + 20, 0,
                                             ctypes.c_void_p(flag.data_ptr()), st))
        end = it0 + 20
        if int(flag):
            break
    check(lib().ba_pcg_solve_pairs_range(ctypes.byref(pa), ctypes.byref(pw), end, end, 1, None, st))
    ist = keep['istate'].cpu()
    assert int(ist_rows[3]) == 1 and int(ist[3]) == 1 and abs(int(ist[2]) - int(ist_rows[2])) <= 1 and end < 60
    # both meet ||r|| <= 1e-10 ||b|| on a system whose smallest eigenvalue is about 1
    assert float((keep['x'] - x_rows).norm() / x_rows.norm()) < 1e-9


@pytest.mark.parametrize('kind', ['batched', 'pairmajor'])
def test_planners_order_the_pairs_by_image(kind):
    """What the product by pair blocks relies on: pairs ascend in (i1, i2) with i1 <= i2, and a row's list holds
    its pairs in that order, so the pairs whose second image it is come first."""
    from blast3r_amd.plan import BAPlan, PMPlan
    from blast3r_amd.synthetic import make_problem
    for cfg, nf, nt in ((0, 9, 200), (1, 30, 300), (2, 40, 900), (3, 24, 500)):
        p = make_problem(cfg, n_frames=nf, n_tracks=nt)
        plan = (BAPlan if kind == 'batched' else PMPlan)(p.infos, p.pids, p.n_tracks, device='cpu')
        n = plan.scalars['n_pairs']
        i1, i2 = (plan.host[k][:n].astype(np.int64) for k in ('pair_i1', 'pair_i2'))
        assert (i1 <= i2).all() and (np.diff(i1 * p.n_imgs + i2) > 0).all()
        row_ptr, ent = plan.host['row_ptr'], plan.host['row_ent']
        for i in range(p.n_imgs):
            row = ent[row_ptr[i]:row_ptr[i + 1]]
            assert (np.diff(row) > 0).all() and (np.diff(row & 1) <= 0).all()
            assert ((np.where(row & 1, i2[row >> 1], i1[row >> 1])) == i).all()


def resident_args(sysm, pa, limit=200_000_000, n_cu=256, m=None):
    """ba_pcg_resident for a block_system, on m images per workgroup (None: the plan's choice); (res, tensors) or None
    where the resident solve does not apply."""
    from blast3r_amd._lib import BaPcgResident, lib
    flat = sysm['umap'].reshape(-1)
    counts = np.bincount(flat[flat >= 0], minlength=sysm['n'])
    shared = np.nonzero(counts >= 2)[0]
    rp = np.cumsum([0] + [len(r) for r in sysm['rows']]).astype(np.int32)
    blk, col = ctypes.c_int32(0), ctypes.c_int32(0)
    plan = lambda cu: lib().ba_pcg_resident_plan(rp.ctypes.data_as(ctypes.c_void_p), sysm['m'], sysm['d'], pa.real32,
                                                 len(shared), cu, ctypes.byref(blk), ctypes.byref(col))
    got = plan(n_cu)
    if got < 1:
        return None
    if m is not None:
        got = min(m, got)
        blk.value = max(int(rp[min(i + got, sysm['m'])] - rp[i]) for i in range(0, sysm['m'], got))
        col.value = min(blk.value + got, sysm['m'])
    nw = int(lib().ba_pcg_resident_words(sysm['m'], sysm['d'], pa.real32, got))
    words = torch.full((nw,), -1, dtype=torch.int64, device=DEV)
    sh = torch.as_tensor(shared if len(shared) else np.zeros(1), dtype=torch.int32, device=DEV)
    res = BaPcgResident(words=words.data_ptr(), shared_u=sh.data_ptr(), n_shared=len(shared), m=got, max_blk=blk.value,
                        max_col=col.value, limit=limit)
    return res, (words, sh)


RESIDENT = [(1, 13, 2, None), (2, 1, 0, 1), (7, 13, 2, None), (7, 13, 2, 3), (40, 13, 2, 1), (61, 10, 2, None), (256, 9, 0, 1),
            (250, 13, 2, None), (40, 16, 2, None), (33, 17, 2, None), (30, 25, 2, None), (29, 22, 0, None), (20, 32, 0, 1), (300, 5, 0, 2), (256, 13, 2, 1), (250, 9, 2, None)]


@pytest.mark.gpu
@pytest.mark.parametrize('real32', [False, True], ids=['fp64', 'fp32'])
@pytest.mark.parametrize('m,d,shared,per', RESIDENT)
def test_resident_solve(m, d, shared, per, real32):
    """ba_pcg_solve_resident against the oracle's loop after 8 updates (tolerance as above) and, to the end of the loop,
    against ba_pcg_solve: the same outcome.  One and several workgroups, ragged last ones, one image per workgroup
    (every column from another workgroup), shared unknowns and parameters that are none, twice in a row."""
    from blast3r_amd._lib import check, lib, stream_ptr
    eps = 1.2e-7 if real32 else 2.3e-16
    for drop in (0.0, 0.3):
        sysm = block_system(m, d, shared, seed=m * 100 + d, density=0.6 if m < 100 else 0.04, drop=drop,
                            dtype=np.float32 if real32 else np.float64)
        if sysm['n'] == 0:
            continue
        for maxiter, tol in ((8, 0.0), (100, 1e-4)):
            pa, keep = pcg_args(sysm, maxiter, tol, real32)
            got = resident_args(sysm, pa, m=per)
            assert got is not None
            res, hold = got
            print(f'resident m={m} d={d} shared={res.n_shared} per={res.m} blk={res.max_blk} col={res.max_col} drop={drop} '
                  f'n={sysm["n"]} maxiter={maxiter}', flush=True)
            check(lib().ba_pcg_solve(ctypes.byref(pa), stream_ptr(DEV)))
            x_rows, ist_rows = keep['x'].clone(), keep['istate'].cpu()
            keep['x'].fill_(float('nan'))
            for _ in range(2):
                check(lib().ba_pcg_solve_resident(ctypes.byref(pa), ctypes.byref(res), stream_ptr(DEV)))
            torch.cuda.synchronize()
            ist = keep['istate'].cpu()
            assert int(ist[6]) == 0
            x, _, _ = oracle_iterate(sysm, maxiter, tol)
            if maxiter == 8:
                assert float((keep['x'].cpu().double() - x).norm() / x.norm()) < 1e4 * eps
                assert ist[:6].tolist() == ist_rows[:6].tolist()
            else:                                      # both meet ||r|| <= tol ||b||; the eigenvalues lie around 1
                assert int(ist[3]) == int(ist_rows[3]) == 1 and abs(int(ist[2]) - int(ist_rows[2])) <= 1
                assert float((keep['x'].cpu().double() - x).norm() / x.norm()) < 10 * tol


@pytest.mark.gpu
@pytest.mark.parametrize('m,d,shared', [(7, 13, 2), (61, 10, 2), (250, 13, 2), (33, 17, 2)])
def test_resident_solve_with_sizes_too_small(m, d, shared):
    """max_blk or max_col one less than the rows need: the kernel gives up before it writes either array, in whichever
    workgroups it is too little for (the others' waits end at their limit); with exactly what they need, the plan's
    solve bit for bit."""
    from blast3r_amd._lib import check, lib, stream_ptr
    sysm = block_system(m, d, shared, seed=m * 100 + d, density=0.6 if m < 100 else 0.04)
    pa, keep = pcg_args(sysm, 8, 0.0, False)
    res, hold = resident_args(sysm, pa)
    blk, per = res.max_blk, res.m
    cols = lambda g: {x for i, j in sysm['pairs'] for x in (i, j) if g[0] <= i < g[1] or g[0] <= j < g[1]} | set(range(*g))
    col = max(len(cols((i, min(i + per, m)))) for i in range(0, m, per))
    solve = lambda: check(lib().ba_pcg_solve_resident(ctypes.byref(pa), ctypes.byref(res), stream_ptr(DEV)))
    solve()
    x = keep['x'].clone()
    res.limit = 1_000_000                              # 10 ms
    for max_blk, max_col in ((blk, col - 1), (blk - 1, col), (blk, 1), (1, col), (blk, col)):
        few = (max_blk < blk and blk > 1) or max_col < col
        if max_blk < 1:
            continue
        print(f'resident sizes m={m} d={d} blk={max_blk} of {blk} col={max_col} of {col}', flush=True)
        res.max_blk, res.max_col = max_blk, max_col
        keep['x'].zero_()
        solve()
        assert bool(keep['istate'][6]) == few
        assert few or torch.equal(keep['x'], x)


@pytest.mark.gpu
def test_resident_solve_gives_up_and_the_launch_sequence_takes_over(monkeypatch):
    """A resident loop whose waits are limited to nothing leaves at once, says so, and solve_delta returns the launch
    sequence's step; with the usual limit it returns the same step to rounding."""
    from blast3r_amd import ba_solver, engine
    from blast3r_amd.synthetic import make_problem
    p = make_problem(0, n_frames=12, n_tracks=600)
    kw = dict(dtype=torch.float64, weight_z=1e-2, huber_delta=2.0)
    steps = {}
    for limit in (0, ba_solver.RESIDENT_LIMIT):
        monkeypatch.setattr(ba_solver, 'RESIDENT_LIMIT', limit)
        g = p.to(DEV)                                  # other tensors: another plan
        for _ in range(2):
            info = {}
            engine._lm_step(**g.lm_inputs(), **kw, info=info)
            assert info['solver'].last['pcg_resident'] == (limit > 0)
            assert info['pcg_istate'].cpu()[2] > 0 and info['pcg_istate'].cpu()[6] == 0
        steps[limit] = info['delta']
    a, b = steps.values()
    assert torch.isfinite(a).all() and float((a - b).norm() / b.norm()) < 1e-4


def test_a_device_whose_resident_solves_give_up_is_left_to_the_launches(monkeypatch):
    """New structures, as an online reconstruction makes them, on a device whose CUs another process holds: after three
    waits in vain the device's solves go by launches, with a try now and then, and back once one succeeds; other devices
    are not concerned.  The library is a stub, so that this runs anywhere."""
    from types import SimpleNamespace

    from blast3r_amd import ba_solver
    stub = SimpleNamespace(ba_pcg_resident_plan=lambda *a: 1, ba_pcg_resident_words=lambda *a: 8,
                           ba_pcg_solve_resident=lambda *a: 0)
    monkeypatch.setattr(ba_solver, 'lib', lambda: stub)
    monkeypatch.setattr(ba_solver, 'ptr', lambda t: t.data_ptr())
    monkeypatch.setattr(torch.cuda, 'is_current_stream_capturing', lambda: False)
    monkeypatch.setattr(torch.cuda, 'get_device_properties', lambda d: SimpleNamespace(multi_processor_count=256))
    pa = SimpleNamespace(maxiter=300, n_imgs=4, d=3, real32=0)
    plan = SimpleNamespace(host=dict(row_ptr=np.arange(5, dtype=np.int32)),
                           workspace=lambda name, shape, dtype: torch.zeros(shape, dtype=dtype))

    def solves(device, n, gave_up, um=None):
        """The number of n solves, each of a new structure (or of um), that waited."""
        tries = 0
        for _ in range(n):
            s = ba_solver.GaussNewtonSolver(1, 4, 4, 10, device)
            u = dict(n_shared=0, shared_u=torch.zeros(1, dtype=torch.int32)) if um is None else um
            if s._run_resident(pa, u, plan, None):
                tries += 1
                assert s._resident_status(torch.tensor([0, 0, 5, 1, 5, 0, int(gave_up), 0]), u, pa) != gave_up
        return tries

    one = dict(n_shared=0, shared_u=torch.zeros(1, dtype=torch.int32))
    assert solves('cuda:6', 5, True, um=one) == 1      # one structure waits in vain once
    assert solves('cuda:6', 1, False) == 1             # and another one still tries
    for _ in range(2):
        assert solves('cuda:6', 3, True) == 3
        assert solves('cuda:6', 1000, True) <= 5
        assert solves('cuda:7', 4, False) == 4
        assert solves('cuda:6', 5000, False) > 0       # the CUs are free again
        assert solves('cuda:6', 10, False) == 10
    assert solves('cuda:6', 2, True) == 2
    assert solves('cuda:6', 3, False) == 3             # waits in a row count
