"""Off-diagonal pair blocks of the pair-major Schur complement: one wave or one workgroup per pair, against the sum
of the products in 64 bits."""
import ctypes

import numpy as np
import pytest
import torch

DEV = 'cuda:0'
COUNTS = (1, 7, 8, 9, 0, 31, 32, 33, 63, 64, 65, 127, 255, 256, 257, 511, 513, 1200, 2, 3)


@pytest.mark.gpu
@pytest.mark.parametrize('real32', [False, True], ids=['fp64', 'fp32'])
@pytest.mark.parametrize('d', [1, 11, 15, 16, 23, 31])
def test_pair_blocks(d, real32):
    """Pairs of every length around the batch of 8 and the four parts of a workgroup (empty ones too), in a schedule
    that is not pair order, diagonal pairs among them left alone.  The sum of n products of rows of 3 has an error of
    at most (3 n + 4) roundings of the sum of magnitudes."""
    from blast3r_amd._lib import check, lib, stream_ptr
    from blast3r_amd.ba_solver import GaussNewtonSolver
    from blast3r_amd.synthetic import make_problem
    from blast3r_amd import cujac
    R, N = (torch.float32, np.float32) if real32 else (torch.float64, np.float64)
    eps = 6e-8 if real32 else 1.2e-16
    p = make_problem(0, n_frames=4, n_tracks=20).to(DEV)           # every other pointer of the call
    out = cujac.compute_residuals_with_rigs(p.infos, p.K, p.P_rig2cam, p.P_w2rig, p.z_coefs, p.pts3d, p.pids, p.pix2d,
                                            p.pix2d_std, p.pix2d_dep, True, 1e-2, 1.0, 50.0, 1.0)
    res, _, w = out.view(-1, 3, 3).unbind(dim=1)
    gs = GaussNewtonSolver(len(p.K), len(p.P_w2rig), p.n_imgs, p.n_tracks, DEV, dtype=R, path='pairmajor')
    J = gs.compute_jacobians(p.infos, p.K, p.P_rig2cam, p.P_w2rig, p.z_coefs, p.pts3d, p.pids, p.pix2d_std,
                             p.pix2d_dep, True, pix2d=p.pix2d,
                             hp=dict(weight_z=1e-2, pnorm=1.0, max_pix_err=50.0, huber_delta=1.0))
    a = gs.prepare(J, res, w)['args']

    rng = np.random.default_rng(d)
    n_runs, dp = 500, 16 if d <= 15 else 32
    V = np.zeros((n_runs, 3, dp), N)
    V[:, :, :d] = rng.normal(0, 1, (n_runs, 3, d))
    n_p = len(COUNTS)
    i1, i2 = np.arange(n_p), np.arange(n_p) + 1
    i2[[4, 7]] = i1[[4, 7]]                                        # diagonal pairs: not this kernel's
    tp = np.cumsum((0,) + COUNTS)
    term = rng.integers(0, n_runs, (tp[-1], 2))
    t = lambda x, dt=torch.int32: torch.as_tensor(np.ascontiguousarray(x), dtype=dt, device=DEV)
    keep = dict(pair_i1=t(i1), pair_i2=t(i2), term_ptr=t(tp), term=t(term), V=t(V, R), pair_sched=t(rng.permutation(n_p)))
    for k, x in keep.items():
        setattr(a, k, x.data_ptr())
    lay = a.lay
    lay.d, lay.hasK, lay.hasP, lay.hasZ, lay.C = d, int(d > 24), int(d > 24), 1, d - 8 * (d > 24)
    lay.off_tau, lay.off_zcf = 2 * lay.hasK, 2 * lay.hasK + 6 * lay.hasP
    a.n_pairs = n_p
    for n_terms in (0, int(tp[-1]), 0, 10 ** 9):                   # not known, as it is, and split whatever the size
        S = torch.full((n_p, d, d), 7.0, dtype=R, device=DEV)
        a.S_pairs, a.n_terms = S.data_ptr(), n_terms
        check(lib().ba_pm_linearize_stage(ctypes.byref(a), 1, stream_ptr(DEV)))
        torch.cuda.synchronize()
        S = S.cpu().double().numpy()
        for q in range(n_p):
            if i1[q] == i2[q]:
                assert (S[q] == 7).all()
                continue
            A, B = (V[term[tp[q]:tp[q + 1], s], :, :d].astype(np.float64).reshape(-1, d) for s in (0, 1))
            bound = (3 * COUNTS[q] + 4) * eps * (np.abs(A).T @ np.abs(B))
            assert (np.abs(S[q] + A.T @ B) <= bound).all(), (q, n_terms)
