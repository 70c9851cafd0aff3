"""The batched Schur pass with each batch's chunks in parts against whole batches."""
import ctypes

import pytest
import torch

from helpers import opts

DEV = 'cuda:0'


def test_parts_rule():
    """Within 1 .. the longest batch, whole batches where these fill the chip, at most 8 items per CU."""
    from blast3r_amd._lib import lib
    rule = lib().ba_schur_parts
    for args in ((0, 0, 0, 256), (1, 1, 1, 256), (10 ** 6, 10 ** 7, 300, 256), (4, 10, 5, 0)):
        assert rule(*args) == 1
    assert rule(1, 14, 14, 256) == 14
    for nb in (1, 2, 3, 17, 95, 200, 255, 256, 257, 383, 600, 2048, 2049):
        for most in (1, 2, 50, 4000):
            for n in (nb, nb * most):
                p = rule(nb, n, most, 256)
                assert 1 <= p <= most and (p == 1 or p * nb <= 8 * 256)


def test_parts_need_the_slot_count():
    """Parts whose partials would all begin at the same place are refused on the host (before any pointer is looked at)."""
    from blast3r_amd._lib import BaLinArgs, lib
    a = BaLinArgs()
    a.L, a.n_chunks, a.n_batches = 4, 4, 2
    a.lay.d, a.lay.C, a.lay.off_tau, a.lay.off_zcf, a.lay.hasK, a.lay.hasP, a.lay.hasZ = 13, 5, 2, 8, 1, 1, 1
    for parts, n_slots, msg in ((2, 0, b'part count'), (2, -1, b'part count'), (2, 3, b'null pointer'),
                                (1, 0, b'null pointer'), (0, 0, b'null pointer')):
        a.parts, a.n_slots = parts, n_slots
        for call in (lambda: lib().ba_linearize_schur(ctypes.byref(a), None),
                     lambda: lib().ba_linearize_stage(ctypes.byref(a), 1, None)):
            assert call() != 0 and msg in lib().ba_last_error(), (parts, n_slots)
    a.parts, a.n_slots, a.n_chunks, a.n_batches = 2, -1, 0, 0
    assert lib().ba_linearize_stage(ctypes.byref(a), 1, None) != 0 and b'part count' in lib().ba_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float64, torch.float32], ids=['fp64', 'fp32'])
@pytest.mark.parametrize('cfg,nf,nt,flags', [(0, 8, 40, {}), (0, 8, 300, {}), (2, 24, 800, {}), (2, 60, 6000, {}),
                                             (2, 24, 800, dict(optim_K=False)), (2, 24, 800, dict(optim_P=False))])
def test_parts_against_whole_batches(cfg, nf, nt, flags, dtype):
    """Parts down to one chunk and past the chunk count (empty parts), with and without the work queue: the same blocks
    but for the order of the additions, the same bits in any order of the work items, and nothing left over in the
    workspace that a part does not write."""
    from blast3r_amd import cujac
    from blast3r_amd._lib import check, lib
    from blast3r_amd.ba_solver import GaussNewtonSolver
    from blast3r_amd.synthetic import make_problem
    p = make_problem(cfg, n_frames=nf, n_tracks=nt).to(DEV)
    o = opts(p)
    out = cujac.compute_residuals_with_rigs(p.infos, p.K, p.P_rig2cam, p.P_w2rig, p.z_coefs, p.pts3d, p.pids, p.pix2d,
                                            p.pix2d_std, p.pix2d_dep, True, o['weight_z'], 1.0, o['clip_pix_err'],
                                            o['huber_delta'])
    res, _, w = out.view(-1, 3, 3).unbind(dim=1)
    hp = dict(weight_z=o['weight_z'], pnorm=1.0, max_pix_err=o['clip_pix_err'], huber_delta=o['huber_delta'])
    gs = GaussNewtonSolver(len(p.K), len(p.P_w2rig), p.n_imgs, p.n_tracks, DEV, dtype=dtype, path='batched')
    J = gs.compute_jacobians(p.infos, p.K, p.P_rig2cam, p.P_w2rig, p.z_coefs, p.pts3d, p.pids, p.pix2d_std,
                             p.pix2d_dep, True, pix2d=p.pix2d, hp=hp, **flags)
    ctx = gs.prepare(J, res, w)
    a, sc, d = ctx['args'], ctx['plan'].scalars, ctx['lay']['d']
    most = sc['max_chunks_per_batch']
    assert a.parts == lib().ba_schur_parts(sc['n_batches'], sc['n_chunks'], most,
                                           torch.cuda.get_device_properties(0).multi_processor_count)
    ctr, eps = a.work_ctr, 1.2e-7 if dtype == torch.float32 else 2.3e-16
    ref = None
    for parts in (0, 1, 2, 3, most, most + 2):
        got = []
        for queue in (ctr, None):
            print(f'schur parts={parts} queue={queue is not None} cfg={cfg} {sc["n_batches"]} batches, {most} chunks', flush=True)
            n = max(parts, 1)
            part = torch.full((n, sc['n_slots'], d, d), float('nan'), dtype=dtype, device=DEV)
            img = torch.full((n, sc['n_batches'], ctx['plan'].L, 2, d), float('nan'), dtype=dtype, device=DEV)
            a.parts, a.partials, a.img_partials, a.work_ctr = parts, part.data_ptr(), img.data_ptr(), queue
            for k in ('S_pairs', 'e_img', 'dg_img'):
                ctx[k].fill_(float('nan'))
            check(lib().ba_linearize_schur(ctypes.byref(a), ctx['stream']))
            for _ in range(2):                         # the reductions may be run again
                check(lib().ba_linearize_stage(ctypes.byref(a), 2, ctx['stream']))
            torch.cuda.synchronize()
            got.append([ctx[k].clone() for k in ('S_pairs', 'e_img', 'dg_img')])
        assert all(torch.equal(x, y) for x, y in zip(*got))
        if ref is None:
            ref = got[0]
        for x, y in zip(got[0], ref):
            assert torch.isfinite(x).all()
            # S = J^T J - V V^T: rounding grows with the terms before their difference; the parts sum the same
            # products, at most as many as the tracks, in another order
            assert float((x - y).abs().max()) <= 4 * nt * eps * float(ref[2].abs().max() + ref[1].abs().max() + ref[0].abs().max())
