"""Per-image sums of the pair-major pass, a wave taking 64 to 512 observations or runs by their number, against the
batched pass, which sums them otherwise."""
import pytest
import torch

from helpers import opts, rel_err

DEV = 'cuda:0'
SPANS = [(24, 800, 64), (60, 19_999, 64), (300, 190_001, 128), (300, 390_003, 256), (300, 590_001, 512)]


def span_of(n):
    """Items per wave: halved from 512 down to 64 while that leaves at most 8192 waves."""
    span = 512
    while span > 64 and n < span * 8192:
        span //= 2
    return span


def test_slot_sizes():
    """Slots: one per wave and one per image, and enough for any smaller number of items too, also where that takes
    shorter spans and so more waves: a buffer sized for the most items ever passed holds every call's."""
    from blast3r_amd._lib import lib
    slots = lambda n: lib().ba_pm_slot_doubles(n, 0, 11) // 256
    waves = lambda n: -(-n // span_of(n))
    assert slots(0) == 0 and slots(1) == 1 and slots(64) == 1 and slots(65) == 2
    assert slots(10 ** 9) == -(-10 ** 9 // 512)
    edges = [span * 8192 + e for span in (128, 256, 512, 1024) for e in (-64, -1, 0, 1, 63, 64)]
    most = 0
    for n in sorted(set(range(1, 400)) | {int(1.07 ** k) + e for k in range(90, 300) for e in (0, 1, 63)} | set(edges)):
        most = max(most, waves(n))
        assert slots(n) == most, n
    assert slots(2 ** 19) == 8192 and slots(2 ** 20) == slots(2 ** 23) == 16384 and slots(2 ** 23 + 1) == 16385
    assert {span_of(int(1.07 ** k)) for k in range(90, 300)} == {64, 128, 256, 512}
    assert lib().ba_pm_slot_doubles(1000, 7, 15) == 23 * 256 and lib().ba_pm_slot_doubles(1000, 7, 16) == 23 * 3 * 256


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float64, torch.float32], ids=['fp64', 'fp32'])
@pytest.mark.parametrize('nf,nt,span', SPANS)
def test_spans_against_batched(nf, nt, span, dtype):
    """Images that end within a span, spans that end within an image, the last one ragged: diag(H_cc) is the same sum in
    another order (n roundings of positive terms); the right-hand sides and S of the two fp64 passes, which also form the
    rows differently, agree to roundings times the condition of the point blocks (1e6 at most here)."""
    from blast3r_amd import cujac
    from blast3r_amd._lib import check, lib
    from blast3r_amd.ba_solver import GaussNewtonSolver
    from blast3r_amd.synthetic import make_problem
    p = make_problem(2, n_frames=nf, n_tracks=nt).to(DEV)
    n_obs = len(p.pids)
    assert span_of(n_obs) == span
    print(f'spans of {span}: {nf} images, {n_obs} observations', flush=True)
    o = opts(p)
    out = cujac.compute_residuals_with_rigs(p.infos, p.K, p.P_rig2cam, p.P_w2rig, p.z_coefs, p.pts3d, p.pids, p.pix2d,
                                            p.pix2d_std, p.pix2d_dep, True, o['weight_z'], 1.0, o['clip_pix_err'],
                                            o['huber_delta'])
    res, _, w = out.view(-1, 3, 3).unbind(dim=1)
    hp = dict(weight_z=o['weight_z'], pnorm=1.0, max_pix_err=o['clip_pix_err'], huber_delta=o['huber_delta'])
    got = {}
    for path in ('batched', 'pairmajor'):
        gs = GaussNewtonSolver(len(p.K), len(p.P_w2rig), p.n_imgs, p.n_tracks, DEV, dtype=dtype, path=path)
        J = gs.compute_jacobians(p.infos, p.K, p.P_rig2cam, p.P_w2rig, p.z_coefs, p.pts3d, p.pids, p.pix2d_std,
                                 p.pix2d_dep, True, pix2d=p.pix2d, hp=hp)
        ctx = gs.prepare(J, res, w)
        if path == 'pairmajor':                        # the slots that the waves leave: up to the last wave's last image
            d = ctx['lay']['d']
            size = lib().ba_pm_slot_doubles(n_obs, p.n_imgs, d)
            slots = ctx['plan'].workspace('jslots', (size // 256, 256), dtype).fill_(float('nan'))
            assert slots.data_ptr() == ctx['args'].jslots
        one = lib().ba_pm_linearize_schur if path == 'pairmajor' else lib().ba_linearize_schur
        check(one(ctx['args'], ctx['stream']))
        torch.cuda.synchronize()
        got[path] = [ctx[k].double().cpu() for k in ('dg_img', 'e_img', 'S_pairs')]
    last_img = int((p.infos[0] < n_obs).sum())
    assert int((slots == slots).any(1).nonzero().max()) == -(-n_obs // span) - 1 + last_img
    counts = torch.diff(p.infos[0].cpu().long(), prepend=torch.zeros(1, dtype=torch.long))
    n = 3 * int(counts.max())
    eps = 1.2e-7 if dtype == torch.float32 else 2.3e-16
    (dg, e, S), (dg0, e0, S0) = got['pairmajor'], got['batched']
    assert (abs(dg - dg0) <= 2 * n * eps * dg0).all()
    if dtype == torch.float64:
        assert S.shape == S0.shape
        assert rel_err(S, S0) < 1e-10 and rel_err(e, e0) < 1e-7
