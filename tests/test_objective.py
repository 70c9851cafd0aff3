"""The line search's objective at the sizes where its launches change, against sorting in 64 bits."""
import math

import pytest
import torch

from test_zz_no_alloc import DEV, _pair

SIZES = (1, 2, 5, 64, 1023, 1025, 16383, 16384, 16385, 17000, 262144, 262145, 1050001)


def _residuals(kind, rows, n):
    gen = torch.Generator().manual_seed(n)
    r = torch.randn((rows, n), generator=gen, dtype=torch.float64)
    if kind == 'ties':                                 # one of three lengths, exact in fp32
        r[:2] = 0
        r[0] = torch.randint(1, 4, (n,), generator=gen).double()
    elif kind == 'wide':                               # every exponent, zeros, and infinities among the upper 20%
        r[:2] *= torch.exp2(torch.randint(-60, 60, (n,), generator=gen).double())
        r[:2, ::7] = 0
        r[0, : n // 10] = math.inf
    elif kind == 'equal':
        r[:2] = 0.75
    return r.float()


@pytest.mark.gpu
@pytest.mark.parametrize('kind', ['normal', 'ties', 'wide', 'equal'])
@pytest.mark.parametrize('n', SIZES)
def test_objective(n, kind):
    """Both entry points give the same bits, and twice in a row; each key and the result are rounded to fp32 (the key
    from two products, a sum and a root: 2 units of 2^-24 each side), the sums are formed in 64 bits."""
    for has_err in (0, 1):
        res = _residuals(kind, 9 if has_err else 3, n).to(DEV)
        print(f'objective n={n} {kind} has_err={has_err}', flush=True)
        a, b = _pair(res, n, has_err)
        assert a.view(torch.int32).tolist() == b.view(torch.int32).tolist() == _pair(res, n, has_err)[0].view(torch.int32).tolist()
        k = n * 80 // 100
        low = res[:2].double().norm(dim=0).sort().values[:k]
        if k:
            assert abs(float(a[1]) - float(low.mean())) <= 4 * 2.0 ** -24 * float(low.mean())
        else:
            assert math.isnan(float(a[1]))
        if has_err:
            want, mag = float(res[3:6].double().mean()), float(res[3:6].double().abs().mean())
            assert abs(float(a[0]) - want) <= 2.0 ** -24 * abs(want) + 1e-12 * mag
        else:
            assert math.isnan(float(a[0]))


@pytest.mark.gpu
def test_objective_of_nothing():
    a, b = _pair(torch.zeros((9, 1), device=DEV), 0, 1)
    assert all(math.isnan(float(v)) for v in (*a, *b))
