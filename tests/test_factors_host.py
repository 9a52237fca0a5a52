"""The factors of a tagged density (factorize_dm) on the CPU."""
import numpy as np
import pytest


@pytest.mark.parametrize('occ', [
    [[2, 2, 2, 0, 0]], [[2, 2, 2, 2, 2]], [[0, 0, 0, 0, 0]], [[2, 0, 2, 0, 1]], [[-1, 2, .5, 0, 0]],
    [[1, 1, 1, 0, 0], [1, 0, 0, 0, 0]], [[1, 1, 1, 1, 1], [0, 0, 1, 0, 1]], [[0, 0, 0, 0, 0], [1, 1, 0, 0, 0]]])
@pytest.mark.parametrize('kind', ['numpy', 'list', 'float64', 'float32', 'bfloat16', 'int64', 'grad'])
def test_tagged_factors(monkeypatch, occ, kind):
    """D = F F^T over the positive occupations, whatever holds them."""
    import torch
    from electrolites_amd import _dev, fastdf
    monkeypatch.setattr(_dev, 'device', lambda: torch.device('cpu'))
    n, nao = len(occ), 6
    rng = np.random.default_rng(0)
    c = rng.standard_normal((n, nao, 5))
    if kind == 'int64':
        occ = np.floor(np.asarray(occ)).tolist()
    o = np.asarray(occ, dtype=float)
    if kind == 'list':
        given = occ
    elif kind == 'numpy':
        given = o
    elif kind == 'grad':
        given = torch.tensor(o, requires_grad=True)
    else:
        given = torch.tensor(o).to(getattr(torch, kind))
    dm = fastdf.tag_array(torch.zeros(n, nao, nao, dtype=torch.float64), mo_coeff=torch.from_numpy(c), mo_occ=given)
    fl, fr = fastdf.factorize_dm(dm, 1)
    num = (o > 0).sum(axis=1)
    assert fr is None and fl.shape == (n, nao, num.max()) and fl.dtype == torch.float64 and fl.is_contiguous()
    fl = fl.detach().numpy()
    for i in range(n):
        want = c[i][:, o[i] > 0] * np.sqrt(o[i][o[i] > 0])
        # a square root and a product, each rounded once
        assert np.allclose(fl[i, :, :num[i]], want, rtol=4.5e-16, atol=0) and not fl[i, :, num[i]:].any()
