"""The metric factor's kernels at the edges of their blocks: 16 x 16 blocks
and 128-wide panels of mdf_potrf, the levels of mdf_trtri."""
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 16, 17, 31, 100, 127, 128, 129, 143, 255, 256, 257, 300, 384, 513, 1100]


def factor(A, ld=None, info=None):
    import torch
    from electrolites_amd import _dev, _lib
    n = A.shape[0]
    ld = ld or n
    low = torch.full((n, ld), float('nan'), dtype=torch.float64, device='cuda')
    low[:, :n] = A
    info = torch.zeros(1, dtype=torch.int32, device='cuda')
    work = torch.full((_lib.query('mdf_potrf_workspace', n) // 8 + 1,), float('nan'), dtype=torch.float64, device='cuda')
    _lib.call('mdf_potrf', _dev.ptr(low), n, ld, _dev.ptr(info), _dev.ptr(work), work.numel() * 8, _dev.stream_ptr())
    return low, info, work


def inverse(low, n, ld, work):
    import torch
    from electrolites_amd import _dev, _lib
    X = torch.full((n, ld), float('nan'), dtype=torch.float64, device='cuda')
    w = torch.full((_lib.query('mdf_trtri_workspace', n) // 8 + 1,), float('nan'), dtype=torch.float64, device='cuda')
    _lib.call('mdf_trtri', _dev.ptr(low), n, ld, _dev.ptr(work), _dev.ptr(X), ld, _dev.ptr(w), w.numel() * 8,
              _dev.stream_ptr())
    return X


def spd(n, seed):
    import torch
    g = torch.Generator(device='cuda').manual_seed(seed)
    q = torch.randn((n, n), generator=g, dtype=torch.float64, device='cuda')
    return q @ q.T + n * torch.eye(n, dtype=torch.float64, device='cuda')


@pytest.mark.parametrize('n', SIZES)
@pytest.mark.parametrize('pad', [0, 3])
def test_factor_and_inverse(n, pad):
    import torch
    print(f'factor n {n} ld {n + pad}', flush=True)
    A = spd(n, n)
    low, info, work = factor(torch.tril(A), n + pad)
    assert int(info) == 0
    L = torch.tril(low[:, :n])
    X = inverse(low, n, n + pad, work)[:, :n]
    # Cholesky in any order of sums: |A - L L^T| <= (n + 1) eps |L| |L^T|; a
    # panel below a diagonal block is A_ip X_pp^T with the block's inverse
    # X_pp, whose error n eps |A_ip| |X_pp^T| <= n eps |L_ip| M_p (M_p =
    # |L_pp^T| |X_pp^T|) meets L_pp^T again: the same bound with |L| M for |L|
    eps = 2.3e-16
    M = torch.zeros_like(A)
    for p in range(0, n, 128):
        b = slice(p, p + 128)
        M[b, b] = L[b, b].abs().T @ X[b, b].abs().T
    W = (L.abs() + L.abs() @ M) @ L.abs().T
    assert float(((A - L @ L.T).abs() - 2 * (n + 1) * eps * W).max()) <= 0
    assert torch.equal(X, torch.tril(X))
    # a triangular inverse by blocks: |L X - I| <= c n eps |L| |X|
    I = torch.eye(n, dtype=torch.float64, device='cuda')
    assert float(((L @ X - I).abs() - 4 * (n + 4) * eps * (L.abs() @ X.abs())).max()) <= 0


@pytest.mark.parametrize('n,bad', [(5, 0), (40, 17), (128, 127), (200, 130), (300, 299)])
def test_factor_reports_the_first_bad_pivot(n, bad):
    import torch
    print(f'bad pivot n {n} at {bad}', flush=True)
    A = spd(n, 1)
    L = torch.linalg.cholesky(A)
    A[bad, bad] = float((L[bad, :bad] ** 2).sum()) - 1.
    low, info, _ = factor(torch.tril(A))
    assert int(info) == bad + 1
